"""Element Hessians of the materials outside the factored form on both sides of the
size from which P1 meshes take two lanes per element (16,384 elements), for the
rules where the lanes differ, against the oracle (SaintVenant) and against the
Hessian-vector product, which keeps its points in one lane."""
import numpy as np
import pytest
from scipy.sparse import csr_matrix

from oracle import pyoracle as po
from polyfem_amd import NLAssembler
from polyfem_amd.mesh import BASE_SEED, kuhn_box, random_lame, smooth_displacement

pytestmark = pytest.mark.gpu
# FP64: the bar of every parity test.  FP32: that of the small meshes (a block entry is the sum of at most 6 points x
# 50 products, sqrt(300) x 6e-8 x a growth of ten from the factors: below 2e-5)
TOL = {"fp64": 1e-10, "mixed": 2e-5}


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("quadrature", [2, 3])
@pytest.mark.parametrize("material", ["SaintVenant", "FixedCorotational", "MooneyRivlin"])
@pytest.mark.parametrize("cells", [(13, 14, 15), (1, 2731, 1), (14, 14, 14)])  # 16,380, 16,386 and 16,464 tets
def test_lanes(cells, material, quadrature, precision):
    m = kuhn_box(*cells, order=1)
    print(f"lanes {material} quadrature {quadrature} {precision} E={m.n_elements}", flush=True)
    lam, mu = random_lame(m.n_elements, seed=BASE_SEED + 1000)
    par = {"params": (0.35 * mu, 0.15 * mu, lam)} if material == "MooneyRivlin" else {"lame": (lam, mu)}
    x = smooth_displacement(m.nodes, 0.02 / max(cells), 0.0, BASE_SEED + 1001)
    a = NLAssembler(material, m, precision=precision, quadrature_order=quadrature, **par)
    v = a.hessian_values(x)
    outer, inner = a.hessian_pattern()
    p = np.random.default_rng(BASE_SEED + 1002).normal(size=m.n_dofs)
    # each row by the sum of its terms' magnitudes
    H = csr_matrix((v.astype(np.float64), inner, outer), shape=(m.n_dofs, m.n_dofs))
    scale = abs(H) @ abs(p)
    assert (np.abs(H @ p - a.hessian_vector_product(x, p)) <= 2 * TOL[precision] * scale.max()).all()
    if material == "SaintVenant":
        ref = po.Oracle(m, lam, mu, material=po.SAINT_VENANT, quad_order=quadrature).hessian(x)[2]
        assert np.abs(v - ref).max() < TOL[precision] * np.abs(ref).max()
