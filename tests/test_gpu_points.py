"""The point-parallel element Hessians (SaintVenant, FixedCorotational,
MooneyRivlin) against the FP64 oracles at the edges of its wavefronts: a
wavefront covers 16 elements at four points and more per element, 64 at one
point, so element counts around 1, 16 and 64 leave it full, one over and
nearly empty."""
import numpy as np
import pytest

from oracle import mooney
from oracle import pyoracle as po
from oracle.fcr import FcrOracle
from polyfem_amd import NLAssembler
from polyfem_amd.mesh import BASE_SEED, kuhn_box, random_lame, smooth_displacement, tet_mesh

pytestmark = pytest.mark.gpu

# FP64: the bar of every parity test.  FP32: a block entry is the sum of at
# most 11 points x 50 products of factors that carry a few roundings each;
# sqrt(550) x 6e-8 x a growth of ten from the factors is below 2e-5.
TOL = {"fp64": 1e-10, "mixed": 2e-5}


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("name", ["SaintVenant", "FixedCorotational", "MooneyRivlin"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65])
def test_wavefront_edges(n, name, order, precision):
    box = kuhn_box(3, 2, 2, order=1)
    m = tet_mesh(box.vertices, box.elem_vertices[:n], order=order)
    lam, mu = random_lame(n, seed=BASE_SEED + 900 + n)
    x = smooth_displacement(m.nodes, 0.05, 1e-3, BASE_SEED + 901)
    print(f"points {name} P{order} {precision} E={n}", flush=True)
    if name == "MooneyRivlin":
        par = (0.35 * mu, 0.15 * mu, lam)
        a, o = NLAssembler(name, m, params=par, precision=precision), mooney.MooneyOracle(m, *par)
    else:
        a = NLAssembler(name, m, lame=(lam, mu), precision=precision)
        o = FcrOracle(m, lam, mu) if name == "FixedCorotational" else po.Oracle(m, lam, mu, material=po.SAINT_VENANT)
    ref = o.hessian(x)[2]
    got = a.hessian_values(x).astype(np.float64)
    assert np.abs(got - ref).max() < TOL[precision] * np.abs(ref).max()
