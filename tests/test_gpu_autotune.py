"""What the autotuner keeps: a gather size that every later call of the handle
accepts, and no configuration twice among the candidates but the two times of the
factored gather."""
import numpy as np
import pytest

from meshes import star_mesh
from oracle import pyoracle as po
from polyfem_amd import NLAssembler
from polyfem_amd.mesh import BASE_SEED, kuhn_box, random_lame, smooth_displacement

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [1, 2])
def test_projected_assembly_after_tuning(order):
    """A node of 70 tets: more than a block gather of 64 threads holds."""
    import torch
    m = star_mesh(35, order=order, seed=5)
    lam, mu = random_lame(m.n_elements, seed=BASE_SEED + 990)
    x = 0.3 * smooth_displacement(m.nodes, 0.05, 1e-3, BASE_SEED + 991)
    print(f"autotune with a node of 70 tets P{order} E={m.n_elements}", flush=True)
    a = NLAssembler("NeoHookean", m, lame=(lam, mu), precision="mixed")
    a.set_tuning("plain", 256, 256)
    want = a.hessian_values(x, project_to_psd=True)
    ref = po.Oracle(m, lam, mu).hessian(x)[2]
    xd = torch.from_numpy(x).cuda()
    for _ in range(12):  # the times decide between equal candidates
        rep = a.autotune_dev(xd.data_ptr())
        assert rep["gather_threads"] in (128, 256, 512)
        assert rep["candidates"] == 9 + 3 + (rep["ms_fused"] is not None)
        assert np.array_equal(a.hessian_values(x, project_to_psd=True), want)
    assert np.abs(a.hessian_values(x) - ref).max() < 1e-6 * np.abs(ref).max()


@pytest.mark.parametrize("material", ["SaintVenant", "FixedCorotational", "MooneyRivlin"])
def test_materials_of_one_hessian_kernel(material):
    import torch
    m = kuhn_box(3, 2, 2, order=2)
    lam, mu = random_lame(m.n_elements, seed=BASE_SEED + 992)
    par = {"params": (0.35 * mu, 0.15 * mu, lam)} if material == "MooneyRivlin" else {"lame": (lam, mu)}
    print(f"autotune {material}", flush=True)
    a = NLAssembler(material, m, precision="mixed", **par)
    rep = a.autotune_dev(torch.zeros(m.n_dofs, dtype=torch.float64, device="cuda").data_ptr())
    assert rep["candidates"] == 3 and rep["hessian_threads"] == 256 and rep["ms_plain_default"] > 0
    assert rep["path"] == "plain" and rep["ms_factored"] is None
