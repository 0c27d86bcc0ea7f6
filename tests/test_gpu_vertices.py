"""The vertex gather of the shape derivative: against the oracle on meshes with
vertices of few and of many elements (the chunked gather holds 256), and under
capture before and after its plan exists."""
import numpy as np
import pytest

from meshes import star_mesh
from oracle import pyoracle as po
from polyfem_amd import NLAssembler
from polyfem_amd.mesh import BASE_SEED, kuhn_box, random_lame, smooth_displacement

pytestmark = pytest.mark.gpu
# the parity tests' bars
TOL = {"fp64": 1e-10, "mixed": 1e-5}
MESHES = {"cell": lambda o: kuhn_box(1, 1, 1, order=o), "box": lambda o: kuhn_box(7, 5, 6, order=o),
          "full": lambda o: star_mesh(128, order=o, seed=6), "over": lambda o: star_mesh(129, order=o, seed=6)}


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("name", MESHES)
def test_shape_derivative(name, order, precision):
    m = MESHES[name](order)
    lam, mu = random_lame(m.n_elements, seed=BASE_SEED + 950)
    x = 0.3 * smooth_displacement(m.nodes, 0.02, 1e-4, BASE_SEED + 951)
    p = np.random.default_rng(BASE_SEED + 952).normal(size=m.n_dofs)
    print(f"shape derivative {name} P{order} {precision}", flush=True)
    a = NLAssembler("LinearElasticity", m, lame=(lam, mu), precision=precision)
    ref = po.Oracle(m, lam, mu, material=po.LINEAR_ELASTICITY).shape_vjp(x, p)
    assert np.abs(a.force_shape_derivative(x, p) - ref).max() < TOL[precision] * np.abs(ref).max()


@pytest.mark.parametrize("planned", [False, True])
def test_shape_derivative_captured(planned):
    torch = pytest.importorskip("torch")
    m = MESHES["box"](1)
    lam, mu = random_lame(m.n_elements, seed=BASE_SEED + 950)
    dev = torch.device("cuda:0")
    a = NLAssembler("NeoHookean", m, lame=(lam, mu), precision="fp64")
    s = torch.cuda.Stream(device=dev)
    a.set_stream(s.cuda_stream)
    dx = torch.tensor(smooth_displacement(m.nodes, 0.02, 1e-4, BASE_SEED + 951), device=dev)
    dp = torch.tensor(np.random.default_rng(BASE_SEED + 952).normal(size=m.n_dofs), device=dev)
    out, ref = (torch.zeros(3 * m.vertices.shape[0], dtype=torch.float64, device=dev) for _ in range(2))
    torch.cuda.synchronize()
    a.gradient_dev(dx.data_ptr(), dp.data_ptr())  # sizes the scratch that the shape derivative uses too
    if planned:
        a.shape_vjp_dev(dx.data_ptr(), dp.data_ptr(), ref.data_ptr())
    a.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        a.shape_vjp_dev(dx.data_ptr(), dp.data_ptr(), out.data_ptr())
    print("captured the shape derivative", flush=True)
    for _ in range(3):
        a.shape_vjp_dev(dx.data_ptr(), dp.data_ptr(), ref.data_ptr())
        a.synchronize()
        out.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            graph.replay()
        s.synchronize()
        assert torch.equal(out, ref)
    a.set_stream(0)
