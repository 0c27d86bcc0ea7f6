"""A node with more elements than any row-unit plan holds: the refusal is kept, so
that later assemblies do not go through the nodes again on the host."""
import time

import numpy as np
import pytest

from meshes import star_mesh
from polyfem_amd import NLAssembler
from polyfem_amd.mesh import BASE_SEED, kuhn_box, random_lame, smooth_displacement
from test_wave_plan import union

pytestmark = pytest.mark.gpu


def enqueue_time(parts):
    """Host time of an assembly's launches, the best of 40, and its results."""
    import torch
    m = union(*parts)
    lam, mu = random_lame(m.n_elements, seed=BASE_SEED + 980)
    a = NLAssembler("NeoHookean", m, lame=(lam, mu), precision="fp64")
    x = torch.from_numpy(0.3 * smooth_displacement(m.nodes, 0.02, 1e-4, BASE_SEED + 981)).cuda()
    e, g, v = (torch.zeros(n, dtype=torch.float64, device="cuda") for n in (1, m.n_dofs, a.nnz))
    torch.cuda.synchronize()
    best = []
    for _ in range(42):
        t = time.perf_counter()
        a.energy_gradient_hessian_dev(x.data_ptr(), e.data_ptr(), g.data_ptr(), v.data_ptr())
        best.append(time.perf_counter() - t)
        a.synchronize()
    return min(best[2:]), a, x.cpu().numpy(), g.cpu().numpy(), v.cpu().numpy()


def test_the_refusal_is_kept():
    box, hub = kuhn_box(20, 20, 20, order=2), star_mesh(35, order=2, seed=5)  # a node of 70 tets
    print(f"refused plan E={box.n_elements + hub.n_elements}", flush=True)
    # the scan for a plan ends at the node that it refuses, here at once and at the end
    first, *_ = enqueue_time([hub, box])
    last, a, x, g, v = enqueue_time([box, hub])
    print(f"enqueued in {1e6 * first:.0f} and {1e6 * last:.0f} us", flush=True)
    assert last < 2 * first
    gh, vh = a.assemble_energy_gradient_hessian(x)[1:]
    assert np.array_equal(gh, g) and np.array_equal(vh, v)
