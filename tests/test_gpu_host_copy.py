"""Results in host arrays: bit for bit what the device entry points write, for
copies below the pinned ring's first size, of one and of many pieces, and from
several threads at once; a non-finite Hessian leaves the caller's values alone."""
import threading

import numpy as np
import pytest

from polyfem_amd import NLAssembler, PfgpuError, _ffi
from polyfem_amd.mesh import BASE_SEED, kuhn_box, random_lame, smooth_displacement

pytestmark = pytest.mark.gpu
# cells: values of 13 KB, 62 KB, 73 KB, 1.0 MB, 2.1 MB, 9.5 MB, 31 MB (FP64)
CELLS = [(1, 1, 1), (2, 2, 3), (2, 3, 3), (9, 9, 9), (12, 12, 11), (20, 20, 20), (30, 30, 29)]


def case(cells, precision):
    m = kuhn_box(*cells, order=1)
    lam, mu = random_lame(m.n_elements, seed=BASE_SEED + 960)
    return m, NLAssembler("NeoHookean", m, lame=(lam, mu), precision=precision), 0.3 * smooth_displacement(m.nodes, 0.02, 1e-4, BASE_SEED + 961)


def on_device(m, a, x):
    import torch
    dx = torch.from_numpy(x).cuda()
    e, g = torch.zeros(1, dtype=torch.float64, device="cuda"), torch.zeros(m.n_dofs, dtype=torch.float64, device="cuda")
    v = torch.zeros(a.nnz, dtype=torch.float32 if a._value_dtype == np.float32 else torch.float64, device="cuda")
    torch.cuda.synchronize()
    a.energy_gradient_hessian_dev(dx.data_ptr(), e.data_ptr(), g.data_ptr(), v.data_ptr())
    a.synchronize()
    return float(e.cpu()[0]), g.cpu().numpy(), v.cpu().numpy()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("cells", CELLS)
def test_host_results_are_the_device_results(cells, precision):
    m, a, x = case(cells, precision)
    print(f"host copy {cells} {precision} values {a.nnz}", flush=True)
    e, g, v = on_device(m, a, x)
    for _ in range(2):
        eh, gh, vh = a.assemble_energy_gradient_hessian(x)
        assert eh == e and np.array_equal(gh, g) and np.array_equal(vh, v)
    assert np.array_equal(a.assemble_gradient(x), g) and a.hessian_values(x).shape == v.shape


def test_threads():
    cases = [case(c, p) for c in CELLS[3:6] for p in ("fp64", "mixed")]
    want = [on_device(*c) for c in cases]
    bad = []

    def work(k):
        m, a, x = cases[k]
        for _ in range(5):
            e, g, v = a.assemble_energy_gradient_hessian(x)
            if not (e == want[k][0] and np.array_equal(g, want[k][1]) and np.array_equal(v, want[k][2])):
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("cells", [CELLS[0], CELLS[4]])
def test_a_non_finite_hessian_is_not_copied(cells):
    m, a, x = case(cells, "fp64")
    x = x.copy()
    x[:] = np.nan
    vals = np.full(a.nnz, 7.0)
    with pytest.raises(PfgpuError):
        _ffi.check(_ffi.lib().pfgpu_hessian_values(a._h, _ffi.C.c_void_p(x.ctypes.data), 0, _ffi.C.c_void_p(vals.ctypes.data)))
    assert (vals == 7.0).all()
