"""The copies of results into host arrays: on the CPU under the sanitizers, with
HIP calls that copy at once and are counted, and on the GPU bit for bit what the
device entry points write."""
import os
import subprocess

import numpy as np
import pytest

from polyfem_amd import PfgpuError, _ffi
from test_gpu_host_copy import CELLS, case, on_device
from test_plans import ROOT

CHECKS = ["pinned_destination", "sizes", "small", "kept_back", "short_lived", "ring_size", "threads", "errors"]


@pytest.fixture(scope="module", params=["address,undefined", "thread"])
def exe(request):
    out = os.path.join(ROOT, "tests", "cpp", "build", "host_copy_check_" + request.param.split(",")[0])
    os.makedirs(os.path.dirname(out), exist_ok=True)
    cmd = ["g++", "-O1", "-g", "-std=c++20", f"-fsanitize={request.param}", "-D__HIP_PLATFORM_AMD__", f"-I{ROOT}/include",
           "-I/opt/rocm/include", os.path.join(ROOT, "tests", "cpp", "host_copy_check.cpp"),
           os.path.join(ROOT, "polyfem_amd", "csrc", "host_copy.cpp"), "-o", out, "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return out


@pytest.mark.parametrize("check", CHECKS)
def test_copies_under_sanitizers(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("OK\n"), (r.stdout[-2000:], r.stderr[-4000:])


def hessian_into(a, x, ptr):
    _ffi.check(_ffi.lib().pfgpu_hessian_values(a._h, _ffi.C.c_void_p(x.ctypes.data), 0, _ffi.C.c_void_p(ptr)))


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [CELLS[0], CELLS[3], CELLS[5]])
def test_pinned_destination(cells):
    import torch
    m, a, x = case(cells, "fp64")
    print(f"pinned destination {cells} values {a.nnz}", flush=True)
    want = a.hessian_values(x)
    for _ in range(3):
        v = torch.zeros(a.nnz, dtype=torch.float64, pin_memory=True)
        hessian_into(a, x, v.data_ptr())
        assert np.array_equal(v.numpy(), want)
    v[:] = 7.0
    with pytest.raises(PfgpuError):
        hessian_into(a, np.full_like(x, np.nan), v.data_ptr())
    assert (v == 7.0).all()


@pytest.mark.gpu
def test_a_ring_given_back_by_a_failed_call():
    """Values of 9.5 and 31 MB held back while their copies are in flight, then
    the same ring under another handle."""
    other = case(CELLS[5], "mixed")
    e, g, v = on_device(*other)
    for cells in CELLS[5:]:
        m, a, x = case(cells, "fp64")
        print(f"held back {cells} values {a.nnz}", flush=True)
        bad = np.full_like(x, np.nan)
        for _ in range(3):
            a.hessian_values(x)
            vals = np.full(a.nnz, 7.0)
            with pytest.raises(PfgpuError):
                hessian_into(a, bad, vals.ctypes.data)
            assert (vals == 7.0).all()
            eh, gh, vh = other[1].assemble_energy_gradient_hessian(other[2])
            assert eh == e and np.array_equal(gh, g) and np.array_equal(vh, v)
