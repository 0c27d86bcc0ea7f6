"""The host loops that build plans and tables: where threads or memory run out, or
a table is refused, inside one of their threads, the caller gets the plan or the
exception and the process goes on."""
import os
import subprocess

import pytest

from meshes import star_mesh
from polyfem_amd.mesh import kuhn_box
from test_plans import ROOT, write_mesh
from test_wave_plan import union

EXE = os.path.join(ROOT, "tests", "cpp", "build", "threads_check")


@pytest.fixture(scope="module")
def exe():
    os.makedirs(os.path.dirname(EXE), exist_ok=True)
    srcs = [os.path.join(ROOT, "tests", "cpp", "threads_check.cpp")]
    srcs += [os.path.join(ROOT, "polyfem_amd", "csrc", s) for s in ("pattern.cpp", "plans.cpp", "fused_tables.cpp")]
    cmd = ["g++", "-O1", "-g", "-std=c++20", "-D__HIP_PLATFORM_AMD__", f"-I{ROOT}/include", "-I/opt/rocm/include", *srcs,
           "-o", EXE, "-lpthread", "-ldl"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return EXE


def run(exe, path, m):
    write_mesh(path, m)
    r = subprocess.run([exe, str(path)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("OK\n"), (r.returncode, r.stdout[-2000:], r.stderr[-2000:])
    return r.stdout


@pytest.mark.parametrize("order", [1, 2])
def test_threads_and_memory_run_out(exe, tmp_path, order):
    n = 18 if order == 1 else 9  # more nodes than the loops do without threads
    assert "patches" in run(exe, tmp_path / "mesh.bin", kuhn_box(n, n, n, order=order))


def test_a_table_refused_in_a_thread(exe, tmp_path):
    """A node with more than 256 neighbours, which the fused path refuses."""
    out = run(exe, tmp_path / "mesh.bin", union(kuhn_box(4, 4, 4, order=2), star_mesh(60, order=2, seed=5)))
    assert "fused tables refused" in out
