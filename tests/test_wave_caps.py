"""The wavefront plans that the library launches, with its own caps of a chunk's
words: every position, descriptor and sum under the sanitizers, on lattices, stars
of many tets with large stages, and unstructured meshes."""
import os
import subprocess

import pytest

from polyfem_amd.mesh import kuhn_box
from test_plans import ROOT, write_mesh
from test_wave_lds import hull_star
from test_wave_plan import MESHES, union
from test_wave_share import unstructured

EXE = os.path.join(ROOT, "tests", "cpp", "build", "wave_caps_check")


@pytest.fixture(scope="module")
def exe():
    os.makedirs(os.path.dirname(EXE), exist_ok=True)
    srcs = [os.path.join(ROOT, "tests", "cpp", "wave_caps_check.cpp")]
    srcs += [os.path.join(ROOT, "polyfem_amd", "csrc", s) for s in ("pattern.cpp", "plans.cpp")]
    cmd = ["g++", "-O1", "-g", "-std=c++20", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
           "-D__HIP_PLATFORM_AMD__", f"-I{ROOT}/include", "-I/opt/rocm/include", *srcs, "-o", EXE, "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return EXE


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("name", [*MESHES, "stars", "lattice", "unstructured"])
def test_plans_as_launched(exe, tmp_path, name, order):
    if name == "stars":
        m = union(*(hull_star(n, order, s) for n in (52, 58, 62, 64) for s in range(3)), kuhn_box(2, 2, 2, order=order))
    elif name == "lattice":
        m = kuhn_box(11, 9, 10, order=order)
    elif name == "unstructured":
        m = unstructured(9 if order == 1 else 6, order, 48)
    else:
        m = MESHES[name](order)
    write_mesh(tmp_path / "mesh.bin", m)
    r = subprocess.run([exe, str(tmp_path / "mesh.bin")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "OK (0 failures)" in r.stdout, (r.stdout[-2000:], r.stderr[-4000:])
    # P2 FP64 refuses stages beyond its LDS
    assert r.stdout.count("chunks checked") >= (0 if name == "fan140" else 1)
