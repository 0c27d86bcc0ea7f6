"""Which gather serves a large P1 mesh: the wavefront gather where rows fill its
chunks (lattices), the row-unit gather on unstructured meshes; on the GPU the
gathers that unstructured meshes take agree with the oracle."""
import os
import re
import subprocess

import numpy as np
import pytest
from scipy.spatial import Delaunay

from oracle import pyoracle as po
from polyfem_amd import NLAssembler
from polyfem_amd.mesh import BASE_SEED, kuhn_box, random_lame, smooth_displacement, tet_mesh
from test_plans import ROOT, write_mesh
from test_wave_lds import hull_star
from test_wave_plan import TOL, union

EXE = os.path.join(ROOT, "tests", "cpp", "build", "wave_share_check")


@pytest.fixture(scope="module")
def exe():
    os.makedirs(os.path.dirname(EXE), exist_ok=True)
    srcs = [os.path.join(ROOT, "tests", "cpp", "wave_share_check.cpp")]
    srcs += [os.path.join(ROOT, "polyfem_amd", "csrc", s) for s in ("pattern.cpp", "plans.cpp")]
    cmd = ["g++", "-O1", "-g", "-std=c++20", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
           "-D__HIP_PLATFORM_AMD__", f"-I{ROOT}/include", "-I/opt/rocm/include", *srcs, "-o", EXE, "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return EXE


def unstructured(cells, order, most=None, seed=0):
    """Delaunay mesh of random points; with most, tets are taken away until no
    vertex lies in more of them."""
    rng = np.random.default_rng(seed)
    X = rng.uniform(size=(cells ** 3, 3)) * cells
    t = Delaunay(X).simplices
    v = np.linalg.det(X[t][:, 1:] - X[t][:, :1])
    t, v = t[np.abs(v) > 2e-3], v[np.abs(v) > 2e-3]
    t[v < 0] = t[v < 0][:, [0, 1, 3, 2]]
    while most and (hub := np.bincount(t.ravel(), minlength=X.shape[0]) > most).any():
        t = t[~(hub[t].any(1) & (rng.random(t.shape[0]) < 0.15))]
    used = np.unique(t)
    new = np.full(X.shape[0], -1)
    new[used] = np.arange(used.size)
    return tet_mesh(X[used] / cells, new[t], order=order)


def chosen(exe, path, m):
    write_mesh(path, m)
    r = subprocess.run([exe, str(path)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-4000:])
    print(r.stdout, flush=True)
    return {(int(q), int(b)): c == "chosen" for q, b, c in re.findall(r"points (\d) bytes (\d): share \S+ (\w+)", r.stdout)}


def test_lattices_take_the_wavefront_gather(exe, tmp_path):
    for g in ((28, 28, 28), (20, 33, 41), (80, 80, 8)):
        got = chosen(exe, tmp_path / "mesh.bin", kuhn_box(*g, order=1))
        assert got == {(1, 8): True, (1, 4): True, (4, 8): False, (4, 4): False}, g
    assert all(chosen(exe, tmp_path / "mesh.bin", kuhn_box(9, 9, 9, order=2)).values())
    # a node in 100 tets: 256 units in a workgroup are the faster ones in FP32
    got = chosen(exe, tmp_path / "mesh.bin", union(kuhn_box(28, 28, 28, order=1), hull_star(100, 1)))
    assert got[1, 8] and not got[1, 4]


@pytest.mark.parametrize("most", [None, 56])
def test_unstructured_meshes(exe, tmp_path, most):
    assert not any(chosen(exe, tmp_path / "mesh.bin", unstructured(20, 1, most)).values())
    got = chosen(exe, tmp_path / "mesh.bin", unstructured(9, 2, 48))
    assert got[1, 4] and got[4, 4]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])  # the innermost: one mesh for both
@pytest.mark.parametrize("quadrature", [0, 2])
@pytest.mark.parametrize("most", [None, 60])
def test_unstructured_against_oracle(most, quadrature, precision):
    m = unstructured(29, 1, most, seed=3)  # more units than the route's line on 256 CUs (131,072 tets)
    assert m.n_elements > 131_072
    print(f"unstructured P1 quadrature {quadrature} {precision} most {most} E={m.n_elements}", flush=True)
    lam, mu = random_lame(m.n_elements, seed=BASE_SEED + 995)
    x = 0.02 * smooth_displacement(m.nodes, 0.05, 0.0, BASE_SEED + 996)
    o = po.Oracle(m, lam, mu, quad_order=quadrature)
    ref, gref = o.hessian(x)[2], o.gradient(x)
    a = NLAssembler("NeoHookean", m, lame=(lam, mu), precision=precision, quadrature_order=quadrature)
    e, g, v = a.assemble_energy_gradient_hessian(x)
    for u in (v, a.hessian_values(x)):
        assert np.abs(u - ref).max() < TOL[precision] * np.abs(ref).max()
    assert np.abs(g - gref).max() < TOL[precision] * np.abs(gref).max()
    assert abs(e - o.energy(x)) < TOL[precision] * abs(o.energy(x))
