"""The LDS of the wavefront gather's workgroup: meshes with a vertex in many
tets and many small blocks around it, whose chunk of one node needs a larger
stage than a chunk of several nodes may have.  On the CPU every plan that is
accepted fits 160 KB, on the GPU such meshes agree with the oracle, whichever
gather serves them."""
import os
import subprocess

import numpy as np
import pytest
from scipy.spatial import ConvexHull

from meshes import star_mesh
from oracle import pyoracle as po
from polyfem_amd import NLAssembler
from polyfem_amd.mesh import BASE_SEED, kuhn_box, random_lame, smooth_displacement, tet_mesh
from test_plans import ROOT, write_mesh
from test_wave_plan import CELLS, TOL, union

EXE = os.path.join(ROOT, "tests", "cpp", "build", "wave_lds_check")


def hull_star(n_tets, order, seed=0):
    """n_tets tets between a centre and the hull of random points of the unit sphere."""
    rng = np.random.default_rng(seed)
    P = rng.normal(size=(n_tets // 2 + 2, 3))
    P /= np.linalg.norm(P, axis=1)[:, None]
    faces = ConvexHull(P).simplices
    assert faces.shape[0] == n_tets
    return tet_mesh(np.concatenate([P, [[0.0, 0.0, 0.0]]]),
                    np.concatenate([faces, np.full((n_tets, 1), P.shape[0])], axis=1), order=order)


@pytest.fixture(scope="module")
def exe():
    os.makedirs(os.path.dirname(EXE), exist_ok=True)
    srcs = [os.path.join(ROOT, "tests", "cpp", "wave_lds_check.cpp")]
    srcs += [os.path.join(ROOT, "polyfem_amd", "csrc", s) for s in ("pattern.cpp", "plans.cpp")]
    cmd = ["g++", "-O1", "-g", "-std=c++20", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
           "-D__HIP_PLATFORM_AMD__", f"-I{ROOT}/include", "-I/opt/rocm/include", *srcs, "-o", EXE, "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    return EXE


def plans(exe, path, m):
    write_mesh(path, m)
    r = subprocess.run([exe, str(path)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "FAIL" not in r.stdout, (r.stdout[-2000:], r.stderr[-4000:])
    return r.stdout


@pytest.mark.parametrize("order", [1, 2])
def test_workgroups_fit(exe, tmp_path, order):
    for n in (40, 48, 52, 56, 58, 60, 62, 64, 100, 126, 128):
        for seed in range(4):
            plans(exe, tmp_path / "mesh.bin", hull_star(n, order, seed))
    for m in (kuhn_box(1, 1, 1, order=order), kuhn_box(6, 5, 7, order=order), star_mesh(30, order=order, seed=5)):
        assert "refused" not in plans(exe, tmp_path / "mesh.bin", m)


def test_a_large_stage_is_refused_at_fp64_alone(exe, tmp_path):
    out = plans(exe, tmp_path / "mesh.bin", union(kuhn_box(4, 4, 4, order=2), hull_star(62, 2)))
    assert out.count("refused") == 2 and out.count("bytes 8: refused") == 2, out


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])  # the innermost: one reference for both
@pytest.mark.parametrize("tets", [62, 64])
@pytest.mark.parametrize("order", [2, 1])
def test_large_stage_against_oracle(order, tets, precision):
    n = CELLS[order]
    parts = [hull_star(tets, order), kuhn_box(n, n, n, order=order), hull_star(56, order, 1), hull_star(52, order, 2)]
    m = union(*parts)
    print(f"large stage P{order} {tets} tets {precision} E={m.n_elements}", flush=True)
    lam, mu = random_lame(m.n_elements, seed=BASE_SEED + 970)
    x = 0.3 * smooth_displacement(m.nodes, 0.05, 1e-3, BASE_SEED + 971)
    o = po.Oracle(m, lam, mu)
    row_ptr, _, ref = o.hessian(x)
    gref = o.gradient(x)
    a = NLAssembler("NeoHookean", m, lame=(lam, mu), precision=precision)
    e, g, v = a.assemble_energy_gradient_hessian(x)
    h = a.hessian_values(x)
    rows = 3 * np.cumsum([0] + [p.nodes.shape[0] for p in parts])
    for i, j in zip(rows[:-1], rows[1:]):  # every part by its own scale
        s, t = row_ptr[i], row_ptr[j]
        for u in (v, h):
            assert np.abs(u[s:t] - ref[s:t]).max() < TOL[precision] * np.abs(ref[s:t]).max()
        assert np.abs(g[i:j] - gref[i:j]).max() < TOL[precision] * np.abs(gref[i:j]).max()
    assert abs(e - o.energy(x)) < TOL[precision] * abs(o.energy(x))


@pytest.mark.gpu
@pytest.mark.parametrize("order,precision,tets", [(2, "mixed", 64), (1, "fp64", 128)])
def test_two_live_handles_of_different_stages(order, precision, tets):
    """The launch limit is the kernel's, which every handle of its order, rule
    and precision shares: a handle of a smaller stage leaves the others alone."""
    n = CELLS[order]

    def handle(m):
        lam, mu = random_lame(m.n_elements, seed=BASE_SEED + 972)
        x = 0.3 * smooth_displacement(m.nodes, 0.05, 1e-3, BASE_SEED + 973)
        a = NLAssembler("NeoHookean", m, lame=(lam, mu), precision=precision)
        return lambda: (*a.assemble_energy_gradient_hessian(x)[1:], a.hessian_values(x))

    box = kuhn_box(n, n, n, order=order)
    print(f"two handles P{order} {precision}", flush=True)
    large = handle(union(box, hull_star(tets, order)))
    first = large()
    small = handle(box)
    other = small()
    for again, want in ((large, first), (small, other), (large, first)):
        for u, w in zip(again(), want):
            assert np.array_equal(u, w)
