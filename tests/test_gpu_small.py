"""The small-mesh kernels of the solve at the edges of their tiles: one workgroup per
slice of 64 rows, rows whose blocks take one pass of 16 entries, exactly one or
several, the last slice with a single row, vector kernels of 256 threads, and meshes
on both sides of the 90,000-vertex line.

Bar: the FP64 true residual of the answer, formed here with scipy from the downloaded
system, meets the solve's tolerance (the library's own check uses one of the kernels
under test), and FP64 and mixed answers agree to a thousand tolerances (the
conditioning of these systems is below that)."""
import numpy as np
import pytest

import eolc
from conftest import GRAV, H, rel_err
from eolc import scene

pytestmark = pytest.mark.gpu


def fan(k):
    """k triangles around one vertex (a row of k + 1 blocks and its opposite apexes)."""
    t = 2 * np.pi * np.arange(k) / k
    X = np.concatenate([[[0.0, 0.0]], 0.5 * np.stack([np.cos(t), np.sin(t)], 1)])
    tri = np.array([[0, 1 + i, 1 + (i + 1) % k] for i in range(k)], dtype=np.int32)
    return X, tri


def strip(n):
    """A band of n vertices in two rows (n even or odd)."""
    X = np.array([[(i // 2) * 0.1 + 0.05 * (i % 2), 0.1 * (i % 2)] for i in range(n)])
    tri = np.array([[i, i + 2, i + 1] if i % 2 == 0 else [i, i + 1, i + 2] for i in range(n - 2)], dtype=np.int32)
    return X, tri


def check(ctx, X, tri, fixed, ml):
    N = len(X)
    hinge = scene.hinges(N, tri)
    rng = np.random.default_rng(N)
    x = np.concatenate([X, np.zeros((N, 1))], axis=1).reshape(-1) + 1e-3 * rng.standard_normal(3 * N)
    v = 0.05 * rng.standard_normal(3 * N)
    fd = (3 * np.asarray(fixed)[:, None] + np.arange(3)).reshape(-1)
    tol, out = 1e-10, []
    for mode in (eolc.SOLVE_FP64_BJ, eolc.SOLVE_MIXED_BJ):
        ctx.set_topology(X, tri, hinge)
        ctx.set_material(0.1, 500.0, 0.3, 1e-5, 0.0, 1.0)
        ctx.set_options(eolc.OPT_SPD_PROJECT_BENDING)
        ctx.upload_state(x, v)
        ctx.forces_fill(GRAV, H)
        A, M = ctx.download_csr(eolc.MAT_MDK), ctx.download_csr(eolc.MAT_M)
        b = M @ v + H * ctx.download_forces()
        rc, st = ctx.velocity_solve(fd, 0.99 * v[fd], tol=tol, mode=mode | (eolc.SOLVE_MULTILEVEL if ml else 0))
        sol = ctx.download_state()[1]
        free = np.ones(3 * N, bool)
        free[fd] = False
        vfix = np.where(free, 0.0, sol)
        assert np.array_equal(sol[fd], 0.99 * v[fd])
        bred = (b - A @ vfix)[free]
        res = np.linalg.norm((b - A @ sol)[free]) / np.linalg.norm(bred)
        print(f"N {N} mode {mode} ml {ml}: {st.iters} iterations, residual {res:.2e}", flush=True)
        assert rc == 0 and res <= 1.001 * tol
        out.append(sol)
    assert rel_err(out[1], out[0]) <= 1e3 * tol


@pytest.mark.parametrize("k", [6, 7, 8, 15, 16, 17, 40])
def test_rows_of_one_and_several_passes(ctx, k):
    X, tri = fan(k)
    check(ctx, X, tri, [1], False)


@pytest.mark.parametrize("n", [3, 63, 64, 65, 128, 129, 255, 256, 257, 513])
def test_slice_and_workgroup_remainders(ctx, n):
    X, tri = strip(n)
    check(ctx, X, tri, [0], False)


@pytest.mark.parametrize("n", [299, 300])
def test_both_sides_of_the_small_mesh_line(ctx, n):
    """300 x 300 vertices are the last small mesh, 301 x 301 the first large one."""
    sc = scene.Scene(n)
    check(ctx, sc.X, sc.tri, sc.fixed, True)
