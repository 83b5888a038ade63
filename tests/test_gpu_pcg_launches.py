"""The PCG by launches per iteration, on grids past the one-launch solve's 576
columns: single handles as two launches (fused_pcg 1) against four, bit for
bit, on scenes whose solves skip strips and columns without FLUID cells; and
the adjoint solves and the projection that allocates nothing on such grids.
"""
import ctypes

import numpy as np
import pytest

import fs2d
from fs2d import scenes
from test_gpu_adjoint import _gpu_gradient
from test_zz_no_alloc import ProjectionArgs, device_field, hip, lib

pytestmark = pytest.mark.gpu

FIELDS = (fs2d.F_U, fs2d.F_V, fs2d.F_P, fs2d.F_CELL, fs2d.F_PARTICLE_POS, fs2d.F_PARTICLE_VEL)


def scene(kind, nx, ny):
    """dam: a block at the lower left.  blocks: 40 rows of every 200 over 70%
    of the width, each 31 columns further left than the one below.  corner: a
    block at the upper right, so that the first strips and columns are empty."""
    c = scenes.walls(nx, ny)
    j, i = np.mgrid[0:ny, 0:nx]
    inner = c != scenes.SOLID
    if kind == "dam":
        on = (i < 0.4 * nx) & (j < 0.6 * ny)
    elif kind == "blocks":
        on = (j % 200 >= 150) & (j % 200 < 190) & ((i + 31 * (j // 200)) % nx > 0.3 * nx)
    else:
        on = (i > 0.7 * nx) & (j > 0.75 * ny)
    c[inner & on] = scenes.FLUID
    return c


def liquid(kind, nx, ny, max_iters=500):
    h = 1.0 / max(nx, ny)
    return (scene(kind, nx, ny),
            dict(k=2, dt=0.002, dx=h, mode=fs2d.PICFLIP, alpha=0.05, tau=0.97, tol=1e-6, max_iters=max_iters))


def stir(sims, seed=3):
    """The same random velocities for the particles of every handle (a block
    that falls freely has nothing to project)."""
    v = sims[0].get(fs2d.F_PARTICLE_VEL)
    v = np.random.default_rng(seed).normal(scale=0.3, size=v.shape).astype(np.float32)
    for s in sims:
        s.set(fs2d.F_PARTICLE_VEL, v)


def empty_strips(cells):
    """Which strips of 64 rows hold no FLUID cell."""
    return [not (cells[j:j + 64] == fs2d.FLUID).any() for j in range(0, cells.shape[0], 64)]


@pytest.mark.parametrize("kind,nx,ny,gap", [
    ("dam", 640, 300, "above"), ("corner", 640, 300, "below"), ("blocks", 700, 1100, "between"),
    ("dam", 577, 64, None), ("blocks", 1000, 450, "between")])
def test_two_launches_with_gaps_match_four(kind, nx, ny, gap):
    cells, kw = liquid(kind, nx, ny)
    sims = [fs2d.Sim(cells, **kw) for _ in range(3)]
    for s, fused in zip(sims, (0, 1, 1)):
        s.set_tuning(pcg_grid=0, fused_pcg=fused)
    sims[2].set_graph(True)
    stir(sims)
    for step in range(4):
        for s in sims:
            s.step()
        want = [sims[0].get(f) for f in FIELDS]
        e = empty_strips(want[3])
        k = [i for i, x in enumerate(e) if not x]
        assert {"above": e[-1] and not e[0], "below": e[0] and not e[-1], None: True,
                "between": any(e[k[0]:k[-1]])}[gap]  # the fluid still leaves the strips it should
        for s in sims[1:]:
            for f, w in zip(FIELDS, want):
                assert s.get(f).tobytes() == w.tobytes(), "%s %dx%d step %d field %d" % (kind, nx, ny, step, f)
            assert s.stats()["pcg_iters"] == sims[0].stats()["pcg_iters"] > 2
    for s in sims:
        s.close()


def test_adjoint_two_launches_match_four():
    n = 640
    target = scenes.target_density(n)
    two = _gpu_gradient(n, 3, 2, target, fused_pcg=1)
    four = _gpu_gradient(n, 3, 2, target, fused_pcg=0)
    for a, b in zip([two[1]] + list(two[2]) + list(two[3]), [four[1]] + list(four[2]) + list(four[3])):
        np.testing.assert_array_equal(a, b)
    assert np.abs(two[2][2]).max() > 0


@pytest.mark.parametrize("kind,nx,ny", [("dam", 640, 400), ("blocks", 640, 400), ("dam", 577, 70)])
def test_noalloc_projection_by_launches_matches_run_stage(kind, nx, ny):
    L, H = lib(), hip()
    cells, kw = liquid(kind, nx, ny)
    for fused in (1, 0):
        g = fs2d.Sim(cells, **kw)
        g.set_tuning(pcg_grid=0, fused_pcg=fused)
        stir([g])
        for _ in range(2):
            g.step()
        for st in (fs2d.STAGE_LEVEL_SET, fs2d.STAGE_P2G, fs2d.STAGE_GRAVITY):
            g.run_stage(st)
        out = ctypes.c_void_p()
        assert H.hipMalloc(ctypes.byref(out), nx * ny * 4) == 0
        try:
            a = ProjectionArgs(
                size_x=nx, size_y=ny, dt=kw["dt"], dx=kw["dx"], rho=997.0, tau=kw["tau"], sigma=0.25,
                pcg_tol=kw["tol"], pcg_max_iters=kw["max_iters"], flags=0, cell=device_field(g, fs2d.F_CELL),
                phi=device_field(g, fs2d.F_PHI), u=device_field(g, fs2d.F_U), v=device_field(g, fs2d.F_V),
                p=out.value, stream=g.L.fs2d_stream(g.h))
            iters, res = ctypes.c_int(-1), ctypes.c_double(-1.0)
            st = L.fs2d_project_noalloc(ctypes.byref(a), ctypes.byref(iters), ctypes.byref(res))
            assert st == fs2d.OK, L.fs2d_last_error(None).decode()
            p = np.empty((ny, nx), dtype=np.float32)
            assert H.hipMemcpy(p.ctypes.data, out.value, nx * ny * 4, 2) == 0  # device to host
        finally:
            H.hipFree(out)
        g.run_stage(fs2d.STAGE_PROJECT)
        s = g.stats()
        assert iters.value == s["pcg_iters"] > 2 and res.value == s["pcg_residual"]
        assert p.tobytes() == g.get(fs2d.F_P).tobytes()
        g.close()
