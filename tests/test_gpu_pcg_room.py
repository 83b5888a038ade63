"""The one-launch PCG's workgroups wait for each other, at most 16 per launch and
one launch per hardware queue.  A process that asks HIP for more queues than the
CUs have room for gets launches per iteration, with the same bits."""
import ctypes

import numpy as np
import pytest

import fs2d
from test_gpu_batch import assert_same
from test_gpu_pcg_launches import liquid, stir
from test_zz_no_alloc import args_for, hip, lib, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("queues,one", [("4", True), ("8", True), ("9", False), ("16", False), ("", True)])
def test_queues_decide_between_one_launch_and_several(queues, one, monkeypatch):
    m = [liquid(kind, nx, ny) for kind, nx, ny in (("dam", 64, 64), ("blocks", 96, 450))]
    plain = [fs2d.Sim(c, **kw) for c, kw in m]
    monkeypatch.setenv("GPU_MAX_HW_QUEUES", queues)  # HIP itself has read its value before
    sims = [fs2d.Sim(c, **kw) for c, kw in m]
    captured = [fs2d.Sim(c, **kw) for c, kw in m]
    batch = fs2d.Batch(m)
    for k in range(2):
        stir((plain[k], sims[k], captured[k], batch.sims[k]))
        captured[k].set_graph(True)
        sims[k].set_timing(True, only=["pcg_one_launch"])
    batch.set_timing(True)
    steps = 3
    for step in range(steps):
        batch.step()
        for k in range(2):
            for s in (plain[k], sims[k], captured[k]):
                s.step()
            for what, s in (("single", sims[k]), ("captured", captured[k]), ("member", batch.sims[k])):
                assert_same(plain[k], s, "%s queues, step %d, %s %d" % (queues, step, what, k))
    for x in sims + [batch]:
        assert x.kernel_times()["pcg_one_launch"][1] == (steps if one else 0)
    batch.close()


def test_noalloc_projection_without_room(monkeypatch):
    L, H = lib(), hip()
    n = 160
    g = scene(n, fs2d.PICFLIP, 3)
    out = ctypes.c_void_p()
    assert H.hipMalloc(ctypes.byref(out), n * n * 4) == 0
    got = []
    try:
        for queues in ("4", "16", "4"):
            monkeypatch.setenv("GPU_MAX_HW_QUEUES", queues)
            a = args_for(g, n, out.value)
            iters, res = ctypes.c_int(-1), ctypes.c_double(-1.0)
            assert L.fs2d_project_noalloc(ctypes.byref(a), ctypes.byref(iters), ctypes.byref(res)) == fs2d.OK
            p = np.empty((n, n), dtype=np.float32)
            assert H.hipMemcpy(p.ctypes.data, out.value, n * n * 4, 2) == 0  # device to host
            got.append((p.tobytes(), iters.value, res.value))
    finally:
        H.hipFree(out)
    g.run_stage(fs2d.STAGE_PROJECT)
    s = g.stats()
    assert got == [(g.get(fs2d.F_P).tobytes(), s["pcg_iters"], s["pcg_residual"])] * 3
    assert s["pcg_iters"] > 2
    g.close()
