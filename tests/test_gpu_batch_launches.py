"""Ensembles with a member past the one-launch solve's limits (577 columns, or
1025 rows): the whole batch then runs its PCG by launches per iteration, the
smaller members with the one-launch solve's order of sums.  Every member must
step bit-identically to its single simulation, whatever the launch shapes.
"""
import numpy as np
import pytest

import fs2d
from test_gpu_batch import assert_same
from test_gpu_pcg_launches import liquid, stir

pytestmark = pytest.mark.gpu


def members(max_iters=500):
    """Sides below and at the limits, and past them; strips and columns without
    FLUID below, between and above others."""
    return [liquid(kind, nx, ny, max_iters) for kind, nx, ny in
            (("dam", 48, 48), ("blocks", 96, 450), ("dam", 600, 200), ("corner", 576, 130), ("blocks", 40, 1030))]


@pytest.mark.parametrize("grid,prefetch,fused,graph", [
    (0, 0, 0, False), (0, 1, 0, True), (64, 1, 1, False), (8, 0, 1, True)])
def test_mixed_batch_members_match_single_steps(grid, prefetch, fused, graph):
    m = members()
    batch = fs2d.Batch(m)
    batch.set_tuning(grid or batch.tuning()["pcg_grid"], prefetch, fused)
    batch.set_graph(graph)
    singles = [fs2d.Sim(c, **kw) for c, kw in m]
    for pair in zip(singles, batch.sims):
        stir(pair)
    for step in range(4):
        batch.step()  # the first chunk or budget of the first steps falls short
        for s in singles:
            s.step()
        for k, (b, s) in enumerate(zip(batch.sims, singles)):
            assert_same(b, s, "step %d member %d" % (step, k))
    assert len({s.stats()["pcg_iters"] for s in singles}) > 2
    batch.close()


def test_mixed_batch_reaches_the_iteration_limit():
    """A limit that the larger members reach and the smallest does not."""
    m = members(max_iters=30)
    batch = fs2d.Batch(m)
    singles = [fs2d.Sim(c, **kw) for c, kw in m]
    for pair in zip(singles, batch.sims):
        stir(pair)
    for step in range(2):
        st = batch.step()
        ss = [s.step() for s in singles]
        assert st == fs2d.WARN_MAXITER and fs2d.WARN_MAXITER in ss
        for k, (b, s) in enumerate(zip(batch.sims, singles)):
            assert_same(b, s, "step %d member %d" % (step, k))
    batch.close()
