"""Per-kernel timing times the kernels that untimed steps run.  A PCG in one
launch is a class of its own, which stays as it is unless one of the phases of
the launches per iteration is timed."""
import pytest

import fs2d
from test_gpu_batch import assert_same
from test_gpu_pcg_launches import liquid, stir

pytestmark = pytest.mark.gpu

PHASES = {"pcg_forward_solve", "pcg_backward_solve", "pcg_spmv_dot", "pcg_axpy_norm"}


def launches(s):
    return {k: n for k, (ms, n) in s.kernel_times().items() if n}


@pytest.mark.parametrize("nx,one", [(96, 1), (576, 1), (577, 0)])
def test_timed_classes_leave_the_solve_as_it_is(nx, one):
    cells, kw = liquid("dam", nx, 90)
    timed, plain = fs2d.Sim(cells, **kw), fs2d.Sim(cells, **kw)
    stir((timed, plain))
    steps = 2
    for only, want in ((["p2g"], {"p2g": steps}),
                       (["p2g", "pcg_one_launch"], {"p2g": steps, **({"pcg_one_launch": steps} if one else {})})):
        timed.reset_kernel_times()
        timed.set_timing(True, only=only)
        for _ in range(steps):
            timed.step()
            plain.step()
        assert launches(timed) == want
        assert_same(timed, plain, "%d columns, timed %s" % (nx, only))
    timed.reset_kernel_times()
    timed.set_timing(True, only=[k for k in timed.kernel_times() if k not in PHASES])
    timed.step()
    plain.step()
    assert ("pcg_one_launch" in launches(timed)) == bool(one) and not PHASES & set(launches(timed))
    for only in (["pcg_spmv_dot"], None):  # the phases asked for, and every class
        timed.reset_kernel_times()
        timed.set_timing(True, only=only)
        timed.step()
        plain.step()
        n = launches(timed)
        assert "pcg_one_launch" not in n and (only is None) == ("pcg_forward_solve" in n)
        if one:
            assert n["pcg_spmv_dot"] >= timed.stats()["pcg_iters"]
        assert_same(timed, plain, "%d columns, timed %s" % (nx, only))


def test_timed_batch_runs_the_kernels_of_untimed_steps():
    m = [liquid(kind, nx, ny) for kind, nx, ny in (("dam", 64, 64), ("blocks", 96, 450))]
    timed, plain = fs2d.Batch(m), fs2d.Batch(m)
    for pair in zip(timed.sims, plain.sims):
        stir(pair)
    timed.set_timing(True)
    for step in range(2):
        timed.step()
        plain.step()
        for k, (a, b) in enumerate(zip(timed.sims, plain.sims)):
            assert_same(a, b, "step %d member %d" % (step, k))
    n = launches(timed)
    assert n["pcg_one_launch"] == 2 and not PHASES & set(n)
