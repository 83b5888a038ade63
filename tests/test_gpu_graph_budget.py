"""Captured steps of grids whose solve runs by launches per iteration (more than
576 columns): the captured part holds a fixed number of iterations, after which
the host reads whether the solve has converged and queues the rest.  Against
uncaptured steps, bit for bit.
"""
import pytest

import fs2d
from test_gpu_graph import assert_same, smoke_pair

pytestmark = pytest.mark.gpu


def test_captured_budget_falls_short():
    """A tighter tolerance after a loose one, on a grid whose captured steps
    have an iteration budget: the solve continues with queued chunks."""
    eager, graph = smoke_pair(600, 5)
    graph.set_graph(True)
    iters = []
    for step, tol in enumerate((1e-2, 1e-2, 1e-7, 1e-7)):
        for s in (eager, graph):
            s.set_solver(tau=0.97, tol=tol, max_iters=1000)
        eager.step()
        graph.step()
        iters.append(graph.stats()["pcg_iters"])
        assert_same(eager, graph, "step %d" % step)
    assert iters[2] > 2 * iters[1] + 64  # past any budget that the second step leaves
    eager.close()
    graph.close()


def test_captured_steps_reach_the_iteration_limit():
    eager, graph = smoke_pair(600, 6)
    graph.set_graph(True)
    for s in (eager, graph):
        s.set_solver(tau=0.97, tol=1e-9, max_iters=12)
    for step in range(3):
        assert eager.step() == fs2d.WARN_MAXITER
        assert graph.step() == fs2d.WARN_MAXITER
        assert_same(eager, graph, "step %d" % step)
    eager.close()
    graph.close()
