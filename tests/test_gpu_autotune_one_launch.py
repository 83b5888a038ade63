"""The autotuner on handles whose PCG is one launch: no launch shape is used, so
it keeps the one that is set, times nothing and leaves the state alone."""
import pytest

import fs2d
from test_gpu_pcg_launches import liquid

pytestmark = pytest.mark.gpu


def test_autotune_keeps_the_set_shapes(tmp_path):
    cache = str(tmp_path / "tune.txt")
    cells, kw = liquid("dam", 300, 300)
    s, again = fs2d.Sim(cells, **kw), fs2d.Sim(cells, **kw)
    s.step()
    p, iters = s.get(fs2d.F_P), s.stats()["pcg_iters"]
    s.set_tuning(pcg_grid=40, fused_pcg=1)
    want = {"pcg_grid": 40, "sweep_prefetch": 0, "fused_pcg": 1}
    assert s.autotune(iters=8, cache=cache) == {**want, "from_cache": False}
    assert s.tuning() == want
    assert s.get(fs2d.F_P).tobytes() == p.tobytes() and s.stats()["pcg_iters"] == iters
    assert again.autotune(iters=8, cache=cache) == {**want, "from_cache": True}

    m = [liquid("dam", 64, 64), liquid("dam", 48, 80)]
    b, again = fs2d.Batch(m), fs2d.Batch(m)
    b.step()
    p = [x.get(fs2d.F_P) for x in b.sims]
    b.set_tuning(40, 1, 1)
    want = {"pcg_grid": 40, "sweep_prefetch": 1, "fused_pcg": 1}
    assert b.autotune(iters=8, cache=cache) == {**want, "from_cache": False}
    assert b.tuning() == want
    assert [x.get(fs2d.F_P).tobytes() for x in b.sims] == [x.tobytes() for x in p]
    assert again.autotune(iters=8, cache=cache) == {**want, "from_cache": True}
    b.close()
    again.close()
