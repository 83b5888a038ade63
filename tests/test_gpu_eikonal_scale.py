"""The eikonal passes' plain root (spacings between 1e-12 and 1e12) and the
general one on both sides of the line: the distances equal the FP64 oracle's
bit for bit."""
import numpy as np
import pytest

import fs2d
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dx", [1.0 / 70, 2e-12, 5e-13])
@pytest.mark.parametrize("nx,ny", [(5, 5), (70, 131)])
def test_eikonal_scale(nx, ny, dx):
    cells = O.dam_break(nx, ny)
    kw = dict(k=2, dt=1e-3, dx=dx, gravity=(0.0, 0.0))
    g = fs2d.Sim(cells, **kw)
    o = O.Oracle(cells, sl_inplace=False, **kw)
    for f, h in ((fs2d.F_PARTICLE_POS, O.F_POS), (fs2d.F_PARTICLE_VEL, O.F_VEL), (fs2d.F_U, fs2d.F_U),
                 (fs2d.F_V, fs2d.F_V)):
        o.set(h, g.get(f).astype(np.float64))
    o.set(O.F_CELL, g.get(fs2d.F_CELL))
    g.run_stage(fs2d.STAGE_LEVEL_SET)
    o.run_stage(O.ST_LEVELSET)
    assert g.get(fs2d.F_PHI, np.float64).tobytes() == o.get(O.F_PHI).tobytes()
    assert np.array_equal(g.get(fs2d.F_CELL), o.get(O.F_CELL))
