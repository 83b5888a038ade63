"""A captured step that holds the whole solve has no iteration budget, so an
ensemble captures it once, however its iteration counts change.  One whose solve
runs by launches per iteration captures again when the budget changes.
"""
import subprocess

import pytest

from test_cpp_wrapper import LIBDIR, ROOT, gxx

SRC = ROOT + "/tests/cpp/graph_captures.cpp"


@pytest.mark.gpu
@pytest.mark.parametrize("nx", [64, 577])
def test_captures_of_an_ensemble(nx, tmp_path):
    exe = str(tmp_path / "graph_captures")
    subprocess.run([gxx(), "-std=c++17", "-O2", "-Wall", "-rdynamic", SRC, "-L" + LIBDIR, "-lfs2d", "-ldl",
                    "-Wl,-rpath," + LIBDIR, "-Wl,-rpath-link,/opt/rocm/lib", "-o", exe], check=True)
    out = subprocess.run([exe, str(nx), "8"], check=True, capture_output=True, text=True, timeout=100).stdout
    rows = [[int(x) for x in line.split()] for line in out.splitlines()]
    print(rows)
    assert len(rows) == 8 and max(r[0] for r in rows) > 32  # past the budget of the first step
    if nx == 64:
        assert [r[1] for r in rows] == [2] * 8  # the two graphs of the first step
    else:
        assert rows[0][1] == 2 and rows[-1][1] > 2
