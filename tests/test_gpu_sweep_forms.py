"""The launch forms of the step that the default sizes of the other tests do
not take (needs an MI355X)."""
import numpy as np
import pytest

import vulture_amd
from vulture_amd import meshgen

pytestmark = pytest.mark.gpu


def _fields(mesh, precision, steps=80):
    """All fields once the source has reached every cell, and the update-once report."""
    with vulture_amd.DeviceSolve(mesh, precision=precision, steps=steps) as ds:
        ds.run(0, steps)
        ds.synchronize()
        return [ds.download(c) for c in range(6)], ds.check_limits(counts=False)


def _write(tmp_path, text):
    p = tmp_path / "m.mesh"
    p.write_text(text)
    return str(p)


@pytest.mark.parametrize("ty", ["1", "3", "5", "8"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_check_counts_the_loops_launches(precision, ty, tmp_path, monkeypatch):
    """The update-once check finds a step clean exactly when the loop's own
    launches, with any number of rows per fast tile, leave the default's
    fields."""
    mesh = _write(tmp_path, meshgen.freespace(n=40, steps=80))
    print(f"case rows per tile {ty} {precision}", flush=True)
    ref, rep = _fields(mesh, precision)
    assert rep["missed"] == rep["repeated"] == rep["outside"] == [0] * 6, rep
    monkeypatch.setenv("VGPU_FAST_TY", ty)
    got, rep = _fields(mesh, precision)
    clean = rep["missed"] == rep["repeated"] == rep["outside"] == [0] * 6
    same = all(np.array_equal(a, b) for a, b in zip(ref, got))
    assert clean == same, (rep, same)
