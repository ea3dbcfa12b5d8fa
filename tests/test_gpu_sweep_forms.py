"""The launch forms of the step that the default sizes of the other tests do
not take (needs an MI355X)."""
import filecmp
import os

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
    tmp_path.mkdir(parents=True, exist_ok=True)
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


@pytest.mark.parametrize("ty", ["1", "3", "5", "8"])
@pytest.mark.parametrize("precision,n", [("fp64", 40), ("fp32", 40), ("fp64", 208)])
def test_rows_per_tile(precision, n, ty, tmp_path, monkeypatch):
    """VGPU_FAST_TY changes no field, where the fast tiles share the sweep's
    launch (40^3) and where they have their own (208^3 in FP64, 85 MB a field)."""
    mesh = _write(tmp_path, meshgen.freespace(n=n, steps=80))
    print(f"case fields of {ty} rows per tile {n} {precision}", flush=True)
    ref, _ = _fields(mesh, precision)
    monkeypatch.setenv("VGPU_FAST_TY", ty)
    got, rep = _fields(mesh, precision)
    assert rep["missed"] == rep["repeated"] == rep["outside"] == [0] * 6, rep
    for a, b in zip(ref, got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("ty", ["2", "8"])
def test_rows_per_tile_packed(ty, tmp_path, monkeypatch):
    """The same for a packed group."""
    meshes = [_write(tmp_path / str(q), meshgen.freespace(n=n, steps=60)) for q, n in enumerate((17, 24, 40))]
    print(f"case packed, {ty} rows per tile", flush=True)
    vulture_amd.run_meshes_group(meshes, [str(tmp_path / f"a{q}") for q in range(3)], precision="fp64")
    monkeypatch.setenv("VGPU_FAST_TY", ty)
    vulture_amd.run_meshes_group(meshes, [str(tmp_path / f"b{q}") for q in range(3)], precision="fp64")
    for q in range(3):
        a, b = str(tmp_path / f"a{q}"), str(tmp_path / f"b{q}")
        files = sorted(os.listdir(a))
        assert files and files == sorted(os.listdir(b))
        assert filecmp.cmpfiles(a, b, files, shallow=False)[0] == files


def _box(n, body, bt="PML 5", steps=40):
    c = n // 2
    lines = ["VM 1.0.0", "CE sweep forms", f"DM {n} {n} {n}", "GS"]
    lines += [f"BT {f} {bt}" for f in ("XLO", "XHI", "YLO", "YHI", "ZLO", "ZHI")]
    lines += ["WF wf1 GAUSSIAN_PULSE 1.0 3.0e-11 1.0e-11",
              f"EX {c} {c + 1} {c} {c + 1} {c} {c + 1} a JZ wf1 1.0 0.0", *body, f"OP {c} {c} {c} {c} {c} {c} t TDOM_ASCII"]
    return "\n".join(lines + ["GE", f"NT {steps}", "CN 0.95", "MS 1e-3", "EN"]) + "\n"


@pytest.mark.parametrize("classes", [True, False])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_listed_debye_site_memory(precision, classes, tmp_path, monkeypatch):
    """Debye sites outside the sweeps' lines (two poles, or one without
    classes) take no more than their list, coefficient and state did in
    launches of their own: 8 bytes and 2 + poles reals a site."""
    if not classes:
        monkeypatch.setenv("VGPU_NO_INDEXED_MEDIA", "1")
    print(f"case Debye site memory {precision} {classes}", flush=True)
    medium = "2.0 0.01 1.0 1e9 -1e9" + (" 4e9 -3e9" if classes else "")
    used = []
    for mt in (f"MT m DEBYE {medium}", "MT m SIMPLE 2.0 0.01 1.0"):
        mesh = _write(tmp_path, _box(112, [mt, "MB 20 90 25 95 30 100 m"]))
        with vulture_amd.DeviceSolve(mesh, precision=precision) as ds:
            st = ds.stats()
            used.append(st["bytes"])
            if len(used) == 1:
                sites, poles = st["debye_sites"], st["debye_poles"]
                assert poles == (2 if classes else 1) and sites > 3 * 70 ** 3 and not st["debye_fused"]
    real = 8 if precision == "fp64" else 4
    assert used[0] - used[1] <= sites * (8 + (2 + poles) * real) + 4096, (used, sites)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_one_pole_site_memory(precision, tmp_path):
    """One-pole sites in the sweeps' lines: a small block in a large grid
    holds currents for its own cells, not for the grid's."""
    print(f"case one-pole site memory {precision}", flush=True)
    used = []
    for mt in ("MT m DEBYE 2.0 0.01 1.0 1e9 -1e9", "MT m SIMPLE 2.0 0.01 1.0"):
        mesh = _write(tmp_path, _box(112, [mt, "MB 40 60 45 65 50 70 m"]))
        with vulture_amd.DeviceSolve(mesh, precision=precision) as ds:
            st = ds.stats()
            used.append(st["bytes"])
            if len(used) == 1:
                sites = st["debye_sites"]
                assert sites >= 3 * 20 ** 3 and st["debye_fused"]
    real = 8 if precision == "fp64" else 4
    assert used[0] - used[1] <= sites * (8 + 3 * real) + 4096, (used, sites)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("body", [
    ["MT m DEBYE 2.0 0.01 1.0 1e9 -1e9", "MB 1 2 1 2 1 2 m"],
    ["MT m DEBYE 2.0 0.01 1.0 1e9 -1e9", "MB 9 10 9 10 9 10 m"],
    ["MT m DEBYE 2.0 0.01 1.0 1e9 -1e9", "MB 0 1 3 9 5 6 m", "EX 2 8 0 10 0 10 b =EZ wf1 0.2 0.0"],
    ["MT m DEBYE 2.0 0.01 1.0 1e9 -1e9", "MT t DEBYE 3.0 0.0 1.0 1e9 -1e9 4e9 -3e9", "MB 0 10 0 10 0 10 m",
     "MB 2 5 2 5 2 5 t", "MB 4 8 4 8 4 8 m"],
], ids=["low", "high", "edge", "mixed"])
@pytest.mark.parametrize("bt", ["PML 5", "MUR", "PEC"])
def test_one_pole_boxes(bt, body, precision, tmp_path, monkeypatch):
    """Currents over the sites' box: blocks at the ends of the grid, flagged
    cells (Mur, sources) outside the box, blocks of other media among them.
    Without classes the same sites are listed; the fields agree bit by bit."""
    mesh = _write(tmp_path, _box(10, body, bt))
    print(f"case one-pole box {bt} {body[1]} {precision}", flush=True)
    a, _ = _fields(mesh, precision, 40)
    monkeypatch.setenv("VGPU_NO_INDEXED_MEDIA", "1")
    b, _ = _fields(mesh, precision, 40)
    assert any(np.count_nonzero(f) for f in a)
    for f, g in zip(a, b):
        assert np.array_equal(f, g)
