"""Corrections beside the sweeps, against the FP64 oracle (needs an MI355X).

A corrected field value is finished by its sweep's thread (Mur faces, zeroed
values, one-pole Debye sites), by an update row in the sweep's launch (small
grids) or by a row behind it (ghosts in groups, everything in larger grids);
SIBC faces run in blocks of 64 in the E sweep's launch.  The meshes here put
corrections where those paths meet: sources on and beside Mur faces, sources on
ghost planes and their sources, several Debye blocks and poles on one edge and
across a TF/SF surface, SIBC surfaces of 63, 64 and 65 faces, and the same mesh
either side of the size to which update rows go.  Bars as for the reference
meshes: FP64 within 1e-12 relative L2, FP32 within 1e-4 or 1.5 times the
float oracle's own error.  With per-cell coefficient arrays instead of classes
and in chunks of steps the files must be those of the first run, byte for byte.
"""
import filecmp
import os
import shutil

import pytest

import oracle
import vulture_amd
from vulture_amd.obsfiles import compare_outputs

from conftest import GOLDEN

pytestmark = pytest.mark.gpu

DM = (18, 13, 11)


def _mesh(dm, bt, body, steps=60, points=()):
    nx, ny, nz = dm
    at = [(nx // 2, ny // 2, nz // 2), (2, 2, 2), (nx - 2, ny - 3, 3), (nx // 3, 1, nz - 2), (1, ny // 2, 1)] + list(points)
    lines = ["VM 1.0.0", "CE corrections", "DM %d %d %d" % dm, "GS"]
    lines += ["BT %s %s" % (f, t) for f, t in zip(("XLO", "XHI", "YLO", "YHI", "ZLO", "ZHI"), bt)]
    lines += ["WF wf1 GAUSSIAN_PULSE 1.0 3.0e-11 1.0e-11"] + body
    for n, (i, j, k) in enumerate(at):
        lines += [f"OP {i} {i} {j} {j} {k} {k} t{n} TDOM_ASCII", f"OP {i} {i} {j} {j} {k} {k} f{n} FDOM_ASCII"]
    return "\n".join(lines + ["GE", f"NT {steps}", "OF 1e9 3e10 16", "CN 0.95", "MS 1e-3", "EN"]) + "\n"


def _sources(nx, ny, nz, step=1):
    """E, J and M sources over a plane that touches y and z faces, hard and soft, and beside the x faces."""
    return [f"EX 4 5 1 {ny - 1} 1 {nz - 1} a JZ wf1 1.0 0.0", f"EX 1 2 1 4 2 5 b EY wf1 1.0 0.0",
            f"EX {nx - 2} {nx - 1} 2 6 1 3 c =EZ wf1 0.5 1.0e-12", f"EX 6 9 {ny - 1} {ny - 1} 2 7 d JMX wf1 380.0 0.0",
            f"EX 7 8 3 5 {nz - 1} {nz - 1} e =JMY wf1 250.0 2.0e-12"]


SURFACES = ['BT s0 SIBC -0.5 0.25 0.25 -0.5', 'BT s1 SIBC "go04.pfe"', 'BT s2 SIBC "go04.pfe"']
MESHES = {
    "mur": _mesh(DM, ["MUR"] * 6, _sources(*DM)),
    "mur_pml": _mesh(DM, ["MUR", "PML 4", "PML 3", "MUR", "PEC", "MUR"], _sources(*DM)),
    "ghosts": _mesh(DM, ["PMC", "PMC", "PERIODIC", "PERIODIC", "PEC", "PMC"],
                    _sources(*DM) + ["EX 0 1 0 1 3 4 g JX wf1 1.0 0.0", "EX 17 18 12 13 5 6 h =EZ wf1 0.4 0.0"],
                    points=[(0, 0, 4), (17, 12, 6), (0, 12, 10)]),
    "debye": _mesh(DM, ["PML 4"] * 6,
                   ["MT one DEBYE 2.0 0.01 1.0 1e9 -1e9", "MT two DEBYE 3.0 0.0 1.0 1e9 -1e9 4e9 -3e9",
                    "MB 3 9 3 8 3 8 one", "MB 7 13 5 10 2 7 two", "MB 8 10 6 9 6 9 one", "MB 12 18 0 4 0 4 one",
                    "PW 5 14 3 10 3 9 pw1 wf1 35.0 20.0 40.0 111111 1.0 0.0", "EX 8 9 6 7 6 7 a JZ wf1 1.0 0.0"]),
    "sibc": _mesh((20, 18, 18), ["PML 3", "PML 3", "MUR", "MUR", "PML 4", "PML 4"],
                  SURFACES + ["TB 10 10 3 10 3 12 s0", "TB 3 11 14 14 4 12 s1", "TB 12 17 3 16 14 14 s2",
                          "EX 6 7 8 9 8 9 a JZ wf1 1.0 0.0", "EX 13 16 9 11 14 14 b JX wf1 0.2 0.0"]),
    "rows_to": _mesh((92, 92, 98), ["PML 4"] * 3 + ["MUR"] * 3,
                     _sources(92, 92, 98) + ["PW 10 80 12 70 9 77 pw1 wf1 35.0 20.0 40.0 111111 1.0 0.0"], steps=40),
    "rows_beyond": _mesh((92, 92, 112), ["PML 4"] * 3 + ["MUR"] * 3,
                         _sources(92, 92, 112) + ["PW 10 80 12 70 9 77 pw1 wf1 35.0 20.0 40.0 111111 1.0 0.0"], steps=40),
}


def _differ(a, b):
    fa, fb = sorted(os.listdir(a)), sorted(os.listdir(b))
    assert fa == fb and fa, (fa, fb)
    return [f for f in fa if not filecmp.cmp(os.path.join(a, f), os.path.join(b, f), shallow=False)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_corrections_against_oracle(name, precision, tmp_path, monkeypatch):
    mesh = str(tmp_path / f"{name}.mesh")
    with open(mesh, "w") as f:
        f.write(MESHES[name])
    shutil.copy(os.path.join(GOLDEN, "ref_inputs", "closedbox_go04", "go04.pfe"), str(tmp_path))
    print(f"case {name} {precision}", flush=True)
    g, o = str(tmp_path / "gpu"), str(tmp_path / "oracle")
    vulture_amd.run_mesh(mesh, g, precision=precision)
    oracle.run_mesh(mesh, o, precision="fp64")
    r = compare_outputs(g, o)
    assert r["files"] >= 10, r
    if precision == "fp64":
        assert r["td"] <= 1e-12 and r["fd_raw"] <= 1e-12, r
    else:
        oracle.run_mesh(mesh, str(tmp_path / "oracle32"), precision="fp32")
        ref = compare_outputs(str(tmp_path / "oracle32"), o)
        assert r["td"] <= max(1e-4, 1.5 * ref["td"]), (r, ref)
    vulture_amd.run_mesh(mesh, str(tmp_path / "chunks"), precision=precision, chunk=14)
    assert not _differ(g, str(tmp_path / "chunks"))
    monkeypatch.setenv("VGPU_NO_INDEXED_MEDIA", "1")
    vulture_amd.run_mesh(mesh, str(tmp_path / "arrays"), precision=precision)
    assert not _differ(g, str(tmp_path / "arrays"))
