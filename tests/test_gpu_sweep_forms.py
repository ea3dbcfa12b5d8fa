"""The launch forms of the step that the default sizes of the other tests do
not take (needs an MI355X)."""
import ctypes
import filecmp
import math
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


class _Grid(ctypes.Structure):
    """vgpu_grid_desc (include/vgpu.h)."""
    _I6, _D = ctypes.c_int * 6, ctypes.POINTER(ctypes.c_double)
    _fields_ = [("nx", ctypes.c_int), ("ny", ctypes.c_int), ("nz", ctypes.c_int), ("gibox", _I6), ("gobox", _I6),
                ("gfilim", _I6 * 6), ("dt", ctypes.c_double), ("c0", ctypes.c_double), ("eps0", ctypes.c_double),
                ("mu0", ctypes.c_double), ("eta0", ctypes.c_double), ("grid_type", ctypes.c_int),
                ("xlines", _D), ("ylines", _D), ("zlines", _D), ("nlines", ctypes.c_int * 3),
                ("dex", _D), ("dey", _D), ("dez", _D), ("idex", _D), ("idey", _D), ("idez", _D),
                ("idhx", _D), ("idhy", _D), ("idhz", _D)]


N, ALPHA, BETA, GAMMA, SIZE = 8, 0.9, 0.4, 0.3, 2.0


def _context(v, lim, ghosts):
    """A uniform N^3 grid of unit edges in FP64, a hard Ez source at (3, 4, 4)
    that holds SIZE from the second step on (a compact step of tiny width)."""
    ones = np.ones(N + 1)
    dp = ones.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    g = _Grid(nx=N, ny=N, nz=N, dt=1.0, c0=1.0, eps0=1.0, mu0=1.0, eta0=1.0, grid_type=0)
    for q in range(6):
        g.gibox[q] = g.gobox[q] = 1 if q % 2 == 0 else N - 1
        for c in range(6):
            g.gfilim[c][q] = lim[c][q]
    g.nlines = (ctypes.c_int * 3)(N, N, N)
    for f in ("xlines", "ylines", "zlines", "dex", "dey", "dez", "idex", "idey", "idez", "idhx", "idhy", "idhz"):
        setattr(g, f, dp)
    ctx = ctypes.c_void_p()
    assert v.vgpu_create(ctypes.byref(g), 0, 0, ctypes.byref(ctx)) == 0
    arrays = [np.full(N ** 3, x) for x in (ALPHA, BETA, GAMMA)]
    p3 = ctypes.c_void_p * 3
    assert v.vgpu_set_media(ctx, *[p3(*[a.ctypes.data] * 3) for a in arrays]) == 0
    assert v.vgpu_set_ghosts(ctx, (ctypes.c_int * 6)(*ghosts)) == 0
    d = ctypes.c_double
    assert v.vgpu_add_waveform(ctx, 8, d(1.0), d(0.0), d(1e-9), d(0.25), None, ctypes.c_ulong(0)) == 0
    assert v.vgpu_add_source(ctx, 2, 0, 0, d(SIZE), 0, d(0.0), (ctypes.c_int * 6)(3, 3, 4, 4, 4, 4)) == 0
    assert v.vgpu_finalize(ctx, ctypes.c_uint64(64), ctypes.c_uint64(64)) == 0, v.vgpu_last_error(ctx)
    return ctx


def _expected(lim, ghosts, steps):
    """The same steps in numpy: sweeps over the limits, source, ghost copies."""
    E, H = np.zeros((3, N, N, N)), np.zeros((3, N, N, N))

    def sweep(F, G, e):
        new = F.copy()
        for c in range(3):
            l = lim[3 * (not e) + c]
            at = tuple(slice(l[2 * a], l[2 * a + 1] + 1) for a in range(3))
            a1, a2 = (c + 1) % 3, (c + 2) % 3
            s = 1 if e else -1  # E reads the value below, H the one above

            def diff(g, a):
                return (g - np.roll(g, s, a))[at] * (1 if e else -1)
            curl = diff(G[a2], a1) - diff(G[a1], a2)
            new[c][at] = (ALPHA * F[c][at] + BETA * curl) if e else F[c][at] - GAMMA * curl
        F[:] = new

    def copy(F, e):
        for f, t in enumerate(ghosts):
            a, hi = f >> 1, f & 1
            if not t:
                continue
            dst, src = (N - 1, N - 2) if hi else (0, 1)
            if t == 3:
                src = 1 if hi else N - 2
            for c in range(3):
                if (c == a) == e:
                    i, j = [slice(None)] * 3, [slice(None)] * 3
                    i[a], j[a] = dst, src
                    F[c][tuple(i)] = (-1.0 if t == 2 else 1.0) * F[c][tuple(j)]

    for n in range(steps):
        sweep(E, H, True)
        # a compact step of no width times sin(2 pi n / 4)
        E[2][3, 4, 4] = SIZE * math.sin(2.0 * 4.0 * math.atan(1.0) * 0.25 * n) if n else 0.0
        copy(E, True)
        sweep(H, E, False)
        copy(H, False)
    return list(E) + list(H)


def _download(v, ctx):
    out = []
    for c in range(6):
        a = np.empty((N, N, N))
        assert v.vgpu_download_field(ctx, c, a.ctypes.data_as(ctypes.c_void_p)) == 0
        out.append(a)
    return out


@pytest.mark.parametrize("ghosts", [(1, 2, 3, 3, 2, 1), (3, 3, 1, 1, 2, 2)])
@pytest.mark.parametrize("inside", [False, True])
def test_ghost_planes_and_limits(inside, ghosts):
    """Ghost planes beside the sweeps' limits, and inside them, where the
    sweep's value is overwritten by the copy: alone and in a group run."""
    vulture_amd.load_host()
    v = vulture_amd.load_vgpu()
    v.vgpu_create.restype = v.vgpu_finalize.restype = v.vgpu_set_media.restype = ctypes.c_int
    v.vgpu_destroy.argtypes = [ctypes.c_void_p]
    steps = 12
    usual = [[1, N - 2] * 3 for _ in range(6)]
    lim = [l[:] for l in usual]
    if inside:  # each ghost component over its ghost planes too
        for c in range(6):
            for a in range(3):
                if (c < 3) == (c % 3 == a):
                    lim[c][2 * a + 1] = N - 1
                    if c < 3:
                        lim[c][2 * a] = 1
    print(f"case ghost planes inside {inside} {ghosts}", flush=True)
    ctxs = [_context(v, l, ghosts) for l in (lim, lim, usual, usual)]
    try:
        for ctx in (ctxs[0], ctxs[2]):
            assert v.vgpu_run(ctx, 0, steps, None) == 0
        first = (ctypes.c_uint64 * 2)(0, 0)
        group = (ctypes.c_void_p * 2)(ctxs[1], ctxs[3])
        for n in range(0, steps, 4):
            first[0] = first[1] = n
            assert v.vgpu_run_group(group, 2, first, ctypes.c_uint64(4)) == 0
        for ctx in ctxs:
            assert v.vgpu_synchronize(ctx) == 0
        alone, grouped = _download(v, ctxs[0]), _download(v, ctxs[1])
        exp = _expected(lim, ghosts, steps)
        for a, b, x in zip(alone, grouped, exp):
            assert np.array_equal(a, b)
            assert np.max(np.abs(a - x)) <= 1e-13 * max(1.0, np.max(np.abs(x)))
        assert any(np.count_nonzero(a) > 100 for a in alone)
    finally:
        for ctx in ctxs:
            v.vgpu_destroy(ctx)


# ---------------------------------------------------------------------------
# The sweeps' forms by size.  The fused leapfrog sweep (VGPU_LEAP=1) keeps the
# corrections in launches of their own, with operands and order of its own
# arrays; its fields are the separate sweeps' to the bit.
# ---------------------------------------------------------------------------
def _mesh(dm, bt, body, steps):
    nx, ny, nz = dm
    lines = ["VM 1.0.0", "CE sweep forms", "DM %d %d %d" % dm, "GS"]
    lines += [f"BT {f} {t}" for f, t in zip(("XLO", "XHI", "YLO", "YHI", "ZLO", "ZHI"), bt)]
    lines += ["WF wf1 GAUSSIAN_PULSE 1.0 3.0e-11 1.0e-11", *body,
              f"PW 5 {nx - 5} 4 {ny - 6} 6 {nz - 4} pw1 wf1 35.0 20.0 40.0 111111 1.0 0.0",
              f"EX 1 3 1 {ny - 1} 1 {nz - 1} b JZ wf1 1.0 0.0", f"EX {nx - 2} {nx - 1} 2 6 1 3 c =EZ wf1 0.5 1.0e-12",
              f"EX 7 8 3 5 {nz - 1} {nz - 1} e =JMY wf1 250.0 2.0e-12",
              f"OP {nx // 2} {nx // 2} {ny // 2} {ny // 2} {nz // 2} {nz // 2} t TDOM_ASCII"]
    return "\n".join(lines + ["GE", f"NT {steps}", "CN 0.95", "MS 1e-3", "EN"]) + "\n"


def _cells(dm, bt, precision):
    """Cells of the allocation: layers and a ghost each side, whole lines in x."""
    layers = [sum(int(t.split()[1]) for t in bt[2 * a:2 * a + 2] if t.startswith("PML")) for a in range(3)]
    n = [dm[a] + layers[a] + 2 for a in range(3)]
    line = 16 if precision == "fp64" else 32
    return (n[0] + line - 1) // line * line * n[1] * n[2]


MEDIA = ["MT one DEBYE 2.0 0.01 1.0 1e9 -1e9", "MT two DEBYE 3.0 0.0 1.0 1e9 -1e9 4e9 -3e9"]
BLOCKS = ["MB 3 40 10 50 12 60 one", "MB 30 60 20 62 5 40 two", "MB 38 46 15 25 20 30 one", "MB 50 55 4 9 60 70 one"]
PML = ["PML 5"] * 6
MIXED = ["PML 4", "MUR", "PMC", "PEC", "MUR", "PML 6"]
MUR = ["MUR"] * 6
ROWS_MAX = 1000000  # cells of the largest grids with update rows
APART = 64 << 20    # bytes of a field beyond which the fast tiles launch apart


def _agree_with_fused_sweep(dm, bt, body, precision, steps, tmp_path, monkeypatch, files=()):
    mesh = _write(tmp_path, _mesh(dm, bt, body, steps))
    for name, text in files:
        (tmp_path / name).write_text(text)
    with vulture_amd.DeviceSolve(mesh, precision=precision, steps=steps) as ds:
        st = ds.stats()
        ds.run(0, steps)
        ds.synchronize()
        a = [ds.download(c) for c in range(6)]
    assert not st["leap"]
    monkeypatch.setenv("VGPU_LEAP", "1")
    with vulture_amd.DeviceSolve(mesh, precision=precision, steps=steps) as ds:
        assert ds.stats()["leap"]
        ds.run(0, steps)
        ds.synchronize()
        for c in range(6):
            b = ds.download(c)
            assert np.count_nonzero(b) > b.size // 20
            assert np.array_equal(a[c], b), c
    return st


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("bt", [PML, MIXED, MUR], ids=["pml", "mixed", "mur"])
@pytest.mark.parametrize("debye", [False, True])
@pytest.mark.parametrize("side", ["below", "above"])
def test_forms_either_side_of_the_update_rows(side, debye, bt, precision, tmp_path, monkeypatch):
    """The largest grid with update rows and the smallest without: the same
    x and y extents, one plane more."""
    dm = [84, 84, 90]
    while _cells(dm, bt, precision) <= ROWS_MAX:
        dm[2] += 1
    dm[2] -= side == "below"
    dm = tuple(dm)
    assert (_cells(dm, bt, precision) <= ROWS_MAX) == (side == "below")
    print(f"case forms at {dm} {bt[1]} Debye {debye} {precision}", flush=True)
    st = _agree_with_fused_sweep(dm, bt, (MEDIA + BLOCKS if debye else []), precision, 30, tmp_path, monkeypatch)
    assert bool(st["debye_fused"]) == debye


@pytest.mark.parametrize("precision,n", [("fp64", 208), ("fp32", 260)])
@pytest.mark.parametrize("bt", [PML, MIXED], ids=["pml", "mixed"])
@pytest.mark.parametrize("debye", [False, True])
def test_forms_with_tiles_apart(debye, bt, precision, n, tmp_path, monkeypatch):
    """Fields past 64 MB: shell and side blocks, then the fast tiles."""
    dm = (n, n, n)
    assert _cells(dm, bt, precision) * (8 if precision == "fp64" else 4) > APART
    print(f"case tiles apart {dm} {bt[1]} Debye {debye} {precision}", flush=True)
    st = _agree_with_fused_sweep(dm, bt, (MEDIA + BLOCKS if debye else []), precision, 100, tmp_path, monkeypatch)
    assert bool(st["debye_fused"]) == debye


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [40, 104])
def test_forms_with_sibc(n, precision, tmp_path, monkeypatch):
    """SIBC faces with their H terms in update rows (40^3) and in rows (104^3)."""
    from vulture_amd import pfe
    dm = (n, n, n)
    assert (_cells(dm, MIXED, precision) <= ROWS_MAX) == (n == 40)
    body = ['BT s0 SIBC "slab.pfe"', "BT s1 SIBC -0.5 0.25 0.25 -0.5", f"TB 12 12 8 {n - 9} 7 {n - 8} s0",
            f"TB 14 {n - 8} 9 {n - 12} 15 15 s0", f"TB 15 {n - 7} 13 13 18 {n - 6} s1"]
    slab = pfe.pfe_text(pfe.fit_slab(1e6, 5e-4, fmax=3e10, per_decade=2))
    print(f"case SIBC {dm} {precision}", flush=True)
    st = _agree_with_fused_sweep(dm, MIXED, body, precision, 60, tmp_path, monkeypatch, [("slab.pfe", slab)])
    assert st["sibc_faces"] > 1000


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("chunk", [0, 14])
def test_corrections_packed(chunk, precision, tmp_path):
    """The meshes of the corrections' oracle tests in one packed group: each
    one's files are its own run's, byte for byte."""
    import shutil

    from conftest import GOLDEN
    from test_gpu_inline import MESHES
    names = sorted(MESHES)
    meshes = []
    for name in names:
        d = tmp_path / name
        meshes.append(_write(d, MESHES[name]))
        shutil.copy(os.path.join(GOLDEN, "ref_inputs", "closedbox_go04", "go04.pfe"), str(d))
    print(f"case packed corrections {precision} {chunk}", flush=True)
    for name, m in zip(names, meshes):
        vulture_amd.run_mesh(m, str(tmp_path / name / "alone"), precision=precision, chunk=chunk)
    vulture_amd.run_meshes_group(meshes, [str(tmp_path / name / "group") for name in names], precision=precision,
                                 chunk=chunk)
    for name in names:
        a, b = str(tmp_path / name / "alone"), str(tmp_path / name / "group")
        files = sorted(os.listdir(a))
        assert files and files == sorted(os.listdir(b))
        assert filecmp.cmpfiles(a, b, files, shallow=False)[0] == files, name
