"""The library's own kernels and planning on the CPU (tests/native/cpu_hip: a
HIP runtime whose device memory is guarded host memory and whose launches run
block by block).

Corrections in line, in update rows, in rows and in groups of rows
(vgpu_inline.h) against the same set-up with its corrections in launches of
their own, over random meshes of every boundary, medium, source and surface
kind: all six fields agree to the bit, in both precisions, with and without
coefficient classes, solo and packed, whatever the order of a launch's blocks.
The update-once check agrees with what it finds of the separate launches."""
import ctypes
import os
import random
import shutil
import subprocess

import numpy as np
import pytest

import vulture_amd
from conftest import GOLDEN, ROOT

CLANG = "/opt/rocm/llvm/bin/clang++"
CSRC = os.path.join(ROOT, "vulture_amd", "csrc")
HOST = os.path.join(ROOT, "vulture_amd", "host")
CPU = os.path.join(ROOT, "tests", "native", "cpu_hip")
HOST_SRC = ["vh_parse.c", "vh_setup.c", "vh_voxel.c", "vh_observe.c", "vh_gpu.c", "vh_serve.c"]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    """Directory of libvgpu.so and libvhost.so, one library for the CPU."""
    if not os.path.exists(CLANG) or shutil.which("gcc") is None:
        pytest.skip("clang++ or gcc not available")
    d = tmp_path_factory.mktemp("cpu")
    cxx = [CLANG, "-std=c++17", "-O2", "-ffp-contract=off", "-fPIC", "-w", "-I" + CPU,
           "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-c"]
    jobs = []
    for src, extra in ((os.path.join(CSRC, "vgpu.hip"), ["-Dvgpu_create=vgpu_create_library"]),
                       (os.path.join(CSRC, "vgpu_k32.hip"), []), (os.path.join(CSRC, "vgpu_k64.hip"), []),
                       (os.path.join(CPU, "cpu_hip.cpp"), []), (os.path.join(CPU, "create.cpp"), [])):
        o = str(d / (os.path.basename(src) + ".o"))
        jobs.append((o, subprocess.Popen(cxx + extra + ["-x", "c++", src, "-o", o], stderr=subprocess.PIPE, text=True)))
    for src in HOST_SRC:
        o = str(d / (src + ".o"))
        jobs.append((o, subprocess.Popen(["gcc", "-std=gnu99", "-O2", "-fPIC", "-ffp-contract=off", "-w",
                                          "-DVH_REAL=double", "-I" + HOST, "-I" + os.path.join(ROOT, "include"), "-c",
                                          os.path.join(HOST, src), "-o", o], stderr=subprocess.PIPE, text=True)))
    for o, p in jobs:
        err = p.communicate()[1]
        assert p.returncode == 0, (o, err[-2000:])
    # its calls stay inside it, whatever else the process has loaded
    subprocess.run([CLANG, "-shared", "-Wl,-Bsymbolic", "-o", str(d / "libvgpu.so")] + [o for o, _ in jobs] +
                   ["-lm", "-lpthread"], check=True)
    os.symlink("libvgpu.so", str(d / "libvhost.so"))
    return str(d)


@pytest.fixture
def cpu(lib, monkeypatch):
    """The Python front end over the CPU build, which the device's library
    neither sees nor is seen by."""
    monkeypatch.setattr(ctypes, "RTLD_GLOBAL", ctypes.RTLD_LOCAL)
    monkeypatch.setattr(vulture_amd, "_LIB", lib)
    monkeypatch.setattr(vulture_amd, "_vgpu", None)
    monkeypatch.setattr(vulture_amd, "_host", None)
    return monkeypatch


def _box(rng, dm, flat=None):
    out = []
    for a in range(3):
        x = sorted((rng.randint(0, dm[a]), rng.randint(0, dm[a])))
        if x[0] == x[1]:
            x = [max(0, x[0] - 1), max(0, x[0] - 1) + 1]
        out += [x[0], x[0]] if a == flat else x
    return " ".join(map(str, out))


def random_mesh(seed, steps):
    """A small mesh of random faces, media, surfaces, sources and a plane wave."""
    rng = random.Random(seed)
    dm = [rng.choice([rng.randint(1, 5), rng.randint(5, 11), rng.randint(10, 16)]) for _ in range(3)]
    bt = []
    for a in range(3):
        if rng.random() < 0.2:
            bt += ["PERIODIC"] * 2
            continue
        bt += [rng.choice(["PEC", "PMC", "MUR", "PML 2", "PML 4"]) for _ in range(2)]
        if any(t.startswith(("MUR", "PML")) for t in bt[-2:]):
            dm[a] = max(dm[a], 4)
    body = []
    surfaces = rng.random() < 0.5
    if surfaces:
        body += ['BT s0 SIBC -0.5 0.25 0.25 -0.5', 'BT s1 SIBC "go04.pfe"']
    body += ["MT one DEBYE 2.0 0.01 1.0 1e9 -1e9", "MT two DEBYE 3.0 0.0 1.0 1e9 -1e9 4e9 -3e9", "MT d SIMPLE 4.0 0.02 1.0"]
    for _ in range(rng.randint(0, 4)):
        body.append(f"MB {_box(rng, dm)} {rng.choice(['one', 'two', 'd'])}{rng.choice(['', ' 101011', ' 111111', ' 000000'])}")
    for _ in range(2 if surfaces else 0):
        a = rng.randint(0, 2)
        if dm[a] < 5:
            continue
        b = _box(rng, dm, a).split()
        b[2 * a] = b[2 * a + 1] = str(rng.randint(2, dm[a] - 2))
        body.append("TB " + " ".join(b) + " " + rng.choice(["s0", "s1", "PEC"]))
    for s in range(rng.randint(1, 4)):
        kind = rng.choice(["EX", "EY", "EZ", "JX", "JY", "JZ", "JMX", "JMY", "HZ", "HX", "IDZ"])
        body.append(f"EX {_box(rng, dm, rng.choice([None, 0, 1, 2]))} s{s} {rng.choice(['', '='])}{kind} wf1 1.0 {rng.choice([0.0, 1e-12])}")
    if rng.random() < 0.5 and min(dm) >= 7:
        m = rng.randint(2, 3)
        body.append("PW " + " ".join(f"{m} {n - m}" for n in dm) +
                    f" pw1 wf1 {rng.uniform(0, 180):.2f} {rng.uniform(0, 360):.2f} {rng.uniform(0, 360):.2f} 111111 1.0 0.0")
    grid = "MS 1e-3"
    if rng.random() < 0.3:  # graded lines: the plane wave's analytic incident field
        grid = "\n".join(f"{ax}L\n" + "\n".join(f"{v:.9e}" for v in np.cumsum([0.0] + [1e-3 * rng.uniform(0.8, 1.2) for _ in range(n)]))
                         for ax, n in zip("XYZ", dm))
    at = [(rng.randint(0, n) for n in dm) for _ in range(4)]
    lines = ["VM 1.0.0", f"CE random mesh {seed}", "DM %d %d %d" % tuple(dm), "GS"]
    lines += [f"BT {f} {t}" for f, t in zip(("XLO", "XHI", "YLO", "YHI", "ZLO", "ZHI"), bt)]
    lines += ["WF wf1 GAUSSIAN_PULSE 1.0 3.0e-12 2.0e-12"] + body
    for q, p in enumerate(at):
        i, j, k = p
        lines += [f"OP {i} {i} {j} {j} {k} {k} t{q} TDOM_ASCII", f"OP {i} {i} {j} {j} {k} {k} f{q} FDOM_ASCII"]
    return "\n".join(lines + ["GE", f"NT {steps}", "OF 1e9 3e10 5", "CN 0.95", grid, "EN"]) + "\n"


def _stage(tmp_path, seed, steps):
    tmp_path.mkdir(parents=True, exist_ok=True)
    p = tmp_path / f"m{seed}.mesh"
    p.write_text(random_mesh(seed, steps))
    shutil.copy(os.path.join(GOLDEN, "ref_inputs", "closedbox_go04", "go04.pfe"), str(tmp_path))
    return str(p)


def _run(mesh, precision, steps):
    with vulture_amd.DeviceSolve(mesh, precision=precision, steps=steps) as ds:
        ds.run(0, steps // 2)
        ds.run(steps // 2, steps - steps // 2)
        ds.synchronize()
        fields = [ds.download(c) for c in range(6)]
        rep, counts = ds.check_limits()
        return fields, rep, counts, ds.stats()


@pytest.mark.parametrize("seed", range(60))
def test_corrections_against_separate_launches(cpu, seed, tmp_path):
    steps = 10
    mesh = _stage(tmp_path, seed, steps)
    precision = ("fp64", "fp32")[seed % 2]
    cpu.setenv("CPU_HIP_SEPARATE", "1")
    ref, rep0, counts0, st0 = _run(mesh, precision, steps)
    cpu.setenv("CPU_HIP_SEPARATE", "0")
    forms = [{}, {"CPU_HIP_ORDER": "reverse"}, {"VGPU_NO_INDEXED_MEDIA": "1"}]
    for env in forms[:1] + [forms[1 + seed // 2 % 2]]:
        with pytest.MonkeyPatch.context() as m:
            for k, v in env.items():
                m.setenv(k, v)
            got, rep, counts, st = _run(mesh, precision, steps)
        assert st["debye_sites"] == st0["debye_sites"] and st["correction_rows"] == st0["correction_rows"]
        assert rep == rep0 and np.array_equal(counts, counts0), env
        for c, (a, b) in enumerate(zip(got, ref)):
            assert np.array_equal(a, b), (env, c, int(np.sum(a != b)))


def test_random_meshes_are_alive(cpu, tmp_path):
    """Most of the random meshes carry fields, and each kind of part occurs."""
    texts = [random_mesh(s, 10) for s in range(60)]
    for word in ("PERIODIC", "PMC", "PEC", "MUR", "PML", " one", " two", "go04", "PW ", "XL", "JMX", "IDZ"):
        assert sum(word in t for t in texts) >= 5, word
    alive = 0
    for s in range(0, 60, 4):
        fields = _run(_stage(tmp_path, s, 10), "fp64", 10)[0]
        alive += all(np.count_nonzero(sum(abs(f) for f in fields[3 * h:3 * h + 3])) > 10 for h in range(2))
    assert alive >= 11


def test_packed_against_alone(cpu, tmp_path):
    """Eight of them in one packed group: the files of each run alone."""
    import filecmp
    for precision in ("fp64", "fp32"):
        meshes = [_stage(tmp_path, s, 12) for s in range(100, 108)]
        alone = [str(tmp_path / f"{precision}a{q}") for q in range(8)]
        grouped = [str(tmp_path / f"{precision}g{q}") for q in range(8)]
        for m, o in zip(meshes, alone):
            vulture_amd.run_mesh(m, o, precision=precision, chunk=4)
        vulture_amd.run_meshes_group(meshes, grouped, precision=precision, chunk=4)
        for a, b in zip(alone, grouped):
            files = sorted(os.listdir(a))
            assert files and files == sorted(os.listdir(b))
            assert filecmp.cmpfiles(a, b, files, shallow=False)[0] == files


@pytest.mark.parametrize("inside", [False, True])
def test_group_reports_failed_launches(cpu, inside):
    """A group run whose launches fail says so, also where no member has its
    corrections in line (ghost planes inside the sweeps' limits)."""
    from test_gpu_sweep_forms import N, _context
    vulture_amd.load_host()
    v = vulture_amd.load_vgpu()
    v.vgpu_create.restype = v.vgpu_finalize.restype = v.vgpu_set_media.restype = ctypes.c_int
    v.vgpu_destroy.argtypes = [ctypes.c_void_p]
    lim = [[1, N - 2] * 3 for _ in range(6)]
    if inside:
        lim[0][1] = N - 1
    ctxs = [_context(v, lim, (1, 1, 3, 3, 2, 2)) for _ in range(2)]
    group, first = (ctypes.c_void_p * 2)(*ctxs), (ctypes.c_uint64 * 2)(0, 0)
    assert v.vgpu_run_group(group, 2, first, ctypes.c_uint64(4)) == 0
    first[0] = first[1] = 4
    cpu.setenv("CPU_HIP_ERROR", "1")
    assert v.vgpu_run_group(group, 2, first, ctypes.c_uint64(4)) == -3
    assert b"kernel launch failed" in v.vgpu_last_error(ctxs[0])
    cpu.setenv("CPU_HIP_ERROR", "0")
    for c in ctxs:
        v.vgpu_destroy(c)
