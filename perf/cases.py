"""The work that a user of this framework has it do, as cases that can be timed.

A case is one mesh (or a group of meshes) of a kind the framework's own
generators write (vulture_amd.meshgen) and a storage precision.  Most cases
step a resident solve through the C-ABI (include/vgpu.h) the way a streaming
host does: `vgpu_run` of one chunk of time steps, then the chunk's volume
samples (`vgpu_run_result`) and the running spectra of its frequency-domain
observers (`vgpu_read_point_observer`).  `prepare` leaves each solve some way
into its run, with the incident pulse on the grid, which is the state that
nearly every step of a real solve meets.  One case is a whole call
(`run_mesh`: parse, set-up, upload, loop, files).

Kinds:
  free       free space, 6-cell UPML, a hard Ez point source
  spheres    cubic mesh with Debye spheres (one voxel object), 8-cell UPML,
             TF/SF plane wave on the auxiliary grid
  cavity     the Debye spheres in a PEC box with a hard point source
  request    graded lines, SIMPLE and Debye blocks, 8-cell UPML, analytic TF/SF
             plane wave: a request of the solve server
  group      up to 16 small requests stepped together (`vgpu_run_group`)
  enclosure  graded shielded enclosure with a slot, 10-cell UPML, analytic TF/SF
             plane wave, a 512-frequency observer
  box        SIBC conductor walls inside Mur faces, dielectric blocks, a dipole
  solve      `run_mesh` on a request
"""
import ctypes
import math
import os
import re
import shutil
import tempfile

import numpy as np
import torch

import vulture_amd
from vulture_amd import meshgen, obsfiles

NT = 200000  # steps of a resident solve: more than one timing of it takes


def listed():
    return [
        # the smallest call: a few steps of a validation-size grid, bound by launches and latency
        dict(name="free_40_fp64", kind="free", precision="fp64", nx=40, ny=40, nz=40, steps=10),
        # a small odd-sized closed resonator: no absorbing layers, ghost planes on every face
        dict(name="cavity_75_fp32", kind="cavity", precision="fp32", nx=75, ny=75, nz=75, spheres=12, steps=20),
        # a small request of the server on its own
        dict(name="request_small_fp32", kind="request", precision="fp32", nx=53, ny=41, nz=62, steps=20),
        # sixteen small requests packed, as the server runs them under load
        dict(name="group_16_fp32", kind="group", precision="fp32", nx=72, ny=72, nz=72, members=16, steps=20),
        # a medium request: a third of its cells in the absorbing layers
        dict(name="request_medium_fp32", kind="request", precision="fp32", nx=101, ny=115, nz=108, steps=20),
        # a large request, ragged on every axis
        dict(name="request_large_fp32", kind="request", precision="fp32", nx=173, ny=211, nz=158, steps=20),
        # the shielded enclosure in the plain FP64 form
        dict(name="enclosure_200_fp64", kind="enclosure", precision="fp64", nx=200, ny=160, nz=120, steps=20),
        # a medium Debye volume in the plain FP64 form
        dict(name="spheres_128_fp64", kind="spheres", precision="fp64", nx=128, ny=128, nz=128, spheres=60, steps=20),
        # the Debye volume of the benchmark, the largest single solve
        dict(name="spheres_256_fp32", kind="spheres", precision="fp32", nx=256, ny=256, nz=256, spheres=200, steps=20),
        # conductor walls and Mur faces: FP32 at size, and the FP64 form's per-filter state
        dict(name="box_256_fp32", kind="box", precision="fp32", nx=256, ny=256, nz=160, steps=20),
        dict(name="box_96_fp64", kind="box", precision="fp64", nx=96, ny=81, nz=64, steps=20),
        # a whole call: mesh file in, observer files out
        dict(name="solve_small_fp32", kind="solve", precision="fp32", nx=48, ny=56, nz=40, steps=1500),
    ]


def draw(rng):
    kind = rng.choice(["free", "spheres", "cavity", "request", "request", "request", "group", "enclosure", "box", "box"])

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    case = dict(kind=kind, precision=rng.choice(["fp32", "fp32", "fp64"]), steps=rng.choice([10, 16, 20, 24, 30]))
    if kind in ("free", "spheres", "cavity"):
        n = size(24, 96) if kind == "free" else size(40, 200) if kind == "spheres" else size(33, 150)
        case.update(nx=n, ny=n, nz=n)
        if kind != "free":
            case["spheres"] = rng.randint(3, 8 if n < 64 else 40)
    elif kind == "request":
        case.update(nx=size(32, 220), ny=size(32, 220), nz=size(32, 220))
    elif kind == "group":
        n = size(40, 80)
        case.update(nx=n, ny=n, nz=n, members=rng.randint(2, 16))
    elif kind == "enclosure":
        case.update(nx=size(48, 220), ny=size(40, 180), nz=size(32, 150))
    else:
        case.update(nx=size(40, 220), ny=size(36, 220), nz=size(32, 160))
    return case


# ---------------------------------------------------------------------------
# meshes
# ---------------------------------------------------------------------------

def _warm_steps(case):
    """Steps before the timed ones: the pulse has entered and spread."""
    across = int(2.4 * max(case["nx"], case["ny"], case["nz"]))  # a uniform grid's wave moves half a cell per step
    want = {"free": 100, "cavity": across, "spheres": across, "request": 300, "group": 300, "enclosure": 400, "box": across}
    s = case["steps"]
    return -(-want[case["kind"]] // s) * s


def _request(rng, n, steps):
    """A serving request of exactly n cells per axis."""
    text, got, _ = meshgen.serving_request(_Fixed(rng, n), steps_min=steps, steps_max=steps)
    assert tuple(got) == tuple(n)
    return text


class _Fixed:
    """A numpy generator whose first draws give wanted axis lengths."""

    def __init__(self, rng, n):
        self._rng, self._n = rng, list(n)

    def uniform(self, *a, **k):
        return math.log(self._n.pop(0)) if self._n else self._rng.uniform(*a, **k)

    def __getattr__(self, name):
        return getattr(self._rng, name)


def _meshes(case, seed):
    """[(mesh text, {file: body})] of a case, from the seed alone."""
    kind = case["kind"]
    n = (case["nx"], case["ny"], case["nz"])
    rng = np.random.default_rng([seed, 77])
    if kind == "free":
        c = n[0] // 2
        text = meshgen.freespace(steps=NT, n=n[0])
        at = [int(c + rng.integers(-2, 3)) for _ in range(3)]
        text = text.replace(f"EX {c} {c} {c} {c} {c} {c + 1} src =EZ wf1 1.0",
                            f"EX {at[0]} {at[0]} {at[1]} {at[1]} {at[2]} {at[2] + 1} src =EZ wf1 {rng.uniform(0.5, 2):.6f}")
        text = text.replace("GE\n", f"OP {c + 4} {c + 4} {c - 5} {c - 5} {c + 3} {c + 3} opf FDOM_ASCII\nGE\nOF 1e7 1e9 64\n")
        out = [(text, {})]
    elif kind in ("spheres", "cavity"):
        closed = kind == "cavity"
        out = [meshgen.debye(steps=NT, n=n[0], spheres=case["spheres"], rmin=min(4, n[0] // 12), rmax=min(20, n[0] // 8),
                             seed=int(rng.integers(1 << 30)), voxel=True, planewave=not closed,
                             boundary="PEC" if closed else "PML")]
    elif kind == "request":
        out = [(_request(rng, n, NT), {})]
    elif kind == "group":
        # members from 32 cells per axis up to the case's, of the same sizes for every seed
        sizes = np.random.default_rng(list(n)).integers(32, np.array(n) + 1, (case["members"], 3)).tolist()
        out = [(_request(rng, m, NT), {}) for m in sizes]
    elif kind == "enclosure":
        text = meshgen.enclosure(steps=NT, nx=n[0], ny=n[1], nz=n[2])
        theta, phi, eta = rng.uniform(20, 160), rng.uniform(20, 160), rng.uniform(0, 180)
        out = [(text.replace("wf1 90 90 90", f"wf1 {theta:.4f} {phi:.4f} {eta:.4f}"), {})]
    elif kind == "box":
        out = [meshgen.sibc_box(steps=NT, nx=n[0], ny=n[1], nz=n[2], seed=int(rng.integers(1 << 30)))]
    else:
        out = [(_request(rng, n, case["steps"]), {})]
    if kind == "solve":
        return out
    done = []
    for text, files in out:
        m = [int(v) for v in re.search(r"^DM (\d+) (\d+) (\d+)", text, re.M).groups()]
        step = [max(1, v // 8) for v in m]
        vol = f"OP 1 {m[0] - 1} 1 {m[1] - 1} 1 {m[2] - 1} lattice TDOM_BINARY {step[0]} {step[1]} {step[2]}\n"
        done.append((text.replace("\nGE\n", "\n" + vol + "GE\n"), files))
    return done


def _write(text, files, folder):
    os.makedirs(folder, exist_ok=True)
    path = os.path.join(folder, "case.mesh")
    with open(path, "w") as f:
        f.write(text)
    for name, body in files.items():
        with open(os.path.join(folder, name), "wb" if isinstance(body, bytes) else "w") as f:
            f.write(body)
    return path


def _observers(text):
    """[(name, type, box, step)] of the OP cards, in order."""
    out = []
    for ln in text.splitlines():
        if ln.startswith("OP "):
            w = ln.split()
            out.append((w[7], w[8], [int(v) for v in w[1:7]], [int(v) for v in w[9:12]] or [1, 1, 1]))
    return out


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

class _Solve:
    """A mesh resident on the device (vh_gpu_open) and its observers' ids."""

    def __init__(self, text, files, precision, chunk):
        self.host, self.v = vulture_amd.load_host(), vulture_amd.load_vgpu()
        self.v.vgpu_run_result.argtypes = [ctypes.c_void_p, ctypes.c_uint64, ctypes.c_int, ctypes.POINTER(ctypes.c_double),
                                           ctypes.POINTER(ctypes.POINTER(ctypes.c_float)), ctypes.POINTER(ctypes.c_uint64)]
        self.v.vgpu_read_point_observer.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_uint64,
                                                    ctypes.c_void_p, ctypes.c_void_p]
        self.v.vgpu_run_group.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_int, ctypes.POINTER(ctypes.c_uint64),
                                          ctypes.c_uint64]
        self.solve, self.ctx = ctypes.c_void_p(), ctypes.c_void_p()
        folder = tempfile.mkdtemp(prefix="case_")
        err = ctypes.create_string_buffer(1024)
        try:
            rc = self.host.vh_gpu_open(os.fsencode(_write(text, files, folder)), 1 if precision == "fp32" else 0, 0, -1, chunk,
                                       ctypes.byref(self.solve), ctypes.byref(self.ctx), err, len(err))
        finally:
            shutil.rmtree(folder, ignore_errors=True)
        if rc != 0:
            raise RuntimeError(err.value.decode(errors="replace"))
        self.chunk, self.next = chunk, 0
        ops = _observers(text)
        points = [o for o in ops if o[1] != "TDOM_BINARY"]
        nf = int(re.search(r"^OF \S+ \S+ (\d+)", text, re.M).group(1))
        self.spectra = [(i, nf) for i, o in enumerate(points) if o[1] == "FDOM_ASCII"]
        (_, _, b, s), = [o for o in ops if o[1] == "TDOM_BINARY"]
        self.nodes = math.prod(1 + (b[2 * a + 1] - b[2 * a]) // s[a] for a in range(3))

    def check(self, rc):
        if rc < 0:
            raise RuntimeError(self.v.vgpu_last_error(self.ctx).decode(errors="replace"))

    def enqueue(self):
        if self.next + self.chunk > NT:
            self.next = 0
        self.check(self.v.vgpu_run(self.ctx, self.next, self.chunk, None))
        self.next += self.chunk

    def results(self):
        """The last chunk's volume samples and every spectrum so far."""
        p = ctypes.POINTER(ctypes.c_float)()
        self.check(self.v.vgpu_run_result(self.ctx, self.next - self.chunk, 1, None, ctypes.byref(p), None))
        out = [np.ctypeslib.as_array(p, (self.chunk, self.nodes, 6)).copy()]
        for i, nf in self.spectra:
            re_im = np.empty((2, 6, nf))
            self.check(self.v.vgpu_read_point_observer(self.ctx, i, None, 0, re_im[0].ctypes.data, re_im[1].ctypes.data))
            out.append(re_im)
        return out

    def __del__(self):
        if self.solve:
            self.host.vh_gpu_close(self.solve, self.ctx)
            self.solve = None


def _enqueue_group(solves):
    n, chunk = len(solves), solves[0].chunk
    if solves[0].next + chunk > NT:
        for s in solves:
            s.next = 0
    ctxs = (ctypes.c_void_p * n)(*[s.ctx for s in solves])
    first = (ctypes.c_uint64 * n)(*[s.next for s in solves])
    rc = solves[0].v.vgpu_run_group(ctxs, n, first, chunk)
    if rc < 0:
        raise RuntimeError(f"vgpu_run_group: {rc}")
    for s in solves:
        s.next += chunk


class _Folder:
    def __init__(self, text, files):
        self.path = tempfile.mkdtemp(prefix="case_")
        self.mesh = _write(text, files, self.path)

    def __del__(self):
        shutil.rmtree(self.path, ignore_errors=True)


def prepare(case, seed):
    meshes = _meshes(case, seed)
    if case["kind"] == "solve":
        return dict(case=case, folder=_Folder(*meshes[0]))
    solves = [_Solve(text, files, case["precision"], case["steps"]) for text, files in meshes]
    state = dict(case=case, solves=solves)
    for _ in range(_warm_steps(case) // case["steps"]):
        _enqueue(state)
    for s in solves:
        s.check(s.v.vgpu_synchronize(s.ctx))
    return state


def _enqueue(state):
    if state["case"]["kind"] == "group":
        _enqueue_group(state["solves"])
    else:
        state["solves"][0].enqueue()


def run(state):
    if "folder" in state:
        f = state["folder"]
        out = os.path.join(f.path, "out")
        vulture_amd.run_mesh(f.mesh, out, precision=state["case"]["precision"])
        return [obsfiles.read_fd(p)[1] for p in obsfiles.observer_files(out, "eh_*_fd.asc")]
    _enqueue(state)
    return [s.results() for s in state["solves"]]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    """Each step reads and writes each field once, reads the two 16-bit
    coefficient classes of every cell, reads and writes the UPML's three
    auxiliaries per component, the Debye edges' currents and the conductor
    walls' filter states.  Flops: 36 per cell's six updates."""
    kind, word = case["kind"], 4 if case["precision"] == "fp32" else 8
    n = [case["nx"], case["ny"], case["nz"]]
    members = case.get("members", 1)
    if kind == "group":  # members are uniform between 32 cells per axis and the case's
        n = [(32 + v) / 2 for v in n]
    pml = {"free": 6, "enclosure": 10, "cavity": 0, "box": 0}.get(kind, 8)
    inner = math.prod(n)
    cells = math.prod(v + 2 * pml for v in n)
    step = cells * (12 * word + 4) + (cells - inner) * 18 * word
    if "spheres" in case:
        lo, hi = min(4, n[0] // 12), min(20, n[0] // 8)
        volume = sum(4 / 3 * math.pi * r ** 3 for r in range(lo, hi + 1)) / (hi - lo + 1)
        step += case["spheres"] * volume * 3 * 2 * word
    if kind == "box":
        w = [v - 4 for v in n]
        faces = 2 * (w[0] * w[1] + w[1] * w[2] + w[2] * w[0])
        step += faces * 4 * 14 * 16
    if kind != "solve":
        step += 9 ** 3 * 6 * 4
    return {"bytes": float(step * case["steps"] * members), "flops": 36.0 * cells * case["steps"] * members}


# ---------------------------------------------------------------------------
# the same steps in plain torch, FP64
# ---------------------------------------------------------------------------

C0 = 299792458.0
MU0 = 4e-7 * math.pi
EPS0 = 1.0 / (MU0 * C0 * C0)
ETA0 = math.sqrt(MU0 / EPS0)


def _limits(box, inc=(1, 1, 1, 1, 1, 1)):
    """Inclusive index limits of the six components over a box of nodes: a
    component lying in a face is included there when the face is."""
    out = []
    for f in range(6):
        lim = []
        for a in range(3):
            lies = (f % 3 != a) if f < 3 else (f % 3 == a)
            lo, hi = box[2 * a], box[2 * a + 1]
            lim.append((lo + 1 if lies and not inc[2 * a] else lo, hi if lies and inc[2 * a + 1] else hi - 1))
        out.append(lim)
    return out


def _cut(lim):
    return tuple(slice(lo, max(lo, hi + 1)) for lo, hi in lim)


def _moved(lim, axis, by):
    return tuple(slice(lo + (by if a == axis else 0), max(lo, hi + 1) + (by if a == axis else 0)) for a, (lo, hi) in enumerate(lim))


class _Fdtd:
    """Yee leapfrog with UPML, Debye media, a hard source and TF/SF plane
    waves, all in FP64, on the cards of one mesh."""

    def __init__(self, text, files):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        lines = text.splitlines()
        card = {}
        for ln in lines:
            w = ln.split()
            if w and re.fullmatch(r"[A-Z]{2}", w[0]):
                card.setdefault(w[0], []).append(w[1:])
        self.m = [int(v) for v in card["DM"][0]]
        self.pml = [int(w[2]) if w[1] == "PML" else 0 for w in card["BT"][:6]][0]
        if any(w[1] not in ("PML", "PEC") for w in card["BT"]):
            raise NotImplementedError(text[:80])
        p, m = self.pml, self.m
        self.gi = [v for a in range(3) for v in (1 + p, 1 + p + m[a])]
        self.go = [v for a in range(3) for v in (1, 1 + 2 * p + m[a])]
        self.shape = [v + 2 * p + 2 for v in m]
        if "XL" in card:
            self.x = []
            for c in "XYZ":
                at = lines.index(c + "L")
                self.x.append(np.array([float(v) for v in lines[at + 1:at + 2 + m["XYZ".index(c)]]]))
        else:
            d = float(card["MS"][0][0])
            self.x = [np.arange(v + 1) * d for v in m]
        self._edges(float(card["CN"][0][0]) if "CN" in card else math.sqrt(3) / 2)
        self._media(card, files)
        self._profiles()
        self.f = [self._zeros() for _ in range(6)]
        if p:
            self.aux = [[self._zeros() for _ in range(2)] for _ in range(3)] + [[self._zeros()] for _ in range(3)]
        w = card["WF"][0]
        self.wf = [float(v) for v in w[2:5]]
        self.hard = [(w[:6], w[8], float(w[9])) for w in card.get("EX", [])]
        self.pw = [self._plane_wave(w) for w in card.get("PW", [])]
        self.n = 0

    def _zeros(self):
        return torch.zeros(self.shape, dtype=torch.float64, device=self.dev)

    def _edges(self, courant):
        self.ide, self.idh, self.de, dmin = [], [], [], []
        p = self.pml
        for a in range(3):
            d = np.diff(self.x[a])
            de = np.concatenate([np.full(p + 1, d[0]), d, np.full(p + 1, d[-1])])
            dh = np.concatenate([de[:1], 0.5 * (de[1:] + de[:-1])])
            dh[0] = dh[1]
            self.de.append((de, dh))
            dmin.append(min(de.min(), dh.min()))
            for to, v in ((self.ide, 1 / de), (self.idh, 1 / dh)):
                s = [1, 1, 1]
                s[a] = -1
                to.append(torch.tensor(v, device=self.dev).reshape(s))
        self.dt = courant / C0 / math.sqrt(sum(1 / v ** 2 for v in dmin))
        self.cubic = all(np.allclose(np.diff(x), self.x[0][1] - self.x[0][0], rtol=0, atol=1e-5) for x in self.x)

    def _media(self, card, files):
        dt = self.dt
        self.alpha = [torch.ones_like(self._zeros()) for _ in range(3)]
        self.beta = [torch.full_like(self.alpha[0], dt / EPS0) for _ in range(3)]
        self.gamma = dt / MU0
        media = {}
        for w in card.get("MT", []):
            if w[1] == "VOXEL":
                continue
            eps, sig = float(w[2]), float(w[3])
            da = db = total = None
            if w[1] == "DEBYE":
                res, pole = float(w[5]), float(w[6])
                da, db = (1 + 0.5 * dt * pole) / (1 - 0.5 * dt * pole), EPS0 * res / (1 - 0.5 * dt * pole)
            total = db or 0.0
            low = 2 * eps * EPS0 + 2 * total * dt + dt * sig
            media[w[0]] = ((low - 2 * dt * sig) / low, 2 * dt / low, da, db)
        p = self.pml
        self.debye = []
        pec = [w[:6] for w in card.get("TB", []) if w[6] == "PEC"]

        def node(box):
            return [int(v) + 1 + p for v in box]

        for a in range(3):  # the grid's outer faces
            for s in range(2):
                b = list(self.go)
                b[2 * a] = b[2 * a + 1] = self.go[2 * a + s]
                self._fill(_limits(b), -1.0, 0.0)
        for w in card.get("MB", []):
            if w[6] not in media:
                self._spheres(files, media)
                continue
            lim = _limits(node(w[:6]))
            al, be, da, db = media[w[6]]
            self._fill(lim, al, be)
            if da is not None:
                for c in range(3):
                    at = _cut(lim[c])
                    z = torch.zeros_like(self.f0(c, at))
                    self.debye.append([c, at, None, da, db, z, z.clone()])
        for b in pec:
            self._fill(_limits(node(b)), -1.0, 0.0)

    def f0(self, c, at):
        return self.alpha[c][at]

    def _fill(self, lim, al, be):
        for c in range(3):
            self.alpha[c][_cut(lim[c])] = al
            self.beta[c][_cut(lim[c])] = be

    def _spheres(self, files, media):
        """The voxel object: each cell's low x, y and z edges, and the z-face
        edges above the last cell of a run along z."""
        head = files["spheres.vox"].splitlines()
        names = [ln.split()[1] for ln in head[5:]]
        keys = np.frombuffer(files["spheres.keys"], dtype="u1" if head[1] == "1" else "<u2").reshape(self.m).astype(np.int64)
        full = np.zeros(self.shape, dtype=np.int64)
        o = 1 + self.pml
        full[tuple(slice(o, o + v) for v in self.m)] = keys
        above = np.where(full > 0, full, np.roll(full, 1, axis=2))
        table = torch.tensor([(1.0, 0.0, 0.0, 0.0)] + [media[v] for v in names], dtype=torch.float64, device=self.dev)
        for c in range(3):
            k = torch.tensor(full if c == 2 else above, device=self.dev)
            inside = k > 0
            row = table[k]
            self.alpha[c] = torch.where(inside, row[..., 0], self.alpha[c])
            self.beta[c] = torch.where(inside, row[..., 1], self.beta[c])
            at = inside.nonzero(as_tuple=True)
            z = torch.zeros(len(at[0]), dtype=torch.float64, device=self.dev)
            self.debye.append([c, at, None, row[..., 2][at], row[..., 3][at], z, z.clone()])
            del row

    def _profiles(self):
        """UPML factors per axis: a_d, b_d at the nodes, a_h, b_h between."""
        self.prof = []
        order, p = 4, self.pml
        for a in range(3):
            de, dh = self.de[a]
            sd, sh = np.zeros(len(de)), np.zeros(len(de))
            for low, up in ((1, -1), (self.gi[2 * a + 1], 1)) if p else ():
                total = de[low:low + p].sum()
                smax = 4.0 * (order + 1) / (5.0 * ETA0 * de[low])
                e, h = (total, total - 0.5 * de[low]) if up < 0 else (0.0, 0.5 * de[low])
                for i in range(low, low + p):
                    sd[i] = 0.5 * self.dt / EPS0 * smax * abs(e / total) ** order
                    sh[i] = 0.5 * self.dt / EPS0 * smax * abs(h / total) ** order
                    e, h = e + up * de[i], h + up * dh[i]
                if up > 0:
                    sd[low + p] = 0.5 * self.dt / EPS0 * smax * (e / total) ** order
            s = [1, 1, 1]
            s[a] = -1
            t = [torch.tensor(v, device=self.dev).reshape(s) for v in ((1 - sd) / (1 + sd), 1 / (1 + sd), (1 - sh) / (1 + sh), 1 / (1 + sh))]
            self.prof.append(t)

    # -- sources -----------------------------------------------------------

    def _pulse(self, t):
        size, delay, width = self.wf
        v = (t - delay) / width
        return size * (torch.exp(-0.5 * v * v) if torch.is_tensor(v) else math.exp(-0.5 * v * v))

    def _phase_velocity(self, theta, phi):
        d = self.x[0][1] - self.x[0][0]
        w = 2 * math.pi / self.dt / 23
        u = [0.5 * d * math.sin(theta) * math.cos(phi), 0.5 * d * math.sin(theta) * math.sin(phi), 0.5 * d * math.cos(theta)]
        b = math.sin(0.5 * w * self.dt) / (C0 * self.dt)
        k = w / C0
        for _ in range(10):
            k -= (sum((math.sin(v * k) / d) ** 2 for v in u) - b * b) / sum(v * math.sin(2 * v * k) / d ** 2 for v in u)
        return w / k

    def _plane_wave(self, w):
        box = [int(v) + 1 + self.pml for v in w[:6]]
        th, ph, et = (math.radians(float(v)) for v in w[8:11])
        ct, st, cp, sp, ce, se = math.cos(th), math.sin(th), math.cos(ph), math.sin(ph), math.cos(et), math.sin(et)
        inc = [ce * sp - se * ct * cp, -ce * cp - se * ct * sp, se * st,
               (se * sp + ce * ct * cp) / ETA0, (-se * cp + ce * ct * sp) / ETA0, -ce * st / ETA0]
        kin = [st * cp, st * sp, ct]
        q = int(min(float(w[9]) // 90, 3)) if float(w[9]) > 0 else 0
        q = q - 1 if float(w[9]) > 0 and float(w[9]) % 90 == 0 else q
        corner = [box[0] if q in (0, 3) else box[1], box[2] if q in (0, 1) else box[3], box[4] if float(w[8]) <= 90 else box[5]]
        pw = dict(rows=([], []))
        if self.cubic:
            d = self.x[0][1] - self.x[0][0]
            rel = self._phase_velocity(0.0, 0.0) / self._phase_velocity(th, ph)
            nx = int(16 + math.sqrt(sum((box[2 * a + 1] - box[2 * a]) ** 2 for a in range(3))))
            s = [0.5 * self.dt / EPS0 * ((np.arange(10) + h) / 10) ** 3.77 * 4 / ETA0 / d for h in (0, 0.5)]
            pw.update(nx=nx, xb=nx - 10, be=self.dt / (EPS0 * d) / rel, ga=self.dt / (MU0 * d) / rel, e=np.zeros(nx + 2), h=np.zeros(nx + 2),
                      pp=np.zeros(10), b=np.zeros(10), sd=s[0], sh=s[1])
        for face in range(6):
            a, up = face // 2, face % 2
            bb = list(box)
            bb[2 * a], bb[2 * a + 1] = (box[face], box[face] + 1) if up else (box[face] - 1, box[face])
            on = [1] * 6
            on[2 * a], on[2 * a + 1] = (1, 0) if up else (0, 1)
            lim = _limits(bb, on)
            t1, t2 = (a + 1) % 3, (a + 2) % 3
            # (corrected component, incident component, offset along the axis, sign): the four curl terms
            # that straddle the face, low faces subtracting the incident field's share and high ones adding it
            sgn = 1 if up else -1
            for e, (fc, ic, s) in ((0, (t1, 3 + t2, -sgn)), (0, (t2, 3 + t1, sgn)), (1, (3 + t1, t2, sgn)), (1, (3 + t2, t1, -sgn))):
                li = [list(v) for v in lim[fc]]
                li[a] = [li[a][up]] * 2
                off = 0 if up else (-1 if e == 0 else 1)
                at = [torch.arange(lo, hi + 1, device=self.dev) for lo, hi in li]
                pos = []
                for ax in range(3):
                    half = (ic == ax) if ic < 3 else (ic - 3 != ax)
                    i = at[ax] + (off if ax == a else 0)
                    if self.cubic:
                        r = i.double() + 0.5 * half - corner[ax]
                    else:
                        x = torch.tensor(self.x[ax], device=self.dev)
                        g = i - self.gi[2 * ax]
                        de = torch.tensor(self.de[ax][0], device=self.dev)
                        r = x[g] + 0.5 * half * de[i] - self.x[ax][corner[ax] - self.gi[2 * ax]]
                    shape = [1, 1, 1]
                    shape[ax] = -1
                    pos.append((kin[ax] * r).reshape(shape))
                dd = pos[0] + pos[1] + pos[2]
                il = (self.idh if e == 0 else self.ide)[a].flatten()[li[a][0]].item()
                row = dict(f=fc, at=_cut(li), amp=s * il * inc[ic], h=ic >= 3)
                if self.cubic:
                    z = dd + (0.5 if ic >= 3 else 0.0)
                    fl = torch.floor(z)
                    row.update(i=fl.long() + (1 if ic >= 3 else 2), w=z - fl)
                else:
                    row.update(delay=dd / C0)
                pw["rows"][e].append(row)
        return pw

    def _incident(self, pw, row, t):
        if not self.cubic:
            return self._pulse(t - row["delay"])
        g = torch.tensor(pw["h"] * ETA0 if row["h"] else pw["e"], device=self.dev)
        return (1 - row["w"]) * g[row["i"]] + row["w"] * g[row["i"] + 1]

    # -- one step ----------------------------------------------------------

    def _aux_e(self, pw, t):
        e, h, xb, nx = pw["e"], pw["h"], pw["xb"], pw["nx"]
        d = pw["be"] * (h[0:nx - 1] - h[1:nx])
        e[1:xb] += d[:xb - 1]
        e[xb:nx] = (1 - pw["sd"]) / (1 + pw["sd"]) * e[xb:nx] + d[xb - 1:] / (1 + pw["sd"])
        e[0] = self._pulse(t)

    def _aux_h(self, pw):
        e, h, xb, nx = pw["e"], pw["h"], pw["xb"], pw["nx"]
        d = pw["ga"] * (e[0:nx] - e[1:nx + 1])
        h[:xb] += d[:xb]
        b = (1 - pw["sh"]) / (1 + pw["sh"]) * pw["b"] + d[xb:] / (1 + pw["sh"])
        h[xb:nx] += b - pw["b"]
        pw["b"] = b

    def _sweep(self, e):
        outer, inner = _limits(self.go), _limits(self.gi)
        new = []
        for c in range(3):
            fc = c + 3 * e
            a1, a2 = (c + 1) % 3, (c + 2) % 3
            at, by = outer[fc], 1 if e else -1
            cut = _cut(at)
            src = [3 - 3 * e + a1, 3 - 3 * e + a2]
            il = self.ide if e else self.idh

            def slope(f, axis):
                d = self.f[f][cut] - self.f[f][_moved(at, axis, by)]
                return d * il[axis][tuple(cut[x] if x == axis else slice(None) for x in range(3))]

            # E: + dHa2/da1 - dHa1/da2 (backward differences); H: the negative curl of E (forward differences)
            curl = slope(src[1], a1) - slope(src[0], a2)
            f = self.f[fc]
            if e == 0:
                al, be = self.alpha[c][cut], self.beta[c][cut]
                val = al * f[cut] + be * curl
            else:
                al, be = 1.0, self.gamma
                val = f[cut] + be * curl
            if self.pml:
                lo = [v[0] for v in at]
                core = tuple(slice(i0 - lo[x], i1 + 1 - lo[x]) for x, (i0, i1) in enumerate(inner[fc]))
                keep = val[core].clone()

                def p(axis, q):
                    return self.prof[axis][q][tuple(cut[x] if x == axis else slice(None) for x in range(3))]

                if e == 0:
                    pp, q = self.aux[c]
                    ppn = al * pp[cut] + be * curl
                    qn = p(a1, 0) * q[cut] + p(a1, 1) * (ppn - pp[cut])
                    val = p(a2, 0) * f[cut] + p(a2, 1) / p(c, 3) * (qn - p(c, 2) * q[cut])
                    pp[cut], q[cut] = ppn, qn
                else:
                    b, = self.aux[3 + c]
                    bn = p(a1, 2) * b[cut] + be * p(a1, 3) * curl
                    val = p(a2, 2) * f[cut] + p(a2, 3) / p(c, 1) * (bn - p(c, 0) * b[cut])
                    b[cut] = bn
                val[core] = keep
            new.append((fc, cut, val))
        for fc, cut, val in new:
            self.f[fc][cut] = val

    def step(self):
        t = self.n * self.dt
        self._sweep(0)
        for d in self.debye:
            c, at, _, da, db, j, last = d
            v = self.f[c][at] - self.beta[c][at] * (1 + da) * j
            d[5] = da * j + db * (v - last)
            d[6] = v
            self.f[c][at] = v
        for pw in self.pw:
            if self.cubic:
                self._aux_e(pw, t)
        for box, wf, size in self.hard:
            b = [int(v) + 1 + self.pml for v in box]
            self.f[2][_cut(_limits(b)[2])] = size * self._pulse(t)
        for e in (0, 1):
            if e:
                self._sweep(1)
            for pw in self.pw:
                for row in pw["rows"][e]:
                    c = row["f"]
                    v = row["amp"] * self._incident(pw, row, t + 0.5 * e * self.dt)
                    old = self.f[c][row["at"]]
                    if e == 0:
                        self.f[c][row["at"]] = self.alpha[c][row["at"]] * old + self.beta[c][row["at"]] * v
                    else:
                        self.f[c][row["at"]] = old + self.gamma * v
        for pw in self.pw:
            if self.cubic:
                self._aux_h(pw)
        self.n += 1


def _reference(text, files, warm, steps):
    """[lattice samples of the last `steps`, spectra of every FDOM observer]."""
    s = _Fdtd(text, files)
    o = 1 + s.pml
    lattice, points = None, []
    for _, typ, b, st in _observers(text):
        if typ == "TDOM_BINARY":
            ax = [torch.arange(b[2 * a] + o, b[2 * a + 1] + o + 1, st[a], device=s.dev) for a in range(3)]
            # nodes run over k, then j, with i fastest
            kk, jj, ii = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
            lattice = (ii.flatten(), jj.flatten(), kk.flatten())
        elif typ == "FDOM_ASCII":
            points.append(tuple(b[2 * a] + o for a in range(3)))
    f0, f1, nf = re.search(r"^OF (\S+) (\S+) (\d+)", text, re.M).groups()
    omega = 2 * math.pi * torch.linspace(float(f0), float(f1), int(nf), dtype=torch.float64, device=s.dev)
    at = tuple(torch.tensor([p[a] for p in points], device=s.dev) for a in range(3))
    dft = torch.zeros(len(points), 2, 6, int(nf), dtype=torch.float64, device=s.dev)
    samples = []
    for n in range(warm + steps):
        if n >= warm:
            samples.append(torch.stack([f[lattice] for f in s.f], dim=-1))
        v = torch.stack([f[at] for f in s.f], dim=-1)[..., None]
        dft[:, 0] += v * torch.cos(omega * (n * s.dt))
        dft[:, 1] -= v * torch.sin(omega * (n * s.dt))
        if n + 1 < warm + steps:
            s.step()
    return [torch.stack(samples)] + list(dft)


def exact(case, seed):
    if case["kind"] in ("box", "solve"):  # conductor walls: recursive convolution; a whole call's files
        return None
    return [_reference(text, files, _warm_steps(case), case["steps"]) for text, files in _meshes(case, seed)]
