// Per-precision time-step driver.  The reference's step (simulation.c:157-222) is
//   observers -> Mur E -> E update (inner grid, UPML) -> Debye blocks -> SIBC E
//   -> sources/TF-SF E -> ghost E -> H update (inner grid, Mur normal H, UPML)
//   -> SIBC H -> sources/TF-SF H -> ghost H
// A step here is the E sweep, the E rows, the H sweep and the H rows.  Each value
// takes its operations in the reference's order: in the sweep's thread, in an
// update row beside it or in a row behind it (XArgs).  What reads and writes
// nothing of a sweep rides in blocks beside it (SideArgs): the observers' samples,
// the values of sources and analytic waves, the aux grids of the plane waves.
// Contexts with the fused sweep, of 2^31 cells and more, or with a set-up that
// the rows do not hold launch the step's parts one after another.
#pragma once
#include "vgpu_kernels.h"
#include <algorithm>
#include <map>
#include <string>
#include <vector>

namespace vgpu {

template <typename T> static T *P(void *p) { return static_cast<T *>(p); }

// Sweep arguments of a step that reads field set `in` and writes set
// c->next(in) (the other set with the fused sweep, the same set otherwise).
template <typename T> static void fill_volume_args(Ctx *c, EArgs<T> &ea, HArgs<T> &ha, int in)
{
  ea.NX = ha.NX = c->NX;
  ea.NY = ha.NY = c->NY;
  ea.NZ = ha.NZ = c->NZ;
  ea.PX = ha.PX = c->PX;
  ea.plane = ha.plane = c->plane;
  const int out = c->next(in);
  for (int d = 0; d < 3; ++d) {
    ea.E[d] = P<T>(c->fld(out, d));
    ea.Ein[d] = P<T>(c->fld(in, d));
    ea.H[d] = P<T>(c->fld(in, 3 + d));
    ha.H[d] = P<T>(c->fld(out, 3 + d));
    ha.Hin[d] = P<T>(c->fld(in, 3 + d));
    ha.E[d] = P<T>(c->fld(out, d));
    ea.alpha[d] = P<T>(c->alpha[d]);
    ea.beta[d] = P<T>(c->beta[d]);
    ha.gamma[d] = P<T>(c->gamma[d]);
    ea.idh[d] = P<T>(c->idh[d]);
    ha.ide[d] = P<T>(c->ide[d]);
    for (int f = 0; f < 6; ++f) ea.in[d][f] = c->grid.gfilim[d][f];
    // ordinary H boxes: inner grid plus the normal H of the two Mur faces on this axis
    for (int f = 0; f < 6; ++f) ha.in[d][0][f] = c->grid.gfilim[3 + d][f];
    for (int s = 0; s < 2; ++s) {
      const int face = 2 * d + s;
      if ((c->murmask >> face) & 1u)
        for (int f = 0; f < 6; ++f) ha.in[d][1 + s][f] = c->fmlim[face][3 + d][f];
      else {
        for (int f = 0; f < 6; ++f) ha.in[d][1 + s][f] = 0;
        ha.in[d][1 + s][1] = -1;
      }
    }
    const int pa = 0;
    (void)pa;
    ea.ad[d] = P<T>(c->prof[0][d]);
    ea.bd[d] = P<T>(c->prof[1][d]);
    ea.ah[d] = P<T>(c->prof[2][d]);
    ea.ibh[d] = P<T>(c->prof[5][d]);
    ha.ad[d] = P<T>(c->prof[0][d]);
    ha.ah[d] = P<T>(c->prof[2][d]);
    ha.bh[d] = P<T>(c->prof[3][d]);
    ha.ibd[d] = P<T>(c->prof[4][d]);
  }
  ea.ecls = P<uint16_t>(c->d_ecls); ea.etab = P<T>(c->d_etab);
  // (without classes the H cells' flags, when some are flagged)
  ha.hcls = P<uint16_t>(c->indexed ? c->d_hcls : c->d_xcls[1]); ha.htab = P<T>(c->d_htab);
  ea.pmlmask = ha.pmlmask = c->pmlmask;
  for (int r = 0; r < 6; ++r)
    for (int d = 0; d < 3; ++d) {
      for (int f = 0; f < 6; ++f) {
        ea.pl[r][d][f] = c->fplim[r][d][f];
        ha.pl[r][d][f] = c->fplim[r][3 + d][f];
      }
      ea.PP[r][d] = P<T>(c->aux1[r][d]);
      ea.P[r][d] = P<T>(c->aux2[r][d]);
      ha.B[r][d] = P<T>(c->auxB[r][d]);
    }
  ea.PPpool = P<T>(c->auxPool[0]);
  ea.Ppool = P<T>(c->auxPool[1]);
  ha.Bpool = P<T>(c->auxPool[2]);
}

// UPML auxiliaries of slab r, component C, carried by a shell run.
template <typename T> static void run_aux(const EArgs<T> &a, int r, int C, void *&x, void *&y)
{
  x = a.PP[r][C];
  y = a.P[r][C];
}
template <typename T> static void run_aux(const HArgs<T> &a, int r, int C, void *&x, void *&y)
{
  x = a.B[r][C];
  y = nullptr;
}

// Shell of a sweep: the cells outside its fast box, cut into pieces.  The
// cut planes on y and z are the limits of the fast box, of every component's
// ordinary-update boxes and of its UPML slabs, so over each product of a y
// and a z interval a cell's regions (classify) depend on x alone.  Such a
// product is one row segment in x (two, either side of the fast box, when
// the rows pass through it), whose regions along x form each component's
// runs; products with equal segments and runs are merged along y, then z.
// The launch blocks are then ordered so that block b runs on XCD b % 8 and
// each XCD gets one contiguous eighth of every piece's blocks.
template <int NB, typename A>
static int build_shell(const A &a, const int (*in)[NB][6], const int *fb, const int N[3], std::vector<ShellPiece> &pcs,
                       std::vector<ShellWork> &work, long long &cells, std::string &err, int lw = 0, int kcPlan = 0)
{
  const bool hasFast = fb[0] <= fb[1] && fb[2] <= fb[3] && fb[4] <= fb[5];
  std::vector<int> cut[3];
  for (int ax = 1; ax < 3; ++ax) {
    auto add = [&](int lo, int hi) {
      if (lo > hi) return;
      cut[ax].push_back(std::max(0, std::min(lo, N[ax])));
      cut[ax].push_back(std::max(0, std::min(hi + 1, N[ax])));
    };
    add(0, N[ax] - 1);
    if (hasFast) add(fb[2 * ax], fb[2 * ax + 1]);
    for (int C = 0; C < 3; ++C) {
      for (int b = 0; b < NB; ++b) add(in[C][b][2 * ax], in[C][b][2 * ax + 1]);
      for (int r = 0; r < 6; ++r)
        if ((a.pmlmask >> r) & 1u) add(a.pl[r][C][2 * ax], a.pl[r][C][2 * ax + 1]);
    }
    std::sort(cut[ax].begin(), cut[ax].end());
    cut[ax].erase(std::unique(cut[ax].begin(), cut[ax].end()), cut[ax].end());
  }
  const int ny = (int)cut[1].size() - 1, nz = (int)cut[2].size() - 1;
  std::vector<ShellPiece> raw;
  long long fastCells = 0, idle = 0;
  std::vector<int> reg[3];
  std::vector<long long> pidx[3];
  for (int tz = 0; tz < nz; ++tz)
    for (int ty = 0; ty < ny; ++ty) {
      const int y0 = cut[1][ty], y1 = cut[1][ty + 1] - 1, z0 = cut[2][tz], z1 = cut[2][tz + 1] - 1;
      const long long rows = (long long)(y1 - y0 + 1) * (z1 - z0 + 1);
      // regions along the row, checked at both corners of the product
      for (int C = 0; C < 3; ++C) {
        reg[C].assign(N[0], -1);
        pidx[C].assign(N[0], 0);
        for (int i = 0; i < N[0]; ++i) {
          long long p1 = 0;
          reg[C][i] = classify<NB>(a, in[C], C, i, y0, z0, pidx[C][i]);
          if (classify<NB>(a, in[C], C, i, y1, z1, p1) != reg[C][i]) {
            err = "shell region not constant over a y-z product";
            return -1;
          }
        }
      }
      const bool through = hasFast && y0 >= fb[2] && y1 <= fb[3] && z0 >= fb[4] && z1 <= fb[5];
      int seg[2][2] = {{0, N[0] - 1}, {1, 0}};
      int nseg = 1;
      if (through) {
        seg[0][1] = fb[0] - 1;
        seg[1][0] = fb[1] + 1;
        seg[1][1] = N[0] - 1;
        nseg = 2;
        fastCells += (long long)(fb[1] - fb[0] + 1) * rows;
      }
      for (int sg = 0; sg < nseg; ++sg) {
        int x0 = seg[sg][0], x1 = seg[sg][1];
        if (x0 > x1) continue;
        const long long segCells = (long long)(x1 - x0 + 1) * rows;
        // trim cells with no component updated from both ends
        auto idleAt = [&](int i) { return reg[0][i] < 0 && reg[1][i] < 0 && reg[2][i] < 0; };
        while (x0 <= x1 && idleAt(x0)) ++x0;
        while (x1 >= x0 && idleAt(x1)) --x1;
        long long used = 0;
        // pieces of at most SHELL_RUNS runs per component
        int xs = x0;
        while (xs <= x1) {
          ShellPiece pc{};
          int xe = xs;
          for (; xe <= x1; ++xe) {
            bool fits = true;
            for (int C = 0; C < 3 && fits; ++C) {
              const bool opens = reg[C][xe] >= 0 && (xe == xs || reg[C][xe] != reg[C][xe - 1]);
              if (opens && pc.nrun[C] == SHELL_RUNS) fits = false;
            }
            if (!fits) break;
            for (int C = 0; C < 3; ++C) {
              const int rg = reg[C][xe];
              if (rg < 0) continue;
              if (xe > xs && rg == reg[C][xe - 1]) {
                pc.run[C][pc.nrun[C] - 1].xb = xe;
                continue;
              }
              ShellRun &rn = pc.run[C][pc.nrun[C]++];
              rn.xa = rn.xb = xe;
              rn.reg = rg;
              if (rg < 6) {
                const int *sl = a.pl[rg][C];
                rn.p0 = pidx[C][xe];
                rn.psy = sl[1] - sl[0] + 1;
                rn.psz = rn.psy * (sl[3] - sl[2] + 1);
                run_aux(a, rg, C, rn.a, rn.b);
              }
            }
          }
          pc.box[0] = xs; pc.box[1] = xe - 1;
          pc.box[2] = y0; pc.box[3] = y1;
          pc.box[4] = z0; pc.box[5] = z1;
          raw.push_back(pc);
          used += (long long)(xe - xs) * rows;
          xs = xe;
        }
        idle += segCells - used;
      }
    }
  // merge along y, then z: a piece extends the last one with the same x
  // range and runs and the same extent on the third axis when adjacent
  auto key_of = [](const ShellPiece &pc, int ax) {
    std::vector<long long> key = {pc.box[0], pc.box[1]};
    const int q = ax == 1 ? 2 : 1;
    key.push_back(pc.box[2 * q]);
    key.push_back(pc.box[2 * q + 1]);
    for (int C = 0; C < 3; ++C) {
      key.push_back(pc.nrun[C]);
      for (int r = 0; r < pc.nrun[C]; ++r) {
        key.push_back(pc.run[C][r].xa);
        key.push_back(pc.run[C][r].xb);
        key.push_back(pc.run[C][r].reg);
      }
    }
    return key;
  };
  auto merge = [&](std::vector<ShellPiece> &v, int ax) {
    std::vector<ShellPiece> out;
    std::map<std::vector<long long>, size_t> last;
    for (const ShellPiece &pc : v) {
      const std::vector<long long> key = key_of(pc, ax);
      auto it = last.find(key);
      if (it != last.end() && out[it->second].box[2 * ax + 1] + 1 == pc.box[2 * ax]) {
        out[it->second].box[2 * ax + 1] = pc.box[2 * ax + 1];
      } else {
        last[key] = out.size();
        out.push_back(pc);
      }
    }
    v.swap(out);
  };
  merge(raw, 1);
  merge(raw, 2);
  // planes per block: up to SHELL_KC, fewer when the shell is too small to
  // give about 512 blocks (two per CU) that way.  A thread re-reads H of the
  // plane below its first plane and redoes its region lookup, so one plane
  // per thread costs more than the occupancy it buys: on 1-2 M-cell grids
  // with an 8-cell UPML, two to four planes ran the step 10-14 % faster
  // than the one a 2048-block target gave them
  long long rawCells = 0;
  for (const ShellPiece &pc : raw)
    rawCells += (long long)(pc.box[1] - pc.box[0] + 1) * (pc.box[3] - pc.box[2] + 1) * (pc.box[5] - pc.box[4] + 1);
  int kcmax = (int)std::max(1LL, std::min((long long)SHELL_KC, rawCells / (256LL * 512)));
  if (const char *ev = getenv("VGPU_SHELL_KC")) kcmax = std::max(1, std::min(atoi(ev), 64));  // tuning override
  if (kcPlan > 0) kcmax = kcPlan;  // a plan for launches shared with other grids (group runs)
  cells = 0;
  pcs.clear();
  for (ShellPiece pc : raw) {
    pc.ni = pc.box[1] - pc.box[0] + 1;
    pc.nj = pc.box[3] - pc.box[2] + 1;
    pc.nk = pc.box[5] - pc.box[4] + 1;
    const long long n = (long long)pc.ni * pc.nj * pc.nk;
    if (n > (1LL << 30)) {
      err = "shell piece too large";
      return -1;
    }
    pc.cells = (int)n;
    // With lw, rows shorter than half a line are padded to whole lines of lw
    // elements, each starting on a line, so a wavefront's loads touch one
    // line per row.  Off by default: since the pieces are read in one batch of
    // scalar loads, the idle lanes' wavefronts cost more (53x41x62 request
    // 40.4 us a step padded, 36.0 packed; 256x256x160 box 342 and 335).
    const bool pad = lw > 0 && 2 * pc.ni < lw;
    pc.xo = pad ? pc.box[0] % lw : 0;
    pc.nip = pad ? (pc.xo + pc.ni + lw - 1) / lw * lw : pc.ni;
    if ((long long)pc.nip * pc.nj > (1LL << 30)) {
      err = "shell piece too large";
      return -1;
    }
    pc.nxy = pc.nip * pc.nj;
    pc.nxyb = (pc.nxy + 255) / 256;
    pc.kc = std::min(pc.nk, kcmax);
    pc.nblk = pc.nxyb * ((pc.nk + pc.kc - 1) / pc.kc);
    cells += n;
    pcs.push_back(pc);
  }
  if (fastCells + idle + cells != (long long)N[0] * N[1] * N[2]) {
    err = "fast box and shell do not tile the grid";
    return -1;
  }
  // launch order: XCD x runs blocks 8*slot + x, slot over its eighths
  std::vector<ShellWork> per[8];
  for (int q = 0; q < (int)pcs.size(); ++q) {
    const int nb = pcs[q].nblk;
    for (int x = 0; x < 8; ++x)
      for (int b = (int)((long long)nb * x / 8); b < (int)((long long)nb * (x + 1) / 8); ++b) per[x].push_back({q, b});
  }
  size_t len = 0;
  for (int x = 0; x < 8; ++x) len = std::max(len, per[x].size());
  work.assign(8 * len, ShellWork{-1, 0});
  for (int x = 0; x < 8; ++x)
    for (size_t t = 0; t < per[x].size(); ++t) work[8 * t + x] = per[x][t];
  return 0;
}

// Pieces as the kernels read them; pool: the pool holding their auxiliaries.
template <typename T> static std::vector<ShellDev> shell_dev(const std::vector<ShellPiece> &pcs, const T *pool)
{
  std::vector<ShellDev> out;
  for (const ShellPiece &p : pcs) {
    ShellDev d{};
    d.x0 = p.box[0]; d.y0 = p.box[2]; d.z0 = p.box[4];
    d.ni = p.ni; d.nip = p.nip; d.xo = p.xo; d.nxy = p.nxy; d.nxyb = p.nxyb; d.kc = p.kc; d.nk = p.nk;
    for (int C = 0; C < 3; ++C)
      for (int r = 0; r < SHELL_RUNS; ++r) {
        ShellDevRun &o = d.run[C][r];
        o.xa = 1;
        if (r >= p.nrun[C]) continue;
        const ShellRun &n = p.run[C][r];
        o.xa = n.xa; o.xb = n.xb; o.reg = n.reg;
        if (n.reg < 6) {
          // the pools hold at most 2^31 elements (vgpu_set_pml)
          o.q0 = (int)(static_cast<const T *>(n.a) - pool + n.p0 - n.xa);
          o.psy = (int)n.psy;
          o.psz = (int)n.psz;
        }
      }
    out.push_back(d);
  }
  return out;
}

// The E and H shells of a context (build_shell); kcPlan > 0 fixes the planes
// per block.
template <typename T>
static int plan_shells(Ctx *c, int kcPlan, std::vector<ShellDev> &ep, std::vector<ShellWork> &ew,
                       std::vector<ShellDev> &hp, std::vector<ShellWork> &hw, long long cells[2], std::string &err)
{
  std::vector<ShellPiece> pe, ph;
  EArgs<T> ea{};
  HArgs<T> ha{};
  fill_volume_args<T>(c, ea, ha, 0);
  const int N[3] = {c->NX, c->NY, c->NZ};
  int ein[3][1][6];
  for (int C = 0; C < 3; ++C)
    for (int q = 0; q < 6; ++q) ein[C][0][q] = ea.in[C][q];
  // VGPU_SHELL_ROWS=1 pads rows shorter than half a line to whole lines
  const int lw = getenv("VGPU_SHELL_ROWS") && getenv("VGPU_SHELL_ROWS")[0] == '1' ? (int)(128 / sizeof(T)) : 0;
  if (build_shell<1>(ea, ein, c->fastE, N, pe, ew, cells[0], err, lw, kcPlan) ||
      build_shell<3>(ha, ha.in, c->fastH, N, ph, hw, cells[1], err, lw, kcPlan))
    return -1;
  ep = shell_dev<T>(pe, ea.PPpool);
  hp = shell_dev<T>(ph, ha.Bpool);
  return 0;
}

// Argument block of the corrections of half-step e.
template <typename T> static void fill_correction_args(Ctx *c, XArgs<T> &x, int e)
{
  x.cls = P<uint16_t>(c->indexed ? (e == 0 ? c->d_ecls : c->d_hcls) : c->d_xcls[e]);
  x.PX = c->PX; x.plane = c->plane;
  x.nupd = c->nXupd[e]; x.nrow = c->nXrow[e]; x.ngroup = c->nXgroup[e];
  x.nsite = e == 0 ? c->nXsite : 0; x.site = P<XSiteDev>(e == 0 ? c->d_xsite : nullptr);
  x.gstart = P<int>(c->d_xgstart[e]); x.row = P<XRow>(c->d_xrow[e]); x.op = P<XOp<T>>(c->d_xop[e]);
  for (int d = 0; d < 3; ++d) {
    x.F[d] = P<T>(c->fld(0, 3 * e + d));
    x.G[d] = P<T>(c->fld(0, 3 - 3 * e + d));
    x.il[d] = P<T>(e == 0 ? c->idh[d] : c->ide[d]);
    x.ca[d] = P<T>(e == 0 ? c->alpha[d] : nullptr);
    x.cb[d] = P<T>(e == 0 ? c->beta[d] : c->gamma[d]);
  }
  x.tab = P<T>(e == 0 ? c->d_etab : c->d_htab);
  x.val = P<T>(c->d_xvals[e]);
  x.aux = P<T>(c->d_aux); x.auxmax = c->auxmax; x.pw = P<PwDev>(c->d_pw); x.eta0 = T(c->grid.eta0);
  x.Etan = P<T>(c->d_setan);
  x.flag0 = ~0u;
  if (e) return;
  x.flag0 = c->xflag0;
  if (c->d_xJ) {
    x.jrow = c->jn[0]; x.jplane = c->jn[0] * c->jn[1];
    x.jfirst = c->jlo[2] * x.jplane + c->jlo[1] * x.jrow + c->jlo[0];
    x.jlast = x.jfirst + c->jn[2] * x.jplane - 1;
    x.J = P<T>(c->d_xJ) - 3ll * x.jfirst;
  }
  x.dtab = P<T>(c->d_xdtab);
  for (int f = 0; f < 6; ++f) x.mzeta[f] = T(c->zeta[f]);
  x.dlast = P<T>(c->d_dlast); x.dJ = P<T>(c->d_dJ); x.dstride = c->debyeSites;
  x.dalpha = P<double>(c->d_dalpha); x.dbeta = P<double>(c->d_dbeta); x.dnp = P<int>(c->d_dnp);
  x.dmaxP = c->debyeMaxPoles; x.dcplx = c->debyeCplx;
}

// Once per context (at finalize): the sweeps' argument blocks go to device
// memory, where the shell kernels and the corrections read them.
template <typename T> int prepare_sweeps(Ctx *c)
{
  for (int e = 0; e < 2; ++e) {
    const int *fb = e == 0 ? c->fastE : c->fastH;
    if (fb[0] <= fb[1] && fb[2] <= fb[3] && fb[4] <= fb[5] &&
        (fb[0] < 1 || fb[2] < 1 || fb[4] < 1 || fb[1] > c->NX - 2 || fb[3] > c->NY - 2 || fb[5] > c->NZ - 2))
      return set_error(c, VGPU_EINVAL, "fast box not inside the grid");
  }
  EArgs<T> ea{}, ea1{};
  HArgs<T> ha{}, ha1{};
  fill_volume_args<T>(c, ea, ha, 0);
  fill_volume_args<T>(c, ea1, ha1, 1);
  std::vector<ShellDev> ep, hp;
  std::vector<ShellWork> ew, hw;
  std::string err;
  if (plan_shells<T>(c, 0, ep, ew, hp, hw, c->shellCells, err)) return set_error(c, VGPU_EINVAL, "%s", err.c_str());
  c->nEpcs = (int)ep.size(); c->nHpcs = (int)hp.size();
  c->nEwork = (int)ew.size(); c->nHwork = (int)hw.size();
  for (int q = 0; q < 2; ++q) {
    c->d_eargs[q] = dev_alloc(c, sizeof(ea));
    c->d_hargs[q] = dev_alloc(c, sizeof(ha));
  }
  c->d_epcs = dev_alloc(c, ep.size() * sizeof(ShellDev));
  c->d_hpcs = dev_alloc(c, hp.size() * sizeof(ShellDev));
  c->d_ework = dev_alloc(c, ew.size() * sizeof(ShellWork));
  c->d_hwork = dev_alloc(c, hw.size() * sizeof(ShellWork));
  if (!c->d_eargs[0] || !c->d_hargs[0] || !c->d_eargs[1] || !c->d_hargs[1] || !c->d_epcs || !c->d_hpcs ||
      !c->d_ework || !c->d_hwork)
    return set_error(c, VGPU_ENOMEM, "sweep arguments");
  auto up = [](void *d, const void *h, size_t n) { return n == 0 || hipMemcpy(d, h, n, hipMemcpyHostToDevice) == hipSuccess; };
  if (!up(c->d_eargs[0], &ea, sizeof(ea)) || !up(c->d_hargs[0], &ha, sizeof(ha)) ||
      !up(c->d_eargs[1], &ea1, sizeof(ea1)) || !up(c->d_hargs[1], &ha1, sizeof(ha1)) ||
      !up(c->d_epcs, ep.data(), ep.size() * sizeof(ShellDev)) ||
      !up(c->d_hpcs, hp.data(), hp.size() * sizeof(ShellDev)) ||
      !up(c->d_ework, ew.data(), ew.size() * sizeof(ShellWork)) ||
      !up(c->d_hwork, hw.data(), hw.size() * sizeof(ShellWork)))
    return set_error(c, VGPU_EDEVICE, "sweep arguments upload");
  if (c->inl) {
    for (int e = 0; e < 2; ++e) {
      XArgs<T> x{};
      fill_correction_args<T>(c, x, e);
      c->d_xargs[e] = dev_alloc(c, sizeof(x));
      if (!c->d_xargs[e]) return set_error(c, VGPU_ENOMEM, "corrections");
      if (!up(c->d_xargs[e], &x, sizeof(x))) return set_error(c, VGPU_EDEVICE, "corrections upload");
    }
    return VGPU_OK;
  }
  // Debye sites, correction rows and SIBC H rows: each one's coefficients, gathered once
  if (c->debyeSites) {
    const T *b[3] = {P<T>(c->beta[0]), P<T>(c->beta[1]), P<T>(c->beta[2])};
    void *db = dev_alloc(c, sizeof(b));
    if (!db) return set_error(c, VGPU_ENOMEM, "Debye coefficients");
    if (!up(db, b, sizeof(b))) return set_error(c, VGPU_EDEVICE, "Debye coefficients upload");
    const long long n = c->debyeSites;
    hipLaunchKernelGGL((k_debye_gather<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, n,
                       P<long long>(c->d_dkey), P<const T *const>(db), c->indexed ? P<uint16_t>(c->d_ecls) : nullptr,
                       c->indexed ? P<T>(c->d_etab) : nullptr, P<T>(c->d_dsbeta));
    if (hipStreamSynchronize(c->stream) != hipSuccess)
      return set_error(c, VGPU_EDEVICE, "Debye coefficients: %s", hipGetErrorString(hipGetLastError()));
  }
  if (c->sibcHRows) {
    const T *g[3] = {P<T>(c->gamma[0]), P<T>(c->gamma[1]), P<T>(c->gamma[2])};
    void *dg = dev_alloc(c, sizeof(g));
    if (!dg) return set_error(c, VGPU_ENOMEM, "SIBC coefficients");
    if (!up(dg, g, sizeof(g))) return set_error(c, VGPU_EDEVICE, "SIBC coefficients upload");
    const long long n = c->sibcHRows;
    hipLaunchKernelGGL((k_corr_gather<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, n,
                       P<long long>(c->d_shkey), 3, P<const T *const>(dg), nullptr, P<T>(c->d_shg), nullptr);
    if (hipStreamSynchronize(c->stream) != hipSuccess)
      return set_error(c, VGPU_EDEVICE, "SIBC coefficients: %s", hipGetErrorString(hipGetLastError()));
  }
  for (int e = 0; e < 2; ++e) {
    if (!c->corrRows[e]) continue;
    const T *coef[3], *alpha[3];
    for (int d = 0; d < 3; ++d) {
      coef[d] = P<T>(e == 0 ? c->beta[d] : c->gamma[d]);
      alpha[d] = P<T>(c->alpha[d]);
    }
    void *dc = dev_alloc(c, sizeof(coef)), *da = dev_alloc(c, sizeof(alpha));
    if (!dc || !da) return set_error(c, VGPU_ENOMEM, "correction coefficients");
    if (!up(dc, coef, sizeof(coef)) || !up(da, alpha, sizeof(alpha)))
      return set_error(c, VGPU_EDEVICE, "correction coefficients upload");
    const long long n = c->corrRows[e];
    hipLaunchKernelGGL((k_corr_gather<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, n,
                       P<long long>(c->d_ckey[e]), 2, P<const T *const>(dc), e == 0 ? P<const T *const>(da) : nullptr,
                       P<T>(c->d_ccoef[e]), P<T>(c->d_calpha[e]));
    if (hipStreamSynchronize(c->stream) != hipSuccess)
      return set_error(c, VGPU_EDEVICE, "correction coefficients: %s", hipGetErrorString(hipGetLastError()));
  }
  return VGPU_OK;
}

// Argument blocks of one solve's step launches, for both field sets (index:
// the set a step reads), built on the host before a run.
template <typename T> struct StepArgs {
  EArgs<T> ea[2];
  HArgs<T> ha[2];
  dim3 vblk, egrid, hgrid, eg1, hg1;   // fast kernels: block, tile grid, padded 1-D launch
  FastE<T> fe[2];
  FastH<T> fh[2];
  const EArgs<T> *eap[2];              // argument blocks in device memory (shells)
  const HArgs<T> *hap[2];
  const ShellDev *epc, *hpc;
  const ShellWork *ewk, *hwk;
  LeapArgs<T> la[2];
  FixArgs<T> fx[2];
  dim3 lgrid, lblk;
  MurArgs<T> ma[2];
  dim3 murGrid;
  DebyeArgs<T> da[2];
  SibcEArgs<T> se[2];
  SibcHArgs<T> sh[2];
  CorrArgs<T> ce[2][2];                // [set][E, H]
  AuxArgs<T> xa;
  bool anyAux;
  ObsArgs<T> oa[2];
  int maxnf;
  SideArgs<T> side[2];                 // what rides with the E and H sweeps
  unsigned nside[2];                   // their blocks
  VolObsArgs<T> va[2];
  unsigned long long *stepp;           // device step counter
};

// Whether a context's fast tiles have launches of their own.  In one launch
// the tiles share the shell's register count (FP32 with Debye sites E 96 and H
// 62 VGPRs against 49 and 53 alone, five and eight wavefronts a SIMD against
// eight), but its blocks fill the device together with
// theirs and one launch fewer is on the step's critical path: 48.6 -> 39.8 us
// a step on a 53x41x62 request, 82 -> 71 on 101x115x108, 298 -> 283 on the
// FP64 200x160x120 enclosure, 377 -> 368 on the 256x256x160 box.  Where the
// fields are past the 256 MB last-level cache the tiles' own occupancy counts
// for more: 537 against 529 us at 272^3 in FP32 (85 MB a field).
static bool sweeps_apart(const Ctx *c) { return c->ncell * c->esz > ((size_t)64 << 20); }

template <typename T> void fill_step_args(Ctx *c, StepArgs<T> &A, const VisitRun *chk, bool packed = false)
{
  const double dt = c->grid.dt;
  // argument sets by the field set a step reads (index 0/1)
  auto &ea = A.ea;
  auto &ha = A.ha;
  for (int q = 0; q < 2; ++q) fill_volume_args<T>(c, ea[q], ha[q], q);
  // Fast kernels: 64x4 tiles (64 x ty) over the fast boxes, marching z in
  // chunks of 4 planes, or 2 where they have launches of their own (272^3 FP32:
  // 505 us a step with 4, 501 with 2, 514 with 8; merged grids within 1 %).
  // Where chunks of 4 make fewer than seven blocks a CU there is little else to
  // run under a block's chain of planes, and one plane a block is faster: a
  // step of the 53x41x62 request 24.8 us against 27.5, 101x115x108 67.6 and
  // 70.9, the FP64 96x81x64 box 49.9 and 52.6; with more blocks the planes' shared loads count (FP64 128^3
  // Debye volume 162 and 167).  Packed launches have their members' blocks
  // together and keep 4 (364 and 383 for 16 requests).
  // Rows per block: four, a wavefront each, in the 256 threads of a launch that
  // the tiles share with the shell and the side blocks.  Launches of their own
  // take another number (tuning override VGPU_FAST_TY: 1..8).
  int ty = 4;
  if (!c->inl || (sweeps_apart(c) && !packed))
    if (const char *ev = getenv("VGPU_FAST_TY")) ty = std::max(1, std::min(atoi(ev), 8));
  A.vblk = dim3(64 * ty);
  auto fast_grid = [&](const int *fb, int &kchunk) {
    if (fb[0] > fb[1] || fb[2] > fb[3] || fb[4] > fb[5]) return dim3(0, 0, 0);
    const int gx = (fb[1] - fb[0] + 64) / 64, gy = (fb[3] - fb[2] + ty) / ty, nz = fb[5] - fb[4] + 1;
    kchunk = std::min(sweeps_apart(c) ? 2 : !packed && gx * gy * ((nz + 3) / 4) < 1792 ? 1 : 4, nz);
    if (const char *ev = getenv("VGPU_FAST_KCHUNK"))  // tuning override: planes per block
      kchunk = std::max(1, std::min(atoi(ev), nz));
    return dim3(gx, gy, (nz + kchunk - 1) / kchunk);
  };
  auto &fe = A.fe;
  auto &fh = A.fh;
  int ekc = 1, hkc = 1;
  const dim3 egrid = A.egrid = fast_grid(c->fastE, ekc), hgrid = A.hgrid = fast_grid(c->fastH, hkc);
  // 1-D launches: an eighth of each z chunk's tiles per XCD (fast_block)
  auto pad8 = [](unsigned long long n) { return dim3((unsigned)((n + 7) / 8 * 8)); };
  const int eper = (int)(egrid.x * egrid.y + 7) / 8, hper = (int)(hgrid.x * hgrid.y + 7) / 8;
  A.eg1 = dim3(8u * eper * egrid.z);
  A.hg1 = dim3(8u * hper * hgrid.z);
  for (int q = 0; q < 2; ++q) {
    FastE<T> &e = fe[q];
    FastH<T> &h = fh[q];
    e.NX = h.NX = c->NX; e.NY = h.NY = c->NY; e.NZ = h.NZ = c->NZ; e.PX = h.PX = c->PX;
    e.plane = h.plane = c->plane;
    e.kchunk = ekc; h.kchunk = hkc; e.per = eper; h.per = hper;
    for (int f = 0; f < 6; ++f) { e.box[f] = c->fastE[f]; h.box[f] = c->fastH[f]; }
    e.nchx = egrid.x; h.nchx = hgrid.x;
    e.gy = egrid.y; e.gz = egrid.z; h.gy = hgrid.y; h.gz = hgrid.z;
    for (int d = 0; d < 3; ++d) {
      e.E[d] = ea[q].E[d]; e.Ein[d] = ea[q].Ein[d]; e.H[d] = ea[q].H[d]; e.idh[d] = ea[q].idh[d];
      e.alpha[d] = ea[q].alpha[d]; e.beta[d] = ea[q].beta[d];
      h.H[d] = ha[q].H[d]; h.Hin[d] = ha[q].Hin[d]; h.E[d] = ha[q].E[d]; h.ide[d] = ha[q].ide[d];
      h.gamma[d] = ha[q].gamma[d];
    }
    e.ecls = ea[q].ecls; e.etab = ea[q].etab;
    h.hcls = ha[q].hcls; h.htab = ha[q].htab;
    if (chk)
      for (int d = 0; d < 3; ++d) { e.vis[d] = chk->vis[d]; h.vis[d] = chk->vis[3 + d]; }
  }
  auto &eap = A.eap;
  auto &hap = A.hap;
  for (int q = 0; q < 2; ++q) {
    eap[q] = P<EArgs<T>>(chk ? chk->eargs : c->d_eargs[q]);
    hap[q] = P<HArgs<T>>(chk ? chk->hargs : c->d_hargs[q]);
  }
  A.epc = P<ShellDev>(c->d_epcs);
  A.hpc = P<ShellDev>(c->d_hpcs);
  A.ewk = P<ShellWork>(c->d_ework);
  A.hwk = P<ShellWork>(c->d_hwork);
  // fused leapfrog sweep: 4 waves of R rows per block, 63-cell x tiles, kz-plane z chunks
  auto &la = A.la;
  auto &fx = A.fx;
  dim3 &lgrid = A.lgrid;
  lgrid = dim3(0);
  A.lblk = dim3(64, 4, 1);
  if (c->leap) {
    const int *fb = c->fastE;
    if (fb[0] <= fb[1] && fb[2] <= fb[3] && fb[4] <= fb[5]) {
      const int R = c->leapR, kz = std::min(c->leapKZ, fb[5] - fb[4] + 1);
      const int ntx = (fb[1] - fb[0] + 63) / 63, ngy = (fb[3] - fb[2] + 4 * R) / (4 * R), ntz = (fb[5] - fb[4] + kz) / kz;
      lgrid = pad8((unsigned long long)ntx * ngy * ntz);
      for (int q = 0; q < 2; ++q) {
        LeapArgs<T> &l = la[q];
        l.NX = c->NX; l.NY = c->NY; l.NZ = c->NZ; l.PX = c->PX; l.plane = c->plane;
        for (int f = 0; f < 6; ++f) l.box[f] = fb[f];
        l.ntx = ntx; l.ngy = ngy; l.ntz = ntz; l.kz = kz;
        for (int d = 0; d < 3; ++d) {
          l.E[d] = ea[q].E[d]; l.Ein[d] = ea[q].Ein[d]; l.H[d] = ha[q].H[d]; l.Hin[d] = ha[q].Hin[d];
          l.idh[d] = ea[q].idh[d]; l.ide[d] = ha[q].ide[d];
          l.alpha[d] = ea[q].alpha[d]; l.beta[d] = ea[q].beta[d]; l.gamma[d] = ha[q].gamma[d];
        }
        l.ecls = ea[q].ecls; l.etab = ea[q].etab; l.hcls = ha[q].hcls; l.htab = ha[q].htab;
        l.discard = (int)c->ncell;
        if (chk)
          for (int d = 0; d < 6; ++d) l.vis[d] = chk->vis[d];
        FixArgs<T> &x = fx[q];
        x.n = c->nFix; x.ent = P<FixEnt>(c->d_fix);
        x.NY = c->NY; x.PX = c->PX; x.plane = c->plane;
        for (int d = 0; d < 3; ++d) {
          x.H[d] = ha[q].H[d]; x.Hin[d] = ha[q].Hin[d]; x.E[d] = ha[q].E[d]; x.ide[d] = ha[q].ide[d];
          x.gamma[d] = ha[q].gamma[d];
        }
        x.hcls = ha[q].hcls; x.htab = ha[q].htab;
      }
    }
  }
  auto &ma = A.ma;
  int murmax1 = 1, murmax2 = 1;
  if (c->murmask) {
    for (int q = 0; q < 2; ++q) {
      MurArgs<T> &m = ma[q];
      m.NX = c->NX; m.NY = c->NY; m.PX = c->PX; m.plane = c->plane;
      for (int d = 0; d < 3; ++d) {
        m.E[d] = ea[q].E[d]; m.Ein[d] = ea[q].Ein[d]; m.H[d] = ea[q].H[d];
        m.alpha[d] = P<T>(c->alpha[d]); m.beta[d] = P<T>(c->beta[d]); m.idh[d] = P<T>(c->idh[d]);
      }
      if (c->indexed) { m.ecls = ea[q].ecls; m.etab = ea[q].etab; }
      if (chk)
        for (int d = 0; d < 3; ++d) m.vis[d] = chk->vis[d];
    }
    static const int order[6][2] = {{1, 2}, {1, 2}, {0, 2}, {0, 2}, {1, 0}, {1, 0}};
    for (int f = 0; f < 6; ++f) {
      for (int q = 0; q < 2; ++q) ma[q].zeta[f] = T(c->zeta[f]);
      for (int u = 0; u < 2; ++u) {
        const int slot = 2 * f + u;
        if ((c->murmask >> f) & 1u) {
          const int comp = order[f][u];
          for (int q = 0; q < 2; ++q) {
            ma[q].comp[slot] = comp;
            for (int e = 0; e < 6; ++e) ma[q].box[slot][e] = c->fmlim[f][comp][e];
          }
          const int ax = f >> 1, a1 = ax == 0 ? 1 : 0, a2 = ax == 2 ? 1 : 2;
          const int *b = ma[0].box[slot];
          murmax1 = std::max(murmax1, b[2 * a1 + 1] - b[2 * a1] + 1);
          murmax2 = std::max(murmax2, b[2 * a2 + 1] - b[2 * a2] + 1);
        } else {
          for (int q = 0; q < 2; ++q) ma[q].comp[slot] = -1;
        }
      }
    }
  }
  A.murGrid = dim3((murmax1 + 15) / 16, (murmax2 + 15) / 16, 12);

  auto &da = A.da;
  if (c->debyeSites) {
    for (int q = 0; q < 2; ++q) {
      DebyeArgs<T> &a = da[q];
      a.key = P<long long>(c->d_dkey); a.sbeta = P<T>(c->d_dsbeta);
      for (int d = 0; d < 3; ++d) a.E[d] = ea[q].E[d];
      a.lastE = P<T>(c->d_dlast); a.J = P<T>(c->d_dJ); a.stride = c->debyeSites;
      a.dalpha = P<double>(c->d_dalpha); a.dbeta = P<double>(c->d_dbeta); a.npoles = P<int>(c->d_dnp);
      a.maxPoles = c->debyeMaxPoles; a.cplx = c->debyeCplx;
    }
  }

  auto &se = A.se;
  auto &sh = A.sh;
  if (c->sibcFaces) {
    for (int q = 0; q < 2; ++q) {
      SibcEArgs<T> &e = se[q];
      SibcHArgs<T> &h = sh[q];
      e.nfaces = c->sibcFaces; e.ijk = P<int>(c->d_sijk); e.surf = P<int>(c->d_ssurf);
      e.blocks = P<SibcBlock>(c->d_sblocks);
      e.adjA = P<unsigned char>(c->d_sadjA); e.adjB = P<unsigned char>(c->d_sadjB);
      e.normal = P<int>(c->d_snormal); e.A = P<double>(c->d_sA); e.B = P<double>(c->d_sB);
      e.filtset = P<int>(c->d_sset); e.npoles = P<int>(c->d_snp); e.asymp = P<double>(c->d_sasymp);
      e.q = P<double>(c->d_sq); e.maxPoles = c->sibcMaxPoles; e.zeta = P<double>(c->d_szeta);
      e.real = c->sibcReal ? 1 : 0;
      e.factored = c->sibcFactored ? 1 : 0;
      e.fbase = P<int>(c->d_sfbase); e.fratio = P<double>(c->d_sfratio);
      e.old = P<double>(c->d_sold); e.Etan = P<T>(c->d_setan);
      // SIBC E runs after the E sweep: it zeroes the new tangential E and
      // reads the old H (sibc.c:444-586)
      for (int d = 0; d < 3; ++d) { e.E[d] = ea[q].E[d]; e.H[d] = ea[q].H[d]; }
      e.NY = c->NY; e.PX = c->PX; e.plane = c->plane;
      h.nrows = c->sibcHRows; h.rowkey = P<long long>(c->d_shkey);
      h.rowstart = P<int>(c->d_shstart); h.rowg = P<T>(c->d_shg);
      h.ent = P<SibcHEnt>(c->d_shent); h.Etan = P<T>(c->d_setan);
      for (int d = 0; d < 3; ++d) { h.H[d] = ha[q].H[d]; h.ide[d] = P<T>(c->ide[d]); }
    }
  }

  auto &ce = A.ce;
  for (int q = 0; q < 2; ++q)
    for (int e = 0; e < 2; ++e) {
      CorrArgs<T> &a = ce[q][e];
      a = CorrArgs<T>{};
      a.nrows = c->corrRows[e];
      a.rowkey = P<long long>(c->d_ckey[e]);
      a.rowstart = P<int>(c->d_cstart[e]); a.ent = P<CorrEnt>(c->d_cent[e]);
      a.rowcoef = P<T>(c->d_ccoef[e]); a.rowalpha = P<T>(c->d_calpha[e]);
      a.electric = e == 0;
      a.wf = P<WaveformDev>(c->d_wf); a.src = P<SourceDev>(c->d_src); a.pw = P<PwDev>(c->d_pw);
      a.aux = P<T>(c->d_aux); a.auxmax = c->auxmax; a.eta0 = c->grid.eta0;
      // the E list corrects the new E, the H list the new H
      for (int d = 0; d < 3; ++d) a.F[d] = e == 0 ? ea[q].E[d] : ha[q].H[d];
    }

  auto &xa = A.xa;
  bool &anyAux = A.anyAux;
  anyAux = false;
  for (auto &p : c->pw) anyAux |= p.d.use_aux != 0;
  if (anyAux) {
    xa.npw = (int)c->pw.size(); xa.pw = P<PwDev>(c->d_pw); xa.aux = P<T>(c->d_aux);
    xa.pml = P<T>(c->d_auxpml); xa.prof = P<T>(c->d_auxprof); xa.auxmax = c->auxmax;
    xa.wf = P<WaveformDev>(c->d_wf);
  }

  // observers sample the fields a step starts from: the set it reads
  auto &oa = A.oa;
  int &maxnf = A.maxnf;
  maxnf = 1;
  if (!c->pobs.empty()) {
    for (int q = 0; q < 2; ++q) {
      ObsArgs<T> &o = oa[q];
      o.nobs = (int)c->pobs.size(); o.cell = P<long long>(c->d_ocell);
      o.first = P<unsigned long long>(c->d_ofirst); o.last = P<unsigned long long>(c->d_olast);
      o.nfreq = P<int>(c->d_onf); o.dftoff = P<long long>(c->d_ooff); o.omega = P<double>(c->d_oomega);
      o.td = P<double>(c->d_otd); o.tdsteps = c->totalSteps; o.dre = P<double>(c->d_odre);
      o.dim = P<double>(c->d_odim);
      for (int d = 0; d < 6; ++d) o.F[d] = P<T>(c->fld(q, d));
    }
    for (auto &o : c->pobs) maxnf = std::max(maxnf, (int)o.omega.size());
  }
  auto &va = A.va;
  if (c->vnodes) {
    for (int q = 0; q < 2; ++q) {
      VolObsArgs<T> &v = va[q];
      v.nodecell = P<long long>(c->d_vcell); v.nodeobs = P<int>(c->d_vobs); v.nnodes = c->vnodes;
      v.first = P<unsigned long long>(c->d_vfirst); v.last = P<unsigned long long>(c->d_vlast);
      v.stage = P<float>(c->d_vstage);
      v.ring = c->vring;
      for (int d = 0; d < 6; ++d) v.F[d] = P<T>(c->fld(q, d));
    }
  }

  // Time-dependent kernels read the step number from the device counter
  // (step n = counter + offset within this run), so the same launches can be
  // captured once in a graph and replayed for later runs.
  unsigned long long *stepp = A.stepp = P<unsigned long long>(c->d_step);
  for (int q = 0; q < 2; ++q) {
    oa[q].step = stepp; oa[q].dt = dt;
    va[q].step = stepp;
    for (int e = 0; e < 2; ++e) { ce[q][e].step = stepp; ce[q][e].dt = dt; ce[q][e].half = e == 0 ? 0.0 : 0.5; }
  }
  xa.step = stepp; xa.dt = dt;
  for (int e = 0; e < 2; ++e) {
    SideArgs<T> &d = A.side[e];
    d.o = oa[0];
    d.v = va[0];
    d.x = xa;
    const int v = 1 - e;  // the E sweep evaluates H values, the H sweep the next step's E values
    d.val.n = c->nXval[v]; d.val.v = P<XVal>(c->d_xval[v]); d.val.out = P<T>(c->d_xvals[v]);
    d.val.wf = P<WaveformDev>(c->d_wf); d.val.half = v == 0 ? 0.0 : 0.5;
    d.electric = e == 0;
    d.nfb = (maxnf + 255) / 256;
    d.b[0] = d.o.nobs * d.nfb;
    d.b[1] = d.b[0] + (int)((d.v.nnodes + 255) / 256);
    d.b[2] = d.b[1] + (int)((d.val.n + 255) / 256);
    d.b[3] = d.b[2] + (anyAux ? xa.npw : 0);
    d.b[4] = d.b[3] + (int)((c->nXupd[e] + 255) / 256);
    A.nside[e] = (unsigned)(d.b[4] + 7) / 8 * 8;
  }
}

// Ghost planes of one half-step (surface.c:569-812), copied within the field
// set the step writes.
template <typename T> void launch_ghosts(Ctx *c, int electric, int q, hipStream_t s)
{
  for (int f = 0; f < 6; ++f) {
    const int t = c->ghost[f];
    if (!t) continue;
    const int a = f >> 1;
    const int inner = (f & 1) ? c->grid.gobox[f] - 1 : c->grid.gobox[f];
    const int opp = (f & 1) ? c->grid.gobox[f - 1] : c->grid.gobox[f + 1] - 1;
    const int dst = (f & 1) ? c->grid.gobox[f] : c->grid.gobox[f] - 1;
    GhostArgs<T> g{};
    g.NX = c->NX; g.NY = c->NY; g.NZ = c->NZ; g.PX = c->PX; g.plane = c->plane;
    g.axis = a; g.dst = dst;
    for (int d = 0; d < 3; ++d) { g.lo[d] = c->grid.gobox[2 * d] - 1; g.hi[d] = c->grid.gobox[2 * d + 1]; }
    const int a1 = a == 0 ? 1 : 0, a2 = a == 2 ? 1 : 2;
    const dim3 gb(16, 16), gg((g.hi[a1] - g.lo[a1] + 16) / 16, (g.hi[a2] - g.lo[a2] + 16) / 16);
    int comps[2], nc;
    if (electric) { comps[0] = a; nc = 1; }
    else { comps[0] = 3 + (a + 1) % 3; comps[1] = 3 + (a + 2) % 3; nc = 2; }
    // E: PEC copy, PMC negate, periodic copy from the opposite side; H: PMC negate, periodic, PEC copy.
    g.src = t == 3 ? opp : inner;
    g.sign = (t == 2) ? T(-1) : T(1);
    for (int u = 0; u < nc; ++u) {
      g.F = P<T>(c->fld(c->next(q), comps[u]));
      hipLaunchKernelGGL(k_ghost<T>, gg, gb, 0, s, g);
    }
  }
}

// The loop (simulation.c:136-230).  With chk, one step of the field sweeps
// only (Mur E, the E sweep, the H sweep), in their update-counting form.
// With the fused sweep, step q of the run reads field set c->par ^ (q & 1)
// and writes the other, and the caller flips c->par by the parity of nsteps
// once the run is enqueued; the separate sweeps read and write set 0.
template <typename T> int run_steps(Ctx *c, uint64_t nsteps, hipStream_t s, bool timeKernels, const VisitRun *chk)
{
  const double pi = 4.0 * atan(1.0);
  timeKernels = timeKernels && !c->evE.empty();
  StepArgs<T> A{};
  fill_step_args<T>(c, A, chk);
  const auto &fe = A.fe;
  const auto &fh = A.fh;
  const dim3 egrid = A.egrid, hgrid = A.hgrid, eg1 = A.eg1, hg1 = A.hg1, vblk = A.vblk;
  const auto &eap = A.eap;
  const auto &hap = A.hap;
  const ShellDev *epc = A.epc, *hpc = A.hpc;
  const ShellWork *ewk = A.ewk, *hwk = A.hwk;
  const XArgs<T> *xe = P<XArgs<T>>(c->d_xargs[0]), *xh = P<XArgs<T>>(c->d_xargs[1]);
  auto fast_e = [&](int q) {
    const FastE<T> &f = fe[q];
    if (!egrid.x) return;
    const int x = c->xlevel();
    // (the check counts Mur's E with level 1's flags)
    if (chk && c->inl && c->indexed) hipLaunchKernelGGL((k_e_fast<T, true, 1, true>), eg1, vblk, 0, s, f, xe);
    else if (chk && c->inl) hipLaunchKernelGGL((k_e_fast<T, false, 1, true>), eg1, vblk, 0, s, f, xe);
    else if (chk && c->indexed) hipLaunchKernelGGL((k_e_fast<T, true, 0, true>), eg1, vblk, 0, s, f, xe);
    else if (chk) hipLaunchKernelGGL((k_e_fast<T, false, 0, true>), eg1, vblk, 0, s, f, xe);
    // (grids whose fast tiles launch apart have no update rows)
    else if (c->indexed && x == 2) hipLaunchKernelGGL((k_e_fast<T, true, 2>), eg1, vblk, 0, s, f, xe);
    else if (c->indexed && x == 1) hipLaunchKernelGGL((k_e_fast<T, true, 1>), eg1, vblk, 0, s, f, xe);
    else if (c->indexed) hipLaunchKernelGGL((k_e_fast<T, true, 0>), eg1, vblk, 0, s, f, xe);
    else if (x) hipLaunchKernelGGL((k_e_fast<T, false, 1>), eg1, vblk, 0, s, f, xe);
    else hipLaunchKernelGGL((k_e_fast<T, false, 0>), eg1, vblk, 0, s, f, xe);
  };
  auto shell_e = [&](int q) {
    const EArgs<T> *a = eap[q];
    const dim3 b(256), g((unsigned)c->nEwork);
    if (!g.x) return;
    if (chk && c->indexed) hipLaunchKernelGGL((k_e_shell<T, true, true>), g, b, 0, s, epc, ewk, a);
    else if (chk) hipLaunchKernelGGL((k_e_shell<T, false, true>), g, b, 0, s, epc, ewk, a);
    else if (c->indexed) hipLaunchKernelGGL((k_e_shell<T, true>), g, b, 0, s, epc, ewk, a);
    else hipLaunchKernelGGL((k_e_shell<T, false>), g, b, 0, s, epc, ewk, a);
  };
  auto fast_h = [&](int q) {
    const FastH<T> &f = fh[q];
    if (!hgrid.x) return;
    if (chk && c->indexed) hipLaunchKernelGGL((k_h_fast<T, true, false, true>), hg1, vblk, 0, s, f);
    else if (chk) hipLaunchKernelGGL((k_h_fast<T, false, false, true>), hg1, vblk, 0, s, f);
    else if (c->indexed) hipLaunchKernelGGL((k_h_fast<T, true, false>), hg1, vblk, 0, s, f);
    else hipLaunchKernelGGL((k_h_fast<T, false, false>), hg1, vblk, 0, s, f);
  };
  auto shell_h = [&](int q) {
    const HArgs<T> *a = hap[q];
    const dim3 b(256), g((unsigned)c->nHwork);
    if (!g.x) return;
    if (chk && c->indexed) hipLaunchKernelGGL((k_h_shell<T, true, true>), g, b, 0, s, hpc, hwk, a);
    else if (chk) hipLaunchKernelGGL((k_h_shell<T, false, true>), g, b, 0, s, hpc, hwk, a);
    else if (c->indexed) hipLaunchKernelGGL((k_h_shell<T, true>), g, b, 0, s, hpc, hwk, a);
    else hipLaunchKernelGGL((k_h_shell<T, false>), g, b, 0, s, hpc, hwk, a);
  };
  // A half-step's sweep in one launch (side blocks, shell, fast tiles), or
  // with `apart` without the fast tiles.
  const bool apart = sweeps_apart(c);
  auto sweep_e = [&](int soff, int last) {
    const unsigned ns = A.nside[0], nw = (unsigned)c->nEwork;
    const unsigned nb = c->sibcFaces ? (unsigned)c->sibcBlocks : 0u, nb8 = (nb + 7) / 8 * 8;
    const dim3 b(256), g(ns + nb8 + nw + (apart ? 0u : eg1.x));
    if (!g.x) return;
    const int x = c->xlevel();
    const FastE<T> &f = fe[0];
    const SideArgs<T> &sd = A.side[0];
    if (chk) {
      auto count = [&](auto k) {
        hipLaunchKernelGGL(k, g, b, 0, s, f, epc, ewk, eap[0], xe, ns, nb8, nw, (unsigned)sd.b[3]);
      };
      if (c->indexed) count(k_e_sweep_chk<T, true>);
      else count(k_e_sweep_chk<T, false>);
      return;
    }
    auto go = [&](auto k) { hipLaunchKernelGGL(k, g, b, 0, s, f, epc, ewk, eap[0], xe, ns, nw, sd, soff, last, pi); };
    auto sibc = [&](auto k) {
      hipLaunchKernelGGL(k, g, b, 0, s, f, epc, ewk, eap[0], xe, ns, nb8, nw, sd, A.se[0], nb, soff, last, pi);
    };
    if (nb && !c->indexed) sibc(k_e_sweep_sibc<T, false, 3>);
    else if (nb && x == 0) sibc(k_e_sweep_sibc<T, true, 0>);
    else if (nb && x == 1) sibc(k_e_sweep_sibc<T, true, 1>);
    else if (nb && x == 2) sibc(k_e_sweep_sibc<T, true, 2>);
    else if (nb && x == 3) sibc(k_e_sweep_sibc<T, true, 3>);
    else if (nb) sibc(k_e_sweep_sibc<T, true, 4>);
    else if (!c->indexed) go(k_e_sweep<T, false, 3>);
    else if (x == 0) go(k_e_sweep<T, true, 0>);
    else if (x == 1) go(k_e_sweep<T, true, 1>);
    else if (x == 2) go(k_e_sweep<T, true, 2>);
    else if (x == 3) go(k_e_sweep<T, true, 3>);
    else go(k_e_sweep<T, true, 4>);
  };
  auto sweep_h = [&](int soff, int last) {
    const unsigned ns = A.nside[1], nw = (unsigned)c->nHwork;
    const dim3 b(256), g(ns + nw + (apart ? 0u : hg1.x));
    if (!g.x) return;
    const SideArgs<T> &sd = A.side[1];
    if (chk) {
      auto count = [&](auto k) {
        hipLaunchKernelGGL(k, g, b, 0, s, fh[0], hpc, hwk, hap[0], xh, ns, nw, (unsigned)sd.b[3]);
      };
      if (c->indexed && c->xflagH) count(k_h_sweep_chk<T, true, true>);
      else if (c->indexed) count(k_h_sweep_chk<T, true, false>);
      else if (c->xflagH) count(k_h_sweep_chk<T, false, true>);
      else count(k_h_sweep_chk<T, false, false>);
      return;
    }
    auto go = [&](auto k) { hipLaunchKernelGGL(k, g, b, 0, s, fh[0], hpc, hwk, hap[0], xh, ns, nw, sd, soff, last, pi); };
    if (c->indexed && c->xflagH) go(k_h_sweep<T, true, true>);
    else if (c->indexed) go(k_h_sweep<T, true, false>);
    else if (c->xflagH) go(k_h_sweep<T, false, true>);
    else go(k_h_sweep<T, false, false>);
  };
  auto rows = [&](int e) {
    const dim3 b(256), g((unsigned)c->row_blocks(e));
    if (!g.x) return;
    if (c->indexed && e == 0 && c->nXsite) hipLaunchKernelGGL((k_rows<T, true, true, true>), g, b, 0, s, xe);
    else if (e == 0 && c->nXsite) hipLaunchKernelGGL((k_rows<T, false, true, true>), g, b, 0, s, xe);
    else if (c->indexed && e == 0) hipLaunchKernelGGL((k_rows<T, true, true>), g, b, 0, s, xe);
    else if (c->indexed) hipLaunchKernelGGL((k_rows<T, true, false>), g, b, 0, s, xh);
    else if (e == 0) hipLaunchKernelGGL((k_rows<T, false, true>), g, b, 0, s, xe);
    else hipLaunchKernelGGL((k_rows<T, false, false>), g, b, 0, s, xh);
  };

  const auto &la = A.la;
  const auto &fx = A.fx;
  const dim3 lgrid = A.lgrid, lblk = A.lblk;
  auto leap = [&](int q) {
    if (!lgrid.x) return;
    const LeapArgs<T> &l = la[q];
    const int R = c->leapR;
    if (chk) {
      if (c->indexed) {
        if (R == 1) hipLaunchKernelGGL((k_leap<T, true, 1, true>), lgrid, lblk, 0, s, l);
        else if (R == 2) hipLaunchKernelGGL((k_leap<T, true, 2, true>), lgrid, lblk, 0, s, l);
        else hipLaunchKernelGGL((k_leap<T, true, 4, true>), lgrid, lblk, 0, s, l);
      } else {
        if (R == 1) hipLaunchKernelGGL((k_leap<T, false, 1, true>), lgrid, lblk, 0, s, l);
        else if (R == 2) hipLaunchKernelGGL((k_leap<T, false, 2, true>), lgrid, lblk, 0, s, l);
        else hipLaunchKernelGGL((k_leap<T, false, 4, true>), lgrid, lblk, 0, s, l);
      }
    } else if (c->indexed) {
      if (R == 1) hipLaunchKernelGGL((k_leap<T, true, 1>), lgrid, lblk, 0, s, l);
      else if (R == 2) hipLaunchKernelGGL((k_leap<T, true, 2>), lgrid, lblk, 0, s, l);
      else hipLaunchKernelGGL((k_leap<T, true, 4>), lgrid, lblk, 0, s, l);
    } else {
      if (R == 1) hipLaunchKernelGGL((k_leap<T, false, 1>), lgrid, lblk, 0, s, l);
      else if (R == 2) hipLaunchKernelGGL((k_leap<T, false, 2>), lgrid, lblk, 0, s, l);
      else hipLaunchKernelGGL((k_leap<T, false, 4>), lgrid, lblk, 0, s, l);
    }
  };
  auto fix = [&](int q) {
    if (!lgrid.x || !c->nFix) return;
    const dim3 g((unsigned)((c->nFix + 3) / 4));
    if (c->indexed) hipLaunchKernelGGL((k_h_fix<T, true>), g, lblk, 0, s, fx[q]);
    else hipLaunchKernelGGL((k_h_fix<T, false>), g, lblk, 0, s, fx[q]);
  };

  const auto &ma = A.ma;
  const dim3 murGrid = A.murGrid;
  if (chk) {
    const int q = c->par;
    if (c->murmask && !c->murPush) hipLaunchKernelGGL((k_mur_e<T, true>), murGrid, dim3(16, 16), 0, s, ma[q]);
    if (c->inl) {
      sweep_e(0, 0);
      if (apart) {
        fast_e(0);
        fast_h(0);
      }
      sweep_h(0, 0);
    } else if (c->leap) {
      leap(q);
      shell_e(q);
      shell_h(q);
    } else {
      fast_e(q);
      shell_e(q);
      fast_h(q);
      shell_h(q);
    }
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return set_error(c, VGPU_EDEVICE, "kernel launch failed: %s", hipGetErrorString(err));
    return VGPU_OK;
  }

  auto &da = A.da;
  const auto &se = A.se;
  const auto &sh = A.sh;
  auto &ce = A.ce;
  auto &xa = A.xa;
  const bool anyAux = A.anyAux;
  auto &oa = A.oa;
  const int maxnf = A.maxnf;
  auto &va = A.va;
  unsigned long long *stepp = A.stepp;
  auto ghost = [&](int electric, int q) { launch_ghosts<T>(c, electric, q, s); };
  int ne = 0, nh = 0;
  auto mark = [&](std::vector<hipEvent_t> &ev, int k) {  // times the fast kernels of the first steps
    if (timeKernels && k < (int)ev.size()) hipEventRecord(ev[k], s);
  };
  // A step: the E sweep and rows, the H sweep and rows, the sweeps with what
  // rides along (SideArgs).  SIBC faces read the old H and write only their
  // own state, so their place before the H sweep is all that matters; so
  // with Mur faces their inner neighbours' threads cannot write, which read
  // the old E.
  if (c->inl && nsteps && A.side[1].b[2])
    hipLaunchKernelGGL(k_first_samples<T>, dim3((unsigned)A.side[1].b[2]), dim3(256), 0, s, A.side[1], pi);
  for (uint64_t n = 0; c->inl && n < nsteps; ++n) {
    const int soff = (int)n, last = n + 1 == nsteps;
    if (c->murmask && !c->murPush) hipLaunchKernelGGL(k_mur_e<T>, murGrid, dim3(16, 16), 0, s, ma[0]);
    // the fast tiles last here and first in the H sweep, which runs them from
    // the top plane down: what the E tiles touched last is still in cache
    if (apart) sweep_e(soff, last);
    mark(c->evE, 2 * ne);
    if (apart) fast_e(0);
    else sweep_e(soff, last);
    mark(c->evE, 2 * ne++ + 1);
    rows(0);
    mark(c->evH, 2 * nh);
    if (apart) fast_h(0);
    else sweep_h(soff, last);
    mark(c->evH, 2 * nh++ + 1);
    if (apart) sweep_h(soff, last);
    rows(1);
  }
  // Steps with corrections in launches of their own: the fused leapfrog sweep,
  // grids of 2^31 cells and more, set-ups that the in-line form does not hold.
  for (uint64_t n = 0; !c->inl && n < nsteps; ++n) {
    const int soff = (int)n;
    const int q = c->leap ? c->par ^ (int)(n & 1) : c->par;  // field set this step reads
    // observers, and the aux grids' E update as extra blocks (k_head)
    if (oa[q].nobs || anyAux) {
      oa[q].soff = soff;
      xa.soff = soff;
      const unsigned gy = (unsigned)(oa[q].nobs + (anyAux ? xa.npw : 0));
      hipLaunchKernelGGL(k_head<T>, dim3(oa[q].nobs ? (maxnf + 63) / 64 : 1, gy), dim3(64), 0, s, oa[q], xa, pi);
    }
    if (va[q].nnodes) {
      va[q].soff = soff;
      hipLaunchKernelGGL(k_observe_volume<T>, dim3((unsigned)((va[q].nnodes + 255) / 256)), dim3(256), 0, s, va[q]);
    }
    if (c->murmask) hipLaunchKernelGGL(k_mur_e<T>, murGrid, dim3(16, 16), 0, s, ma[q]);
    // events bracket the fast kernels (the dominant launches): the fused
    // sweep and its fix-up, or the fast E and H kernels
    if (timeKernels && ne < (int)c->evE.size() / 2) hipEventRecord(c->evE[2 * ne], s);
    if (c->leap) leap(q);
    else fast_e(q);
    if (timeKernels && ne < (int)c->evE.size() / 2) { hipEventRecord(c->evE[2 * ne + 1], s); ++ne; }
    shell_e(q);
    // Layers 0 and 1 hold each cell's first block, inside and outside the
    // fast E box, so their sites never share an edge: they go in one launch.
    // Later layers follow one launch each, in block order.
    for (int l = 0; l < c->debyeLayers;) {
      const int l1 = l == 0 && c->debyeLayers > 1 ? 2 : l + 1;
      da[q].base = c->debyeLayerStart[l];
      da[q].n = c->debyeLayerStart[l1] - c->debyeLayerStart[l];
      l = l1;
      if (da[q].n == 0) continue;
      hipLaunchKernelGGL(k_debye<T>, dim3((unsigned)((da[q].n + 255) / 256)), dim3(256), 0, s, da[q]);
    }
    if (c->sibcFaces) hipLaunchKernelGGL((k_sibc_e<T, true>), dim3((unsigned)c->sibcBlocks), dim3(256), 0, s, se[q]);
    if (ce[q][0].nrows) {
      ce[q][0].soff = soff;
      hipLaunchKernelGGL(k_corr<T>, dim3((unsigned)((ce[q][0].nrows + 255) / 256)), dim3(256), 0, s, ce[q][0], pi);
    }
    ghost(1, q);
    if (c->leap) shell_h(q);
    if (timeKernels && nh < (int)c->evH.size() / 2) hipEventRecord(c->evH[2 * nh], s);
    if (c->leap) fix(q);
    else fast_h(q);
    if (timeKernels && nh < (int)c->evH.size() / 2) { hipEventRecord(c->evH[2 * nh + 1], s); ++nh; }
    if (!c->leap) shell_h(q);
    if (c->sibcFaces)
      hipLaunchKernelGGL(k_sibc_h<T>, dim3((unsigned)((sh[q].nrows + 255) / 256)), dim3(256), 0, s, sh[q]);
    // H corrections, and the aux grids' H update as extra blocks
    if (ce[q][1].nrows || anyAux) {
      ce[q][1].soff = soff;
      const int nb = (int)((ce[q][1].nrows + 255) / 256);
      const dim3 g((unsigned)(nb + (anyAux ? xa.npw : 0)));
      if (anyAux) hipLaunchKernelGGL(k_corr_aux<T>, g, dim3(256), 0, s, ce[q][1], pi, xa, nb);
      else hipLaunchKernelGGL(k_corr<T>, g, dim3(256), 0, s, ce[q][1], pi);
    }
    ghost(0, q);
  }
  hipLaunchKernelGGL(k_advance_step, dim3(1), dim3(64), 0, s, stepp, (unsigned long long)nsteps);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return set_error(c, VGPU_EDEVICE, "kernel launch failed: %s", hipGetErrorString(err));
  return VGPU_OK;
}

// A solve's argument blocks for packed launches (field set 0), uploaded once
// after set-up.  Contexts with the fused sweep take no part in group runs.
template <typename T> int upload_pack(Ctx *c)
{
  StepArgs<T> A{};
  fill_step_args<T>(c, A, nullptr, true);
  // shells at SHELL_KC planes per block: a packed launch fills the device
  // with many grids' blocks, where a small grid's own plan used one plane
  std::vector<ShellDev> ep, hp;
  std::vector<ShellWork> ew, hw;
  std::string err;
  long long cells[2];
  if (plan_shells<T>(c, SHELL_KC, ep, ew, hp, hw, cells, err)) return set_error(c, VGPU_EINVAL, "%s", err.c_str());
  c->d_epcsPk = dev_alloc(c, ep.size() * sizeof(ShellDev));
  c->d_hpcsPk = dev_alloc(c, hp.size() * sizeof(ShellDev));
  c->d_eworkPk = dev_alloc(c, ew.size() * sizeof(ShellWork));
  c->d_hworkPk = dev_alloc(c, hw.size() * sizeof(ShellWork));
  if (!c->d_epcsPk || !c->d_hpcsPk || !c->d_eworkPk || !c->d_hworkPk)
    return set_error(c, VGPU_ENOMEM, "group-run shells");
  auto up = [](void *d, const void *h, size_t n) {
    return n == 0 || hipMemcpy(d, h, n, hipMemcpyHostToDevice) == hipSuccess;
  };
  if (!up(c->d_epcsPk, ep.data(), ep.size() * sizeof(ShellDev)) ||
      !up(c->d_hpcsPk, hp.data(), hp.size() * sizeof(ShellDev)) ||
      !up(c->d_eworkPk, ew.data(), ew.size() * sizeof(ShellWork)) ||
      !up(c->d_hworkPk, hw.data(), hw.size() * sizeof(ShellWork)))
    return set_error(c, VGPU_EDEVICE, "group-run shells upload");
  c->nEworkPk = (int)ew.size();
  c->nHworkPk = (int)hw.size();
  PackArgs<T> p{};
  p.fe = A.fe[0];
  p.fh = A.fh[0];
  p.epc = P<ShellDev>(c->d_epcsPk); p.hpc = P<ShellDev>(c->d_hpcsPk);
  p.ewk = P<ShellWork>(c->d_eworkPk); p.hwk = P<ShellWork>(c->d_hworkPk);
  p.ea = A.eap[0]; p.ha = A.hap[0];
  p.xe = P<XArgs<T>>(c->d_xargs[0]); p.xh = P<XArgs<T>>(c->d_xargs[1]);
  p.nEside = A.nside[0]; p.nHside = A.nside[1];
  p.nEshell = (unsigned)c->nEworkPk; p.nHshell = (unsigned)c->nHworkPk;
  p.se = A.side[0]; p.sh = A.side[1];
  c->d_pack = dev_alloc(c, sizeof(p));
  if (!c->d_pack) return set_error(c, VGPU_ENOMEM, "group-run arguments");
  if (hipMemcpy(c->d_pack, &p, sizeof(p), hipMemcpyHostToDevice) != hipSuccess)
    return set_error(c, VGPU_EDEVICE, "group-run arguments: %s", hipGetErrorString(hipGetLastError()));
  return VGPU_OK;
}

// Steps of several solves in lockstep on one stream (vgpu_run_group): the
// same kernels in the same order per solve as run_steps, with the sweeps and
// what rides along, and the rows, of all solves in one packed launch each; SIBC
// E, and Mur E where it keeps its launch, stay one per solve.  Solves share no
// memory, so only each solve's own order matters, and every block does what it
// does in the solve's own launch.  Members without PackArgs (corrections in
// launches of their own) run alone.
template <typename T> int run_group_steps(Ctx *const *all, int nall, uint64_t nsteps, hipStream_t s)
{
  const double pi = 4.0 * atan(1.0);
  Ctx *cs[PACK_MAX];
  int n = 0;
  for (int i = 0; i < nall; ++i) {
    if (all[i]->d_pack) {
      cs[n++] = all[i];
    } else if (const int r = run_steps<T>(all[i], nsteps, s, false)) {
      return r;
    }
  }
  std::vector<StepArgs<T>> A(n);
  for (int i = 0; i < n; ++i) fill_step_args<T>(cs[i], A[i], nullptr, true);
  // One packed launch: the solves with a positive block count, in order.
  auto plan = [&](auto blocks) {
    PackMap m{};
    unsigned tot = 0;
    for (int i = 0; i < n; ++i) {
      const long long k = blocks(i);
      if (k <= 0) continue;
      m.args[m.n] = cs[i]->d_pack;
      m.start[m.n++] = tot;
      tot += (unsigned)k;
    }
    m.start[m.n] = tot;
    return m;
  };
  // packs by kernel form: with classes, the E sweep's by the level of its
  // in-line corrections
  PackMap sweepE[6], sweepH[4], rowE[4], rowH[2];
  for (int x = 0; x < 6; ++x)
    sweepE[x] = plan([&](int i) {
      return (cs[i]->indexed ? cs[i]->xlevel() : 5) == x ? (long long)A[i].nside[0] + cs[i]->nEworkPk + A[i].eg1.x : 0LL; });
  for (int x = 0; x < 2; ++x) {
    const bool idx = x == 0;
    for (int f = 0; f < 2; ++f)  // with flagged H cells or without
      sweepH[2 * x + f] = plan([&](int i) {
        return cs[i]->indexed == idx && cs[i]->xflagH == (f == 0)
                   ? (long long)A[i].nside[1] + cs[i]->nHworkPk + A[i].hg1.x : 0LL; });
    auto nrows = [&](int i, int e) { return cs[i]->indexed == idx ? cs[i]->row_blocks(e) : 0LL; };
    for (int f = 0; f < 2; ++f)  // with Debye sites of the list or without
      rowE[2 * x + f] = plan([&](int i) { return (cs[i]->nXsite > 0) == (f == 0) ? nrows(i, 0) : 0LL; });
    rowH[x] = plan([&](int i) { return nrows(i, 1); });
  }
  const PackMap first = plan([&](int i) { return (long long)A[i].side[1].b[2]; });
  auto blocks = [](const PackMap &m) { return dim3(m.start[m.n]); };  // a packed launch's 1-D grid
  const dim3 b(256);
  if (first.n && nsteps) hipLaunchKernelGGL(k_first_samples_pk<T>, blocks(first), b, 0, s, first, pi);
  for (uint64_t st = 0; n && st < nsteps; ++st) {
    for (PackMap &m : sweepE) m.soff = (int)st, m.last = st + 1 == nsteps;
    for (PackMap &m : sweepH) m.soff = (int)st, m.last = st + 1 == nsteps;
    for (int i = 0; i < n; ++i)
      if (cs[i]->murmask && !cs[i]->murPush)
        hipLaunchKernelGGL(k_mur_e<T>, A[i].murGrid, dim3(16, 16), 0, s, A[i].ma[0]);
    if (sweepE[0].n) hipLaunchKernelGGL((k_e_sweep_pk<T, true, 0>), blocks(sweepE[0]), b, 0, s, sweepE[0], pi);
    if (sweepE[1].n) hipLaunchKernelGGL((k_e_sweep_pk<T, true, 1>), blocks(sweepE[1]), b, 0, s, sweepE[1], pi);
    if (sweepE[2].n) hipLaunchKernelGGL((k_e_sweep_pk<T, true, 2>), blocks(sweepE[2]), b, 0, s, sweepE[2], pi);
    if (sweepE[3].n) hipLaunchKernelGGL((k_e_sweep_pk<T, true, 3>), blocks(sweepE[3]), b, 0, s, sweepE[3], pi);
    if (sweepE[4].n) hipLaunchKernelGGL((k_e_sweep_pk<T, true, 4>), blocks(sweepE[4]), b, 0, s, sweepE[4], pi);
    if (sweepE[5].n) hipLaunchKernelGGL((k_e_sweep_pk<T, false, 3>), blocks(sweepE[5]), b, 0, s, sweepE[5], pi);
    if (rowE[0].n) hipLaunchKernelGGL((k_rows_pk<T, true, true, true>), blocks(rowE[0]), b, 0, s, rowE[0]);
    if (rowE[1].n) hipLaunchKernelGGL((k_rows_pk<T, true, true>), blocks(rowE[1]), b, 0, s, rowE[1]);
    if (rowE[2].n) hipLaunchKernelGGL((k_rows_pk<T, false, true, true>), blocks(rowE[2]), b, 0, s, rowE[2]);
    if (rowE[3].n) hipLaunchKernelGGL((k_rows_pk<T, false, true>), blocks(rowE[3]), b, 0, s, rowE[3]);
    for (int i = 0; i < n; ++i)
      if (cs[i]->sibcFaces)
        hipLaunchKernelGGL((k_sibc_e<T, false>), dim3((unsigned)cs[i]->sibcBlocks), dim3(256), 0, s, A[i].se[0]);
    if (sweepH[0].n) hipLaunchKernelGGL((k_h_sweep_pk<T, true, true>), blocks(sweepH[0]), b, 0, s, sweepH[0], pi);
    if (sweepH[1].n) hipLaunchKernelGGL((k_h_sweep_pk<T, true, false>), blocks(sweepH[1]), b, 0, s, sweepH[1], pi);
    if (sweepH[2].n) hipLaunchKernelGGL((k_h_sweep_pk<T, false, true>), blocks(sweepH[2]), b, 0, s, sweepH[2], pi);
    if (sweepH[3].n) hipLaunchKernelGGL((k_h_sweep_pk<T, false, false>), blocks(sweepH[3]), b, 0, s, sweepH[3], pi);
    if (rowH[0].n) hipLaunchKernelGGL((k_rows_pk<T, true, false>), blocks(rowH[0]), b, 0, s, rowH[0]);
    if (rowH[1].n) hipLaunchKernelGGL((k_rows_pk<T, false, false>), blocks(rowH[1]), b, 0, s, rowH[1]);
  }
  // (the step counters advance with the group's close)
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return set_error(all[0], VGPU_EDEVICE, "kernel launch failed: %s", hipGetErrorString(err));
  return VGPU_OK;
}

// Update-once check (the reference's CHECK_LIMITS build: grid.h:181-191, and
// checkGrid, grid.c:951-1025).  One step of the field sweeps -- Mur E, the E
// sweep, the H sweep, in the grids that the loop launches them in -- runs in
// its counting form, which adds one to a per-cell count for each update instead
// of storing it: a value left to an update row counts there, a Mur value where
// its inner neighbour's thread or Mur's own launch writes it.  Each component's
// counts are then tallied against its outer field limits folim.  Fields, UPML auxiliaries and Debye state are left as they were.
// Bytes of device memory one update-once check uses: visit counts per
// component (device layout), the two sweep argument blocks, the tally and,
// with counts, their staging in the counts layout; each part 256-byte aligned.
template <typename T> size_t check_limits_bytes(const Ctx *c, bool counts, size_t off[4])
{
  auto al = [](size_t n) { return (n + 255) / 256 * 256; };
  const size_t cells = (size_t)c->plane * c->NZ, ncell = (size_t)c->NX * c->NY * c->NZ;
  off[0] = 0;
  off[1] = al(6 * cells * sizeof(unsigned));
  off[2] = off[1] + al(al(sizeof(EArgs<T>)) + sizeof(HArgs<T>));
  off[3] = off[2] + al(24 * sizeof(unsigned long long));
  return off[3] + (counts ? al(6 * ncell) : 0);
}

template <typename T>
int check_limits(Ctx *c, const int folim[6][6], vgpu_limits_report *rep, unsigned char *counts, void *scratch,
                 size_t scratchBytes)
{
  const size_t cells = (size_t)c->plane * c->NZ;      // device layout, padded rows
  const size_t ncell = (size_t)c->NX * c->NY * c->NZ; // counts layout, x fastest
  unsigned *vis = nullptr;
  char *args = nullptr;
  unsigned long long *tally = nullptr;
  unsigned char *dcounts = nullptr;
  int r = VGPU_OK;
  const size_t hoff = (sizeof(EArgs<T>) + 255) / 256 * 256;
  size_t off[4];
  const size_t need = check_limits_bytes<T>(c, counts != nullptr, off);
  if (scratch && need > scratchBytes)
    return set_error(c, VGPU_EINVAL,
                     "update-once check of this grid needs %zu bytes of scratch, more than the %zu the "
                     "no-allocation entry point holds",
                     need, scratchBytes);
  if (hipDeviceSynchronize() != hipSuccess) return set_error(c, VGPU_EDEVICE, "device error before the check");
  bool have;
  if (scratch) {
    // the caller's buffer: no allocation
    char *b = static_cast<char *>(scratch);
    vis = reinterpret_cast<unsigned *>(b + off[0]);
    args = b + off[1];
    tally = reinterpret_cast<unsigned long long *>(b + off[2]);
    dcounts = counts ? reinterpret_cast<unsigned char *>(b + off[3]) : nullptr;
    have = true;
  } else {
    have = hipMalloc((void **)&vis, 6 * cells * sizeof(unsigned)) == hipSuccess &&
           hipMalloc((void **)&args, hoff + sizeof(HArgs<T>)) == hipSuccess &&
           hipMalloc((void **)&tally, 24 * sizeof(unsigned long long)) == hipSuccess &&
           (!counts || hipMalloc((void **)&dcounts, 6 * ncell) == hipSuccess);
  }
  if (!have) {
    r = set_error(c, VGPU_ENOMEM, "update-once check buffers");
  } else {
    EArgs<T> ea;
    HArgs<T> ha;
    unsigned long long init[24];
    for (int q = 0; q < 24; ++q) init[q] = (q & 3) == 3 ? ~0ull : 0ull;
    bool ok = hipMemcpy(&ea, c->d_eargs[c->par], sizeof ea, hipMemcpyDeviceToHost) == hipSuccess &&
              hipMemcpy(&ha, c->d_hargs[c->par], sizeof ha, hipMemcpyDeviceToHost) == hipSuccess;
    VisitRun vr{};
    for (int q = 0; q < 6; ++q) vr.vis[q] = vis + q * cells;
    for (int d = 0; d < 3; ++d) { ea.vis[d] = vr.vis[d]; ha.vis[d] = vr.vis[3 + d]; }
    vr.eargs = args;
    vr.hargs = args + hoff;
    // the counts start at zero (a fill kernel: no memset node if captured)
    const size_t nv = 6 * cells;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)std::min<size_t>((nv + 255) / 256, 65535)), dim3(256), 0, c->stream,
                       vis, nv, 0u);
    ok = ok && hipStreamSynchronize(c->stream) == hipSuccess &&
         hipMemcpy(args, &ea, sizeof ea, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(args + hoff, &ha, sizeof ha, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(tally, init, sizeof init, hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) r = set_error(c, VGPU_EDEVICE, "update-once check set-up");
    if (!r) r = run_steps<T>(c, 1, c->stream, false, &vr);
    if (!r) {
      for (int C = 0; C < 6; ++C) {
        Lim6 lim;
        for (int f = 0; f < 6; ++f) lim.v[f] = folim[C][f];
        hipLaunchKernelGGL(k_visit_tally, dim3((c->NX + 255) / 256, c->NY, c->NZ), dim3(256), 0, c->stream,
                           vr.vis[C], c->NX, c->NY, c->NZ, (long long)c->PX, lim, tally + 4 * C,
                           dcounts ? dcounts + C * ncell : nullptr);
      }
      unsigned long long out[24];
      if (hipStreamSynchronize(c->stream) != hipSuccess ||
          hipMemcpy(out, tally, sizeof out, hipMemcpyDeviceToHost) != hipSuccess ||
          (counts && hipMemcpy(counts, dcounts, 6 * ncell, hipMemcpyDeviceToHost) != hipSuccess)) {
        r = set_error(c, VGPU_EDEVICE, "update-once check: %s", hipGetErrorString(hipGetLastError()));
      } else {
        for (int C = 0; C < 6; ++C) {
          rep->missed[C] = out[4 * C];
          rep->repeated[C] = out[4 * C + 1];
          rep->outside[C] = out[4 * C + 2];
          rep->first[C] = out[4 * C + 3] == ~0ull ? -1 : (int64_t)out[4 * C + 3];
        }
      }
    }
  }
  if (!scratch) {
    (void)hipFree(vis);
    (void)hipFree(args);
    (void)hipFree(tally);
    (void)hipFree(dcounts);
  }
  return r;
}

}  // namespace vgpu
