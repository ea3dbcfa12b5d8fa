// Corrections, set-up (XArgs, vgpu_internal.h): from the Debye sites, SIBC
// edges and faces, source and TF/SF rows, Mur faces and ghost planes of a
// context, what the sweeps' threads apply in line and the rows of the rest, in
// the reference's order: Mur E, the update, Debye blocks, SIBC, sources and
// TF/SF, ghosts (simulation.c:157-222).
#pragma once
#include "vgpu_kernels.h"
#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <unordered_map>
#include <vector>

namespace vgpu {

// Where the sweeps update and where ghosts are written, from the host's limits.
template <typename T> struct InlineGeom {
  const Ctx *c;
  EArgs<T> ea{};
  HArgs<T> ha{};
  int ein[3][1][6];
  struct Ghost { int axis, dst, src; double sign; };
  std::vector<Ghost> ghosts[6];  // per component, in face order
  int glo[3], ghi[3];            // the copied planes' extents

  explicit InlineGeom(Ctx *ctx) : c(ctx)
  {
    fill_volume_args<T>(ctx, ea, ha, 0);
    for (int C = 0; C < 3; ++C)
      for (int q = 0; q < 6; ++q) ein[C][0][q] = ea.in[C][q];
    // ghost planes as launch_ghosts copies them (surface.c:569-812)
    const int N[3] = {c->NX, c->NY, c->NZ};
    for (int a = 0; a < 3; ++a) {
      glo[a] = std::max(0, c->grid.gobox[2 * a] - 1);
      ghi[a] = std::min(N[a] - 1, c->grid.gobox[2 * a + 1]);
    }
    for (int f = 0; f < 6; ++f) {
      const int t = c->ghost[f], a = f >> 1;
      if (!t) continue;
      const int *go = c->grid.gobox;
      const int inner = (f & 1) ? go[f] - 1 : go[f], opp = (f & 1) ? go[f - 1] : go[f + 1] - 1;
      const Ghost g{a, (f & 1) ? go[f] : go[f] - 1, t == 3 ? opp : inner, t == 2 ? -1.0 : 1.0};
      for (int C = 0; C < 6; ++C)
        if (C < 3 ? C == a : C - 3 != a) ghosts[C].push_back(g);
    }
  }
  // region of component C (0-2 E, 3-5 H): 6 ordinary, 0-5 UPML, -1 not swept
  int region(int C, const int n[3]) const
  {
    long long p;
    return C < 3 ? classify<1>(ea, ein[C], C, n[0], n[1], n[2], p) : classify<3>(ha, ha.in[C - 3], C - 3, n[0], n[1], n[2], p);
  }
  void unlin(long long cell, int n[3]) const
  {
    n[0] = (int)(cell % c->PX);
    n[1] = (int)(cell / c->PX % c->NY);
    n[2] = (int)(cell / c->plane);
  }
  bool ghost_dst(int C, const int n[3]) const
  {
    for (int a = 0; a < 3; ++a)
      if (n[a] < glo[a] || n[a] > ghi[a]) return false;
    for (const Ghost &g : ghosts[C])
      if (n[g.axis] == g.dst) return true;
    return false;
  }
  // the Mur face an E value lies on (-1 none), and its inner neighbour
  int mur_face(int C, const int n[3], int nb[3]) const
  {
    for (int f = 0; f < 6; ++f) {
      if (!((c->murmask >> f) & 1u) || (f >> 1) == C) continue;
      const int *b = c->fmlim[f][C], a = f >> 1;
      const int at = (f & 1) ? b[2 * a + 1] : b[2 * a];
      if (n[a] != at || !in_box(b, n[0], n[1], n[2])) continue;
      for (int q = 0; q < 3; ++q) nb[q] = n[q];
      nb[a] += (f & 1) ? -1 : 1;
      return f;
    }
    return -1;
  }
};

// Stable sort by the 64-bit key of each element, least significant digit first.
template <typename V> static void sort_by_key(std::vector<V> &v)
{
  long long top = 0;
  bool sorted = true;
  for (size_t k = 0; k < v.size(); ++k) {
    top = std::max(top, v[k].key);
    sorted = sorted && (k == 0 || v[k - 1].key <= v[k].key);
  }
  if (sorted) return;
  constexpr int BITS = 11;
  std::vector<V> w(v.size());
  std::vector<size_t> at(1 << BITS);
  for (int shift = 0; shift < 63 && (top >> shift) > 0; shift += BITS) {
    std::fill(at.begin(), at.end(), 0);
    for (const V &x : v) ++at[(x.key >> shift) & ((1 << BITS) - 1)];
    size_t sum = 0;
    for (size_t &n : at) {
      const size_t m = n;
      n = sum;
      sum += m;
    }
    for (const V &x : v) w[at[(x.key >> shift) & ((1 << BITS) - 1)]++] = x;
    v.swap(w);
  }
}

template <typename T> int build_inline(Ctx *c)
{
  if (!c->inl) return VGPU_OK;
  using Ent = Ctx::XEnt;
  const InlineGeom<T> geo(c);
  const int N[3] = {c->NX, c->NY, c->NZ};
  auto fail = [&](const char *what) { return set_error(c, VGPU_ENOMEM, "corrections: %s", what); };
  auto up = [&](void *&d, const void *h, size_t bytes) {
    d = dev_alloc(c, bytes);
    return d && (bytes == 0 || hipMemcpy(d, h, bytes, hipMemcpyHostToDevice) == hipSuccess);
  };
  auto kind = [](const Ent &x) { return x.code & 7; };

  // Mur faces: each E value on one is written by the thread of its inner
  // neighbour when that takes the ordinary update; else the whole context
  // keeps Mur's own launch before the sweep
  struct Flag { long long key; unsigned fl; };  // key: cell
  std::vector<Flag> flags[2];
  c->murPush = c->murmask != 0;
  for (int f = 0; f < 6 && c->murPush; ++f)
    for (int C = 0; C < 3 && c->murPush; ++C) {
      if (!((c->murmask >> f) & 1u) || (f >> 1) == C) continue;
      const int *b = c->fmlim[f][C], a = f >> 1;
      int lo[3] = {b[0], b[2], b[4]}, hi[3] = {b[1], b[3], b[5]};
      lo[a] = hi[a] = (f & 1) ? b[2 * a + 1] : b[2 * a];
      int n[3];
      for (n[2] = lo[2]; n[2] <= hi[2]; ++n[2])
        for (n[1] = lo[1]; n[1] <= hi[1]; ++n[1])
          for (n[0] = lo[0]; n[0] <= hi[0]; ++n[0]) {
            int nb[3];
            if (geo.mur_face(C, n, nb) != f || geo.region(C, nb) != 6 || geo.region(C, n) >= 0) {
              c->murPush = false;
              continue;
            }
            flags[0].push_back({c->lin(nb[0], nb[1], nb[2]), (unsigned)XF_MUR << (2 * f + (C - a + 5) % 3)});
          }
    }
  if (!c->murPush) flags[0].clear();
  sort_by_key(flags[0]);
  // whether a Mur face takes component C of a cell
  auto feeds_mur = [&](long long cell, int C) {
    auto it = std::lower_bound(flags[0].begin(), flags[0].end(), cell, [](const Flag &x, long long k) { return x.key < k; });
    for (; it != flags[0].end() && it->key == cell; ++it)
      for (int f = 0; f < 6; ++f)
        for (int s = 0; s < 2; ++s)
          if (((it->fl >> (XF_MUR_SHIFT + 2 * f + s)) & 1u) && (f / 2 + 1 + s) % 3 == C) return true;
    return false;
  };

  // operations but Debye, by value; an H set to zero by SIBC takes none of its
  // terms; a ghost value takes its source's, so what else would change it is lost
  for (int e = 0; e < 2; ++e) {
    std::vector<Ent> &v = c->xent[e];
    sort_by_key(v);
    size_t k = 0;
    long long corrected = -1, zeroed = -1;
    c->corrRows[e] = 0;
    for (const Ent &x : v) {
      const int what = kind(x);
      if (what == XO_ZERO) {
        if (k && kind(v[k - 1]) == XO_ZERO && v[k - 1].key == x.key) continue;
        zeroed = x.value();
      } else if (what == XO_SIBC) {
        if (zeroed == x.value()) continue;
      } else if (corrected != x.value()) {  // sources and TF/SF
        corrected = x.value();
        ++c->corrRows[e];
      }
      if (!geo.ghosts[3 * e + x.comp()].empty()) {
        int n[3];
        geo.unlin(x.cell(), n);
        if (geo.ghost_dst(3 * e + x.comp(), n)) continue;
      }
      v[k++] = x;
    }
    v.resize(k);
  }

  // Debye sites: one one-pole site alone on a swept value goes to the class
  // table, the others are operations
  std::vector<Ctx::XSite> simple;
  long long listed = 0;
  {
    std::vector<Ctx::XSite> &st = c->xsite;
    sort_by_key(st);
    std::vector<Ent> add;
    const std::vector<Ent> &v = c->xent[0];
    size_t q = 0;
    simple.reserve(st.size());
    for (size_t a = 0; a < st.size();) {
      size_t b = a;
      while (b < st.size() && st[b].key == st[a].key) ++b;
      while (q < v.size() && v[q].value() < st[a].key) ++q;
      const bool ops = q < v.size() && v[q].value() == st[a].key;
      const int C = (int)(st[a].key % 3), m = st[a].med;
      int n[3];
      geo.unlin(st[a].key / 3, n);
      if (!geo.ghost_dst(C, n)) {
        if (b == a + 1 && !ops && c->dsimple[m] && geo.region(C, n) >= 0) {
          simple.push_back(st[a]);
        } else {
          for (size_t k = a; k < b; ++k) {
            if (st[k].med >= 1 << 21) return set_error(c, VGPU_EINVAL, "Debye site index out of range");
            add.push_back({st[k].key * 4, XO_DEBYE | st[k].med << 8, 0, 0, 0});
            ++listed;
          }
        }
      }
      a = b;
    }
    std::vector<Ctx::XSite>().swap(st);
    c->xent[0].insert(c->xent[0].end(), add.begin(), add.end());
  }

  // ghosts of every value that changes
  for (int e = 0; e < 2; ++e) {
    sort_by_key(c->xent[e]);
    std::vector<Ent> add;
    const std::vector<Ent> &v = c->xent[e];
    for (int C = 0; C < 3; ++C) {
      const auto &gs = geo.ghosts[3 * e + C];
      for (size_t g = 0; g < gs.size(); ++g) {
        int lo[3], hi[3], n[3];
        for (int a = 0; a < 3; ++a) {
          lo[a] = geo.glo[a];
          hi[a] = geo.ghi[a];
        }
        lo[gs[g].axis] = hi[gs[g].axis] = gs[g].dst;
        for (n[2] = lo[2]; n[2] <= hi[2]; ++n[2])
          for (n[1] = lo[1]; n[1] <= hi[1]; ++n[1])
            for (n[0] = lo[0]; n[0] <= hi[0]; ++n[0]) {
              // copied face by face, each over the whole plane: a value on two
              // ghost planes takes the value both maps lead to
              int s[3] = {n[0], n[1], n[2]}, nb[3];
              double sign = 1.0;
              bool first = true;
              for (size_t h = 0; h < gs.size(); ++h) {
                if (n[gs[h].axis] != gs[h].dst) continue;
                first = first && h >= g;
                s[gs[h].axis] = gs[h].src;
                sign *= gs[h].sign;
              }
              if (!first) continue;
              if (geo.region(3 * e + C, n) >= 0)
                return set_error(c, VGPU_EINVAL, "ghost plane inside the sweeps' limits");
              const long long src = c->lin(s[0], s[1], s[2]), val = src * 3 + C;
              if (geo.region(3 * e + C, s) < 0 && !(e == 0 && geo.mur_face(C, s, nb) >= 0)) {
                auto it = std::lower_bound(v.begin(), v.end(), val, [](const Ent &x, long long k) { return x.value() < k; });
                if (it == v.end() || it->value() != val) continue;
              }
              add.push_back({(c->lin(n[0], n[1], n[2]) * 3 + C) * 4 + 3, XO_GHOST, (int)src, sign, 0});
            }
      }
    }
    c->xent[e].insert(c->xent[e].end(), add.begin(), add.end());
    sort_by_key(c->xent[e]);
  }

  // The cells the sweeps correct in line, in cell order: their flags and Debye
  // media; and each value's operations [a, b): update rows, rows, and zeros
  // alone on a swept value, which are a flag.  Update rows take values of the
  // ordinary update with both neighbours inside on every axis, unless a Mur
  // face takes them too: its thread, the sweep's, reads the old value.
  // They pay where a launch is what a step waits for: 53x41x62 request 35.6 ->
  // 28.9 us a step, 40^3 free space FP64 28.6 -> 26.5.  In large grids reading
  // the other field's neighbours again costs more than the rows' launch: 256^3
  // Debye volume 497 -> 531, 173x211x158 request 204 -> 215.  The line is drawn
  // at a million cells; between there and about three million it depends on
  // what is corrected.  Sources and TF/SF would still gain (2.0 M-cell request
  // 71.4 -> 66.2, 2.7 M-cell Debye volume FP64 156.5 -> 153.7, 140^3 with a
  // one-pole block FP32 63.4 -> 59.3), sites of several poles lose (the same
  // block, two poles: 75.3 -> 92.4 FP32, 133 -> 186 FP64; 108^3 44.6 -> 51.0).
  const bool small = c->xskip = c->ncell <= 1000000;
  struct Value { size_t a, b; bool ghost; };
  struct Entry { int cell; int med[3]; unsigned fl; };
  std::vector<Value> upd[2], rest[2];
  std::vector<Entry> ents[2];
  auto plan = [&](int e) {
    const std::vector<Ent> &v = c->xent[e];
    std::vector<Flag> fl = flags[e];
    upd[e].clear();
    rest[e].clear();
    for (size_t a = 0; a < v.size();) {
      size_t b = a;
      while (b < v.size() && v[b].value() == v[a].value()) ++b;
      size_t from = a;
      if (!small && (e == 1 || kind(v[a]) != XO_ZERO)) {  // a row wherever it lies
        rest[e].push_back({a, b, kind(v[a]) == XO_GHOST});
        a = b;
        continue;
      }
      const long long cell = v[a].cell();
      const int C = v[a].comp();
      int n[3];
      geo.unlin(cell, n);
      const int reg = geo.region(3 * e + C, n);
      const bool inside = n[0] > 0 && n[1] > 0 && n[2] > 0 && n[0] < N[0] - 1 && n[1] < N[1] - 1 && n[2] < N[2] - 1;
      if (reg >= 0 && kind(v[a]) == XO_ZERO && (small || e == 0) && (b == a + 1 || !small || reg != 6 || !inside)) {
        fl.push_back({cell, (unsigned)XF_ZERO << C});
        ++from;
      }
      if (from < b) {
        if (small && reg == 6 && inside && !(e == 0 && feeds_mur(cell, C))) {
          fl.push_back({cell, (unsigned)XF_SKIP << C});
          upd[e].push_back({from, b, false});
        } else {
          rest[e].push_back({from, b, kind(v[a]) == XO_GHOST});
        }
      }
      a = b;
    }
    sort_by_key(fl);
    std::vector<Entry> &ent = ents[e];
    ent.clear();
    const size_t ns = e == 0 ? simple.size() : 0;
    for (size_t qs = 0, qf = 0; qs < ns || qf < fl.size();) {
      const long long cs = qs < ns ? simple[qs].key / 3 : INT64_MAX, cf = qf < fl.size() ? fl[qf].key : INT64_MAX;
      const long long cell = std::min(cs, cf);
      Entry x{(int)cell, {-1, -1, -1}, 0};
      for (; qs < ns && simple[qs].key / 3 == cell; ++qs) {
        x.med[simple[qs].key % 3] = simple[qs].med;
        x.fl |= XF_DEBYE << simple[qs].key % 3;
      }
      for (; qf < fl.size() && fl[qf].key == cell; ++qf) x.fl |= fl[qf].fl;
      ent.push_back(x);
    }
  };
  // kinds of flagged cells: (old class when withOld), Debye media, flags
  using Kind = std::array<int, 5>;
  struct Hash {
    size_t operator()(const Kind &k) const
    {
      uint64_t h = 1469598103934665603ull;
      for (int x : k) h = (h ^ (uint32_t)x) * 1099511628211ull;
      return (size_t)(h ^ h >> 29);
    }
  };
  std::vector<Kind> made[2];
  std::vector<int> of[2];
  auto kinds = [&](int e, bool withOld) {
    const std::vector<uint32_t> &cls = e == 0 ? c->ecls : c->hcls;
    const std::vector<Entry> &ent = ents[e];
    std::unordered_map<Kind, int, Hash> ids;
    made[e].clear();
    of[e].resize(ent.size());
    Kind prev{};
    int prevId = -1;
    for (size_t k = 0; k < ent.size(); ++k) {
      const Kind key{withOld ? (int)cls[ent[k].cell] : 0, ent[k].med[0], ent[k].med[1], ent[k].med[2], (int)ent[k].fl};
      if (prevId < 0 || key != prev) {
        auto it = ids.find(key);
        if (it == ids.end()) {
          it = ids.emplace(key, (int)made[e].size()).first;
          made[e].push_back(key);
        }
        prev = key;
        prevId = it->second;
      }
      of[e][k] = prevId;
    }
  };
  // Coefficient classes are kept when the flagged cells' own fit beside them:
  // with the one-pole sites' media in them, else with those sites as
  // operations.  Without classes every site is one, and a flagged cell's number
  // is its flags'.
  const size_t baseE = c->etab.size() / 6, baseH = c->htab.size() / 3;
  bool indexed = baseE <= 65536 && baseH <= 65536 && !getenv("VGPU_NO_INDEXED_MEDIA");
  auto fits = [&] {
    kinds(0, true);
    kinds(1, true);
    return baseE + made[0].size() <= 65536 && baseH + made[1].size() <= 65536;
  };
  plan(0);
  plan(1);
  if (!(indexed && fits())) {
    for (const Ctx::XSite &s : simple) c->xent[0].push_back({s.key * 4, XO_DEBYE | s.med << 8, 0, 0, 0});
    listed += (long long)simple.size();
    simple.clear();
    sort_by_key(c->xent[0]);
    plan(0);
    indexed = indexed && fits();
    if (!indexed) {
      kinds(0, false);
      kinds(1, false);
    }
  }
  c->indexed = indexed;
  c->debyeSimple = (long long)simple.size();
  c->debyeFast = 0;
  int jhi[3] = {-1, -1, -1};
  for (const Ctx::XSite &s : simple) {
    int n[3];
    geo.unlin(s.key / 3, n);
    c->debyeFast += in_box(c->fastE, n[0], n[1], n[2]);
    for (int a = 0; a < 3; ++a) {
      c->jlo[a] = jhi[a] < 0 ? n[a] : std::min(c->jlo[a], n[a]);
      jhi[a] = std::max(jhi[a], n[a]);
    }
  }
  for (int a = 0; a < 3; ++a) c->jn[a] = jhi[a] < 0 ? 0 : jhi[a] - c->jlo[a] + 1;
  c->debyeSites = listed;
  if (listed > INT32_MAX) return set_error(c, VGPU_EINVAL, "too many Debye sites");
  if (listed) {
    c->d_dlast = dev_alloc(c, (size_t)listed * c->esz);
    c->d_dJ = dev_alloc(c, (size_t)listed * c->debyeMaxPoles * (c->debyeCplx ? 2 : 1) * c->esz);
    if (!c->d_dlast || !c->d_dJ) return fail("Debye state");
  }

  for (int e = 0; e < 2; ++e) {
    const std::vector<Ent> &v = c->xent[e];
    if (v.size() > (1u << 30) - 1) return set_error(c, VGPU_EINVAL, "too many corrections");
    // rows with ghosts behind them go in groups
    struct Src { long long key; size_t q; };  // the value a row changes, or its ghosts' source
    std::vector<Src> by;
    const std::vector<Value> &R = rest[e];
    bool ghosts = false;
    for (size_t q = 0; q < R.size(); ++q) ghosts = ghosts || R[q].ghost;
    std::vector<char> grouped(R.size(), 0);
    if (ghosts) {
      for (size_t q = 0; q < R.size(); ++q) {
        const Ent &x = v[R[q].a];
        by.push_back({(R[q].ghost ? (long long)x.arg * 3 + x.comp() : x.value()) * 2 + R[q].ghost, q});
      }
      sort_by_key(by);
      for (size_t a = 0; a < by.size();) {
        size_t b = a;
        while (b < by.size() && by[b].key / 2 == by[a].key / 2) ++b;
        if (b > a + 1 && !R[by[a].q].ghost)
          for (size_t q = a; q < b; ++q) grouped[by[q].q] = 1;
        a = b;
      }
    }
    // Debye sites alone on their value, component by component; the sites of
    // rows hold the state slots behind theirs
    auto alone = [&](size_t q) { return !grouped[q] && R[q].b == R[q].a + 1 && kind(v[R[q].a]) == XO_DEBYE; };
    std::vector<XSiteDev> site;
    for (int C = 0; C < 3 && e == 0; ++C)
      for (size_t q = 0; q < R.size(); ++q)
        if (alone(q) && v[R[q].a].comp() == C)
          site.push_back({(int)v[R[q].a].cell(), (unsigned)(v[R[q].a].code >> 8) << 2 | (unsigned)C});
    if (e == 0) {
      c->nXsite = (long long)site.size();
      if (!site.empty() && !up(c->d_xsite, site.data(), site.size() * sizeof(XSiteDev))) return fail("Debye sites");
    }
    int slot = (int)site.size();
    std::vector<XRow> row;
    std::vector<XOp<T>> op;
    std::vector<int> gstart;
    row.reserve(upd[e].size() + R.size() - site.size() + 1);
    op.reserve(v.size() - site.size());
    auto take = [&](const Value &r) {
      row.push_back({(int)v[r.a].cell(), (unsigned)op.size() << 2 | (unsigned)v[r.a].comp()});
      for (size_t k = r.a; k < r.b; ++k)
        op.push_back({v[k].code, kind(v[k]) == XO_DEBYE ? slot++ : v[k].arg, T(v[k].a), T(v[k].b)});
    };
    for (const Value &r : upd[e]) take(r);
    c->nXupd[e] = (long long)row.size();
    for (size_t q = 0; q < R.size(); ++q)
      if (!grouped[q] && !alone(q)) take(R[q]);
    c->nXrow[e] = (long long)row.size() - c->nXupd[e];
    for (const Src &s : by)
      if (grouped[s.q]) {
        if (!R[s.q].ghost) gstart.push_back((int)(row.size() - c->nXupd[e]));
        take(R[s.q]);
      }
    c->nXgroup[e] = (long long)gstart.size();
    gstart.push_back((int)(row.size() - c->nXupd[e]));
    row.push_back({0, (unsigned)op.size() << 2});
    if (!up(c->d_xgstart[e], gstart.data(), gstart.size() * sizeof(int)) ||
        !up(c->d_xrow[e], row.data(), row.size() * sizeof(XRow)) || !up(c->d_xop[e], op.data(), op.size() * sizeof(op[0])))
      return fail("rows");
    std::vector<Ent>().swap(c->xent[e]);
    // values evaluated ahead
    c->nXval[e] = (long long)c->xval[e].size();
    if (c->nXval[e]) {
      c->d_xvals[e] = dev_alloc(c, c->xval[e].size() * sizeof(T));
      if (!c->d_xvals[e] || !up(c->d_xval[e], c->xval[e].data(), c->xval[e].size() * sizeof(XVal))) return fail("values");
    }
    std::vector<XVal>().swap(c->xval[e]);

    // classes of the flagged cells: their coefficients, Debye media and flags
    const std::vector<Entry> &ent = ents[e];
    if (ent.empty()) continue;
    if (indexed) {
      std::vector<uint32_t> &cls = e == 0 ? c->ecls : c->hcls;
      std::vector<double> &tab = e == 0 ? c->etab : c->htab;
      const size_t base = e == 0 ? baseE : baseH, w = e == 0 ? 6 : 3;
      for (const Kind &k : made[e])
        for (size_t s = 0; s < w; ++s) tab.push_back(tab[(size_t)k[0] * w + s]);
      for (size_t k = 0; k < ent.size(); ++k) cls[ent[k].cell] = (uint32_t)(base + of[e][k]);
    } else {
      std::vector<uint16_t> f(c->ncell, 0);
      for (size_t k = 0; k < ent.size(); ++k) f[ent[k].cell] = (uint16_t)(e == 0 ? 1 + of[e][k] : ent[k].fl);
      if (!up(c->d_xcls[e], f.data(), f.size() * sizeof(uint16_t))) return fail("flags");
    }
    if (e == 1) {
      c->xflagH = true;
      c->hflags.assign(baseH, 0.0);
      if (indexed)
        for (const Kind &k : made[e]) c->hflags.push_back((double)k[4]);
      continue;
    }
    c->xflag0 = indexed ? (unsigned)baseE : 1u;
    std::vector<T> dt(made[e].size() * DTAB_STRIDE, T(0));
    for (size_t k = 0; k < made[e].size(); ++k) {
      for (int C = 0; C < 3; ++C)
        if (made[e][k][1 + C] >= 0) {
          dt[k * DTAB_STRIDE + 2 * C] = T(c->dhost[0][made[e][k][1 + C]]);
          dt[k * DTAB_STRIDE + 2 * C + 1] = T(c->dhost[1][made[e][k][1 + C]]);
        }
      dt[k * DTAB_STRIDE + 6] = T(made[e][k][4]);
    }
    if (!up(c->d_xdtab, dt.data(), dt.size() * sizeof(T))) return fail("class table");
    if (!simple.empty() && !(c->d_xJ = dev_alloc(c, (size_t)c->jn[0] * c->jn[1] * c->jn[2] * 3 * sizeof(T))))
      return fail("Debye state");
  }
  return VGPU_OK;
}

}  // namespace vgpu
