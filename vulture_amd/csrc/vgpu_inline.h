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

  explicit InlineGeom(Ctx *ctx) : c(ctx)
  {
    fill_volume_args<T>(ctx, ea, ha, 0);
    for (int C = 0; C < 3; ++C)
      for (int q = 0; q < 6; ++q) ein[C][0][q] = ea.in[C][q];
    // ghost planes as launch_ghosts copies them (surface.c:569-812)
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

template <typename T> int build_inline(Ctx *c)
{
  if (!c->inl) return VGPU_OK;
  using Ent = Ctx::XEnt;
  const InlineGeom<T> geo(c);
  auto fail = [&](const char *what) { return set_error(c, VGPU_ENOMEM, "corrections: %s", what); };
  auto up = [&](void *&d, const void *h, size_t bytes) {
    d = dev_alloc(c, bytes);
    return d && (bytes == 0 || hipMemcpy(d, h, bytes, hipMemcpyHostToDevice) == hipSuccess);
  };
  auto less = [](const Ent &a, const Ent &b) {
    if (a.cell != b.cell) return a.cell < b.cell;
    if (a.comp != b.comp) return a.comp < b.comp;
    if (a.order != b.order) return a.order < b.order;
    return a.seq < b.seq;
  };
  auto same = [](const Ent &a, const Ent &b) { return a.cell == b.cell && a.comp == b.comp; };

  // Mur faces: each E value on one is written by the thread of its inner
  // neighbour when that takes the ordinary update; else the whole context
  // keeps Mur's own launch before the sweep
  struct Mur { long long cell; unsigned fl; };  // a neighbour, its flag of one face and component
  std::vector<Mur> mur;
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
            mur.push_back({c->lin(nb[0], nb[1], nb[2]), (unsigned)XF_MUR << (2 * f + (C - a + 5) % 3)});
          }
    }
  if (!c->murPush) mur.clear();
  std::sort(mur.begin(), mur.end(), [](const Mur &a, const Mur &b) { return a.cell < b.cell; });

  // E operations but Debye, then the Debye sites: one one-pole site alone on a
  // swept value goes to the class table, others are listed
  auto tidy = [&](int e) {
    std::vector<Ent> &v = c->xent[e];
    std::sort(v.begin(), v.end(), less);
    v.erase(std::unique(v.begin(), v.end(),
                        [&](const Ent &a, const Ent &b) {
                          return same(a, b) && (a.code & 7) == XO_ZERO && (b.code & 7) == XO_ZERO;
                        }),
            v.end());
    // a ghost value takes its source's: what else would change it is lost
    v.erase(std::remove_if(v.begin(), v.end(),
                           [&](const Ent &a) {
                             int n[3];
                             geo.unlin(a.cell, n);
                             return geo.ghost_dst(3 * e + a.comp, n);
                           }),
            v.end());
  };
  tidy(0);
  tidy(1);
  struct Simple { long long cell; int comp, med; };
  std::vector<Simple> simple;
  long long listed = 0;
  {
    std::vector<Ctx::XSite> &st = c->xsite;
    std::stable_sort(st.begin(), st.end(), [](const Ctx::XSite &a, const Ctx::XSite &b) {
      return a.cell != b.cell ? a.cell < b.cell : a.comp < b.comp;
    });
    std::vector<Ent> add;
    const std::vector<Ent> &v = c->xent[0];
    size_t q = 0;
    simple.reserve(st.size());
    for (size_t a = 0; a < st.size();) {
      size_t b = a;
      while (b < st.size() && st[b].cell == st[a].cell && st[b].comp == st[a].comp) ++b;
      while (q < v.size() && (v[q].cell < st[a].cell || (v[q].cell == st[a].cell && v[q].comp < st[a].comp))) ++q;
      const bool rows = q < v.size() && v[q].cell == st[a].cell && v[q].comp == st[a].comp;
      int n[3];
      geo.unlin(st[a].cell, n);
      if (!geo.ghost_dst(st[a].comp, n)) {
        const int m = st[a].med;
        if (b == a + 1 && !rows && c->dsimple[m] && geo.region(st[a].comp, n) >= 0) {
          simple.push_back({st[a].cell, st[a].comp, m});
        } else {
          for (size_t k = a; k < b; ++k) {
            if (st[k].med >= 1 << 21) return set_error(c, VGPU_EINVAL, "Debye site index out of range");
            add.push_back({st[k].cell, (long long)k, st[k].comp, 0, XO_DEBYE | st[k].med << 8, (int)listed++, 0, 0});
          }
        }
      }
      a = b;
    }
    std::vector<Ctx::XSite>().swap(st);
    c->xent[0].insert(c->xent[0].end(), add.begin(), add.end());
    std::sort(c->xent[0].begin(), c->xent[0].end(), less);
  }
  // zeroed E of swept values, when nothing comes before: a flag of the class
  struct Zero { long long cell; int comp; };
  std::vector<Zero> zero;
  {
    std::vector<Ent> &v = c->xent[0];
    std::vector<Ent> keep;
    keep.reserve(v.size());
    for (size_t a = 0; a < v.size(); ++a) {
      int n[3];
      geo.unlin(v[a].cell, n);
      if ((v[a].code & 7) == XO_ZERO && (a == 0 || !same(v[a - 1], v[a])) && geo.region(v[a].comp, n) >= 0)
        zero.push_back({v[a].cell, v[a].comp});
      else keep.push_back(v[a]);
    }
    v.swap(keep);
  }
  // ghosts of every value that changes
  for (int e = 0; e < 2; ++e) {
    std::vector<Ent> add;
    const std::vector<Ent> &v = c->xent[e];
    const int N[3] = {c->NX, c->NY, c->NZ};
    for (int C = 0; C < 3; ++C) {
      const auto &gs = geo.ghosts[3 * e + C];
      for (size_t g = 0; g < gs.size(); ++g) {
        int lo[3] = {0, 0, 0}, hi[3] = {N[0] - 1, N[1] - 1, N[2] - 1}, n[3];
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
              const long long cell = c->lin(n[0], n[1], n[2]), src = c->lin(s[0], s[1], s[2]);
              const Ent key{src, -1, C, -1, 0, 0, 0, 0};
              auto it = std::lower_bound(v.begin(), v.end(), key, less);
              if (geo.region(3 * e + C, s) < 0 && !(e == 0 && geo.mur_face(C, s, nb) >= 0) &&
                  !(it != v.end() && it->cell == src && it->comp == C))
                continue;
              add.push_back({cell, 0, C, 3, XO_GHOST, (int)src, sign, 0});
            }
      }
    }
    c->xent[e].insert(c->xent[e].end(), add.begin(), add.end());
    std::sort(c->xent[e].begin(), c->xent[e].end(), less);
  }

  // the cells the E sweep corrects in line, in cell order
  struct Entry { int cell; int med[3]; unsigned fl; };
  std::vector<Entry> ent;
  auto plan = [&] {
    ent.clear();
    size_t qs = 0, qz = 0, qm = 0;
    for (;;) {
      long long cell = INT64_MAX;
      if (qs < simple.size()) cell = std::min(cell, simple[qs].cell);
      if (qz < zero.size()) cell = std::min(cell, zero[qz].cell);
      if (qm < mur.size()) cell = std::min(cell, mur[qm].cell);
      if (cell == INT64_MAX) break;
      Entry x{(int)cell, {-1, -1, -1}, 0};
      for (; qs < simple.size() && simple[qs].cell == cell; ++qs) {
        x.med[simple[qs].comp] = simple[qs].med;
        x.fl |= XF_DEBYE << simple[qs].comp;
      }
      for (; qz < zero.size() && zero[qz].cell == cell; ++qz) x.fl |= XF_ZERO << zero[qz].comp;
      for (; qm < mur.size() && mur[qm].cell == cell; ++qm) x.fl |= mur[qm].fl;
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
  std::vector<Kind> made;
  std::vector<int> of;
  auto kinds = [&](bool withOld) {
    std::unordered_map<Kind, int, Hash> ids;
    made.clear();
    of.resize(ent.size());
    Kind prev{};
    int prevId = -1;
    for (size_t k = 0; k < ent.size(); ++k) {
      const Kind key{withOld ? (int)c->ecls[ent[k].cell] : 0, ent[k].med[0], ent[k].med[1], ent[k].med[2], (int)ent[k].fl};
      if (prevId < 0 || key != prev) {
        auto it = ids.find(key);
        if (it == ids.end()) {
          it = ids.emplace(key, (int)made.size()).first;
          made.push_back(key);
        }
        prev = key;
        prevId = it->second;
      }
      of[k] = prevId;
    }
  };
  // Coefficient classes are kept when the flagged cells' own fit beside them:
  // with the one-pole sites' media in them, else with those sites in rows.
  // Without classes every site is in a row, and a flagged cell's number is
  // its flags'.
  const size_t baseE = c->etab.size() / 6;
  bool indexed = baseE <= 65536 && c->htab.size() / 3 <= 65536 && !getenv("VGPU_NO_INDEXED_MEDIA");
  auto fits = [&] {
    kinds(true);
    return baseE + made.size() <= 65536;
  };
  plan();
  if (!(indexed && fits())) {
    long long seq = 0;
    for (const Simple &s : simple)
      c->xent[0].push_back({s.cell, seq++, s.comp, 0, XO_DEBYE | s.med << 8, (int)listed++, 0, 0});
    simple.clear();
    std::sort(c->xent[0].begin(), c->xent[0].end(), less);
    plan();
    indexed = indexed && fits();
    if (!indexed) kinds(false);
  }
  c->indexed = indexed;
  c->debyeSimple = (long long)simple.size();
  c->debyeSites = listed;
  if (listed) {
    c->d_dlast = dev_alloc(c, (size_t)listed * c->esz);
    c->d_dJ = dev_alloc(c, (size_t)listed * c->debyeMaxPoles * (c->debyeCplx ? 2 : 1) * c->esz);
    if (!c->d_dlast || !c->d_dJ) return fail("Debye state");
  }

  // rows, those with ghosts behind them in groups
  for (int e = 0; e < 2; ++e) {
    const std::vector<Ent> &v = c->xent[e];
    if (v.size() > (1u << 30) - 1) return set_error(c, VGPU_EINVAL, "too many corrections");
    struct Row { long long src; int ghost; size_t a, b; };  // src: value the row changes, or its ghosts' source
    std::vector<Row> R;
    for (size_t a = 0; a < v.size();) {
      size_t b = a;
      while (b < v.size() && same(v[b], v[a])) ++b;
      const bool g = (v[a].code & 7) == XO_GHOST;
      R.push_back({(g ? v[a].arg : v[a].cell) * 3 + v[a].comp, g, a, b});
      a = b;
    }
    std::vector<size_t> by(R.size());
    for (size_t q = 0; q < by.size(); ++q) by[q] = q;
    std::sort(by.begin(), by.end(), [&](size_t a, size_t b) {
      return R[a].src != R[b].src ? R[a].src < R[b].src : R[a].ghost != R[b].ghost ? R[a].ghost < R[b].ghost : a < b;
    });
    std::vector<char> grouped(R.size(), 0);
    for (size_t a = 0; a < by.size();) {
      size_t b = a;
      while (b < by.size() && R[by[b]].src == R[by[a]].src) ++b;
      if (b > a + 1 && !R[by[a]].ghost)
        for (size_t q = a; q < b; ++q) grouped[by[q]] = 1;
      a = b;
    }
    std::vector<XRow> row;
    std::vector<XOp<T>> op;
    std::vector<int> gstart;
    row.reserve(R.size() + 1);
    op.reserve(v.size());
    auto take = [&](const Row &r) {
      row.push_back({(int)v[r.a].cell, (unsigned)op.size() << 2 | (unsigned)v[r.a].comp});
      for (size_t k = r.a; k < r.b; ++k) op.push_back({v[k].code, v[k].arg, T(v[k].a), T(v[k].b)});
    };
    for (size_t q = 0; q < R.size(); ++q)
      if (!grouped[q]) take(R[q]);
    c->nXrow[e] = (long long)row.size();
    for (size_t q = 0; q < by.size(); ++q)
      if (grouped[by[q]]) {
        if (!R[by[q]].ghost) gstart.push_back((int)row.size());
        take(R[by[q]]);
      }
    c->nXgroup[e] = (long long)gstart.size();
    gstart.push_back((int)row.size());
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
  }
  if (ent.empty()) return VGPU_OK;

  if (!simple.empty() && !(c->d_xJ = dev_alloc(c, 3 * c->ncell * sizeof(T)))) return fail("Debye state");
  // classes of the flagged cells: their coefficients, Debye media and flags
  c->xflag0 = indexed ? (unsigned)baseE : 1u;
  if (indexed) {
    for (const Kind &k : made)
      for (int s = 0; s < 6; ++s) c->etab.push_back(c->etab[(size_t)k[0] * 6 + s]);
    for (size_t k = 0; k < ent.size(); ++k) c->ecls[ent[k].cell] = (uint32_t)(baseE + of[k]);
  } else {
    std::vector<uint16_t> f(c->ncell, 0);
    for (size_t k = 0; k < ent.size(); ++k) f[ent[k].cell] = (uint16_t)(1 + of[k]);
    if (!up(c->d_xcls, f.data(), f.size() * sizeof(uint16_t))) return fail("flags");
  }
  std::vector<T> dt(made.size() * DTAB_STRIDE, T(0));
  for (size_t k = 0; k < made.size(); ++k) {
    for (int C = 0; C < 3; ++C)
      if (made[k][1 + C] >= 0) {
        dt[k * DTAB_STRIDE + 2 * C] = T(c->dhost[0][made[k][1 + C]]);
        dt[k * DTAB_STRIDE + 2 * C + 1] = T(c->dhost[1][made[k][1 + C]]);
      }
    dt[k * DTAB_STRIDE + 6] = T(made[k][4]);
  }
  if (!up(c->d_xdtab, dt.data(), dt.size() * sizeof(T))) return fail("class table");
  return VGPU_OK;
}

}  // namespace vgpu
