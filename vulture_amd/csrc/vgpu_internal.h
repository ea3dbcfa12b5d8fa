// Internal declarations of the MI355X FDTD core library (not part of the C-ABI).
//
// Device layout: every 3-D array is x-fastest, index (k*NY + j)*PX + i, with
// PX the x extent rounded up to 128 bytes so rows start on cache-line
// boundaries.  Extents NX,NY,NZ are the reference's allocation extents
// (gobox plus one ghost layer each side), so grid indices i,j,k are the
// reference's own.
//
// With the fused leapfrog sweep the fields are held twice.  A step reads the
// fields of step n from one set and writes those of step n+1 to the other
// (the sweeps, Mur E); the corrections after each sweep (Debye, SIBC,
// sources, TF/SF, ghosts) then modify the new set in place.  Nothing a
// kernel reads from the old set is written during the step, so a sweep may
// recompute a neighbour's new value from the old fields at any time, in any
// block, without racing the block that stores it.  The separate sweeps
// update one set in place, as the reference does.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstddef>
#include <string>
#include <mutex>
#include <vector>
#include "vgpu.h"

namespace vgpu {

// ---- kernel argument blocks (passed by value) ----

struct WaveformDev;
struct PwDev;

// Full argument block of the E sweep, kept in device memory and read through
// a pointer by the shell blocks.
template <typename T> struct EArgs {
  int NX, NY, NZ, PX;
  long long plane;
  T *E[3];               // new E (written)
  const T *Ein[3];       // old E (read)
  const T *H[3];         // old H
  const T *alpha[3], *beta[3];
  const T *idh[3];
  int in[3][6];          // inner-grid limits per E component
  unsigned pmlmask;
  int pl[6][3][6];       // UPML slab limits [region][component][face]
  T *PP[6][3], *P[6][3]; // UPML auxiliaries, x-fastest within each slab box
  T *PPpool, *Ppool;     // the pools holding them (same layout: a slab is at the same offset in both)
  const T *ad[3], *bd[3], *ah[3], *ibh[3];
  // coefficient classes: per-cell class, [class][8] alpha/beta (6 used)
  const uint16_t *ecls;
  const T *etab;
  unsigned *vis[3];      // update-once check: visit counts per component (null in ordinary runs)
};

template <typename T> struct HArgs {
  int NX, NY, NZ, PX;
  long long plane;
  T *H[3];               // new H (written)
  const T *Hin[3];       // old H (read)
  const T *E[3];         // new E
  const T *gamma[3];
  const T *ide[3];
  int in[3][3][6];       // ordinary-update boxes per H component (inner grid, two Mur faces)
  unsigned pmlmask;
  int pl[6][3][6];
  T *B[6][3];
  T *Bpool;              // the pool holding the B slabs
  const T *ad[3], *ah[3], *bh[3], *ibd[3];
  const uint16_t *hcls;  // coefficient classes: per-cell class, [class][4] gamma (3 used)
  const T *htab;
  unsigned *vis[3];      // update-once check (null in ordinary runs)
};

// ---- corrections ----
//
// The updates that follow a sweep (Debye sites, SIBC edges and faces, sources,
// TF/SF, ghost planes) each change single field values and read no field but
// that value, or a ghost's source.  Two forms:
//
//  - In line: the thread that sweeps a cell applies them right after its
//    update, with no second pass over the field.  This takes what needs no
//    look-up chain: a single one-pole Debye site per value (its alpha and beta
//    in the class table, its J in a dense array over the sites' box, its
//    previous E the old E the sweep has in a register), an E to zero (SIBC), and Mur's E, which the
//    thread of the face's inner neighbour writes, having both of that
//    neighbour's values Mur's equation takes.  Such cells have coefficient
//    classes of their own (from `flag0` on), so the others pay one comparison.
//  - Update rows, for the other operations on values of the ordinary update
//    (TF/SF faces, sources, SIBC's H terms): the sweep leaves the value alone
//    (a flag of the cell's class) and a thread of its own, in blocks beside
//    the sweep's, makes the whole update and then the value's operations in
//    the reference's order.  An update reads no value of its own kind but its
//    own, so this needs no order between them.  (Operations walked by the
//    sweep's threads measured slower: each costs four dependent loads, one
//    lane of a wavefront at a time at the x faces.)
//  - Rows, for what is left (ghost planes, values that are not ordinary
//    updates): a launch after the sweep, a thread per value, ghosts behind the
//    row of their source.  Debye sites alone on their value (of several poles,
//    or without classes) have a list of their own in it.
enum XKind { XO_SRC, XO_AUX, XO_WAVE, XO_ZERO, XO_DEBYE, XO_GHOST, XO_SIBC };
// flags of a flagged class (E: dtab slot 6, H: the class table's slot 3):
// one-pole Debye sites of components 0-2 (bits 0-2), zeroed components (3-5),
// components left to update rows (6-8), and per Mur face f the components
// (f/2 + 1) % 3 and (f/2 + 2) % 3 it takes from the cell (bits 9+2f, 10+2f)
enum XFlag { XF_DEBYE = 1, XF_ZERO = 8, XF_SKIP = 64, XF_MUR = 512, XF_MUR_SHIFT = 9 };
constexpr int DTAB_STRIDE = 8;

// code: kind (bits 0-2), then
//   SRC:   density (3), soft (4); arg value
//   AUX:   incident component (3-5), negative sign (6), plane wave (8-); arg aux cell, a dp, b inverse edge length
//   WAVE:  negative sign (6); arg value, b inverse edge length
//   DEBYE: medium (8-); arg site
//   GHOST: arg source cell, a sign
//   SIBC:  SibcHEnt's bits (3-); arg face, a/b the two inverse edge lengths
template <typename T> struct XOp {
  int code, arg;
  T a, b;
};

struct XRow {
  int cell;
  unsigned opc;          // first operation << 2 | component
};

// A Debye site that is its value's only operation: what a row would have to
// look up -- its one operation, where that ends -- is known.
struct XSiteDev {
  int cell;
  unsigned mc;           // medium << 2 | component
};

// A value of the incident field or of a source at one time: scale *
// wf_value(t) in double, rounded once (a source), or its two factors rounded
// first, the time less `geo` (an analytic plane wave's, at one edge).
struct XVal {
  double geo, delay, scale;
  int wf, wave;
};

template <typename T> struct XArgs {
  unsigned flag0;        // first flagged class (E)
  const uint16_t *cls;   // per cell: class, or without classes E 0 / 1 + dtab row, H its flags
  const T *dtab;         // [class - flag0][8]: alpha, beta of J per component, flags
  T *J;                  // [cell of the one-pole sites' box][component], from the box's would-be cell (0, 0, 0)
  int PX;
  long long plane;
  T mzeta[6];            // Mur factors
  long long nupd, nrow, ngroup;  // update rows, rows, then groups of rows (a row and its ghosts)
  const int *gstart;     // first row of each group
  const XRow *row;
  const XOp<T> *op;
  T *F[3];               // the half-step's fields
  const T *G[3], *il[3]; // the other fields, the inverse lengths of the update
  const T *tab;          // class table (null: per-cell arrays)
  const T *ca[3], *cb[3];  // alpha and beta, or gamma in cb
  const T *val;          // source and analytic incident values
  const T *aux;          // aux grids [pw][2][auxmax]
  int auxmax;
  const PwDev *pw;
  T eta0;
  T *dlast, *dJ;         // Debye sites of rows
  long long dstride;
  const double *dalpha, *dbeta;
  const int *dnp;
  int dmaxP, dcplx;
  const T *Etan;
  long long nsite;       // sites alone on their value (E); they hold the first state slots
  const XSiteDev *site;
  int jrow, jplane;      // the one-pole sites' box: cells a row and a plane
  int jfirst, jlast;     // the places of its first and last cell
};

// Values of a half-step's sources and analytic plane waves, evaluated ahead
// of it at t = (n + half) * dt.
template <typename T> struct ValArgs {
  long long n;
  const XVal *v;
  T *out;
  const WaveformDev *wf;
  double half;
};

// Lean by-value arguments of the fast sweep kernels.
template <typename T> struct FastE {
  int NX, NY, NZ, PX;
  long long plane;
  int box[6];            // fast box (every E component inner-grid)
  int kchunk, nchx;      // planes per block; 64-cell x chunks from box[0]
  int gy, gz;            // y blocks, z chunks
  int per;               // blocks of a z chunk per XCD
  T *E[3];               // new E (written)
  const T *Ein[3];       // old E
  const T *H[3];         // old H
  const T *idh[3];
  const uint16_t *ecls;  // coefficient classes
  const T *etab;
  const T *alpha[3], *beta[3];  // per-cell arrays when there are no classes
  unsigned *vis[3];      // update-once check (null in ordinary runs)
};

template <typename T> struct FastH {
  int NX, NY, NZ, PX;
  long long plane;
  int box[6];
  int kchunk, nchx;
  int gy, gz, per;
  T *H[3];               // new H (written)
  const T *Hin[3];       // old H
  const T *E[3];         // new E
  const T *ide[3];
  const uint16_t *hcls;
  const T *htab;
  const T *gamma[3];
  unsigned *vis[3];      // update-once check (null in ordinary runs)
};

// Fused leapfrog sweep over the fused box (E and H of every cell inside take
// the ordinary update).  A wave owns a tile of 63 x-cells by R rows and
// marches over kz planes; it computes E on 64 x 1+R cells per plane (its
// tile and the x and y neighbours its H needs) and H of the plane below.
template <typename T> struct LeapArgs {
  int NX, NY, NZ, PX;
  long long plane;
  int box[6];            // fused box
  int ntx, ngy, ntz, kz; // x tiles (63 cells), y tiles (4 waves of R rows per block), z chunks of kz planes
  T *E[3];               // new E, H (written)
  T *H[3];
  const T *Ein[3];       // old E, H
  const T *Hin[3];
  const T *idh[3], *ide[3];
  const uint16_t *ecls, *hcls;  // coefficient classes
  const T *etab, *htab;
  const T *alpha[3], *beta[3], *gamma[3];  // per-cell arrays when there are no classes
  int discard;           // first element of the discard area past every field array's cells
  unsigned *vis[6];      // update-once check (null in ordinary runs)
};

// Elements past the cells of every field array that the fused sweep writes
// the values of cells a lane does not own to (never read).
constexpr int FIELD_DISCARD = 65536;

// H cells of the fused box whose new value the fused sweep cannot give
// (an E input of theirs is corrected after the sweep -- a Debye site, a
// source or TF/SF row, an SIBC face -- or is not an ordinary update): one
// 64-cell x chunk of one row per entry, with a mask of its cells.  They are
// updated again after the E corrections, from the old H and the final E.
struct FixEnt {
  int i0, j, k, pad_;    // first cell of the chunk
  unsigned long long mask;  // cells i0 + lane to update
};
template <typename T> struct FixArgs {
  long long n;
  const FixEnt *ent;
  int NY, PX;
  long long plane;
  T *H[3];
  const T *Hin[3];
  const T *E[3];
  const T *ide[3];
  const uint16_t *hcls;
  const T *htab;
  const T *gamma[3];
};

// A piece of a sweep's shell (the cells outside its fast box): a box whose
// rows share, per component, one sequence of x runs, each run one region
// (ordinary update or one UPML slab) over a range of x.  A block covers 256
// consecutive cells of the piece's x-y plane (x fastest) and marches over
// `kc` planes; block b of the piece is x-y block b % nxyb of z chunk
// b / nxyb.
constexpr int SHELL_RUNS = 4;
constexpr int SHELL_KC = 4;  // planes a shell thread marches over
struct ShellRun {
  int xa, xb;            // inclusive x range
  int reg, pad_;         // 6 ordinary, 0..5 UPML slab
  long long p0;          // UPML: slab index of (xa, box[2], box[4])
  long long psy, psz;    // slab index strides of j and k (1 for i)
  void *a, *b;           // UPML auxiliaries of the slab: E sweep PP and P, H sweep B
};
struct ShellPiece {
  int box[6];            // inclusive cell limits
  int ni, nj, nk, cells; // extents, cell count
  int nxy, nxyb, kc, nblk;  // x-y plane lanes (nip per row), its 256-lane blocks, planes per block, blocks
  int nrun[3];           // runs per component (cells outside every run are not updated)
  int nip, xo;           // lanes per row (a whole number of 128-byte lines) and the row's first cell's lane
  int pad_;
  ShellRun run[3][SHELL_RUNS];
};

// A piece as the kernels read it: everything a block needs in consecutive
// words, so one batch of scalar loads brings it, in place of one load after
// another along the runs.  A run's q0 is its element offset in the
// auxiliaries' pools at x = 0, row 0, plane 0 of the piece; a run past the
// component's last has xa > xb.
struct ShellDevRun {
  int xa, xb, reg, q0, psy, psz;
};
struct ShellDev {
  int x0, y0, z0, ni, nip, xo, nxy, nxyb, kc, nk;
  int pad_[2];
  ShellDevRun run[3][SHELL_RUNS];
};

// One block of a shell launch: its piece and the piece's block (piece < 0:
// nothing to do).
struct ShellWork {
  int piece, block;
};

// Mur tangential-E faces (mur.c:135-395): one box per (face, component).
template <typename T> struct MurArgs {
  int NX, NY, PX;
  long long plane;
  T *E[3];               // new E (written on the face)
  const T *Ein[3];       // old E
  const T *H[3];         // old H
  const T *alpha[3], *beta[3];
  const T *idh[3];
  int box[12][6];        // limits of face f component slot s at [2f+s]
  int comp[12];          // component of each slot (-1 unused)
  T zeta[6];
  const uint16_t *ecls;  // coefficient classes (null: read the per-cell alpha/beta arrays)
  const T *etab;
  unsigned *vis[3];      // update-once check (null in ordinary runs)
};

// Debye sites of one layer (debye.c:243-307): a layer holds at most one site
// per E cell, layers run in block order.
template <typename T> struct DebyeArgs {
  long long n;           // sites in this layer
  const long long *key;  // per site: medium << 42 | device linear index << 2 | component
  const T *sbeta;        // per site: beta of the site's edge
  T *E[3];
  T *lastE;              // per site
  T *J;                  // [pole][site] (real poles) or [pole][site][2]
  long long stride;      // sites in the whole state block (J pole stride)
  long long base;        // first site of this layer in the state block
  const double *dalpha, *dbeta;  // [medium][maxPoles][2]
  const int *npoles;     // [medium]
  int maxPoles;
  int cplx;
};

// A block of the SIBC E launch: up to SIBC_FACES faces of one surface, so the
// surface, its filters and its matrices are uniform across the block.
struct SibcBlock {
  int surf, pad_;
  long long f0, f1;      // first face of the block, end of the surface's faces
};

// SIBC faces (sibc.c:443-586): per-face geometry, per-surface constants.
template <typename T> struct SibcEArgs {
  long long nfaces;
  const SibcBlock *blocks;
  const int *ijk;        // [face][3]
  const int *surf;       // [face]
  const unsigned char *adjA, *adjB;  // [face][4]
  const int *normal;     // [surface]
  const double *A, *B;   // [surface][16]
  const int *filtset;    // [surface] -> filter set
  const int *npoles;     // [set][16]
  const double *asymp;   // [set][16]
  const double *q;       // [set][16][maxPoles][3][2]
  int maxPoles;
  int real;              // all coefficients real: zeta holds real states only
  int factored;          // one state per (input, pole): zeta [(input*maxPoles + pole)][face]
  const int *fbase;      // factored: [set][input] filter whose coefficients drive the input's states, or -1
  const double *fratio;  // factored: [set][16][maxPoles] each filter's residue over its base filter's
  double *zeta;          // [(filter*maxPoles + pole)][face][2], or [..][face] when real
  double *old;           // [input][face]: the previous step's filter input
  T *Etan;               // [face][4]
  T *E[3];
  const T *H[3];
  int NY, PX;
  long long plane;
};

// Gathered SIBC H corrections (sibc.c:616-776): one row per touched H cell,
// entries in the reference's application order.
// Device form (16 bytes).  bits: kind (bit 0: 0 edge term, 1 parallel-
// adjacent term), Etan slots ea (bits 1-2) and eb (3-4), negative sign (5),
// full edge weight (6: weight 1, else 1/2 = 0.5*(1 + PMC edge)), !isAdjA
// (7), !isAdjB (8), axis of the inverse lengths (9-10); ia/ib index the
// inverse primary edge lengths of that axis.
struct SibcHEnt {
  int face;
  int bits;
  int ia, ib;
};

template <typename T> struct SibcHArgs {
  long long nrows;
  const long long *rowkey;   // cell << 3 | zero << 2 | component; zero: normal H of a face, set to 0
  const int *rowstart;   // [nrows+1]
  const T *rowg;         // the row cell's gamma
  const SibcHEnt *ent;
  const T *Etan;
  T *H[3];
  const T *ide[3];
};

// Sources and TF/SF corrections applied after the volume update, one row
// per touched cell, entries in reference order (sources first, then plane
// waves face by face, planewave.c:576-1007, source.c:602-753).
struct CorrEntry {
  int kind;              // 0 field source, 1 density source, 2 TF/SF aux grid, 3 TF/SF analytic
  int idx;               // source or plane-wave index
  int inc;               // incident field component (TF/SF)
  int auxid;             // floor(d) (aux grid)
  double sign;           // TF/SF sign
  double il;             // inverse edge length (TF/SF)
  double geo;            // dp (aux grid) or d/v (analytic)
};

// Device form of a correction entry (24 bytes).  code: kind (bits 0-1),
// incident component (bits 2-4), negative sign (bit 5), source or plane-wave
// index (bits 8-31).
struct CorrEnt {
  int code;
  int auxid;
  double geo;            // dp (aux grid) or d/v (analytic)
  double il;             // inverse edge length (TF/SF)
};

struct WaveformDev {
  int type;
  double size, delay, width, frequency;
  const double *table;   // [n][3]
  unsigned long n;
};

struct SourceDev {
  int kind, soft, waveform;
  double size, delay;
};

struct PwDev {
  double Finc[6];
  int waveform;
  double delay;
  int use_aux, nx, xb;
  double beta, gamma;
};

template <typename T> struct CorrArgs {
  long long nrows;
  const long long *rowkey;   // cell << 2 | component, ascending
  const int *rowstart;
  const CorrEnt *ent;
  const T *rowcoef;      // the row cell's beta (E) or gamma (H)
  const T *rowalpha;     // the row cell's alpha (E only)
  T *F[3];               // E or H components
  int electric;
  const unsigned long long *step;  // device step counter: n = *step + soff
  int soff;
  double dt, half;       // t = (n + half) * dt: timeE (half 0) or timeH (half 0.5)
  const WaveformDev *wf;
  const SourceDev *src;
  const PwDev *pw;
  const T *aux;          // aux grids [pw][2][auxmax]: Eyi then Hzi
  int auxmax;
  double eta0;
};

template <typename T> struct AuxArgs {
  int npw;
  const PwDev *pw;
  T *aux;                // [pw][2][auxmax]
  T *pml;                // [pw][3][10]: PPyi, Pyi, Bzi
  const T *prof;         // [pw][4][10]: adx, bdx, ahx, bhx
  int auxmax;
  const WaveformDev *wf;
  const unsigned long long *step;  // t = (*step + soff) * dt (timeE)
  int soff;
  double dt;
};

// Point observers and DFT (observer.c:622-650, 857-899).
template <typename T> struct ObsArgs {
  int nobs;
  const long long *cell; // [obs]
  const unsigned long long *first, *last;
  const int *nfreq;
  const long long *dftoff;   // offset of the observer's [6][nfreq] block
  const double *omega;       // concatenated per observer
  double *td;                // [obs][nsteps][6]
  unsigned long long tdsteps;
  double *dre, *dim;
  const T *F[6];
  const unsigned long long *step;  // n = *step + soff, t = n * dt
  int soff;
  double dt;
};

template <typename T> struct VolObsArgs {
  const long long *nodecell; // [node] for all volume observers
  const int *nodeobs;
  long long nnodes;
  const unsigned long long *first, *last;
  float *stage;              // [row][node][6], row = step modulo ring
  const T *F[6];
  const unsigned long long *step;  // n = *step + soff
  int soff;
  unsigned long long ring;   // staging rows: two runs' worth
};

// What rides along with a half-step's sweep, in blocks of its own: things the
// sweep neither reads nor writes: its update rows; in the E sweep the H half
// of the observers' samples of its step, the aux grids' E update and the values
// of its step's H sources and analytic waves; in the H sweep the E half of the
// next step's samples and the next step's E values -- E is final then -- and the
// aux grids' H update.  A run's first E samples and values have a launch of
// their own before it, and its last step takes none.
template <typename T> struct SideArgs {
  ObsArgs<T> o;
  VolObsArgs<T> v;
  AuxArgs<T> x;
  ValArgs<T> val;
  int electric;          // rides with the E sweep
  int nfb;               // 256-frequency blocks per observer
  int b[5];              // first block past the observers, volume samples, values, aux grids, update rows
};

// ---- packed launches over several solves (vgpu_run_group) ----

constexpr int PACK_MAX = VGPU_GROUP_MAX;  // solves in one group run

// The end of a group run, one launch over its solves: the step counters, and
// the run's rows of volume samples (8-byte pairs: n of them, from `at` on in
// a ring of `ring`) to their place in pinned host memory.
struct GroupClose {
  int n;
  unsigned start[PACK_MAX + 1];  // first block of each solve; start[n] is the grid
  unsigned long long by, *step[PACK_MAX];
  const double *src[PACK_MAX];
  double *dst[PACK_MAX];
  long long at[PACK_MAX], pairs[PACK_MAX], ring[PACK_MAX];
};

// One solve's by-value argument blocks for the packed launches, for field set
// 0 (the one the separate sweeps read and write), kept in device memory.  A
// packed launch passes the step offset itself.
template <typename T> struct PackArgs {
  FastE<T> fe;
  FastH<T> fh;
  const ShellDev *epc, *hpc;
  const ShellWork *ewk, *hwk;
  const EArgs<T> *ea;
  const HArgs<T> *ha;
  const XArgs<T> *xe, *xh;  // corrections
  unsigned nEside, nHside, nEshell, nHshell;  // blocks
  SideArgs<T> se, sh;
};

// Argument of a packed launch: the solves it covers, in launch order, and
// the first launch block (or block row) of each: solve d owns blocks
// start[d] .. start[d+1]-1 and runs them as its own launch would run blocks
// 0 .. start[d+1]-start[d]-1.
struct PackMap {
  int n;                         // solves in this launch
  int soff, last;                // step offset within the run, its last step
  unsigned start[PACK_MAX + 1];
  const void *args[PACK_MAX];    // each solve's PackArgs
};

template <typename T> struct GhostArgs {
  int NX, NY, NZ, PX;
  long long plane;
  T *F;
  int axis, dst, src;
  T sign;
  int lo[3], hi[3];
};

// ---- context ----

struct Region { int lim[6]; };

// Fast boxes of the two sweeps: where every E (H) component takes the
// ordinary update (the intersection of the inner-grid limits gfilim), kept
// one cell inside the allocation so the fast kernels never test bounds.
// With lw > 0 the x range is cut to whole lines of lw elements (when that
// keeps most of it): then no line is shared by the fast kernel and the
// shell, and the shell's row ends fill their lines.
inline void fast_boxes(const int gfilim[6][6], const int N[3], int fastE[6], int fastH[6], int lw = 0)
{
  for (int e = 0; e < 2; ++e) {
    int *fb = e == 0 ? fastE : fastH;
    for (int a = 0; a < 3; ++a) {
      fb[2 * a] = 1;
      fb[2 * a + 1] = N[a] - 2;
      for (int d = 0; d < 3; ++d) {
        fb[2 * a] = fb[2 * a] > gfilim[3 * e + d][2 * a] ? fb[2 * a] : gfilim[3 * e + d][2 * a];
        fb[2 * a + 1] = fb[2 * a + 1] < gfilim[3 * e + d][2 * a + 1] ? fb[2 * a + 1] : gfilim[3 * e + d][2 * a + 1];
      }
    }
    if (lw > 0) {
      const int x0 = (fb[0] + lw - 1) / lw * lw, x1 = (fb[1] + 1) / lw * lw - 1;
      if (fb[1] - fb[0] + 1 >= 4 * lw && x1 - x0 + 1 >= 2 * lw) {
        fb[0] = x0;
        fb[1] = x1;
      }
    }
  }
}

// Fused box of the leapfrog sweep: where E and H both take the ordinary
// update, its x range cut to whole 63-cell tiles when that leaves at most 16
// columns to the shells.
inline void leap_box(const int gfilim[6][6], const int N[3], int fb[6])
{
  int fe[6], fh[6];
  fast_boxes(gfilim, N, fe, fh, 0);
  for (int a = 0; a < 3; ++a) {
    fb[2 * a] = fe[2 * a] > fh[2 * a] ? fe[2 * a] : fh[2 * a];
    fb[2 * a + 1] = fe[2 * a + 1] < fh[2 * a + 1] ? fe[2 * a + 1] : fh[2 * a + 1];
  }
  const int w = fb[1] - fb[0] + 1;
  if (w >= 63 && w % 63 <= 16) fb[1] = fb[0] + w / 63 * 63 - 1;
}

// The in-line form of a context's corrections (XArgs).
struct InlineState {
  // every context but those with the fused sweep, those too large for it, and
  // those whose set-up it does not hold
  bool inl = false;
  bool murPush = false;                      // Mur E written by its inner neighbour's thread
  // in-line corrections of the E sweep: 0 none, 1 Mur and zeros, 2 Debye
  // sites as well; 3 and 4 the same with update rows
  int xlevel() const { return xflag0 == ~0u ? 0 : (debyeSimple ? 2 : 1) + (xskip ? 2 : 0); }
  long long debyeSimple = 0;                 // one-pole Debye sites applied from the class table
  long long debyeFast = 0;                   // those of them in the fast E box
  // an operation on one field value, before rows are made of them
  // (key: ((cell * 3 + component) * 4 + order); kept in the reference's order within one key)
  struct XEnt {
    long long key;
    int code, arg;
    double a, b;
    long long value() const { return key / 4; }
    long long cell() const { return key / 12; }
    int comp() const { return (int)(key / 4 % 3); }
  };
  std::vector<XEnt> xent[2];
  struct XSite { long long key; int med; };  // key: cell * 3 + component
  std::vector<XSite> xsite;                  // Debye sites in block order
  long long debyeAll = 0;                    // all Debye sites
  std::vector<char> dsimple;                 // per Debye medium: one real pole
  std::vector<double> dhost[2];              // its alpha and beta (real part)
  std::vector<XVal> xval[2];
  unsigned xflag0 = ~0u;
  int jlo[3] = {}, jn[3] = {};               // box of the one-pole sites
  bool xskip = false;                        // values may be left to update rows
  bool xflagH = false;                       // some H cells are flagged (with xskip)
  void *d_xargs[2] = {}, *d_xval[2] = {}, *d_xvals[2] = {}, *d_xcls[2] = {};
  void *d_xgstart[2] = {}, *d_xrow[2] = {}, *d_xop[2] = {}, *d_xsite = nullptr;
  void *d_xdtab = nullptr, *d_xJ = nullptr;
  long long nXval[2] = {}, nXupd[2] = {}, nXrow[2] = {}, nXgroup[2] = {}, nXsite = 0;
  // blocks of half-step e's launch of rows: rows and groups, then sites
  long long row_blocks(int e) const
  {
    return (nXrow[e] + nXgroup[e] + 255) / 256 + (e == 0 ? (nXsite + 255) / 256 : 0);
  }
  std::vector<double> hflags;                // [H class] flags
};

struct Ctx : InlineState {
  std::string err;
  vgpu_prec prec;
  int device;
  size_t esz;            // bytes per stored real
  int NX, NY, NZ, PX;
  long long plane;
  size_t ncell;          // PX*NY*NZ
  vgpu_grid_desc grid;
  std::vector<double> xl, yl, zl, dex, dey, dez, idex, idey, idez, idhx, idhy, idhz;
  hipStream_t stream = nullptr;
  std::vector<hipEvent_t> evE, evH;
  double last_total_ms = 0, last_e_ms = 0, last_h_ms = 0;
  bool finalized = false;
  size_t bytes = 0;

  // device allocations
  std::vector<void *> allocs;
  // the field sets (Ex..Hz each): set `par` holds the current fields; with
  // the fused sweep there are two and every step flips it, otherwise F1 is F
  void *F[6] = {}, *F1[6] = {};
  int par = 0;
  void *fld(int set, int d) const { return set ? F1[d] : F[d]; }
  int next(int set) const { return leap ? set ^ 1 : set; }  // the set a step writes
  void *alpha[3] = {}, *beta[3] = {}, *gamma[3] = {};
  void *ide[3] = {}, *idh[3] = {};
  bool media_set = false;

  // Coefficient classes (the reference's indexed-media representation,
  // grid.h:108-135): every cell's (alpha, beta) triple of E components and
  // gamma triple of H components is one entry of a small table.  Built on
  // the host in vgpu_set_media, refined in vgpu_finalize with what the sweeps
  // do in line (build_inline), uploaded as uint16 per cell when both tables fit.
  std::vector<uint32_t> ecls, hcls;          // host, per device cell
  std::vector<double> etab, htab;            // host: [class][6] alpha/beta, [class][3] gamma (device: padded to 8, 4)
  bool indexed = false;
  void *d_ecls = nullptr, *d_hcls = nullptr, *d_etab = nullptr, *d_htab = nullptr;
  int nEcls = 0, nHcls = 0;
  // fused leapfrog sweep: the fast boxes are its fused box, H cells to
  // update again after the E corrections
  bool leap = false;
  int leapR = 4, leapKZ = 8;
  long long nFix = 0, fixCells = 0;
  void *d_fix = nullptr;
  std::vector<long long> eTouched;           // E values (cell * 3 + component) changed after the E sweep
  int fastE[6] = {}, fastH[6] = {};          // boxes of the sweeps' fast kernels
  void *d_eargs[2] = {}, *d_hargs[2] = {};   // argument blocks in device memory, by the set read
  void *d_epcs = nullptr, *d_ework = nullptr;   // E shell: pieces, launch blocks
  void *d_hpcs = nullptr, *d_hwork = nullptr;   // H shell
  int nEwork = 0, nHwork = 0, nEpcs = 0, nHpcs = 0;
  // the same shells at the most planes per block, for the packed launches of
  // group runs, which hold many grids' blocks
  void *d_epcsPk = nullptr, *d_eworkPk = nullptr, *d_hpcsPk = nullptr, *d_hworkPk = nullptr;
  int nEworkPk = 0, nHworkPk = 0;
  long long shellCells[2] = {};              // cells of the E and H shell pieces

  // UPML
  unsigned pmlmask = 0;
  int fplim[6][6][6];
  void *aux1[6][3] = {}, *aux2[6][3] = {}, *auxB[6][3] = {};
  // UPML auxiliaries live in three pools (E: PP and P with the same layout,
  // H: B); aux1/aux2/auxB point into them, each slab 256-byte aligned.
  void *auxPool[3] = {};
  void *prof[6][3] = {};   // ad, bd, ah, bh, ibd, ibh per axis

  // Mur
  unsigned murmask = 0;
  double zeta[6] = {};
  int fmlim[6][6][6];

  // ghosts
  int ghost[6] = {};

  // Debye blocks (host side until finalize)
  struct DebyeBlock { int flim[3][6]; int np; std::vector<double> da, db; };
  std::vector<DebyeBlock> debye;
  int debyeLayers = 0;
  std::vector<long long> debyeLayerStart;
  long long debyeSites = 0;
  int debyeMaxPoles = 0, debyeCplx = 0;
  void *d_dkey = nullptr, *d_dsbeta = nullptr, *d_dlast = nullptr, *d_dJ = nullptr;
  void *d_dalpha = nullptr, *d_dbeta = nullptr, *d_dnp = nullptr;

  // SIBC
  struct SibcSurf { vgpu_sibc_desc d; std::vector<unsigned char> adjA, adjB;
                    std::vector<double> q0[16], q1[16], q2[16]; };
  std::vector<SibcSurf> sibc;
  long long sibcFaces = 0;
  int sibcMaxPoles = 1;
  bool sibcReal = false;                     // all filter coefficients real: real filter state
  bool sibcFactored = false;                 // FP32 form: one state per (input, pole)
  void *d_sfbase = nullptr, *d_sfratio = nullptr, *d_sblocks = nullptr;
  int sibcBlocks = 0;
  void *d_sijk = nullptr, *d_ssurf = nullptr, *d_sadjA = nullptr, *d_sadjB = nullptr, *d_snormal = nullptr;
  void *d_sA = nullptr, *d_sB = nullptr, *d_sset = nullptr, *d_snp = nullptr, *d_sasymp = nullptr, *d_sq = nullptr;
  void *d_szeta = nullptr, *d_sold = nullptr, *d_setan = nullptr;
  long long sibcHRows = 0;
  void *d_shkey = nullptr, *d_shstart = nullptr, *d_shent = nullptr, *d_shg = nullptr;

  // waveforms, sources, plane waves
  std::vector<WaveformDev> wf;
  std::vector<std::vector<double>> wftab;
  struct Src { int field, kind, soft, waveform; double size, delay; int flim[6]; };
  std::vector<Src> src;
  struct Pw { vgpu_pw_desc d; double prof[4][10]; };
  std::vector<Pw> pw;
  void *d_wf = nullptr, *d_src = nullptr, *d_pw = nullptr, *d_aux = nullptr, *d_auxpml = nullptr, *d_auxprof = nullptr;
  int auxmax = 0;
  long long corrRows[2] = {0, 0};
  void *d_ckey[2] = {}, *d_cstart[2] = {}, *d_cent[2] = {}, *d_ccoef[2] = {}, *d_calpha[2] = {};

  // observers
  struct PObs { int i, j, k; uint64_t first, last; std::vector<double> omega; };
  std::vector<PObs> pobs;
  struct VObs { int box[6]; int step[3]; uint64_t first, last; long long nodes; };
  std::vector<VObs> vobs;
  uint64_t totalSteps = 0, maxRun = 0, lastRunSteps = 0, lastRunFirst = 0;
  // device step counter (read by the time-dependent kernels) and the host's
  // view of its value once the enqueued work has run
  void *d_step = nullptr;
  void *d_pack = nullptr;  // PackArgs for group runs (separate sweeps only)
  uint64_t stepHost = 0;
  // a captured graph of graphSteps whole steps (replayed by vgpu_run)
  hipGraph_t graph = nullptr;
  hipGraphExec_t graphExec = nullptr;
  uint64_t graphSteps = 0;
  int graphPar = 0;                          // field set current when the graph was captured
  uint64_t graphRuns = 0;                    // runs replayed from it
  bool graphTried = false, lastRunTimed = false;
  // group runs led by this context: the last group's members (context
  // serials, never reused) and length, and a graph captured once the same
  // group runs twice in a row
  uint64_t serial = 0;
  std::vector<uint64_t> groupKey;
  uint64_t groupSteps = 0;
  hipGraph_t groupGraph = nullptr;
  hipGraphExec_t groupExec = nullptr;
  bool groupTried = false;
  // replaced group graphs, freed once the event recorded after their last
  // launch has completed
  struct RetiredGraph { hipGraph_t graph; hipGraphExec_t exec; hipEvent_t done; };
  std::vector<RetiredGraph> retired;
  void *d_ocell = nullptr, *d_ofirst = nullptr, *d_olast = nullptr, *d_onf = nullptr, *d_ooff = nullptr;
  void *d_oomega = nullptr, *d_otd = nullptr, *d_odre = nullptr, *d_odim = nullptr;
  long long vnodes = 0;
  void *d_vcell = nullptr, *d_vobs = nullptr, *d_vfirst = nullptr, *d_vlast = nullptr, *d_vstage = nullptr;
  std::vector<long long> vobsNodeStart;
  // Volume samples stream out without a sync per run: the device staging
  // holds 2*maxRun rows (row = step modulo that), each run's rows are copied
  // asynchronously into its slot of a pinned host ring after its kernels,
  // and a record of each of the last two runs (first step, length, start and
  // end events) lets the host finish one run while the next one runs.
  uint64_t vring = 0;
  float *h_vring = nullptr;  // [2][maxRun][vnodes][6], pinned
  struct RunRec { uint64_t first = 0, n = 0; bool valid = false; hipEvent_t start = nullptr, end = nullptr; };
  RunRec runs[2];
  uint64_t runCount = 0;
  const RunRec &last_run() const { return runs[runCount ? (runCount - 1) & 1 : 0]; }
  // Point spectra are read through a pinned buffer: one observer's, re then
  // im, gathered by one kernel on the context's stream.
  std::mutex specMu;
  double *h_spec = nullptr;  // [2][6][most frequencies of an observer]

  long long lin(int i, int j, int k) const { return ((long long)k * NY + j) * PX + i; }
};

int set_error(Ctx *c, int code, const char *fmt, ...);
void *dev_alloc(Ctx *c, size_t bytes);

// Update-once check: visit-count arrays per component (device layout) and
// sweep argument blocks in device memory that carry them.
struct VisitRun {
  unsigned *vis[6];
  void *eargs, *hargs;
};

// Corrections of a finalized set-up: rows, flagged classes, device arrays
// (vgpu_inline.h).
template <typename T> int build_inline(Ctx *c);

// Per-precision step driver, instantiated for double and float.
// Enqueues nsteps steps that start at the device step counter, then advances
// it; with timeKernels the volume sweeps of the first steps are timed.  With
// chk it enqueues one step of the field sweeps only, counting updates.
template <typename T>
int run_steps(Ctx *c, uint64_t nsteps, hipStream_t s, bool timeKernels, const VisitRun *chk = nullptr);
// Uploads the sweeps' argument blocks (once, at finalize).
template <typename T> int prepare_sweeps(Ctx *c);
// Uploads the context's argument blocks for packed launches (once, at finalize).
template <typename T> int upload_pack(Ctx *c);
// Enqueues nsteps steps of n contexts in lockstep on stream s, with packed
// launches, then advances each one's step counter.
template <typename T> int run_group_steps(Ctx *const *cs, int n, uint64_t nsteps, hipStream_t s);
// Update-once check of the field sweeps against the outer field limits.  Its
// buffers come from `scratch` (scratchBytes long) when given, else they are
// allocated for the call.
template <typename T>
int check_limits(Ctx *c, const int folim[6][6], vgpu_limits_report *rep, unsigned char *counts, void *scratch,
                 size_t scratchBytes);
template <typename T> size_t check_limits_bytes(const Ctx *c, bool counts, size_t off[4]);

}  // namespace vgpu
