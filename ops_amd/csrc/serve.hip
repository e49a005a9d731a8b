// Batched multi-block CG engine with a continuous-batching scheduler
// (include/ops_mi355x_serve.h).
//
// Device side.  Each active solve (one block) is described by a SolveDev
// (field pointers, strides, sizes, tile grid) and a SolveStat (CG scalars
// and status) in device memory.  A tile table lists (solve, tile) pairs of
// every active solve, contiguous per solve.  One CG iteration is two
// launches, each persistent (a fixed grid walks the tile table; blocks are
// renumbered so each XCD walks a contiguous stretch of tiles):
//   sk_sweep     rrn = fold of r.r ; beta = rrn / rro, stop test ;
//                w = A (beta p + r) per tile, partial p.w per tile
//   sk_update    pw = fold of p.w ; alpha = rro / pw ;
//                p = beta p + r ; u += alpha p ; r -= alpha w, partial r.r
// Every workgroup folds the partials of each solve it works on itself, in the
// same fixed order, so no launch waits for a fold of its own; the sweep forms the new p at the
// points its stencil reads and the update, pointwise, stores it.  (Five
// launches, with folds and p update of their own, took 17.5 us an iteration
// on a small solve.)  The CG scalars alternate between two copies: a launch
// reads one, and its solve's first tile writes the other.  sk_finish folds
// the last r.r of a batch of iterations and tests it.
// Solves that are done skip all work, so a graph of K iterations stops each
// solve exactly where it converges.  A solve's numbers do not depend on the
// rest of the batch.  3D heat tiles are 128 x 4 x chunk columns marched along
// z in registers, 2D Poisson tiles 128 x (4 chunk) rows, two points per lane.
//
// Host side.  Fields live in one arena of the HBM budget (first-fit, 256 B
// granules, coalescing).  A step admits queued solves in FIFO order while a
// slot and memory are free (set-up kernels generate inputs, coefficients
// and the first residual on the device), rebuilds the tile table if the
// batch changed, launches K iterations (one graph launch), reads back the
// per-solve status and retires converged solves.  Tables are read by the
// kernels from device memory, so one captured graph serves every batch.
#include <deque>
#include <map>

#include "../../include/ops_mi355x_serve.h"
#include "../apps/problems.h"
#include "box.h"
#include "engine.h"
#include "column.h"

using namespace opsmi;

namespace {

// Default tile parameter per size class (size_class): rows per wave of a 2D
// tile, z planes of a 3D tile.  A tile is worked through serially, so small
// solves take short tiles (more workgroups) and large ones long tiles (fewer
// rim re-reads).  Microseconds per CG iteration of one FP64 solve alone:
//   2D side   1 row   2 rows  4 rows  8 rows |  3D side  4      8      16     32 planes
//     128      12.6    13.8    15.8    19.3  |    32    16.5   21.9   32.2   53.4
//     256      12.5    13.6    15.8    20.0  |    64    17.8   22.1   33.5   54.4
//     512      14.3    14.7    16.6    20.5  |    96    27.4   31.3   38.3   60.3
//     700      20.0    17.4    19.1    23.2  |   128    45.8   45.5   47.2   64.2
//    1000      28.7    24.2    22.0    24.6  |   200   226    260    213    221
//    2000      85      71      63      64    |   256   427    401    386    391
//    4096     377     324     309     302    |   512  3059   3009   2995   2987
// A class's value is within 10 % of its sides' best; opsmi_serve_autotune
// measures on the card at hand.
constexpr int kRows2D[3] = {1, 2, 4};
constexpr int kChunk3D[3] = {4, 4, 16};
constexpr int kPart = 4;  // partial sums per tile: planes 0-2 of the update, plane 3 p.w

struct SolveDev {
  double *u, *p, *r, *w, *kx, *ky, *kz;  // element (0,0,0) of each field
  long sy, sz;
  int kind, nx, ny, nz;
  int tx, ty;   // tiles along x and y
  int chunk;    // 3D: z planes per tile; 2D: rows per wave
  int sv;       // points per lane along x (kSV; kSV32 for FP32-inner solves)
  int tile0, ntiles;
  int active;
  double rx, ry, rz;
  // FP32-inner refinement: u = x and f (FP64), and the FP32 inner fields
  // e, rr, p, w (3D heat: also the face coefficients rounded to float) with
  // their own row and plane pitch
  int mixed;
  double *f;
  float *e32, *r32, *p32, *w32;
  float *kx32, *ky32, *kz32;
  long sy32, sz32;
};

// phases of a mixed solve: the next iteration runs an inner FP32 PCG step,
// or applies the correction x += e and recomputes the FP64 residual
// (3D heat: applies it in one iteration, PH_CORR, and recomputes in the next)
enum { PH_INNER = 0, PH_RESID = 1, PH_CORR = 2 };

struct SolveStat {
  double rro, rr0, stop, pw, alpha, beta;
  int iters, done, max_iters;
  int pending;  // an update's sums are still to be folded
  // mixed: inner r.z, inner stop threshold, |f|, targets
  double rz, istop, fn, tol, inner_tol;
  int phase, outer, max_outer, axpby;  // axpby: the next p update runs
};

struct TileBox {
  int x0, y0, z0, z1;
};

// Points per lane along x: every field's x = 0 is 256-byte aligned and its
// row pitch a multiple of 256 bytes, so a lane's points are one aligned
// load: kSV doubles (16 bytes) for FP64 solves and FP32-inner 3D heat
// solves (8-byte FP32 loads; their 3D grids, sides 32-256, would leave most
// lanes of 256-point tiles idle: the wider form measured 0.73 s against
// 0.59 s on a 30-request heat stream), kSV32 floats (16 bytes) for the FP32
// fields of an FP32-inner 2D Poisson solve, whose FP64 fields a lane then
// reads as two 16-byte loads (40-request Poisson stream: 1.20 s against
// 1.35 s with 8-byte lanes).  A tile is (64 sv) points wide.
constexpr int kSV = 2;
constexpr int kSV32 = 4;

__device__ __forceinline__ TileBox tile_box(const SolveDev &d, int li) {
  TileBox b;
  const int tx = li % d.tx, rest = li / d.tx;
  b.x0 = tx * kWave * d.sv;
  if (d.kind == OPSMI_SOLVE_HEAT3D) {
    b.y0 = (rest % d.ty) * kWavesPerBlock;
    b.z0 = (rest / d.ty) * d.chunk;
    b.z1 = min(b.z0 + d.chunk, d.nz);
  } else {
    b.y0 = rest * kWavesPerBlock * d.chunk;
    b.z0 = 0;
    b.z1 = 1;
  }
  return b;
}

// f(x, y, z, n) over this thread's groups of the tile: V consecutive points
// from x (V = the solve's points per lane), n (1..V) of them inside the block
//
// A lane whose group is whole (n == V: every lane but those at a solve's
// right edge) calls f with the literal V, so the element-count branches in
// f's vector loads and stores fold away: a branch join makes the compiler
// wait for every load in flight, which would serialise a group's loads.
template <int V, class F>
__device__ __forceinline__ void tile_groups(const SolveDev &d, const TileBox &b, F f) {
  const int x = b.x0 + V * (int)threadIdx.x;
  const int n = min(V, d.nx - x);
  if (n <= 0) return;
  auto g = [&](int y, int z) {
    if (n == V) f(x, y, z, V);
    else f(x, y, z, n);
  };
  if (d.kind == OPSMI_SOLVE_HEAT3D) {
    const int y = b.y0 + (int)threadIdx.y;
    if (y >= d.ny) return;
    for (int z = b.z0; z < b.z1; z++) g(y, z);
  } else {
    for (int i = 0; i < d.chunk; i++) {
      const int y = b.y0 + (int)threadIdx.y + kWavesPerBlock * i;
      if (y < d.ny) g(y, 0);
    }
  }
}

__device__ __forceinline__ Ptr<double> P(double *a, const SolveDev &d) { return Ptr<double>{a, d.sy, d.sz}; }
__device__ __forceinline__ Ptr<const double> PC(const double *a, const SolveDev &d) {
  return Ptr<const double>{a, d.sy, d.sz};
}

__device__ __forceinline__ void store_partial(double v, double *dst, double (*sh)[1]) {
  double acc[1] = {v};
  block_reduce<double, OPS_INC, 1>(acc, sh);
  if (threadIdx.x == 0 && threadIdx.y == 0) *dst = acc[0];
}

__device__ __forceinline__ Ptr<float> PF32(float *a, const SolveDev &d) { return Ptr<float>{a, d.sy32, d.sz32}; }
__device__ __forceinline__ Ptr<const float> PF32C(const float *a, const SolveDev &d) {
  return Ptr<const float>{a, d.sy32, d.sz32};
}

// output stage of the FP64 heat column for a mixed heat solve's residual
// pass: r = f - A x, the inner start rr = (float) r, e = 0, p = rr (no
// preconditioner), sums (r.r, rr.rr, rr.rr) in FP64
struct HeatOutResid {
  const Ptr<const double> &f;
  const Ptr<float> &rr, &e, &p;
  double acc[3] = {0.0, 0.0, 0.0};
  __device__ __forceinline__ void operator()(int x, int y, int z, int nn, const double (&v)[kSV],
                                             const double (&pc)[kSV]) {
    double fv[kSV];
    ldv<double, kSV>(f.at(x, y, z), nn, fv);
    float q32[kSV], zero[kSV];
#pragma unroll
    for (int j = 0; j < kSV; j++) {
      const double r = fv[j] - v[j];
      q32[j] = (float)r;
      zero[j] = 0.0f;
      if (j < nn) {
        acc[0] = acc[0] + r * r;
        acc[1] = acc[1] + (double)q32[j] * (double)q32[j];
        acc[2] = acc[2] + (double)q32[j] * (double)q32[j];
      }
    }
    stv<float, kSV, false>(e.at(x, y, z), nn, zero);
    stv<float, kSV, false>(rr.at(x, y, z), nn, q32);
    stv<float, kSV, false>(p.at(x, y, z), nn, q32);
  }
};

// the 2D 5-point operator over a group: the group's row and the rows above
// and below, and the neighbours just left and right of the group
template <class T, int V>
struct Row5 {
  T c[V], up[V], dn[V];
  T l, r;
};
template <class T, int V>
__device__ __forceinline__ void load5(const Ptr<const T> &p, int x, int y, int n, Row5<T, V> &R) {
  ldv<T, V>(p.at(x, y, 0), n, R.c);
  ldv<T, V>(p.at(x, y - 1, 0), n, R.up);
  ldv<T, V>(p.at(x, y + 1, 0), n, R.dn);
  R.l = p(x - 1, y, 0);
  R.r = p(x + n, y, 0);
}
// 4 p - (p(x-1) + p(x+1)) - (p(y-1) + p(y+1)) at point j of the group
template <class T, int V>
__device__ __forceinline__ T op5(const Row5<T, V> &R, int j, int n) {
  const T xm = j == 0 ? R.l : R.c[j > 0 ? j - 1 : 0];
  const T xp = j + 1 < n ? R.c[j + 1 < V ? j + 1 : j] : R.r;
  return (T)4.0 * R.c[j] - (xm + xp) - (R.up[j] + R.dn[j]);
}

// First tile of this workgroup.  XCD k takes the k-th contiguous eighth of
// the tiles in flight: of the whole grid's when the table is longer than the
// grid, otherwise of the table's.  (Numbered over the grid, a table of 504
// tiles filled 2 of the 8 XCDs: a 1000^2 Poisson iteration took 64.9 us,
// spread over all eight 28.0; a 128^3 heat iteration 222.6 and 60.8.)
__device__ __forceinline__ int first_tile(int nt) {
  const int nb = min(nt, (int)gridDim.x);
  return (int)blockIdx.x < nb ? (int)xcd_tile(blockIdx.x, (unsigned)nb) : nt;
}

// ------------------------------------------------------------ iteration
// Sums of a solve's partials [tile0, tile0 + ntiles) of planes first ..
// first + D - 1, in thread 0.  Thread i adds partials i, i + 256, ... in that
// order; eight are loaded before they are added (eight loads in flight, the
// same sums).
template <int D>
__device__ __forceinline__ void fold_partials(const double *part, size_t np, int first, int t0, int n,
                                              double (&acc)[D], double (*sh)[D]) {
  const int tid = (int)(threadIdx.x + threadIdx.y * blockDim.x);
#pragma unroll
  for (int k = 0; k < D; k++) acc[k] = 0.0;
  for (int i0 = tid; i0 < n; i0 += 8 * 256) {
    double t8[8][D];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int i = i0 + u * 256;
#pragma unroll
      for (int k = 0; k < D; k++) t8[u][k] = i < n ? part[(first + k) * np + t0 + i] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (i0 + u * 256 < n)
#pragma unroll
        for (int k = 0; k < D; k++) acc[k] = acc[k] + t8[u][k];
  }
  block_reduce<double, OPS_INC, D>(acc, sh);
}

// The CG scalars after an update whose sums are sum[]: iteration count, beta
// and stop test.  Mixed solves follow the refinement loop of the FP64-IR /
// FP32-PCG solver:
//   PH_RESID: residual r, |r|/|f| <= tol stops; else the inner solve starts
//             with rz and its stop threshold max(inner_tol, tol / (2 relres)) |rr_0|
//   PH_INNER: stop the inner solve at its threshold (the next sweep corrects
//             x), else b = (float)(rzn / rz) and p = Mi rr + b p
__device__ __forceinline__ void advance(SolveStat &q, const SolveDev &d, const double *sum) {
  q.pending = 0;
  if (!d.mixed) {
    const double rrn = sum[0];
    q.beta = rrn / q.rro;
    q.rro = rrn;
    q.iters = q.iters + 1;
    if (sqrt(rrn) <= q.stop) q.done = 1;
    else if (q.iters >= q.max_iters) q.done = 2;
    return;
  }
  if (q.phase == PH_INNER) {
    const double rzn = sum[0], rrn = sum[1];
    q.iters = q.iters + 1;
    q.rro = rrn;
    if (sqrt(rrn) <= q.istop) {
      q.phase = d.kind == OPSMI_SOLVE_HEAT3D ? PH_CORR : PH_RESID;
      q.outer = q.outer + 1;
    } else if (q.iters >= q.max_iters) {
      q.done = 2;
    } else {
      q.beta = (double)(float)(rzn / q.rz);
      q.rz = rzn;
      q.axpby = 1;
    }
    return;
  }
  const double rrd = sum[0];
  if (q.outer == 0) {
    q.fn = sqrt(rrd);
    q.rr0 = rrd;
  }
  q.rro = rrd;
  const double rel = sqrt(rrd) / q.fn;
  if (rel <= q.tol) q.done = 1;
  else if (q.outer >= q.max_outer) q.done = 2;
  else {
    q.rz = sum[1];
    q.istop = fmax(q.inner_tol, 0.5 * q.tol / rel) * sqrt(sum[2]);
    q.phase = PH_INNER;
    q.axpby = 0;
  }
}

// what a launch's workgroups need of their solve's scalars
struct Step {
  double a, b;   // p_new = a p + b r
  double alpha;  // u += alpha p_new, r -= alpha w (update)
  int done, phase;
};
__device__ __forceinline__ Step step_of(const SolveStat &q, const SolveDev &d) {
  Step c;
  c.a = q.beta;
  c.b = 1.0;
  if (d.mixed) {
    // p = Mi rr + b p, or p as the residual pass left it
    c.a = q.axpby ? q.beta : 1.0;
    c.b = q.axpby ? (d.kind == OPSMI_SOLVE_HEAT3D ? 1.0 : 0.25) : 0.0;
  }
  c.alpha = 0.0;
  c.done = q.done;
  c.phase = q.phase;
  return c;
}

// LDS of an iteration launch: sums being folded, the step all threads read,
// and the tile's own sums
struct IterLds {
  double fold[16][3];
  double one[16][1];
  double tile3[16][3];
  double tile1[16][1];
  Step step;
};

// the new scalars in sweep (folds a pending update's sums) and in update
// (folds p.w); all threads of the workgroup call it for each tile.  A
// workgroup's tiles of one solve follow each other, so only the first of them
// (fresh) folds and the others find the step in LDS: a fold reads as many sums
// as the solve has tiles, and once a tile that is their square (2D 8192^2,
// 32768 tiles: 1831 us an iteration folding for every tile, 1188 now).
// The solve's first tile, always a fresh one, stores the scalars.
__device__ __forceinline__ Step sweep_step(IterLds &L, const SolveDev &d, const SolveStat &in, SolveStat &out,
                                           const double *part, size_t np, bool first_of_solve, bool fresh) {
  if (!fresh) return L.step;
  const bool pending = in.pending != 0;
  double sum[3] = {0.0, 0.0, 0.0};
  if (pending) {
    if (d.mixed) {
      fold_partials<3>(part, np, 0, d.tile0, d.ntiles, sum, L.fold);
    } else {
      double s1[1];
      fold_partials<1>(part, np, 0, d.tile0, d.ntiles, s1, L.one);
      sum[0] = s1[0];
    }
  }
  if (threadIdx.x == 0 && threadIdx.y == 0) {
    SolveStat q = in;
    if (pending) advance(q, d, sum);
    L.step = step_of(q, d);
    if (first_of_solve) out = q;
  }
  __syncthreads();
  return L.step;
}
__device__ __forceinline__ Step update_step(IterLds &L, const SolveDev &d, const SolveStat &in, SolveStat &out,
                                            const double *part, size_t np, bool first_of_solve, bool fresh) {
  if (!fresh) return L.step;
  double pw[1] = {0.0};
  const bool inner = !d.mixed || in.phase == PH_INNER;
  if (inner) fold_partials<1>(part, np, 3, d.tile0, d.ntiles, pw, L.one);
  if (threadIdx.x == 0 && threadIdx.y == 0) {
    SolveStat q = in;
    Step c = step_of(q, d);
    if (inner) {
      q.pw = pw[0];
      q.alpha = d.mixed ? (double)(float)(q.rz / pw[0]) : q.rro / pw[0];
      c.alpha = q.alpha;
    }
    // a heat solve's correction has no sums: its residual comes next
    q.pending = q.phase == PH_CORR ? 0 : 1;
    if (q.phase == PH_CORR) q.phase = PH_RESID;
    L.step = c;
    if (first_of_solve) out = q;
  }
  __syncthreads();
  return L.step;
}

// V points of a row with their neighbours in the rows below and above and to
// the left and right, at element offset o.  Loads are whole vectors whatever
// part of them lies inside the solve: a vector starts on its own size, so it
// never leaves the field's allocation, and what lies past the last point is
// the zero halo or padding.
template <class T, int V>
struct Star {
  T c[V], dn[V], up[V], l, r;
  __device__ __forceinline__ void load(const T *p, long o, long sy) {
    ldv<T, V>(p + o, V, c);
    ldv<T, V>(p + o - sy, V, dn);
    ldv<T, V>(p + o + sy, V, up);
    l = p[o - 1];
    r = p[o + V];
  }
  // this = a this + b h
  __device__ __forceinline__ void combine(const Star &h, T a, T b) {
#pragma unroll
    for (int j = 0; j < V; j++) {
      c[j] = a * c[j] + b * h.c[j];
      dn[j] = a * dn[j] + b * h.dn[j];
      up[j] = a * up[j] + b * h.up[j];
    }
    l = a * l + b * h.l;
    r = a * r + b * h.r;
  }
};

// w = A (a p + b r) of the 2D operator over a tile.  start() issues the first
// row's loads (before the scalars are known), run() keeps the next row's in
// flight while a row is computed.
template <class T, int V>
struct Sweep5 {
  const SolveDev &d;
  const T *p, *r;
  long sy, xo;
  int x, y0, n;
  Star<T, V> P, R;
  __device__ __forceinline__ Sweep5(const SolveDev &d_, const TileBox &b, const T *p_, const T *r_, long sy_)
      : d(d_), p(p_), r(r_), sy(sy_) {
    x = b.x0 + V * (int)threadIdx.x;
    y0 = b.y0 + (int)threadIdx.y;
    n = max(0, min(V, d.nx - x));
    xo = n > 0 ? x : 0;
  }
  __device__ __forceinline__ long at(int y) const { return xo + (long)min(y, d.ny - 1) * sy; }
  __device__ __forceinline__ void start() {
    P.load(p, at(y0), sy);
    R.load(r, at(y0), sy);
  }
  __device__ __forceinline__ double run(T a, T bb, T *w) {
    double acc = 0.0;
    for (int i = 0; i < d.chunk; i++) {
      const int y = y0 + kWavesPerBlock * i;
      Star<T, V> C = P;
      C.combine(R, a, bb);
      if (i + 1 < d.chunk) {
        P.load(p, at(y + kWavesPerBlock), sy);
        R.load(r, at(y + kWavesPerBlock), sy);
      }
      const int m = y < d.ny ? n : 0;
      T v[V];
#pragma unroll
      for (int j = 0; j < V; j++) {
        const T xm = j == 0 ? C.l : C.c[j > 0 ? j - 1 : 0];
        const T xp = j + 1 < V ? C.c[j + 1 < V ? j + 1 : j] : C.r;
        v[j] = (T)4.0 * C.c[j] - (xm + xp) - (C.up[j] + C.dn[j]);
        if (j < m) acc = acc + (double)v[j] * (double)C.c[j];
      }
      stv<T, V, false>(w + at(y), m, v);
    }
    return acc;
  }
};

// A column of the 3D heat operator on q = a p + b r (CHAIN) or on p, marched
// along z with three planes of q in registers; neighbours along y come from
// the caches, one plane of loads ahead.  No LDS and no barriers: at these
// sizes (sides of 32 to 256, mostly in the caches) a plane of the LDS column
// waited for its loads at a barrier (128^3, 16 planes: 60.8 us an iteration).
// Arithmetic as HeatColumn (column.h).
template <class T, int V, bool CHAIN>
struct HeatMarch {
  struct Plane {  // loaded for one z: centre of the next plane, rims and coefficients of this one
    T p[V], ylp[V], yhp[V], xlp, xhp;
    T r[V], ylr[V], yhr[V], xlr, xhr;
    T kx[V], ky[V], kyh[V], kzn[V], kxh;
  };
  const SolveDev &d;
  const T *p, *r, *kx, *ky, *kz;
  long sy, sz, o0;
  int x, y, z0, z1, n;
  T pm[V], rm[V], pc[V], rc[V], kzc[V];
  Plane A;
  __device__ __forceinline__ HeatMarch(const SolveDev &d_, const TileBox &b, const T *p_, const T *r_, const T *kx_,
                                       const T *ky_, const T *kz_, long sy_, long sz_)
      : d(d_), p(p_), r(r_), kx(kx_), ky(ky_), kz(kz_), sy(sy_), sz(sz_) {
    x = b.x0 + V * (int)threadIdx.x;
    y = b.y0 + (int)threadIdx.y;
    z0 = b.z0;
    z1 = b.z1;
    n = y < d.ny ? max(0, min(V, d.nx - x)) : 0;
    o0 = (x < d.nx ? x : 0) + (long)min(y, d.ny - 1) * sy;
  }
  __device__ __forceinline__ void load(int z, Plane &A) const {
    const long o = o0 + (long)z * sz;
    ldv<T, V>(p + o + sz, V, A.p);
    ldv<T, V>(p + o - sy, V, A.ylp);
    ldv<T, V>(p + o + sy, V, A.yhp);
    A.xlp = p[o - 1];
    A.xhp = p[o + V];
    if constexpr (CHAIN) {
      ldv<T, V>(r + o + sz, V, A.r);
      ldv<T, V>(r + o - sy, V, A.ylr);
      ldv<T, V>(r + o + sy, V, A.yhr);
      A.xlr = r[o - 1];
      A.xhr = r[o + V];
    }
    ldv<T, V>(kx + o, V, A.kx);
    ldv<T, V>(ky + o, V, A.ky);
    ldv<T, V>(ky + o + sy, V, A.kyh);
    ldv<T, V>(kz + o + sz, V, A.kzn);
    A.kxh = kx[o + V];
  }
  __device__ __forceinline__ void start() {
    const long o = o0 + (long)z0 * sz;
    ldv<T, V>(p + o - sz, V, pm);
    ldv<T, V>(p + o, V, pc);
    if constexpr (CHAIN) {
      ldv<T, V>(r + o - sz, V, rm);
      ldv<T, V>(r + o, V, rc);
    }
    ldv<T, V>(kz + o, V, kzc);
    load(z0, A);
  }
  template <class OUT>
  __device__ __forceinline__ void run(T a, T b, T rx, T ry, T rz, OUT &out) {
    auto q = [&](T pv, T rv) {
      if constexpr (CHAIN) return a * pv + b * rv;
      else return pv;
    };
    if constexpr (CHAIN) {
#pragma unroll
      for (int j = 0; j < V; j++) {
        pm[j] = q(pm[j], rm[j]);
        pc[j] = q(pc[j], rc[j]);
      }
    }
    for (int z = z0; z < z1; z++) {
      Plane C = A;
      if (z + 1 < z1) load(z + 1, A);
      T pn[V], v[V];
      const T xl = q(C.xlp, C.xlr), xh = q(C.xhp, C.xhr);
#pragma unroll
      for (int j = 0; j < V; j++) pn[j] = q(C.p[j], C.r[j]);
#pragma unroll
      for (int j = 0; j < V; j++) {
        const T pxm = j == 0 ? xl : pc[j > 0 ? j - 1 : 0];
        const T pxp = j + 1 < V ? pc[j + 1 < V ? j + 1 : j] : xh;
        const T kxn = j + 1 < V ? C.kx[j + 1 < V ? j + 1 : j] : C.kxh;
        const T pym = q(C.ylp[j], C.ylr[j]), pyp = q(C.yhp[j], C.yhr[j]);
        v[j] = ((T)1.0 + ry * (C.kyh[j] + C.ky[j]) + rx * (kxn + C.kx[j]) + rz * (C.kzn[j] + kzc[j])) * pc[j] -
               ry * (C.kyh[j] * pyp + C.ky[j] * pym) - rx * (kxn * pxp + C.kx[j] * pxm) -
               rz * (C.kzn[j] * pn[j] + kzc[j] * pm[j]);
      }
      out(x, y, z, n, v, pc);
#pragma unroll
      for (int j = 0; j < V; j++) {
        pm[j] = pc[j];
        pc[j] = pn[j];
        kzc[j] = C.kzn[j];
      }
    }
  }
};

// x = x + (double) e over a tile
template <int V>
__device__ __forceinline__ void correct_tile(const SolveDev &d, const TileBox &b) {
  const Ptr<double> x = P(d.u, d);
  const Ptr<const float> ev = PF32C(d.e32, d);
  tile_groups<V>(d, b, [&](int i, int j, int k, int n) {
    double xv[V];
    float evv[V];
    ldv<double, V>(x.at(i, j, k), n, xv);
    ldv<float, V>(ev.at(i, j, k), n, evv);
#pragma unroll
    for (int q = 0; q < V; q++) xv[q] = xv[q] + (double)evv[q];
    stv<double, V, false>(x.at(i, j, k), n, xv);
  });
}

// Both launches: latency-bound on small solves (a tile entry, its solve and
// the partials are loaded one after the other, then two block reductions:
// 5.2 us a launch at 64^2), bandwidth-bound on large ones.  A tile's first
// loads are issued before its solve's sums are folded.  Microseconds per CG
// iteration of one solve alone, five launches and now:
//   2D 64^2 17.8 and 12.3, 512^2 19.6 and 14.7, 1000^2 28.0 and 24.0, 2000^2
//   76.5 and 63 (5.1 TB/s of 80 bytes a point), 4096^2 335 and 309, 8192^2
//   1392 and 1188; FP32-inner 1000^2 25.0 and 19.3, 8192^2 721 and 634
//   3D 64^3 24.7 and 17.7, 128^3 60.8 and 47.2, 200^3 245 and 214, 300^3 719
//   and 724, 512^3 2995 and 3002; FP32-inner 200^3 278 and 121, 384^3 769 and 772
// Between them 3D solves whose fields straddle the Infinity Cache lose: 240^3
// 313 and 330, 256^3 365 and 386, FP32-inner 256^3 196 and 210.  The sweep
// there takes 223 us for 48 bytes a point (3.6 TB/s; the update 165, 5.7): it
// fetches 1.23 times its arrays, the five launches' LDS column 1.14 times.
// Tried there: neighbours along x by lane shuffles and uniform row addresses,
// 382 at 256^3 (FP32-inner 202); with the coefficients loaded past the caches
// 390 (189), 5 % slower at 128^3; tiles of 64 planes 374, 20 % slower at 200^3;
// four waves a SIMD, which spill, 524.
__global__ __launch_bounds__(256) void sk_sweep(const SolveDev *__restrict__ S, const SolveStat *__restrict__ in,
                                                SolveStat *__restrict__ out, const int2 *__restrict__ tiles,
                                                const int *__restrict__ ntiles, double *part, size_t np) {
  __shared__ IterLds L;
  const int nt = *ntiles;
  for (int t = first_tile(nt); t < nt; t += (int)gridDim.x) {
    const int s = __builtin_amdgcn_readfirstlane(tiles[t].x), li = __builtin_amdgcn_readfirstlane(tiles[t].y);
    const SolveDev &d = S[s];
    if (in[s].done) {
      if (li == 0 && threadIdx.x == 0 && threadIdx.y == 0) out[s] = in[s];
      continue;
    }
    const TileBox b = tile_box(d, li);
    const bool fresh = t < (int)gridDim.x || tiles[t - (int)gridDim.x].x != s;
    __syncthreads();  // the previous tile's sums and step have been read
    if (!d.mixed) {
      double acc;
      if (d.kind == OPSMI_SOLVE_HEAT3D) {
        HeatMarch<double, kSV, true> m(d, b, d.p, d.r, d.kx, d.ky, d.kz, d.sy, d.sz);
        m.start();
        const Step c = sweep_step(L, d, in[s], out[s], part, np, li == 0, fresh);
        if (c.done) continue;
        const Ptr<double> w = P(d.w, d);
        HeatOutW<double, kSV, false> o{w};
        m.run(c.a, c.b, d.rx, d.ry, d.rz, o);
        acc = o.acc;
      } else {
        Sweep5<double, kSV> m(d, b, d.p, d.r, d.sy);
        m.start();
        const Step c = sweep_step(L, d, in[s], out[s], part, np, li == 0, fresh);
        if (c.done) continue;
        acc = m.run(c.a, c.b, d.w);
      }
      store_partial(acc, part + 3 * np + t, L.tile1);
      continue;
    }
    if (d.kind == OPSMI_SOLVE_HEAT3D) {
      HeatMarch<float, kSV, true> m(d, b, d.p32, d.r32, d.kx32, d.ky32, d.kz32, d.sy32, d.sz32);
      m.start();
      const Step c = sweep_step(L, d, in[s], out[s], part, np, li == 0, fresh);
      if (c.done) continue;
      if (c.phase == PH_CORR) {
        correct_tile<kSV>(d, b);
      } else if (c.phase == PH_RESID) {
        // FP64 residual of the corrected x and the inner start; the sums go
        // where the update's do (this launch reads none)
        const Ptr<const double> f = PC(d.f, d);
        const Ptr<float> rr = PF32(d.r32, d), ev = PF32(d.e32, d), p = PF32(d.p32, d);
        HeatOutResid o{f, rr, ev, p};
        HeatMarch<double, kSV, false> md(d, b, d.u, nullptr, d.kx, d.ky, d.kz, d.sy, d.sz);
        md.start();
        md.run(1.0, 0.0, d.rx, d.ry, d.rz, o);
        block_reduce<double, OPS_INC, 3>(o.acc, L.tile3);
        if (threadIdx.x == 0 && threadIdx.y == 0) {
          part[t] = o.acc[0];
          part[np + t] = o.acc[1];
          part[2 * np + t] = o.acc[2];
        }
      } else {
        const Ptr<float> w = PF32(d.w32, d);
        HeatOutW<float, kSV, false> o{w};
        m.run((float)c.a, (float)c.b, (float)d.rx, (float)d.ry, (float)d.rz, o);
        store_partial(o.acc, part + 3 * np + t, L.tile1);
      }
    } else {
      Sweep5<float, kSV32> m(d, b, d.p32, d.r32, d.sy32);
      m.start();
      const Step c = sweep_step(L, d, in[s], out[s], part, np, li == 0, fresh);
      if (c.done) continue;
      if (c.phase == PH_RESID) {
        // the correction (pointwise; the residual follows in sk_update once
        // every tile has applied it)
        correct_tile<kSV32>(d, b);
      } else {
        const double acc = m.run((float)c.a, (float)c.b, d.w32);
        store_partial(acc, part + 3 * np + t, L.tile1);
      }
    }
  }
}

// p = a p + b r ; u += alpha p ; r -= alpha w over a tile, sums of r r (and,
// MIXED, of r.Mi r and r.r).  start() issues the first group's loads.
template <class T, int V, bool MIXED>
struct UpdateTile {
  const SolveDev &d;
  T *u, *p, *r;
  const T *w;
  long sy, sz, xo;
  int y0, z0, n, groups;
  bool heat;
  T uv[V], pv[V], rv[V], wv[V];
  __device__ __forceinline__ UpdateTile(const SolveDev &d_, const TileBox &b, T *u_, T *p_, T *r_, const T *w_,
                                        long sy_, long sz_)
      : d(d_), u(u_), p(p_), r(r_), w(w_), sy(sy_), sz(sz_) {
    const int x = b.x0 + V * (int)threadIdx.x;
    heat = d.kind == OPSMI_SOLVE_HEAT3D;
    y0 = b.y0 + (int)threadIdx.y;
    z0 = b.z0;
    n = max(0, min(V, d.nx - x));
    xo = n > 0 ? x : 0;
    groups = heat ? b.z1 - b.z0 : d.chunk;
  }
  __device__ __forceinline__ int row(int i) const { return heat ? y0 : y0 + kWavesPerBlock * i; }
  __device__ __forceinline__ long at(int i) const {
    return xo + (long)min(row(i), d.ny - 1) * sy + (heat ? (long)(z0 + i) * sz : 0);
  }
  __device__ __forceinline__ void load(int i) {
    const long o = at(i);
    ldv<T, V>(u + o, V, uv);
    ldv<T, V>(p + o, V, pv);
    ldv<T, V>(r + o, V, rv);
    ldv<T, V>(w + o, V, wv);
  }
  __device__ __forceinline__ void run(T a, T b, T alpha, T mi, double (&acc)[3]) {
    for (int i = 0; i < groups; i++) {
      const int m = row(i) < d.ny ? n : 0;
      const long o = at(i);
      T un[V], pn[V], rn[V];
#pragma unroll
      for (int q = 0; q < V; q++) {
        pn[q] = a * pv[q] + b * rv[q];
        un[q] = uv[q] + alpha * pn[q];
        rn[q] = rv[q] - alpha * wv[q];
        if (q < m) {
          if constexpr (MIXED) {
            const T z = mi * rn[q];
            acc[0] = acc[0] + (double)rn[q] * (double)z;
            acc[1] = acc[1] + (double)rn[q] * (double)rn[q];
          } else {
            acc[0] = acc[0] + rn[q] * rn[q];
          }
        }
      }
      if (i + 1 < groups) load(i + 1);
      stv<T, V, false>(u + o, m, un);
      stv<T, V, false>(p + o, m, pn);
      stv<T, V, false>(r + o, m, rn);
    }
  }
};

// the inner FP32 step of a mixed solve, V points per lane
template <int V>
__device__ __forceinline__ void update_inner(IterLds &L, const SolveDev &d, const TileBox &b, const SolveStat &in,
                                             SolveStat &out, const double *part, size_t np, bool first_of_solve,
                                             bool fresh, float mi, double (&acc)[3]) {
  UpdateTile<float, V, true> m(d, b, d.e32, d.p32, d.r32, d.w32, d.sy32, d.sz32);
  m.load(0);
  const Step c = update_step(L, d, in, out, part, np, first_of_solve, fresh);
  m.run((float)c.a, (float)c.b, (float)c.alpha, mi, acc);
}

__global__ __launch_bounds__(256) void sk_update(const SolveDev *__restrict__ S, const SolveStat *__restrict__ in,
                                                 SolveStat *__restrict__ out, const int2 *__restrict__ tiles,
                                                 const int *__restrict__ ntiles, double *part, size_t np) {
  __shared__ IterLds L;
  const int nt = *ntiles;
  for (int t = first_tile(nt); t < nt; t += (int)gridDim.x) {
    const int s = __builtin_amdgcn_readfirstlane(tiles[t].x), li = __builtin_amdgcn_readfirstlane(tiles[t].y);
    const SolveDev &d = S[s];
    if (in[s].done) {
      if (li == 0 && threadIdx.x == 0 && threadIdx.y == 0) out[s] = in[s];
      continue;
    }
    const TileBox b = tile_box(d, li);
    double acc[3] = {0.0, 0.0, 0.0};
    const bool fresh = t < (int)gridDim.x || tiles[t - (int)gridDim.x].x != s;
    __syncthreads();  // the previous tile's sums and step have been read
    if (!d.mixed) {
      UpdateTile<double, kSV, false> m(d, b, d.u, d.p, d.r, d.w, d.sy, d.sz);
      m.load(0);
      const Step c = update_step(L, d, in[s], out[s], part, np, li == 0, fresh);
      m.run(c.a, c.b, c.alpha, 1.0, acc);
      store_partial(acc[0], part + t, L.tile1);
      continue;
    }
    // 2D Poisson: Jacobi, 1 / diag of the 5-point operator; 3D heat: none
    const bool heat = d.kind == OPSMI_SOLVE_HEAT3D;
    const float mi = heat ? 1.0f : 0.25f;
    const int phase = in[s].phase;
    if (phase == PH_INNER) {
      if (d.sv == kSV32) update_inner<kSV32>(L, d, b, in[s], out[s], part, np, li == 0, fresh, mi, acc);
      else update_inner<kSV>(L, d, b, in[s], out[s], part, np, li == 0, fresh, mi, acc);
    } else {
      update_step(L, d, in[s], out[s], part, np, li == 0, fresh);
      if (heat) continue;  // its correction and residual ran in the sweep
      // FP64 residual r = f - A x, then the inner start from it:
      // rr = (float) r, e = 0, p = Mi rr; (r.r, rr . Mi rr, rr . rr).
      // Runs once per correction: the tile is covered in halves of 64 kSV
      // points (two doubles per lane, fewer registers for the kernel).
      const Ptr<float> ev = PF32(d.e32, d), rr = PF32(d.r32, d), p = PF32(d.p32, d);
      const Ptr<const double> x = PC(d.u, d), f = PC(d.f, d);
      TileBox bh = b;
      for (int h = 0; h < kSV32 / kSV; h++, bh.x0 += kWave * kSV)
        tile_groups<kSV>(d, bh, [&](int i, int j, int k, int n) {
          Row5<double, kSV> R;
          load5<double, kSV>(x, i, j, n, R);
          double fv[kSV];
          ldv<double, kSV>(f.at(i, j, k), n, fv);
          float q32[kSV], z32[kSV], zero[kSV];
#pragma unroll
          for (int q = 0; q < kSV; q++) {
            const double ax = op5<double, kSV>(R, q, n);
            const double v = fv[q] - ax;
            const float qv = (float)v;
            const float z = mi * qv;
            q32[q] = qv;
            z32[q] = z;
            zero[q] = 0.0f;
            if (q < n) {
              acc[0] = acc[0] + v * v;
              acc[1] = acc[1] + (double)qv * (double)z;
              acc[2] = acc[2] + (double)qv * (double)qv;
            }
          }
          stv<float, kSV, false>(ev.at(i, j, k), n, zero);
          stv<float, kSV, false>(rr.at(i, j, k), n, q32);
          stv<float, kSV, false>(p.at(i, j, k), n, z32);
        });
    }
    block_reduce<double, OPS_INC, 3>(acc, L.tile3);
    if (threadIdx.x == 0 && threadIdx.y == 0) {
      part[t] = acc[0];
      part[np + t] = acc[1];
      part[2 * np + t] = acc[2];
    }
  }
}

// the last update's sums of a batch of iterations, one workgroup a solve
__global__ __launch_bounds__(256) void sk_finish(const SolveDev *__restrict__ S, SolveStat *st, const double *part,
                                                 size_t np) {
  __shared__ double sh[16][3];
  const int s = (int)blockIdx.x;
  if (!S[s].active || st[s].done || !st[s].pending) return;
  double sum[3];
  if (S[s].mixed) {
    fold_partials<3>(part, np, 0, S[s].tile0, S[s].ntiles, sum, sh);
  } else {
    __shared__ double one[16][1];
    double s1[1];
    fold_partials<1>(part, np, 0, S[s].tile0, S[s].ntiles, s1, one);
    sum[0] = s1[0];
  }
  if (threadIdx.x == 0) advance(st[s], S[s], sum);
}

// ------------------------------------------------------------ set-up
__global__ __launch_bounds__(256) void sk_zero(double *a, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) a[i] = 0.0;
}

// heat: w = 1/K over the extended box ([-1, n] per side), u = u0 = rhs inside
__global__ __launch_bounds__(256) void sk_heat_inputs(SolveDev d, uint64_t seed) {
  const long ne = (long)(d.nx + 2) * (d.ny + 2) * (d.nz + 2);
  for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < ne; q += (long)gridDim.x * blockDim.x) {
    const int x = (int)(q % (d.nx + 2)) - 1;
    const long rest = q / (d.nx + 2);
    const int y = (int)(rest % (d.ny + 2)) - 1, z = (int)(rest / (d.ny + 2)) - 1;
    P(d.w, d)(x, y, z) = 1.0 / opsapp::heat_K(seed, x, y, z, d.nx, d.ny);
    if (x >= 0 && x < d.nx && y >= 0 && y < d.ny && z >= 0 && z < d.nz)
      P(d.u, d)(x, y, z) = opsapp::heat_rhs(seed, x, y, z, d.nx, d.ny, d.nz, 3);
  }
}

// heat: face coefficients over [0, n] per side (tea_leaf_common_init_Kx_Ky_Kz
// on the app's ext range), then the zeroed external faces x, y, z in {0, n}
__global__ __launch_bounds__(256) void sk_heat_coefs(SolveDev d) {
  const long ne = (long)(d.nx + 1) * (d.ny + 1) * (d.nz + 1);
  const Ptr<const double> w = PC(d.w, d);
  for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < ne; q += (long)gridDim.x * blockDim.x) {
    const int x = (int)(q % (d.nx + 1));
    const long rest = q / (d.nx + 1);
    const int y = (int)(rest % (d.ny + 1)), z = (int)(rest / (d.ny + 1));
    const double c = w(x, y, z);
    double kx = (w(x - 1, y, z) + c) / (2.0 * w(x - 1, y, z) * c);
    double ky = (w(x, y - 1, z) + c) / (2.0 * w(x, y - 1, z) * c);
    double kz = (w(x, y, z - 1) + c) / (2.0 * w(x, y, z - 1) * c);
    if (x == 0 || x == d.nx) kx = 0.0;
    if (y == 0 || y == d.ny) ky = 0.0;
    if (z == 0 || z == d.nz) kz = 0.0;
    P(d.kx, d)(x, y, z) = kx;
    P(d.ky, d)(x, y, z) = ky;
    P(d.kz, d)(x, y, z) = kz;
  }
}

// first residual, p = r, partial r.p per tile (grid = the solve's tiles)
__global__ __launch_bounds__(256) void sk_first_residual(SolveDev d, uint64_t seed, double *part) {
  __shared__ double sh[16][1];
  const int li = (int)blockIdx.x;
  const TileBox b = tile_box(d, li);
  if (d.kind == OPSMI_SOLVE_HEAT3D) {
    const Ptr<double> w0 = P(d.w, d), r0 = P(d.r, d);
    HeatOutInit<double, kSV, false> out{w0, r0};
    HeatMarch<double, kSV, false> m(d, b, d.u, nullptr, d.kx, d.ky, d.kz, d.sy, d.sz);
    m.start();
    m.run(1.0, 0.0, d.rx, d.ry, d.rz, out);
  }
  const Ptr<double> r = P(d.r, d), p = P(d.p, d);
  const bool poisson = d.kind == OPSMI_SOLVE_POISSON2D;
  double acc = 0.0;
  tile_groups<kSV>(d, b, [&](int x, int y, int z, int n) {
#pragma unroll
    for (int q = 0; q < kSV; q++) {
      if (q >= n) continue;
      if (poisson) r(x + q, y, z) = opsapp::poisson_rhs(seed, x + q, y, 0, d.nx, d.ny);
      const double v = r(x + q, y, z);
      p(x + q, y, z) = v;
      acc = acc + v * v;
    }
  });
  store_partial(acc, part + li, sh);
}

// mixed 3D heat, after sk_heat_inputs and sk_heat_coefs wrote 1/K into f's
// storage, x = rhs and the face coefficients: f = rhs inside, and the face
// coefficients rounded to float over the extended box
__global__ __launch_bounds__(256) void sk_mixed_heat_finish(SolveDev d) {
  const long ne = (long)(d.nx + 2) * (d.ny + 2) * (d.nz + 2);
  for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < ne; q += (long)gridDim.x * blockDim.x) {
    const int x = (int)(q % (d.nx + 2)) - 1;
    const long rest = q / (d.nx + 2);
    const int y = (int)(rest % (d.ny + 2)) - 1, z = (int)(rest / (d.ny + 2)) - 1;
    if (x >= 0 && x < d.nx && y >= 0 && y < d.ny && z >= 0 && z < d.nz) P(d.f, d)(x, y, z) = P(d.u, d)(x, y, z);
    PF32(d.kx32, d)(x, y, z) = (float)P(d.kx, d)(x, y, z);
    PF32(d.ky32, d)(x, y, z) = (float)P(d.ky, d)(x, y, z);
    PF32(d.kz32, d)(x, y, z) = (float)P(d.kz, d)(x, y, z);
  }
}

// mixed 2D Poisson: f = rhs inside (x and the FP32 fields start at zero);
// the first iteration's residual pass finds r = f
__global__ __launch_bounds__(256) void sk_mixed_inputs(SolveDev d, uint64_t seed) {
  const long n = (long)d.nx * d.ny;
  for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
    const int x = (int)(q % d.nx), y = (int)(q / d.nx);
    P(d.f, d)(x, y, 0) = opsapp::poisson_rhs(seed, x, y, 0, d.nx, d.ny);
  }
}

__global__ void sk_mixed_stat(SolveStat *q, double tol, double inner_tol, int max_iters, int max_outer) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  q->rro = q->rr0 = q->stop = q->pw = q->alpha = q->beta = 0.0;
  q->iters = 0;
  q->done = 0;
  q->max_iters = max_iters;
  q->pending = 0;
  q->rz = q->istop = q->fn = 0.0;
  q->tol = tol;
  q->inner_tol = inner_tol;
  q->phase = PH_RESID;
  q->outer = 0;
  q->max_outer = max_outer;
  q->axpby = 0;
}

__global__ __launch_bounds__(256) void sk_first_fold(SolveStat *q, const double *part, int n, double tol,
                                                     int max_iters) {
  __shared__ double sh[16][1];
  double acc[1] = {0.0};
  for (int i = (int)threadIdx.x; i < n; i += (int)blockDim.x) acc[0] = acc[0] + part[i];
  block_reduce<double, OPS_INC, 1>(acc, sh);
  if (threadIdx.x == 0) {
    q->rro = acc[0];
    q->rr0 = acc[0];
    q->stop = tol * sqrt(acc[0]);
    q->pw = q->alpha = q->beta = 0.0;
    q->iters = 0;
    q->done = 0;
    q->max_iters = max_iters;
    q->pending = 0;
    q->phase = PH_INNER;
    q->outer = 0;
    q->axpby = 0;
  }
}

// ------------------------------------------------------------ host
struct Arena {
  size_t size = 0;
  std::map<size_t, size_t> free_;  // offset -> length
  void init(size_t n) {
    size = n;
    free_.clear();
    free_[0] = n;
  }
  bool alloc(size_t n, size_t *off) {
    for (auto it = free_.begin(); it != free_.end(); ++it) {
      if (it->second < n) continue;
      *off = it->first;
      const size_t rest = it->second - n, o = it->first + n;
      free_.erase(it);
      if (rest) free_[o] = rest;
      return true;
    }
    return false;
  }
  void release(size_t off, size_t n) {
    auto it = free_.emplace(off, n).first;
    auto nx = std::next(it);
    if (nx != free_.end() && it->first + it->second == nx->first) {
      it->second += nx->second;
      free_.erase(nx);
    }
    if (it != free_.begin()) {
      auto pv = std::prev(it);
      if (pv->first + pv->second == it->first) {
        pv->second += it->second;
        free_.erase(it);
      }
    }
  }
};

struct Geometry {
  int nfields, nx, ny, nz;
  long pitch, plane, field;        // double fields, elements
  int nfields32;                   // FP32 fields (mixed solves)
  long pitch32, plane32, field32;  // elements
  size_t bytes;
};

Geometry geometry(const opsmi_solve_req &q) {
  Geometry g;
  const bool heat = q.kind == OPSMI_SOLVE_HEAT3D;
  // FP64 fields: u, p, r, w [, kx, ky, kz]; mixed: x, f [, kx, ky, kz]
  g.nfields = heat ? (q.mixed ? 5 : 7) : (q.mixed ? 2 : 4);
  g.nx = g.ny = q.n;
  g.nz = heat ? q.n : 1;
  g.pitch = ((long)g.nx + 2 + 31) / 32 * 32;
  g.plane = g.pitch * (g.ny + 2);
  // 32 lead elements put x = 0 on a 256-byte boundary; round to 256 bytes
  g.field = (g.plane * (heat ? g.nz + 2 : 1) + 32 + 31) / 32 * 32;
  // FP32 fields of a mixed solve: e, rr, p, w [, kx, ky, kz]
  g.nfields32 = q.mixed ? (heat ? 7 : 4) : 0;
  g.pitch32 = ((long)g.nx + 2 + 63) / 64 * 64;
  g.plane32 = g.pitch32 * (g.ny + 2);
  // 64 lead elements put x = 0 on a 256-byte boundary
  g.field32 = (g.plane32 * (heat ? g.nz + 2 : 1) + 64 + 63) / 64 * 64;
  g.bytes = (size_t)g.nfields * g.field * sizeof(double) + (size_t)g.nfields32 * g.field32 * sizeof(float);
  return g;
}

struct Req {
  opsmi_solve_req q;
  int state = 0;  // 0 queued, 1 active, 2 done (memory held until fetch/release)
  int slot = -1;
  size_t off = 0, bytes = 0;
  SolveDev dev{};
};

}  // namespace

struct opsmi_server_s {
  hipStream_t stream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int iters_per_launch = 8, use_graph = 1, max_slots = 0, grid = 0;
  size_t budget = 0, in_use = 0;
  size_t max_tiles = 0, cap_tiles = 0;  // tiles a full arena can need, tiles the tables hold now
  char *arena_base = nullptr;
  Arena arena;
  SolveDev *d_solves = nullptr;
  SolveStat *d_stat = nullptr;  // two copies of max_slots
  int2 *d_tiles = nullptr;
  int *d_ntiles = nullptr;
  double *d_part = nullptr;  // kPart planes of cap_tiles; set-up sums too (no iteration leaves any behind)
  SolveStat *h_stat = nullptr;  // pinned
  Staging staging;              // fetched solutions
  std::vector<SolveDev> h_solves;
  std::vector<int> slot_req;
  std::vector<int2> h_tiles;
  int h_ntiles = 0;
  bool dirty = true;
  std::deque<int> queue;
  std::map<int, Req> reqs;
  std::deque<opsmi_solve_done> completed;
  int next_id = 0, n_active = 0;
  long tiles_active = 0;  // tiles of the admitted solves (the next table)
  // tile parameter per size class (defaults; opsmi_serve_autotune measures)
  int chunk3d[3] = {kChunk3D[0], kChunk3D[1], kChunk3D[2]};
  int chunk3d_mixed[3] = {kChunk3D[0], kChunk3D[1], kChunk3D[2]};  // FP32-inner heat solves
  int rows2d[3] = {kRows2D[0], kRows2D[1], kRows2D[2]};
  int rows2d_mixed[3] = {kRows2D[0], kRows2D[1], kRows2D[2]};  // FP32-inner solves
};

namespace {

void check_req(const opsmi_solve_req &q) {
  if (q.kind != OPSMI_SOLVE_POISSON2D && q.kind != OPSMI_SOLVE_HEAT3D)
    fail(OPS_INVALID_ARGUMENT, cat("opsmi_serve_submit: unknown solve kind ", q.kind));
  if (q.n < 2 || q.n > (q.kind == OPSMI_SOLVE_HEAT3D ? 2048 : 65536))
    fail(OPS_INVALID_ARGUMENT, cat("opsmi_serve_submit: grid side ", q.n, " out of range"));
  if (!(q.tol > 0.0) || q.max_iters < 1)
    fail(OPS_INVALID_ARGUMENT, "opsmi_serve_submit: tol must be > 0 and max_iters >= 1");
  if (q.mixed != 0 && q.mixed != 1)
    fail(OPS_INVALID_ARGUMENT, "opsmi_serve_submit: mixed must be 0 (FP64) or 1 (FP32-inner refinement)");
}

// tile parameter of a solve: z planes per 3D tile, rows per wave of a 2D
// tile; one value per size class (three classes per kind)
int size_class(int kind, int n) {
  if (kind == OPSMI_SOLVE_HEAT3D) return n < 64 ? 0 : (n < 128 ? 1 : 2);
  return n < 256 ? 0 : (n < 1024 ? 1 : 2);
}
int tile_param(opsmi_server S, int kind, int n, int mixed) {
  if (kind == OPSMI_SOLVE_HEAT3D) return mixed ? S->chunk3d_mixed[size_class(kind, n)] : S->chunk3d[size_class(kind, n)];
  return mixed ? S->rows2d_mixed[size_class(kind, n)] : S->rows2d[size_class(kind, n)];
}

long tiles_of(const opsmi_solve_req &q, int param, int *tx, int *ty) {
  const Geometry g = geometry(q);
  const int w = kWave * (q.mixed && q.kind == OPSMI_SOLVE_POISSON2D ? kSV32 : kSV);  // tile width in points
  *tx = (g.nx + w - 1) / w;
  if (q.kind == OPSMI_SOLVE_HEAT3D) {
    *ty = (g.ny + kWavesPerBlock - 1) / kWavesPerBlock;
    return (long)*tx * *ty * ((g.nz + param - 1) / param);
  }
  *ty = (g.ny + kWavesPerBlock * param - 1) / (kWavesPerBlock * param);
  return (long)*tx * *ty;
}

void launch_iterations(opsmi_server S, hipStream_t st, int iters) {
  const dim3 blk(kWave, kWavesPerBlock);
  for (int k = 0; k < iters; k++) {
    hipLaunchKernelGGL(sk_sweep, dim3(S->grid), blk, 0, st, S->d_solves, S->d_stat, S->d_stat + S->max_slots,
                       S->d_tiles, S->d_ntiles, S->d_part, S->cap_tiles);
    hipLaunchKernelGGL(sk_update, dim3(S->grid), blk, 0, st, S->d_solves, S->d_stat + S->max_slots, S->d_stat,
                       S->d_tiles, S->d_ntiles, S->d_part, S->cap_tiles);
  }
  hipLaunchKernelGGL(sk_finish, dim3(S->max_slots), dim3(256), 0, st, S->d_solves, S->d_stat, S->d_part,
                     S->cap_tiles);
}

// Tables (tile list and partial sums) for `need` tiles; false when there is no
// memory for them.  Sized for every tile the arena could ever hold they would
// take 0.5 % of the budget beside it (1.2 GB at 200 GB), most of it never used:
// they start at kFirstTiles and at least double.
constexpr size_t kFirstTiles = 16384;
bool have_tables(opsmi_server S, size_t need) {
  if (need <= S->cap_tiles) return true;
  OPSMI_HIP(hipStreamSynchronize(S->stream));  // set-up kernels use the sums
  for (size_t cap : {std::min(S->max_tiles, std::max(need, 2 * S->cap_tiles)), need}) {
    int2 *tiles = nullptr;
    double *part = nullptr;
    hipError_t e = hipMalloc(&tiles, sizeof(int2) * cap);
    if (e == hipSuccess) e = hipMalloc(&part, sizeof(double) * kPart * cap);
    if (e == hipSuccess) {
      (void)hipFree(S->d_tiles);
      (void)hipFree(S->d_part);
      S->d_tiles = tiles;
      S->d_part = part;
      S->cap_tiles = cap;
      S->dirty = true;
      // the captured launches hold the old addresses
      if (S->exec) OPSMI_HIP(hipGraphExecDestroy(S->exec));
      if (S->graph) OPSMI_HIP(hipGraphDestroy(S->graph));
      S->exec = nullptr;
      S->graph = nullptr;
      return true;
    }
    (void)hipFree(tiles);
    if (e != hipErrorOutOfMemory) OPSMI_HIP(e);
    (void)hipGetLastError();
  }
  return false;
}

// admits the queue head while a slot and memory are free; sets up on device
void admit(opsmi_server S) {
  while (!S->queue.empty()) {
    const int id = S->queue.front();
    Req &R = S->reqs[id];
    int slot = -1;
    for (int s = 0; s < S->max_slots; s++)
      if (S->slot_req[s] < 0) {
        slot = s;
        break;
      }
    if (slot < 0) return;
    const Geometry g = geometry(R.q);
    size_t off;
    if (!S->arena.alloc(g.bytes, &off)) return;
    int tx, ty;
    const int param = tile_param(S, R.q.kind, R.q.n, R.q.mixed);
    const long nt = tiles_of(R.q, param, &tx, &ty);
    if ((size_t)(S->tiles_active + nt) > S->max_tiles) {
      S->arena.release(off, g.bytes);
      return;
    }
    if (!have_tables(S, (size_t)(S->tiles_active + nt))) {
      S->arena.release(off, g.bytes);
      if (S->n_active == 0) fail(OPS_RUNTIME_ERROR, "opsmi_serve: no device memory for the tile tables of a solve");
      return;  // with the tables there are, once the solves before it are done
    }
    S->tiles_active += nt;
    S->queue.pop_front();
    R.state = 1;
    R.slot = slot;
    R.off = off;
    R.bytes = g.bytes;
    S->in_use += g.bytes;
    S->slot_req[slot] = id;
    // fields: u, p, r, w [, kx, ky, kz]; mixed: x, f [, kx, ky, kz], then
    // FP32 e, rr, p, w [, kx, ky, kz]
    double *base = (double *)(S->arena_base + off);
    double *f[7] = {};
    for (int i = 0; i < g.nfields; i++) f[i] = base + (size_t)i * g.field;
    // element (-1,-1,-1) sits at field + 31, so x = 0 starts a 256-byte line
    const long lead = 32 + g.pitch + (R.q.kind == OPSMI_SOLVE_HEAT3D ? g.plane : 0);
    SolveDev d{};
    const bool heat = R.q.kind == OPSMI_SOLVE_HEAT3D;
    if (R.q.mixed) {
      float *b32 = (float *)(base + (size_t)g.nfields * g.field);
      // float element (-1,-1[,-1]) at +63
      const long lead32 = 64 + g.pitch32 + (heat ? g.plane32 : 0);
      d.u = f[0] + lead;
      d.f = f[1] + lead;
      d.e32 = b32 + lead32;
      d.r32 = b32 + g.field32 + lead32;
      d.p32 = b32 + 2 * g.field32 + lead32;
      d.w32 = b32 + 3 * g.field32 + lead32;
      if (heat) {
        d.kx = f[2] + lead;
        d.ky = f[3] + lead;
        d.kz = f[4] + lead;
        d.kx32 = b32 + 4 * g.field32 + lead32;
        d.ky32 = b32 + 5 * g.field32 + lead32;
        d.kz32 = b32 + 6 * g.field32 + lead32;
      }
      d.sy32 = g.pitch32;
      d.sz32 = heat ? g.plane32 : 0;
      d.mixed = 1;
    } else {
      d.u = f[0] + lead;
      d.p = f[1] + lead;
      d.r = f[2] + lead;
      d.w = f[3] + lead;
    }
    if (heat && !R.q.mixed) {
      d.kx = f[4] + lead;
      d.ky = f[5] + lead;
      d.kz = f[6] + lead;
    }
    d.sy = g.pitch;
    d.sz = g.plane;
    d.kind = R.q.kind;
    d.nx = g.nx;
    d.ny = g.ny;
    d.nz = g.nz;
    d.tx = tx;
    d.ty = ty;
    d.chunk = param;
    d.sv = R.q.mixed && R.q.kind == OPSMI_SOLVE_POISSON2D ? kSV32 : kSV;
    d.tile0 = 0;
    d.ntiles = (int)nt;
    d.active = 1;
    d.rx = d.ry = d.rz = 1.0;
    R.dev = d;
    hipStream_t st = S->stream;
    const size_t nall = g.bytes / sizeof(double);
    hipLaunchKernelGGL(sk_zero, dim3((unsigned)std::min<size_t>((nall + 255) / 256, 4096)), dim3(256), 0, st, base,
                       nall);
    if (R.q.mixed && heat) {
      // 1/K into f's storage and x = rhs (sk_heat_inputs), the face
      // coefficients from them, then f = rhs and the float coefficients
      SolveDev dk = d;
      dk.w = d.f;
      const long ne = (long)(g.nx + 2) * (g.ny + 2) * (g.nz + 2);
      const unsigned gb = (unsigned)std::min<long>((ne + 255) / 256, 4096);
      hipLaunchKernelGGL(sk_heat_inputs, dim3(gb), dim3(256), 0, st, dk, R.q.seed);
      hipLaunchKernelGGL(sk_heat_coefs, dim3(gb), dim3(256), 0, st, dk);
      hipLaunchKernelGGL(sk_mixed_heat_finish, dim3(gb), dim3(256), 0, st, d);
    } else if (R.q.mixed) {
      const long ni = (long)g.nx * g.ny;
      hipLaunchKernelGGL(sk_mixed_inputs, dim3((unsigned)std::min<long>((ni + 255) / 256, 4096)), dim3(256), 0, st, d,
                         R.q.seed);
    }
    if (R.q.mixed) {
      // inner FP32 solves run to 1e-6 of their initial residual (or
      // tol / (2 relres)): on the 60-request serving mix 1e-4 took 100 502
      // iterations, 1e-5 96 018, 1e-6 90 305, 1e-7 91 951, 1e-8 96 738
      // (OPSMI_SERVE_INNER_TOL overrides)
      static const double inner_tol = [] {
        const char *e = getenv("OPSMI_SERVE_INNER_TOL");
        return e ? atof(e) : 1e-6;
      }();
      hipLaunchKernelGGL(sk_mixed_stat, dim3(1), dim3(64), 0, st, S->d_stat + slot, R.q.tol, inner_tol,
                         R.q.max_iters, 30);
      OPSMI_HIP(hipGetLastError());
      S->dirty = true;
      S->n_active++;
      continue;
    }
    if (R.q.kind == OPSMI_SOLVE_HEAT3D) {
      const long ne = (long)(g.nx + 2) * (g.ny + 2) * (g.nz + 2);
      const unsigned gb = (unsigned)std::min<long>((ne + 255) / 256, 4096);
      hipLaunchKernelGGL(sk_heat_inputs, dim3(gb), dim3(256), 0, st, d, R.q.seed);
      hipLaunchKernelGGL(sk_heat_coefs, dim3(gb), dim3(256), 0, st, d);
    }
    hipLaunchKernelGGL(sk_first_residual, dim3((unsigned)nt), dim3(kWave, kWavesPerBlock), 0, st, d, R.q.seed,
                       S->d_part);
    hipLaunchKernelGGL(sk_first_fold, dim3(1), dim3(256), 0, st, S->d_stat + slot, (const double *)S->d_part,
                       (int)nt, R.q.tol, R.q.max_iters);
    OPSMI_HIP(hipGetLastError());
    S->dirty = true;
    S->n_active++;
  }
}

void rebuild_tables(opsmi_server S) {
  S->h_tiles.clear();
  for (int s = 0; s < S->max_slots; s++) {
    SolveDev &d = S->h_solves[s];
    const int rid = S->slot_req[s];
    if (rid < 0) {
      d = SolveDev{};
      continue;
    }
    d = S->reqs[rid].dev;
    d.tile0 = (int)S->h_tiles.size();
    for (int i = 0; i < d.ntiles; i++) S->h_tiles.push_back(make_int2(s, i));
  }
  S->h_ntiles = (int)S->h_tiles.size();
  OPSMI_HIP(hipMemcpyAsync(S->d_solves, S->h_solves.data(), sizeof(SolveDev) * S->max_slots, hipMemcpyHostToDevice,
                           S->stream));
  if (S->h_ntiles)
    OPSMI_HIP(hipMemcpyAsync(S->d_tiles, S->h_tiles.data(), sizeof(int2) * S->h_ntiles, hipMemcpyHostToDevice,
                             S->stream));
  OPSMI_HIP(hipMemcpyAsync(S->d_ntiles, &S->h_ntiles, sizeof(int), hipMemcpyHostToDevice, S->stream));
  OPSMI_HIP(hipStreamSynchronize(S->stream));  // host vectors may change after this
  S->dirty = false;
}

Req &find(opsmi_server S, int id) {
  auto it = S->reqs.find(id);
  if (it == S->reqs.end()) fail(OPS_INVALID_ARGUMENT, cat("opsmi_serve: unknown solve id ", id));
  return it->second;
}

void free_req(opsmi_server S, int id) {
  Req &R = find(S, id);
  if (R.state != 2) fail(OPS_INVALID_ARGUMENT, cat("opsmi_serve: solve ", id, " has not completed"));
  S->arena.release(R.off, R.bytes);
  S->in_use -= R.bytes;
  S->reqs.erase(id);
}

}  // namespace

extern "C" {

size_t opsmi_serve_request_bytes(const opsmi_solve_req *req) {
  OPSMI_API_BEGIN
  if (!req) fail(OPS_INVALID_ARGUMENT, "opsmi_serve_request_bytes: NULL request");
  check_req(*req);
  return geometry(*req).bytes;
  OPSMI_API_END(0)
}

opsmi_server opsmi_serve_create(size_t hbm_budget, int max_slots, int iters_per_launch, int use_graph) {
  OPSMI_API_BEGIN
  require_init();
  if (max_slots < 1 || max_slots > 65536 || iters_per_launch < 1 || iters_per_launch > 1024)
    fail(OPS_INVALID_ARGUMENT, "opsmi_serve_create: max_slots in [1, 65536], iters_per_launch in [1, 1024]");
  if (hbm_budget < (1u << 20)) fail(OPS_INVALID_ARGUMENT, "opsmi_serve_create: budget below 1 MiB");
  opsmi_server S = new opsmi_server_s();
  S->budget = hbm_budget / 256 * 256;
  S->max_slots = max_slots;
  S->iters_per_launch = iters_per_launch;
  S->use_graph = use_graph ? 1 : 0;
  // OPSMI_SERVE_GRAPH=0 forces direct launches (same kernels; for profilers)
  if (const char *e = getenv("OPSMI_SERVE_GRAPH"))
    if (e[0] == '0') S->use_graph = 0;
  S->grid = inst().num_cus * 8;
  // the least memory a tile stands for: 128 x 4 points (one row per wave)
  // over 4 fields, half of it used in the worst row (129 points in rows of
  // 160); solves of fewer points than that have at most 8 tiles
  S->max_tiles = std::min<size_t>(S->budget / 8192 + (size_t)max_slots * 8,
                                  (size_t)1 << 25);
  OPSMI_HIP(hipStreamCreateWithFlags(&S->stream, hipStreamNonBlocking));
  OPSMI_HIP(hipMalloc(&S->arena_base, S->budget));
  S->arena.init(S->budget);
  OPSMI_HIP(hipMalloc(&S->d_solves, sizeof(SolveDev) * max_slots));
  OPSMI_HIP(hipMalloc(&S->d_stat, 2 * sizeof(SolveStat) * max_slots));
  OPSMI_HIP(hipMalloc(&S->d_ntiles, sizeof(int)));
  if (!have_tables(S, std::min(S->max_tiles, kFirstTiles))) OPSMI_HIP(hipErrorOutOfMemory);
  OPSMI_HIP(hipHostMalloc((void **)&S->h_stat, sizeof(SolveStat) * max_slots, hipHostMallocDefault));
  OPSMI_HIP(hipMemsetAsync(S->d_stat, 0, 2 * sizeof(SolveStat) * max_slots, S->stream));
  S->h_solves.assign(max_slots, SolveDev{});
  S->slot_req.assign(max_slots, -1);
  rebuild_tables(S);
  return S;
  OPSMI_API_END(nullptr)
}

int opsmi_serve_submit(opsmi_server S, const opsmi_solve_req *req) {
  OPSMI_API_BEGIN
  if (!S || !req) fail(OPS_INVALID_ARGUMENT, "opsmi_serve_submit: NULL argument");
  check_req(*req);
  const Geometry g = geometry(*req);
  if (g.bytes > S->budget)
    fail(OPS_INVALID_ARGUMENT, cat("opsmi_serve_submit: solve needs ", g.bytes, " bytes, budget is ", S->budget));
  int tx, ty;
  if ((size_t)tiles_of(*req, tile_param(S, req->kind, req->n, req->mixed),
                       &tx, &ty) > S->max_tiles)
    fail(OPS_INVALID_ARGUMENT, "opsmi_serve_submit: solve has more tiles than the tile table holds");
  const int id = S->next_id++;
  Req R;
  R.q = *req;
  S->reqs[id] = R;
  S->queue.push_back(id);
  return id;
  OPSMI_API_END(-1)
}

int opsmi_serve_step(opsmi_server S) {
  OPSMI_API_BEGIN
  if (!S) fail(OPS_INVALID_ARGUMENT, "opsmi_serve_step: NULL server");
  // admission: queue head first; set-up kernels run on the server stream
  admit(S);
  if (S->dirty) rebuild_tables(S);
  if (S->n_active > 0) {
    if (S->use_graph) {
      if (!S->exec) {
        OPSMI_HIP(hipStreamBeginCapture(S->stream, hipStreamCaptureModeThreadLocal));
        launch_iterations(S, S->stream, S->iters_per_launch);
        OPSMI_HIP(hipStreamEndCapture(S->stream, &S->graph));
        OPSMI_HIP(hipGraphInstantiate(&S->exec, S->graph, nullptr, nullptr, 0));
      }
      OPSMI_HIP(hipGraphLaunch(S->exec, S->stream));
    } else {
      launch_iterations(S, S->stream, S->iters_per_launch);
      OPSMI_HIP(hipGetLastError());
    }
    OPSMI_HIP(hipMemcpyAsync(S->h_stat, S->d_stat, sizeof(SolveStat) * S->max_slots, hipMemcpyDeviceToHost,
                             S->stream));
    OPSMI_HIP(hipStreamSynchronize(S->stream));
    for (int s = 0; s < S->max_slots; s++) {
      const int rid = S->slot_req[s];
      if (rid < 0 || !S->h_stat[s].done) continue;
      Req &R = S->reqs[rid];
      R.state = 2;
      R.slot = -1;
      S->slot_req[s] = -1;
      S->n_active--;
      S->tiles_active -= R.dev.ntiles;
      S->dirty = true;
      opsmi_solve_done c;
      c.id = rid;
      c.status = S->h_stat[s].done;
      c.iters = S->h_stat[s].iters;
      c.outer = S->h_stat[s].outer;
      c.rr0 = S->h_stat[s].rr0;
      c.rr = S->h_stat[s].rro;
      S->completed.push_back(c);
    }
  }
  return S->n_active + (int)S->queue.size();
  OPSMI_API_END(-1)
}

int opsmi_serve_completed(opsmi_server S, opsmi_solve_done *out, int cap) {
  OPSMI_API_BEGIN
  if (!S || (!out && cap > 0)) fail(OPS_INVALID_ARGUMENT, "opsmi_serve_completed: NULL argument");
  int n = 0;
  while (n < cap && !S->completed.empty()) {
    out[n++] = S->completed.front();
    S->completed.pop_front();
  }
  return n;
  OPSMI_API_END(-1)
}

int opsmi_serve_fetch(opsmi_server S, int id, double *out) {
  OPSMI_API_BEGIN
  if (!S || !out) fail(OPS_INVALID_ARGUMENT, "opsmi_serve_fetch: NULL argument");
  Req &R = find(S, id);
  if (R.state != 2) fail(OPS_INVALID_ARGUMENT, cat("opsmi_serve_fetch: solve ", id, " has not completed"));
  const SolveDev &d = R.dev;
  Box b;
  b.base = (char *)d.u;
  b.pitch = d.sy * 8;
  b.plane = d.sz * 8;
  b.width = (size_t)d.nx * 8;
  b.rows = (unsigned)d.ny;
  b.planes = (unsigned)d.nz;
  if (device_pointer(out)) {
    for (int z = 0; z < d.nz; z++)
      OPSMI_HIP(hipMemcpy2DAsync(out + (size_t)z * d.nx * d.ny, b.width, d.u + (long)z * d.sz, b.pitch, b.width,
                                 (size_t)d.ny, hipMemcpyDeviceToDevice, S->stream));
    OPSMI_HIP(hipStreamSynchronize(S->stream));
  } else {
    box_copy(S->staging, S->stream, b, (char *)out, false);
  }
  free_req(S, id);
  return 0;
  OPSMI_API_END(-1)
}

int opsmi_serve_release(opsmi_server S, int id) {
  OPSMI_API_BEGIN
  if (!S) fail(OPS_INVALID_ARGUMENT, "opsmi_serve_release: NULL server");
  free_req(S, id);
  return 0;
  OPSMI_API_END(-1)
}

// Tile-shape autotuner: for each kind and size class, a solve of a
// representative size is set up alone and `iters` CG iterations are timed
// (HIP events on the server stream, after two untimed ones) for each
// candidate tile parameter; the fastest is kept for that class.  Classes whose
// representative does not fit the budget keep their default.
int opsmi_serve_autotune(opsmi_server S, int iters) {
  OPSMI_API_BEGIN
  if (!S) fail(OPS_INVALID_ARGUMENT, "opsmi_serve_autotune: NULL server");
  if (S->n_active || !S->queue.empty()) fail(OPS_INVALID_ARGUMENT, "opsmi_serve_autotune: the server must be idle");
  if (iters < 1 || iters > 1000) fail(OPS_INVALID_ARGUMENT, "opsmi_serve_autotune: iters in [1, 1000]");
  static const int rep[2][3] = {{160, 512, 1536}, {48, 96, 192}};
  static const int cand2[] = {1, 2, 4, 8}, cand3[] = {4, 8, 16, 32};
  hipEvent_t e0, e1;
  OPSMI_HIP(hipEventCreate(&e0));
  OPSMI_HIP(hipEventCreate(&e1));
  // FP64 and FP32-inner solves get their own tables (the FP32 kernels move
  // half the bytes per point and may prefer other tiles): km 0 Poisson,
  // 1 heat, 2 FP32-inner Poisson, 3 FP32-inner heat
  for (int km = 0; km < 4; km++)
    for (int cls = 0; cls < 3; cls++) {
      const int kind = km % 2 == 1 ? OPSMI_SOLVE_HEAT3D : OPSMI_SOLVE_POISSON2D, mixed = km >= 2;
      opsmi_solve_req q{kind, rep[kind][cls], 12345, 1e-300, 1 << 30, mixed};
      if (geometry(q).bytes > S->budget) continue;
      int *slot_param = kind == OPSMI_SOLVE_HEAT3D ? (mixed ? &S->chunk3d_mixed[cls] : &S->chunk3d[cls])
                                                   : (mixed ? &S->rows2d_mixed[cls] : &S->rows2d[cls]);
      const int *cand = kind == OPSMI_SOLVE_HEAT3D ? cand3 : cand2;
      const int nc = 4;
      int best = *slot_param;
      float best_ms = 1e30f;
      for (int c = 0; c < nc; c++) {
        *slot_param = cand[c];
        int tx, ty;
        if ((size_t)tiles_of(q, cand[c], &tx, &ty) > S->max_tiles) continue;
        const int id = S->next_id++;
        Req R;
        R.q = q;
        S->reqs[id] = R;
        S->queue.push_back(id);
        admit(S);
        if (S->n_active != 1) {  // memory held by results not yet fetched
          S->queue.pop_back();
          S->reqs.erase(id);
          continue;
        }
        rebuild_tables(S);
        launch_iterations(S, S->stream, 2);
        OPSMI_HIP(hipEventRecord(e0, S->stream));
        launch_iterations(S, S->stream, iters);
        OPSMI_HIP(hipEventRecord(e1, S->stream));
        OPSMI_HIP(hipEventSynchronize(e1));
        float ms = 0;
        OPSMI_HIP(hipEventElapsedTime(&ms, e0, e1));
        if (ms < best_ms) {
          best_ms = ms;
          best = cand[c];
        }
        Req &T = S->reqs[id];
        S->slot_req[T.slot] = -1;
        S->tiles_active -= T.dev.ntiles;
        S->n_active--;
        T.state = 2;
        free_req(S, id);
        rebuild_tables(S);
      }
      *slot_param = best;
    }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return 0;
  OPSMI_API_END(-1)
}

int opsmi_serve_tile_param(opsmi_server S, int kind, int n) {
  OPSMI_API_BEGIN
  if (!S) fail(OPS_INVALID_ARGUMENT, "opsmi_serve_tile_param: NULL server");
  if (kind != OPSMI_SOLVE_POISSON2D && kind != OPSMI_SOLVE_HEAT3D)
    fail(OPS_INVALID_ARGUMENT, cat("opsmi_serve_tile_param: unknown solve kind ", kind));
  return tile_param(S, kind, n, 0);
  OPSMI_API_END(-1)
}

size_t opsmi_serve_bytes_in_use(opsmi_server S) { return S ? S->in_use : 0; }
int opsmi_serve_active(opsmi_server S) { return S ? S->n_active : 0; }
int opsmi_serve_queued(opsmi_server S) { return S ? (int)S->queue.size() : 0; }

void opsmi_serve_destroy(opsmi_server S) {
  if (!S) return;
  if (S->stream) (void)hipStreamSynchronize(S->stream);
  if (S->exec) (void)hipGraphExecDestroy(S->exec);
  if (S->graph) (void)hipGraphDestroy(S->graph);
  (void)hipFree(S->arena_base);
  (void)hipFree(S->d_solves);
  (void)hipFree(S->d_stat);
  (void)hipFree(S->d_tiles);
  (void)hipFree(S->d_ntiles);
  (void)hipFree(S->d_part);
  (void)hipHostFree(S->h_stat);
  S->staging.release();
  if (S->stream) (void)hipStreamDestroy(S->stream);
  delete S;
}

}  // extern "C"
