// Batched tridiagonal solves behind ops_tridMultiDimBatch[_Inc]
// (ops/c/include/ops_tridiag.h:45-83, ops/c/src/tridiag/ops_tridiag.cpp:
// 78-249).  The reference hands raw pointers to the external libtrid
// (tridDmtsvStridedBatch); this file is the backend's own solver.
//
// Thomas: one thread per system.  Lines are numbered so that consecutive
// threads take systems that are neighbours in x (for solves along y and z the
// loads of a wave are then contiguous).  The forward sweep keeps the modified
// super-diagonal c' and right-hand side d' in a step-major scratch array
// ([step][line]), so scratch traffic is coalesced for every direction.
// Arithmetic is the reciprocal form
//   r = 1/(b_i - a_i c'_{i-1});  d'_i = r (d_i - a_i d'_{i-1});  c'_i = r c_i
//   x_i = d'_i - c'_i x_{i+1}
// with contraction off, so results equal the CPU restatement bit for bit.
//
// PCR (strategy PCR): log2(n) steps of parallel cyclic reduction (Hockney
// 1965) in registers and LDS; a_0 and c_{n-1} are taken as 0.
#include "engine.h"

using namespace opsmi;

struct ops_tridsolver_params_c {
  int strategy;
};

namespace {

struct LineGeo {
  long n;         // system length
  long stride;    // element stride along the solve dimension
  long count;     // number of systems
  int e0;         // extent of the first other dimension (fastest)
  long s0, s1;    // element strides of the two other dimensions
};

__device__ __forceinline__ long line_offset(const LineGeo &g, long id) {
  // (a 64-bit division takes some hundred instructions)
  const long i1 = id >> 32 ? id / g.e0 : (long)((unsigned)id / (unsigned)g.e0), i0 = id - i1 * g.e0;
  return i0 * g.s0 + i1 * g.s1;
}

// The recurrence is serial per system but its loads are not: the passes
// run in blocks of P steps, and while a block's recurrence runs the next
// block's loads are already in flight (two register sets, the loop unrolled
// by two so each set has fixed registers), so a thread waits on memory once
// per pass rather than once per block.  Loads of the block past the end are
// clamped to the last step (in bounds, never used), so the loads and the
// recurrence of full blocks carry no branches (a branch join would make the
// compiler wait for every load in flight); the last, partial block runs with
// per-step conditions.  The arithmetic and its order are those of the plain
// loop.  Without _Inc, d' is written in place into d (the backward pass
// overwrites it with x), so only c' goes through the scratch; _Inc leaves d
// untouched and keeps d' in scratch too.  The forward pass reads a, b, c, d
// once, with the non-temporal hint.
constexpr int kPre = 8;

template <class T, int P>
struct FwdBuf {
  T a[P], b[P], c[P], d[P];
};
template <class T, int P>
struct BwdBuf {
  T c[P], d[P], u[P];
};

template <class T, bool INC, int P>
__global__ __launch_bounds__(256) void k_thomas(const T *__restrict__ a, const T *__restrict__ b,
                                                const T *__restrict__ c, T *__restrict__ d, T *__restrict__ u,
                                                T *__restrict__ cs, T *__restrict__ ds, LineGeo g) {
  const long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= g.count) return;
  const long o = line_offset(g, id);
  const long s = g.stride, L = g.count, n = g.n;
  const T *ap = a + o, *bp = b + o, *cp = c + o;
  T *dp = d + o;
  T bb = (T)1.0 / bp[0];
  T cprev = bb * cp[0];
  T dprev = bb * dp[0];
  cs[id] = cprev;
  if (INC) ds[id] = dprev;
  else dp[0] = dprev;
  // ---- forward: steps 1 .. n-1
  auto fload = [&](long i0, FwdBuf<T, P> &f) {
#pragma unroll
    for (int k = 0; k < P; k++) {
      const long i = min(i0 + k, n - 1);
      f.a[k] = ldg<T, true>(ap + i * s);
      f.b[k] = ldg<T, true>(bp + i * s);
      f.c[k] = ldg<T, true>(cp + i * s);
      f.d[k] = ldg<T, true>(dp + i * s);
    }
  };
  auto fstep = [&](const FwdBuf<T, P> &f, int k, long i) {
    bb = (T)1.0 / (f.b[k] - f.a[k] * cprev);
    dprev = bb * (f.d[k] - f.a[k] * dprev);
    cprev = bb * f.c[k];
    cs[i * L + id] = cprev;
    if (INC) ds[i * L + id] = dprev;
    else dp[i * s] = dprev;
  };
  auto ffull = [&](const FwdBuf<T, P> &f, long i0) {
#pragma unroll
    for (int k = 0; k < P; k++) fstep(f, k, i0 + k);
  };
  auto ftail = [&](const FwdBuf<T, P> &f, long i0) {
#pragma unroll
    for (int k = 0; k < P; k++)
      if (i0 + k < n) fstep(f, k, i0 + k);
  };
  if (n > 1) {
    FwdBuf<T, P> X, Y;
    long i0 = 1;
    fload(i0, X);
    while (true) {
      if (i0 + P > n) {
        ftail(X, i0);
        break;
      }
      fload(i0 + P, Y);
      ffull(X, i0);
      i0 += P;
      if (i0 >= n) break;
      if (i0 + P > n) {
        ftail(Y, i0);
        break;
      }
      fload(i0 + P, X);
      ffull(Y, i0);
      i0 += P;
      if (i0 >= n) break;
    }
  }
  // ---- backward: x_{n-1} = d'_{n-1}, then steps n-2 .. 0
  T x = dprev;
  if (INC) u[o + (n - 1) * s] = u[o + (n - 1) * s] + x;
  else dp[(n - 1) * s] = x;
  auto bload = [&](long i1, BwdBuf<T, P> &w) {
#pragma unroll
    for (int k = 0; k < P; k++) {
      const long i = max(i1 - k, 0L);
      w.c[k] = cs[i * L + id];
      w.d[k] = INC ? ds[i * L + id] : dp[i * s];
      if (INC) w.u[k] = u[o + i * s];
    }
  };
  auto bstep = [&](const BwdBuf<T, P> &w, int k, long i) {
    x = w.d[k] - w.c[k] * x;
    if (INC) u[o + i * s] = w.u[k] + x;
    else dp[i * s] = x;
  };
  auto bfull = [&](const BwdBuf<T, P> &w, long i1) {
#pragma unroll
    for (int k = 0; k < P; k++) bstep(w, k, i1 - k);
  };
  auto btail = [&](const BwdBuf<T, P> &w, long i1) {
#pragma unroll
    for (int k = 0; k < P; k++)
      if (i1 - k >= 0) bstep(w, k, i1 - k);
  };
  if (n > 1) {
    BwdBuf<T, P> X, Y;
    long i1 = n - 2;
    bload(i1, X);
    while (true) {
      if (i1 - P + 1 < 0) {
        btail(X, i1);
        break;
      }
      bload(i1 - P, Y);
      bfull(X, i1);
      i1 -= P;
      if (i1 < 0) break;
      if (i1 - P + 1 < 0) {
        btail(Y, i1);
        break;
      }
      bload(i1 - P, X);
      bfull(Y, i1);
      i1 -= P;
      if (i1 < 0) break;
    }
  }
}

// Solves along x (element stride 1).  One thread per system would make each
// load of a wave touch 64 rows (64 cache lines); here a one-wave workgroup
// takes NS systems (64, or 32 where 64 would leave SIMDs without a wave) and
// moves them through LDS in chunks of kChunk steps: the
// wave loads a chunk of a, b, c, d with row-contiguous V-wide loads (kChunk/V
// lanes per system), stores it transposed ([step][system]) in LDS, and each
// lane runs the same recurrence as k_thomas on its system from LDS, writing
// c' and d' to the step-major scratch.  The next chunk's loads are issued
// before the recurrence runs.  The backward pass reads c', d' per step
// (coalesced), puts a chunk of x in LDS and writes it (or adds it to u) with
// row-contiguous stores.  Same operations in the same order as k_thomas.
constexpr int kChunk = 16;

template <class T, int V, int NS>
struct XChunk {
  static constexpr int kLanesPerSys = kChunk / V;      // lanes covering one system's chunk
  static constexpr int kSysPerLoad = 64 / kLanesPerSys;  // systems per wave-wide load
  static constexpr int kLoads = NS / kSysPerLoad;        // loads per array per chunk
};

template <class T, int V, int NS, bool INC>
__global__ __launch_bounds__(64) void k_thomas_x(const T *__restrict__ a, const T *__restrict__ b,
                                                 const T *__restrict__ c, T *__restrict__ d, T *__restrict__ u,
                                                 T *__restrict__ cs, T *__restrict__ ds, LineGeo g) {
  using XC = XChunk<T, V, NS>;
  __shared__ T LA[kChunk][NS + 1], LB[kChunk][NS + 1], LC[kChunk][NS + 1], LD[kChunk][NS + 1];
  const int lane = (int)threadIdx.x;
  const long first = (long)blockIdx.x * NS;
  const long id = first + lane;  // this lane's system in the recurrence
  const long L = g.count, n = g.n;
  // the systems and chunk positions this lane covers in row-contiguous loads
  const int sub = lane % XC::kLanesPerSys, sys0 = lane / XC::kLanesPerSys;
  long rowoff[XC::kLoads];
  bool rowok[XC::kLoads];
#pragma unroll
  for (int k = 0; k < XC::kLoads; k++) {
    const long sid = first + sys0 + k * XC::kSysPerLoad;
    rowok[k] = sid < L;
    rowoff[k] = rowok[k] ? line_offset(g, sid) : 0;
  }
  T ra[XC::kLoads][V], rb[XC::kLoads][V], rc[XC::kLoads][V], rd[XC::kLoads][V];
  // every system of the workgroup exists (workgroup-uniform)
  const bool all_rows = first + NS <= L;
  auto load_chunk = [&](long i0) {
    if (all_rows && i0 + kChunk <= n) {
      // a full chunk: no per-row branches, so the loads of all rows are in
      // flight together (a branch join makes the compiler wait for every
      // outstanding load, which serialised the rows: 241 us along x at 256^3)
#pragma unroll
      for (int k = 0; k < XC::kLoads; k++) {
        using VT = vec_t<T, V>;
        const long i = i0 + sub * V;
        const VT va = ldg<VT, true>((const VT *)(a + rowoff[k] + i));
        const VT vb = ldg<VT, true>((const VT *)(b + rowoff[k] + i));
        const VT vc = ldg<VT, true>((const VT *)(c + rowoff[k] + i));
        const VT vd = ldg<VT, true>((const VT *)(d + rowoff[k] + i));
#pragma unroll
        for (int j = 0; j < V; j++) {
          ra[k][j] = va[j];
          rb[k][j] = vb[j];
          rc[k][j] = vc[j];
          rd[k][j] = vd[j];
        }
      }
      return;
    }
#pragma unroll
    for (int k = 0; k < XC::kLoads; k++) {
      const long i = i0 + sub * V;
      if (rowok[k] && i + V <= n) {
        using VT = vec_t<T, V>;
        const VT va = ldg<VT, true>((const VT *)(a + rowoff[k] + i));
        const VT vb = ldg<VT, true>((const VT *)(b + rowoff[k] + i));
        const VT vc = ldg<VT, true>((const VT *)(c + rowoff[k] + i));
        const VT vd = ldg<VT, true>((const VT *)(d + rowoff[k] + i));
#pragma unroll
        for (int j = 0; j < V; j++) {
          ra[k][j] = va[j];
          rb[k][j] = vb[j];
          rc[k][j] = vc[j];
          rd[k][j] = vd[j];
        }
      } else {
#pragma unroll
        for (int j = 0; j < V; j++) {
          const bool ok = rowok[k] && i + j < n;
          ra[k][j] = ok ? a[rowoff[k] + i + j] : (T)0;
          rb[k][j] = ok ? b[rowoff[k] + i + j] : (T)1;
          rc[k][j] = ok ? c[rowoff[k] + i + j] : (T)0;
          rd[k][j] = ok ? d[rowoff[k] + i + j] : (T)0;
        }
      }
    }
  };
  auto stage_chunk = [&]() {
#pragma unroll
    for (int k = 0; k < XC::kLoads; k++) {
      const int sy = sys0 + k * XC::kSysPerLoad;
#pragma unroll
      for (int j = 0; j < V; j++) {
        LA[sub * V + j][sy] = ra[k][j];
        LB[sub * V + j][sy] = rb[k][j];
        LC[sub * V + j][sy] = rc[k][j];
        LD[sub * V + j][sy] = rd[k][j];
      }
    }
  };
  const bool live = lane < NS && id < L;
  T cprev = 0, dprev = 0;
  load_chunk(0);
  for (long i0 = 0; i0 < n; i0 += kChunk) {
    stage_chunk();
    __syncthreads();
    if (i0 + kChunk < n) load_chunk(i0 + kChunk);
    if (live && i0 > 0 && i0 + kChunk <= n) {
      // an inner full chunk: no per-step branches (their joins would make
      // the compiler wait for the next chunk's loads already in flight)
#pragma unroll
      for (int k = 0; k < kChunk; k++) {
        const long i = i0 + k;
        const T av = LA[k][lane], bv = LB[k][lane], cv = LC[k][lane], dv = LD[k][lane];
        const T bb = (T)1.0 / (bv - av * cprev);
        dprev = bb * (dv - av * dprev);
        cprev = bb * cv;
        cs[i * L + id] = cprev;
        ds[i * L + id] = dprev;
      }
    } else if (live) {
#pragma unroll
      for (int k = 0; k < kChunk; k++) {
        const long i = i0 + k;
        if (i < n) {
          const T av = LA[k][lane], bv = LB[k][lane], cv = LC[k][lane], dv = LD[k][lane];
          if (i == 0) {
            const T bb = (T)1.0 / bv;
            cprev = bb * cv;
            dprev = bb * dv;
          } else {
            const T bb = (T)1.0 / (bv - av * cprev);
            dprev = bb * (dv - av * dprev);
            cprev = bb * cv;
          }
          cs[i * L + id] = cprev;
          ds[i * L + id] = dprev;
        }
      }
    }
    __syncthreads();
  }
  // backward: chunks from the last one down; x of a chunk goes to LA.  The
  // c', d' of the next chunk are loaded while this one is solved (two
  // register sets used in turn).
  T x = dprev;
  const long last0 = (n - 1) / kChunk * kChunk;
  T cv[2][kChunk], dv[2][kChunk];
  auto load_back = [&](int q, long i0) {
    if (!live || i0 < 0) return;
#pragma unroll
    for (int k = 0; k < kChunk; k++) {
      const long i = i0 + k;
      if (i < n - 1) {
        cv[q][k] = cs[i * L + id];
        dv[q][k] = ds[i * L + id];
      }
    }
  };
  load_back(0, last0);
  int q = 0;
  for (long i0 = last0; i0 >= 0; i0 -= kChunk, q ^= 1) {
    if (q == 0) load_back(1, i0 - kChunk);
    else load_back(0, i0 - kChunk);
    if (live) {
#pragma unroll
      for (int k = kChunk - 1; k >= 0; k--) {
        const long i = i0 + k;
        const T cq = q == 0 ? cv[0][k] : cv[1][k];
        const T dq = q == 0 ? dv[0][k] : dv[1][k];
        if (i == n - 1) LA[k][lane] = x;
        else if (i < n - 1) {
          x = dq - cq * x;
          LA[k][lane] = x;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < XC::kLoads; k++) {
      const long i = i0 + sub * V;
      const int sy = sys0 + k * XC::kSysPerLoad;
      if (!rowok[k]) continue;
      if (i + V <= n) {
        using VT = vec_t<T, V>;
        VT v;
#pragma unroll
        for (int j = 0; j < V; j++) v[j] = LA[sub * V + j][sy];
        if (INC) {
          const VT uo = *(const VT *)(u + rowoff[k] + i);
#pragma unroll
          for (int j = 0; j < V; j++) v[j] = uo[j] + v[j];
          *(VT *)(u + rowoff[k] + i) = v;
        } else {
          *(VT *)(d + rowoff[k] + i) = v;
        }
      } else {
#pragma unroll
        for (int j = 0; j < V; j++)
          if (i + j < n) {
            const T xv = LA[sub * V + j][sy];
            if (INC) u[rowoff[k] + i + j] = u[rowoff[k] + i + j] + xv;
            else d[rowoff[k] + i + j] = xv;
          }
      }
    }
    __syncthreads();
  }
}

// PCR.  A workgroup takes S neighbouring systems of n rows; J threads share a
// system, thread j holding rows j, j + J, ... (at most ROWS) in registers.
// The steps of distance below J find their neighbours through LDS, those of
// J and above in the thread's own registers.  Lanes run along the systems for
// solves along y and z and along the rows for solves along x (ALONG), so a
// load takes whole segments either way (one workgroup per system read 8 bytes
// of every 128-byte line along y and z).  Bounded by vector arithmetic, 62
// instructions a row and step, two divisions among them: sharing their
// reciprocals (same quotients by Markstein's correction) saved nothing after
// its range checks.  Microseconds along x / y / z, one workgroup per system and
// now: 256^3 366 / 774 / 887 and 323 / 317 / 310, 200 x 130 x 97 63 / 118 / 148
// and 64 / 61 / 53.  Two rows a thread (pcr_rows).  The operations of a row are the
// algorithm's, in its order.

template <class T>
struct PcrRow {
  T a, b, c, d;
};

// one step of a row: lo, hi its neighbours where they exist
template <class T>
__device__ __forceinline__ PcrRow<T> pcr_step(const PcrRow<T> &x, bool lo, const PcrRow<T> &l, bool hi,
                                              const PcrRow<T> &h) {
  const T k1 = lo ? x.a / l.b : (T)0;
  const T k2 = hi ? x.c / h.b : (T)0;
  T bv = x.b, dv = x.d;
  if (lo) {
    bv = bv - l.c * k1;
    dv = dv - l.d * k1;
  }
  if (hi) {
    bv = bv - h.a * k2;
    dv = dv - h.d * k2;
  }
  return PcrRow<T>{lo ? -l.a * k1 : (T)0, bv, hi ? -h.c * k2 : (T)0, dv};
}

template <class T, bool INC, bool ALONG, int ROWS>
__global__ __launch_bounds__(512) void k_pcr(const T *__restrict__ a, const T *__restrict__ b,
                                             const T *__restrict__ c, T *__restrict__ d, T *__restrict__ u,
                                             LineGeo g, int S, int J) {
  extern __shared__ unsigned char smem[];
  const int n = (int)g.n, tid = (int)threadIdx.x;
  const int s = ALONG ? tid / J : tid & (S - 1), j = ALONG ? tid & (J - 1) : tid / S;
  const long id = (long)xcd_tile(blockIdx.x, gridDim.x) * S + s;
  const bool live = id < g.count;
  const long o = live ? line_offset(g, id) : 0;
  // LDS: rows of a system one after the other, or systems of a row; this
  // thread's rows are kstep apart in it and gstep apart in memory
  const int lr = ALONG ? 1 : S, kstep = J * lr, all = n * S;
  const int at = (ALONG ? s * n : s) + j * lr;
  typedef vec_t<T, 2> Pair;
  Pair *L = (Pair *)smem + at;
  const long q0 = o + j * g.stride, gstep = J * g.stride;
  PcrRow<T> r[ROWS];
#pragma unroll
  for (int k = 0; k < ROWS; k++) {
    const int i = j + k * J;
    r[k] = PcrRow<T>{(T)0, (T)1, (T)0, (T)0};
    if (live && i < n) {
      const long q = q0 + k * gstep;
      r[k] = PcrRow<T>{a[q], b[q], c[q], d[q]};
      if (i == 0) r[k].a = (T)0;
      if (i == n - 1) r[k].c = (T)0;
    }
  }
  const int top = min(J, n);
  for (int st = 1; st < top; st *= 2) {
#pragma unroll
    for (int k = 0; k < ROWS; k++)
      if (j + k * J < n) {
        Pair *p = L + k * kstep;
        p[0] = Pair{r[k].a, r[k].b};
        p[all] = Pair{r[k].c, r[k].d};
      }
    __syncthreads();
    const int away = st * lr;
#pragma unroll
    for (int k = 0; k < ROWS; k++) {
      const int i = j + k * J;
      if (i < n) {
        const bool lo = i >= st, hi = i + st < n;
        const Pair *l = L + (k * kstep - (lo ? away : 0)), *h = L + (k * kstep + (hi ? away : 0));
        const Pair l0 = l[0], l1 = l[all], h0 = h[0], h1 = h[all];
        r[k] = pcr_step(r[k], lo, PcrRow<T>{l0[0], l0[1], l1[0], l1[1]}, hi, PcrRow<T>{h0[0], h0[1], h1[0], h1[1]});
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int m = 1; m < ROWS; m *= 2) {
    if (m * J >= n) break;
    PcrRow<T> x[ROWS];
#pragma unroll
    for (int k = 0; k < ROWS; k++) {
      const bool lo = k >= m, hi = k + m < ROWS && j + (k + m) * J < n;
      const int l = k >= m ? k - m : k, h = k + m < ROWS ? k + m : k;
      x[k] = r[k];
      // along x a wave without rows here, or whose rows have no neighbour left,
      // skips the divisions (257 rows 78 -> 76 us); across systems every wave
      // has some (256 rows 56 us, 58 with the condition)
      if (!ALONG || (j + k * J < n && (lo || hi))) x[k] = pcr_step(r[k], lo, r[l], hi, r[h]);
    }
#pragma unroll
    for (int k = 0; k < ROWS; k++) r[k] = x[k];
  }
#pragma unroll
  for (int k = 0; k < ROWS; k++) {
    const int i = j + k * J;
    if (live && i < n) {
      const T x = r[k].d / r[k].b;
      const long q = q0 + k * gstep;
      if (INC) u[q] = u[q] + x;
      else d[q] = x;
    }
  }
}

// rows a thread holds.  4 took 368 / 333 / 321 us along x / y / z at 256^3 in
// FP64, 2 323 / 317 / 310, and 71 / 61 / 53 and 64 / 61 / 53 at 200 x 130 x 97.
// Longer systems across y and z, of which a workgroup would have one or two,
// take 4; along x they take 2 all the same (3e6 points in FP64, one workgroup
// per system first, then 4 rows and 2: 257 rows 74, 81 and 76 us, 400 rows 70,
// 76 and 69, 512 rows 61, 68 and 60, 1024 rows 76, 74 and 65; in FP32 512 rows
// 45, 37 and 35).
inline int pcr_rows(int n, bool along) { return along || n <= 256 ? 2 : 4; }

// threads per system and systems per workgroup
struct PcrShape {
  int S, J;
  size_t lds;
};
inline PcrShape pcr_shape(int n, size_t es, int rows) {
  PcrShape p;
  p.J = 1;
  while (p.J * rows < n) p.J *= 2;
  // 128 bytes of systems where their rows then fit the 64 KiB of LDS a
  // workgroup may ask for, at most 512 threads; fewer systems for long ones
  p.S = (int)(128 / es);
  const size_t row = 4 * es;  // bytes in LDS
  while (p.S > 1 && (p.S * p.J > 512 || n * p.S * row > (64u << 10))) p.S /= 2;
  // short systems: at least four waves a workgroup
  while (p.S * p.J < 256 && n * p.S * 2 * row <= (40u << 10)) p.S *= 2;
  p.lds = p.J > 1 ? n * p.S * row : 0;
  return p;
}

struct TridScratch {
  void *p = nullptr;
  size_t bytes = 0;
};
TridScratch g_scratch;

void *trid_scratch(size_t bytes) {
  if (bytes > g_scratch.bytes) {
    if (g_scratch.p) {
      OPSMI_HIP(hipStreamSynchronize(inst().stream));
      OPSMI_HIP(hipFree(g_scratch.p));
    }
    OPSMI_HIP(hipMalloc(&g_scratch.p, bytes));
    g_scratch.bytes = bytes;
  }
  return g_scratch.p;
}

// Scratch of the entry point that allocates nothing
// (ops_tridMultiDimBatch_noalloc): c' and d' of every system, step-major, as
// the library scratch above.  Each GPU holds its own copy for the life of the
// process; host code reaches it only through the address that
// hipGetSymbolAddress returned on that device (the array's name in host code
// is not a device address).  Calls on one GPU share it, so calls that overlap
// on one GPU race.
constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
__device__ __align__(256) char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
char *g_noalloc_ptr[kMaxDevices];

// trid_run with fixed_scr set: no flush, no library scratch, no timing events
// or statistics records, so nothing is allocated on the host or the device.
void trid_run(int ndim, int solvedim, int *range, ops_dat a, ops_dat b, ops_dat c, ops_dat d, ops_dat u,
              ops_tridsolver_params_c *ctx, char *fixed_scr = nullptr) {
  require_init();
  if (!fixed_scr) flush_all();
  else if (!queue_empty())
    fail(OPS_RUNTIME_ERROR, "ops_tridMultiDimBatch_noalloc: loops are queued; call ops_execute() first "
                            "(running them may allocate)");
  if (!a || !b || !c || !d || !range || !ctx) fail(OPS_INVALID_ARGUMENT, "Tridsolver error: NULL argument");
  if (ndim < 1 || ndim > 3 || ndim != a->block->dims)
    fail(OPS_INVALID_ARGUMENT, "Tridsolver error: ndim must match the block (1-3D)");
  if (solvedim < 0 || solvedim >= ndim) fail(OPS_INVALID_ARGUMENT, "Tridsolver error: solvedim out of range");
  ops_dat all[5] = {a, b, c, d, u};
  int nd = u ? 5 : 4;
  // ops/c/src/tridiag/ops_tridiag.cpp:91-101
  for (int i = 0; i < ndim; i++)
    for (int k = 1; k < nd; k++)
      if (all[k]->size[i] != a->size[i])
        fail(OPS_RUNTIME_ERROR, "Tridsolver error: the a,b,c,d datasets all need to be the same size");
  for (int k = 1; k < nd; k++)
    if (strcmp(all[k]->type, a->type) != 0)
      fail(OPS_RUNTIME_ERROR, "Tridsolver error: the a,b,c,d datasets must all be of the same type");
  DType dt = dtype_of(a->type, a->type_size);
  if (dt != DT_F64 && dt != DT_F32)
    fail(OPS_RUNTIME_ERROR, "Tridsolver error: unsupported type. Dataset type must either be \"double\" or \"float\"");
  for (int k = 0; k < nd; k++) {
    if (all[k]->dim != 1) fail(OPS_NOT_IMPLEMENTED, "Tridsolver error: multi-component dats are not supported");
    if (all[k]->locked_hd) fail(OPS_RUNTIME_ERROR, cat("Tridsolver error: dat ", all[k]->name, " is locked"));
  }
  int dims[3] = {1, 1, 1};
  long offset = 0;
  long st[3] = {1, a->size[0], (long)a->size[0] * a->size[1]};
  for (int i = 0; i < ndim; i++) {
    dims[i] = range[2 * i + 1] - range[2 * i];
    int first = a->d_m[i] + a->base[i], last = a->size[i] + a->d_m[i] + a->base[i];
    if (dims[i] < 0 || range[2 * i] < first || range[2 * i + 1] > last)
      fail(OPS_INVALID_ARGUMENT, cat("Tridsolver error: range outside the dats in dimension ", i));
    offset += (long)range[2 * i] * st[i];
  }
  for (int k = 0; k < nd; k++) {
    if (fixed_scr && all[k]->dirty_hd == 1)
      fail(OPS_RUNTIME_ERROR, cat("ops_tridMultiDimBatch_noalloc: dat ", all[k]->name,
                                  " has newer data on the host; upload it first (ops_execute, or any loop)"));
    sync_to_device(all[k]);
  }
  LineGeo g;
  g.n = dims[solvedim];
  g.stride = st[solvedim];
  int od[2], q = 0;
  for (int i = 0; i < 3; i++)
    if (i != solvedim) od[q++] = i;
  g.e0 = dims[od[0]];
  g.s0 = st[od[0]];
  g.s1 = st[od[1]];
  g.count = (long)dims[od[0]] * dims[od[1]];
  // statistics per solve direction (the timing table's loop name)
  static const char *names[2][3] = {{"ops_tridMultiDimBatch x", "ops_tridMultiDimBatch y", "ops_tridMultiDimBatch z"},
                                    {"ops_tridMultiDimBatch_Inc x", "ops_tridMultiDimBatch_Inc y",
                                     "ops_tridMultiDimBatch_Inc z"}};
  const char *nm = names[u ? 1 : 0][solvedim];
  double bytes = (double)g.n * g.count * a->type_size * (u ? 6.0 : 5.0);
  if (g.n <= 0 || g.count <= 0) {
    if (!fixed_scr) run_loop(nm, 0.0, [](hipStream_t) {});
    return;
  }
  if (fixed_scr && (double)g.n * g.count * a->type_size * 2.0 > (double)kNoAllocScratchBytes)
    fail(OPS_INVALID_ARGUMENT,
         cat("ops_tridMultiDimBatch_noalloc: ", g.count, " systems of ", g.n, " rows need ",
             2 * g.n * g.count * (long)a->type_size, " bytes of scratch; the maximum is ", kNoAllocScratchBytes,
             " (", kNoAllocScratchBytes / 16, " points in double, ", kNoAllocScratchBytes / 8, " in float)"));
  // the launch: through run_loop (statistics, timing events) or, for the
  // no-allocation entry point, straight onto the library's stream
  auto launch = [&](const std::function<void(hipStream_t)> &fn) {
    if (fixed_scr) {
      fn(inst().stream);
      OPSMI_HIP(hipGetLastError());
    } else {
      run_loop(nm, bytes, fn);
    }
  };
  size_t es = a->type_size;
  char *pa = a->data_d + a->base_offset + offset * es, *pb = b->data_d + b->base_offset + offset * es;
  char *pc = c->data_d + c->base_offset + offset * es, *pd = d->data_d + d->base_offset + offset * es;
  char *pu = u ? u->data_d + u->base_offset + offset * es : nullptr;
  bool pcr = ctx && ctx->strategy == 3;
  if (pcr) {
    if (g.n > 1024) fail(OPS_NOT_IMPLEMENTED, "Tridsolver error: PCR supports systems of at most 1024 rows");
    const int per = pcr_rows((int)g.n, solvedim == 0);
    const PcrShape ps = pcr_shape((int)g.n, es, per);
    const unsigned nb = (unsigned)((g.count + ps.S - 1) / ps.S);
    const dim3 block((unsigned)(ps.S * ps.J));
    launch([&](hipStream_t s) {
      auto go = [&](auto kern, auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        hipLaunchKernelGGL(kern, dim3(nb), block, ps.lds, s, (const T *)pa, (const T *)pb, (const T *)pc, (T *)pd,
                           (T *)pu, g, ps.S, ps.J);
      };
      auto rows = [&](auto r, auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        constexpr int ROWS = decltype(r)::value;
        const bool x = solvedim == 0;
        if (u) go(x ? k_pcr<T, true, true, ROWS> : k_pcr<T, true, false, ROWS>, t);
        else go(x ? k_pcr<T, false, true, ROWS> : k_pcr<T, false, false, ROWS>, t);
      };
      auto type = [&](auto *t) {
        if (per == 2) rows(std::integral_constant<int, 2>{}, t);
        else rows(std::integral_constant<int, 4>{}, t);
      };
      if (dt == DT_F64) type((double *)nullptr);
      else type((float *)nullptr);
    });
  } else {
    size_t sb = (size_t)g.n * g.count * es;
    char *scr = fixed_scr ? fixed_scr : (char *)trid_scratch(2 * sb);
    // one-wave workgroups while each then has a CU to itself (100^3 in FP64:
    // 29 us instead of 46 in 40 workgroups of four waves); beyond that four
    // waves share a CU better (45 000 systems of 203 in FP32: 83 and 91 us)
    const int tpb = g.count <= 64L * inst().num_cus ? 64 : 256;
    int nblk = (int)((g.count + tpb - 1) / tpb);
    if (solvedim == 0) {
      // x solves: LDS-staged chunks, 16-byte row loads when every array's
      // rows start 16-byte aligned (30 450 systems of 301 in FP32: 143 us
      // instead of 164 with single elements)
      const long per16 = 16 / (long)es;
      bool v16 = g.s0 % per16 == 0 && g.s1 % per16 == 0;
      for (char *p : {pa, pb, pc, pd, pu})
        if (p && (uintptr_t)p % 16 != 0) v16 = false;
      // half-filled waves (32 systems) while each of those finds a SIMD of its
      // own, in FP32, whose rows are half as long, up to a quarter more.  FP64,
      // 32 and 64 systems a wave: 30 450 systems of 301 147 and 201 us, 32 000
      // of 256 111 and 113, 40 000 of 301 238 and 180, 65 536 of 256 261 and
      // 217.  FP32: 30 450 of 301 123 and 143, 33 124 of 300 138 and 158,
      // 40 000 134 and 138, 42 000 152 and 143, 65 536 193 and 183
      const bool half = g.count <= (dt == DT_F32 ? 160L : 128L) * inst().num_cus;
      const int nw = (int)((g.count + (half ? 31 : 63)) / (half ? 32 : 64));
      launch([&](hipStream_t s) {
        auto go = [&](auto v, auto ns, auto *t) {
          using T = std::remove_pointer_t<decltype(t)>;
          constexpr int V = decltype(v)::value, NS = decltype(ns)::value;
          hipLaunchKernelGGL((u ? k_thomas_x<T, V, NS, true> : k_thomas_x<T, V, NS, false>), dim3(nw), dim3(64), 0, s,
                             (const T *)pa, (const T *)pb, (const T *)pc, (T *)pd, (T *)pu, (T *)scr,
                             (T *)(scr + sb), g);
        };
        auto width = [&](auto ns, auto *t) {
          using T = std::remove_pointer_t<decltype(t)>;
          if (v16) go(std::integral_constant<int, 16 / (int)sizeof(T)>{}, ns, t);
          else go(std::integral_constant<int, 1>{}, ns, t);
        };
        auto type = [&](auto ns) {
          if (dt == DT_F64) width(ns, (double *)nullptr);
          else width(ns, (float *)nullptr);
        };
        if (half) type(std::integral_constant<int, 32>{});
        else type(std::integral_constant<int, 64>{});
      });
      mark_device_dirty(u ? u : d);
      note_external_write(u ? u : d);
      return;
    }
    launch([&](hipStream_t s) {
      if (dt == DT_F64) {
        if (u) hipLaunchKernelGGL((k_thomas<double, true, kPre>), dim3(nblk), dim3(tpb), 0, s, (double *)pa, (double *)pb, (double *)pc, (double *)pd, (double *)pu, (double *)scr, (double *)(scr + sb), g);
        else hipLaunchKernelGGL((k_thomas<double, false, kPre>), dim3(nblk), dim3(tpb), 0, s, (double *)pa, (double *)pb, (double *)pc, (double *)pd, (double *)pu, (double *)scr, (double *)(scr + sb), g);
      } else {
        if (u) hipLaunchKernelGGL((k_thomas<float, true, kPre>), dim3(nblk), dim3(tpb), 0, s, (float *)pa, (float *)pb, (float *)pc, (float *)pd, (float *)pu, (float *)scr, (float *)(scr + sb), g);
        else hipLaunchKernelGGL((k_thomas<float, false, kPre>), dim3(nblk), dim3(tpb), 0, s, (float *)pa, (float *)pb, (float *)pc, (float *)pd, (float *)pu, (float *)scr, (float *)(scr + sb), g);
      }
    });
  }
  mark_device_dirty(u ? u : d);
  note_external_write(u ? u : d);
}

}  // namespace

namespace opsmi {
// Called by ops_init with the library's device current: the device address
// of this device's copy of the no-allocation scratch.
void trid_noalloc_setup(int dev) {
  if (dev < 0 || dev >= kMaxDevices) fail(OPS_RUNTIME_CONFIGURATION_ERROR, cat("device ", dev, " out of range"));
  if (g_noalloc_ptr[dev]) return;
  void *ptr = nullptr;
  OPSMI_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  if (!ptr) fail(OPS_RUNTIME_ERROR, "hipGetSymbolAddress returned no address for the tridiagonal scratch");
  g_noalloc_ptr[dev] = (char *)ptr;
}
}  // namespace opsmi

extern "C" {

ops_tridsolver_params_c *ops_tridsolver_params_create(ops_block block, int strategy) {
  (void)block;
  ops_tridsolver_params_c *p = new ops_tridsolver_params_c;
  p->strategy = strategy;
  return p;
}

void ops_tridsolver_params_destroy(ops_tridsolver_params_c *p) { delete p; }

void ops_tridMultiDimBatch_c(int ndim, int solvedim, int *range, ops_dat a, ops_dat b, ops_dat c, ops_dat d,
                             ops_tridsolver_params_c *ctx) {
  OPSMI_API_BEGIN
  trid_run(ndim, solvedim, range, a, b, c, d, nullptr, ctx);
  OPSMI_API_END()
}

void ops_tridMultiDimBatch_Inc_c(int ndim, int solvedim, int *range, ops_dat a, ops_dat b, ops_dat c, ops_dat d,
                                 ops_dat u, ops_tridsolver_params_c *ctx) {
  OPSMI_API_BEGIN
  if (!u) fail(OPS_INVALID_ARGUMENT, "Tridsolver error: NULL u");
  trid_run(ndim, solvedim, range, a, b, c, d, u, ctx);
  OPSMI_API_END()
}

// The reference's C-linkage entry points: the params object's one data
// member points at the solver settings.
void ops_tridMultiDimBatch(int ndim, int solvedim, int *range, ops_dat a, ops_dat b, ops_dat c, ops_dat d,
                           ops_tridsolver_params *tridsolver_ctx) {
  OPSMI_API_BEGIN
  if (!tridsolver_ctx) fail(OPS_INVALID_ARGUMENT, "Tridsolver error: NULL ops_tridsolver_params");
  trid_run(ndim, solvedim, range, a, b, c, d, nullptr, *(ops_tridsolver_params_c **)tridsolver_ctx);
  OPSMI_API_END()
}

void ops_tridMultiDimBatch_Inc(int ndim, int solvedim, int *range, ops_dat a, ops_dat b, ops_dat c, ops_dat d,
                               ops_dat u, ops_tridsolver_params *tridsolver_ctx) {
  OPSMI_API_BEGIN
  if (!tridsolver_ctx) fail(OPS_INVALID_ARGUMENT, "Tridsolver error: NULL ops_tridsolver_params");
  if (!u) fail(OPS_INVALID_ARGUMENT, "Tridsolver error: NULL u");
  trid_run(ndim, solvedim, range, a, b, c, d, u, *(ops_tridsolver_params_c **)tridsolver_ctx);
  OPSMI_API_END()
}

// ops_tridMultiDimBatch (u NULL) or ops_tridMultiDimBatch_Inc (u given) on
// the same kernels, with the c'/d' scratch in the library's fixed device
// array instead of library-allocated memory: at most 64 MiB of scratch,
// i.e. 2 * rows * systems * sizeof(element) <= 64 MiB.
void ops_tridMultiDimBatch_noalloc(int ndim, int solvedim, int *range, ops_dat a, ops_dat b, ops_dat c, ops_dat d,
                                   ops_dat u, ops_tridsolver_params *tridsolver_ctx) {
  OPSMI_API_BEGIN
  if (!tridsolver_ctx) fail(OPS_INVALID_ARGUMENT, "Tridsolver error: NULL ops_tridsolver_params");
  require_init();
  const int dev = inst().device;
  char *ptr = dev >= 0 && dev < kMaxDevices ? g_noalloc_ptr[dev] : nullptr;
  if (!ptr) fail(OPS_RUNTIME_ERROR, "ops_tridMultiDimBatch_noalloc: scratch address not set up (ops_init)");
  trid_run(ndim, solvedim, range, a, b, c, d, u, *(ops_tridsolver_params_c **)tridsolver_ctx, ptr);
  OPSMI_API_END()
}

}  // extern "C"
