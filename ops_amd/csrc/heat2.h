// The 2D TeaLeaf operator (5-point, coefficients Kx, Ky) with two points per
// lane: the device code of calc_w, of common_init and of the 2D CG chain.
//
// A workgroup owns 128 x 16 points, wave v its rows 4 v .. 4 v + 3, lane l the
// points x0 + 2 l, x0 + 2 l + 1.  Each wave loads its four rows of every array,
// the row above and the row below p (and Ky's fifth row) as 16-byte vectors,
// all before the first use and none under a condition; the x neighbours across
// lanes come from the neighbouring lane, at the wave's two ends from one more
// load per row.  Bound by memory: at 3001 x 2003 calc_w's 192 MB take 31 us
// (6.2 TB/s, part of it from the Infinity Cache), common_init's 240 MB 47 us;
// one point per lane and one row after the other (the general engine) took 46.5
// and 52.6 us.  The chain's 385 MB take 67.5 us there (73 without NT) and its
// 2.3 GB 457 us at 6000 x 6000 (pair and calc_w alone: 72 and 489 us); it needs
// 141 registers, and squeezed into 128, for a fourth wave per SIMD, it spills
// and takes 494 us there.
//
// NT: Kx, Ky and u, which no other loop of the iteration touches, pass the
// caches by, which leaves them to p, r and w: for a chain whose seven arrays
// outgrow the Infinity Cache (chain and r.r loop at 3001 x 2003 101 us instead
// of 107, at 4000 x 3000 209 instead of 216, at 6000 x 6000 617 and 613; where
// they fit, at 1500 x 1000, it would take 33 us instead of 28).
//
// The sums of w p are the general engine's, bit for bit: its workgroup owns
// 64 x 16 points, wave j rows j, j + 4, j + 8, j + 12 one after the other, then
// a butterfly over the columns and a sum over waves 0 .. 3, and one partial per
// workgroup in hardware order.  Here row j of every wave goes through LDS to
// wave j, which adds the four in that order; the butterfly runs over half a
// wave for each of a lane's two columns and ends by adding the two.
#pragma once

#include "engine.h"

namespace opsmi {

template <bool NT, class T>
__device__ __forceinline__ void stg(T *p, T v) {
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

constexpr int kHeat2Rows = 4;  // rows of a wave
enum Heat2Mode { HEAT2_W, HEAT2_INIT, HEAT2_CHAIN, HEAT2_CHAIN_AXPY };

struct Heat2Args {
  Ptr<double> w, r, pnew, u;  // r: common_init's; pnew, u: the chain's
  Ptr<const double> Kx, Ky, p, rr;  // p: the operand (chain: p before the axpby); rr: the chain's r
  double rx, ry, alpha_u, a, b;
};

inline unsigned heat2_tiles(const Range3 &r) { return (unsigned)((r.x1 - r.x0 + kWave - 1) / kWave); }
inline dim3 heat2_grid(const Range3 &r) {
  const int rows = kHeat2Rows * kWavesPerBlock;
  return dim3((heat2_tiles(r) + 1) / 2, (unsigned)((r.y1 - r.y0 + rows - 1) / rows), 1);
}
// partials of the reduction: one per 64 x 16 points
inline unsigned heat2_parts(const Range3 &r) { return heat2_tiles(r) * heat2_grid(r).y; }

// the hardware block that takes logical tile l of nb (inverse of xcd_tile)
__device__ __forceinline__ unsigned xcd_block(unsigned l, unsigned nb) {
  const unsigned q8 = nb >> 3, r8 = nb & 7u, big = r8 * (q8 + 1);
  if (l < big) return (l % (q8 + 1)) * 8 + l / (q8 + 1);
  return ((l - big) % q8) * 8 + r8 + (l - big) / q8;
}

template <int MODE, bool NT = false>
__global__ __launch_bounds__(kWave *kWavesPerBlock) void k_heat2(Heat2Args f, Range3 R, unsigned tiles, RedCtl ctl) {
  constexpr bool CHAIN = MODE == HEAT2_CHAIN || MODE == HEAT2_CHAIN_AXPY;
  constexpr int N = kHeat2Rows;
  using D2 = vec_t<double, 2>;
  const TileId t = tile_id();
  const int lane = (int)threadIdx.x, wv = (int)threadIdx.y;
  const int x = R.x0 + (int)t.x * 2 * kWave + 2 * lane;
  const int y = R.y0 + (int)t.y * N * kWavesPerBlock + N * wv;
  // lanes past the end load from the last pair that a point of the range
  // needs; it may start on the far rim, and its second element lie in the
  // next row or the allocation's padding
  const int lx = min(x, R.x0 + ((R.x1 - R.x0) & ~1));
  // the one element beyond the wave's ends: lane 0 x - 1, lane 63 x + 2
  const int ex = lane == 0 ? x - 1 : lane == kWave - 1 ? min(x + 2, R.x1) : lx;
  auto row = [&](int k) { return min(y + k, R.y1); };  // k = -1 .. N, up to the far rim
  D2 p[N + 2], ky[N + 1], kx[N];
  double pe[N], kxe[N];
#pragma unroll
  for (int k = 0; k < N + 2; k++) p[k] = *(const D2 *)f.p.at(lx, row(k - 1), R.z0);
#pragma unroll
  for (int k = 0; k < N + 1; k++) ky[k] = ldg<D2, NT>((const D2 *)f.Ky.at(lx, row(k), R.z0));
#pragma unroll
  for (int k = 0; k < N; k++) {
    const int yk = min(y + k, R.y1 - 1);
    kx[k] = ldg<D2, NT>((const D2 *)f.Kx.at(lx, yk, R.z0));
    kxe[k] = *f.Kx.at(lane == kWave - 1 ? ex : lx, yk, R.z0);
    pe[k] = *f.p.at(ex, yk, R.z0);
  }
  if constexpr (CHAIN) {
    // p = a p + b r where the axpby runs, the old p on the rim
    const bool in0 = x < R.x1, in1 = x + 1 < R.x1;
    // r has no rim: stay on its rows and columns
    const int cx = min(lx, R.x1 - 1 - ((R.x1 - 1 - R.x0) & 1));
    const bool ein = ex >= R.x0 && ex < R.x1;
    D2 q[N + 2], uo[N];
    double qe[N];
#pragma unroll
    for (int k = 0; k < N + 2; k++) {
      const int yk = max(R.y0, min(y + k - 1, R.y1 - 1));
      q[k] = *(const D2 *)f.rr.at(cx, yk, R.z0);
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
      const int yk = min(y + k, R.y1 - 1);
      qe[k] = *f.rr.at(max(R.x0, min(ex, R.x1 - 1)), yk, R.z0);
      if constexpr (MODE == HEAT2_CHAIN_AXPY) uo[k] = ldg<D2, NT>((const D2 *)f.u.at(cx, yk, R.z0));
    }
    if constexpr (MODE == HEAT2_CHAIN_AXPY) {
#pragma unroll
      for (int k = 0; k < N; k++)
        if (y + k < R.y1) {
          const double v0 = uo[k][0] + f.alpha_u * p[k + 1][0], v1 = uo[k][1] + f.alpha_u * p[k + 1][1];
          if (in1) stg<NT>((D2 *)f.u.at(x, y + k, R.z0), D2{v0, v1});
          else if (in0) *f.u.at(x, y + k, R.z0) = v0;
        }
    }
#pragma unroll
    for (int k = 0; k < N + 2; k++) {
      const bool yin = y + k - 1 >= R.y0 && y + k - 1 < R.y1;
      const double n0 = f.a * p[k][0] + f.b * q[k][0], n1 = f.a * p[k][1] + f.b * q[k][1];
      p[k][0] = yin && in0 ? n0 : p[k][0];
      p[k][1] = yin && in1 ? n1 : p[k][1];
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
      const double n = f.a * pe[k] + f.b * qe[k];
      pe[k] = ein ? n : pe[k];
      if (y + k < R.y1) {
        if (in1) *(D2 *)f.pnew.at(x, y + k, R.z0) = p[k + 1];
        else if (in0) *f.pnew.at(x, y + k, R.z0) = p[k + 1][0];
      }
    }
  }
  double sum[N][2];
#pragma unroll
  for (int k = 0; k < N; k++) {
    const D2 c = p[k + 1], dn = p[k], up = p[k + 2];
    const double sl = __shfl_up(c[1], 1, kWave), sr = __shfl_down(c[0], 1, kWave), sk = __shfl_down(kx[k][0], 1, kWave);
    const double pl = lane == 0 ? pe[k] : sl;
    const double pr = lane == kWave - 1 ? pe[k] : sr, kr = lane == kWave - 1 ? kxe[k] : sk;
    const double v0 = (1.0 + f.ry * (ky[k + 1][0] + ky[k][0]) + f.rx * (kx[k][1] + kx[k][0])) * c[0] -
                      f.ry * (ky[k + 1][0] * up[0] + ky[k][0] * dn[0]) - f.rx * (kx[k][1] * c[1] + kx[k][0] * pl);
    const double v1 = (1.0 + f.ry * (ky[k + 1][1] + ky[k][1]) + f.rx * (kr + kx[k][1])) * c[1] -
                      f.ry * (ky[k + 1][1] * up[1] + ky[k][1] * dn[1]) - f.rx * (kr * pr + kx[k][1] * c[0]);
    const bool in = y + k < R.y1;
    sum[k][0] = in && x < R.x1 ? v0 * c[0] : 0.0;
    sum[k][1] = in && x + 1 < R.x1 ? v1 * c[1] : 0.0;
    if (in && x + 1 < R.x1) {
      *(D2 *)f.w.at(x, y + k, R.z0) = D2{v0, v1};
      if constexpr (MODE == HEAT2_INIT) *(D2 *)f.r.at(x, y + k, R.z0) = D2{c[0] - v0, c[1] - v1};
    } else if (in && x < R.x1) {
      *f.w.at(x, y + k, R.z0) = v0;
      if constexpr (MODE == HEAT2_INIT) *f.r.at(x, y + k, R.z0) = c[0] - v0;
    }
  }
  if constexpr (MODE != HEAT2_INIT) {
    __shared__ D2 sh[N][kWavesPerBlock][kWave];
    __shared__ double fold[2][N];
#pragma unroll
    for (int k = 0; k < N; k++) sh[k][wv][lane] = D2{sum[k][0], sum[k][1]};
    __syncthreads();
    double s0 = 0.0, s1 = 0.0;
#pragma unroll
    for (int v = 0; v < kWavesPerBlock; v++) {
      const D2 q = sh[wv][v][lane];
      s0 = s0 + q[0];
      s1 = s1 + q[1];
    }
#pragma unroll
    for (int off = kWave / 4; off > 0; off >>= 1) {
      s0 = s0 + __shfl_xor(s0, off, kWave);
      s1 = s1 + __shfl_xor(s1, off, kWave);
    }
    if ((lane & (kWave / 2 - 1)) == 0) fold[lane / (kWave / 2)][wv] = s0 + s1;
    __syncthreads();
    const unsigned tx = 2 * t.x + (unsigned)lane;
    if (wv == 0 && lane < 2 && tx < tiles) {
      const double *q = fold[lane];
      double s = q[0];
#pragma unroll
      for (int j = 1; j < N; j++) s = s + q[j];
      ((double *)ctl.partials)[xcd_block(t.y * tiles + tx, tiles * gridDim.y)] = s;
    }
  }
}

// host: every array allows the 16-byte loads
inline bool heat2_ok(const Range3 &r, std::initializer_list<ops_dat> dats) {
  bool ok = use_vec() && r.z1 - r.z0 == 1;
  for (ops_dat d : dats) ok = ok && vec16_ok(d, r.x0);
  return ok;
}

}  // namespace opsmi
