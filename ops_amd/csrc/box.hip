// Boxes of points between device arrays and host memory (fetch, set, slabs,
// declarations with data, a finished solve's solution).
//
// A box is rows of a pitched array; host buffers hold it densely.  A 2D copy
// call moves such a box row by row (7 us a row to pageable memory: a 1000^2
// solution took 7.4 ms, a 128^3 one 108 ms), so one kernel packs or unpacks
// the box instead, straight into or out of pinned host memory, in pieces of
// kPiece bytes over two buffers: while the kernel works on one piece the host
// copies the other from or to the caller's memory.  Fetches of FP64 fields,
// before and after: 64^2 0.49 and 0.04 ms, 1000^2 7.4 and 1.0 ms, 64^3 27
// and 0.17 ms, 128^3 108 and 1.6 ms.
#include "box.h"

#include <string.h>

#include <algorithm>
#include <chrono>

using namespace opsmi;

namespace {

// Two pieces in flight; 4 MiB takes the kernel about 80 us at link speed,
// several times a launch, and the host about 400 us to copy.
constexpr size_t kPiece = (size_t)4 << 20;
// Wide rows on their way to the device go by a copy call, which takes them
// straight from the caller's pages (29 GB/s) while the pieces wait for the
// host's copy into them (27).  Sets, copy call and pieces: one row of 800 KB 43
// and 47 us, of 80 MB 2660 and 2820; 50 rows of 2.4 MB 3970 and 4290; 400 rows
// of 512 KB 7210 and 7220, and below that every row's 7 us show.
constexpr size_t kWideRow = (size_t)512 << 10;
constexpr unsigned kPerThread = 4;

template <int U>
struct unit_of;
template <>
struct unit_of<1> { typedef unsigned char type; };
template <>
struct unit_of<2> { typedef unsigned short type; };
template <>
struct unit_of<4> { typedef unsigned type; };
template <>
struct unit_of<8> { typedef unsigned long long type; };
template <>
struct unit_of<16> { typedef unsigned type __attribute__((ext_vector_type(4))); };

// units [0, n) of a piece whose first one is unit `col` of row `row`.
// Bounded by the link (one load and one store per unit): the widest unit the
// box's alignment allows, kPerThread units a thread 256 apart.
template <int U, bool TO_DEVICE, bool SOA>
__global__ __launch_bounds__(256) void k_box(Box b, char *host, unsigned row, size_t col, unsigned n) {
  typedef typename unit_of<U>::type T;
  const unsigned i0 = blockIdx.x * (256u * kPerThread) + threadIdx.x;
#pragma unroll
  for (unsigned k = 0; k < kPerThread; k++) {
    const unsigned i = i0 + k * 256u;
    if (i >= n) continue;
    const size_t at = col + i, wu = b.width;  // units per row
    size_t r, c;
    if ((at | wu) >> 32) {
      r = at / wu;
      c = at % wu;
    } else {
      r = (unsigned)at / (unsigned)wu;
      c = (unsigned)at % (unsigned)wu;
    }
    r += row;
    const unsigned y = (unsigned)r % b.rows, z = (unsigned)r / b.rows;
    char *p = b.base + (long)z * b.plane + (long)y * b.pitch;
    if constexpr (SOA) {
      const size_t m = b.elem / U, sub = c % m, q = c / m;
      p += (long)(q / b.comps * b.elem) + (long)(q % b.comps) * b.cstride + (long)(sub * U);
    } else {
      p += (long)(c * U);
    }
    if constexpr (TO_DEVICE) *(T *)p = ((const T *)host)[i];
    else ((T *)host)[i] = *(const T *)p;
  }
}

// a whole array's rows outside [r0, r1) x [y0, y1) x [z0, z1) of raw units,
// rows and planes: a wave per row and kSegment of its units, which copies all
// of them or those left and right of the range
constexpr unsigned kSegment = 1024;
template <int U>
__global__ __launch_bounds__(256) void k_outside(char *dst, const char *src, unsigned pitch, unsigned rows,
                                                 unsigned total, unsigned r0, unsigned r1, unsigned y0, unsigned y1,
                                                 unsigned z0, unsigned z1) {
  typedef typename unit_of<U>::type T;
  const unsigned row = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x % 64;
  if (row >= total) return;
  const unsigned y = row % rows, z = row / rows;
  const bool inside = y >= y0 && y < y1 && z >= z0 && z < z1;
  const T *s = (const T *)src + (size_t)row * pitch;
  T *d = (T *)dst + (size_t)row * pitch;
  const unsigned lo = blockIdx.y * kSegment, hi = min(lo + kSegment, pitch);
  if (inside && lo >= r0 && hi <= r1) return;
  for (unsigned i = lo + lane; i < hi; i += 64)
    if (!inside || i < r0 || i >= r1) d[i] = s[i];
}

template <int U>
void launch(const Box &b, char *host, bool to_device, unsigned row, size_t col, unsigned n, hipStream_t s) {
  const dim3 g((n + 256u * kPerThread - 1) / (256u * kPerThread));
  const bool soa = b.comps > 1;
  auto k = to_device ? (soa ? k_box<U, true, true> : k_box<U, true, false>)
                     : (soa ? k_box<U, false, true> : k_box<U, false, false>);
  hipLaunchKernelGGL(k, g, dim3(256), 0, s, b, host, row, col, n);
  OPSMI_HIP(hipGetLastError());
}

void wait_event(hipEvent_t e) {
  const auto t0 = std::chrono::steady_clock::now();
  for (;;) {
    const hipError_t r = hipEventQuery(e);
    if (r == hipSuccess) return;
    if (r != hipErrorNotReady) OPSMI_HIP(r);
    if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(50)) {
      OPSMI_HIP(hipEventSynchronize(e));
      return;
    }
  }
}

}  // namespace

namespace opsmi {

void Staging::release() {
  for (int q = 0; q < 2; q++) {
    if (host[q]) (void)hipHostFree(host[q]);
    if (ev[q]) (void)hipEventDestroy(ev[q]);
    host[q] = dev[q] = nullptr;
    ev[q] = nullptr;
  }
}

void Staging::ensure() {
  for (int q = 0; q < 2; q++) {
    if (!host[q]) {
      OPSMI_HIP(hipHostMalloc((void **)&host[q], kPiece, hipHostMallocMapped | hipHostMallocCoherent));
      OPSMI_HIP(hipHostGetDevicePointer((void **)&dev[q], host[q], 0));
    }
    if (!ev[q]) OPSMI_HIP(hipEventCreateWithFlags(&ev[q], hipEventDisableTiming));
  }
}

void copy_outside(ops_dat d, char *dst, const char *src, const Range3 &r) {
  const int nd = d->block->dims;
  const int lo[3] = {r.x0, r.y0, r.z0}, hi[3] = {r.x1, r.y1, r.z1};
  unsigned a[3] = {0, 0, 0}, b[3] = {1, 1, 1};
  for (int q = 0; q < nd; q++) {  // raw indexes
    const int first = d->d_m[q] + d->base[q];
    a[q] = (unsigned)std::min(std::max(lo[q] - first, 0), d->size[q]);
    b[q] = (unsigned)std::min(std::max(hi[q] - first, 0), d->size[q]);
  }
  const size_t total = (size_t)d->size[1] * d->size[2];
  int U = 16;
  const size_t es = d->elem_size;
  // units that whole points and the allocation's start are multiples of (the
  // range's ends fall on points)
  while (es % U || (uintptr_t)src % U || (uintptr_t)dst % U) U /= 2;
  const size_t per = es / U, pitch = d->size[0] * per;
  if (total >> 31 || pitch / kSegment > 65000) {
    OPSMI_HIP(hipMemcpyAsync(dst, src, d->mem, hipMemcpyDeviceToDevice, inst().stream));
    return;
  }
  const dim3 g((unsigned)((total + 3) / 4), (unsigned)((pitch + kSegment - 1) / kSegment));
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, g, dim3(256), 0, inst().stream, dst, src, (unsigned)pitch, (unsigned)d->size[1],
                       (unsigned)total, (unsigned)(a[0] * per), (unsigned)(b[0] * per), a[1], b[1], a[2], b[2]);
  };
  if (U == 16) go(k_outside<16>);
  else if (U == 8) go(k_outside<8>);
  else if (U == 4) go(k_outside<4>);
  else if (U == 2) go(k_outside<2>);
  else go(k_outside<1>);
  OPSMI_HIP(hipGetLastError());
}

void box_copy(Staging &st, hipStream_t s, Box b, char *buf, bool to_device) {
  const size_t total = (size_t)b.width * b.rows * b.planes;  // bytes
  if (total == 0) return;
  if ((size_t)b.rows * b.planes >> 32) {  // row numbers are 32 bits
    const unsigned planes = b.planes;
    b.planes = 1;
    for (unsigned z = 0; z < planes; z++, b.base += b.plane, buf += b.width * b.rows)
      box_copy(st, s, b, buf, to_device);
    return;
  }
  if (to_device && b.comps == 1 && b.width > kWideRow) {
    for (unsigned z = 0; z < b.planes; z++)
      OPSMI_HIP(hipMemcpy2DAsync(b.base + (long)z * b.plane, b.pitch, buf + (size_t)z * b.width * b.rows, b.width,
                                 b.width, b.rows, hipMemcpyHostToDevice, s));
    OPSMI_HIP(hipStreamSynchronize(s));
    return;
  }
  st.ensure();
  // the widest unit that every row start (and, by component, every element)
  // is a multiple of
  int U = 16;
  const bool soa = b.comps > 1;
  const unsigned long long all = (unsigned long long)(uintptr_t)b.base | (unsigned long long)b.pitch |
                                 (unsigned long long)b.plane |
                                 (soa ? (unsigned long long)b.cstride | b.elem : (unsigned long long)b.width);
  while (all % U) U /= 2;
  const size_t width_bytes = b.width;
  b.width = width_bytes / U;
  const size_t pieces = (total + kPiece - 1) / kPiece;
  auto bytes_of = [&](size_t k) { return std::min(kPiece, total - k * kPiece); };
  auto start = [&](size_t k) {
    const int q = (int)(k & 1);
    const size_t at = k * kPiece;
    const unsigned row = (unsigned)(at / width_bytes);
    const size_t col = at % width_bytes / U;
    const unsigned n = (unsigned)(bytes_of(k) / U);
    if (U == 16) launch<16>(b, st.dev[q], to_device, row, col, n, s);
    else if (U == 8) launch<8>(b, st.dev[q], to_device, row, col, n, s);
    else if (U == 4) launch<4>(b, st.dev[q], to_device, row, col, n, s);
    else if (U == 2) launch<2>(b, st.dev[q], to_device, row, col, n, s);
    else launch<1>(b, st.dev[q], to_device, row, col, n, s);
    OPSMI_HIP(hipEventRecord(st.ev[q], s));
  };
  if (to_device) {
    for (size_t k = 0; k < pieces; k++) {
      if (k >= 2) wait_event(st.ev[k & 1]);
      memcpy(st.host[k & 1], buf + k * kPiece, bytes_of(k));
      start(k);
    }
    // both buffers are free again on return
    wait_event(st.ev[(pieces - 1) & 1]);
    return;
  }
  start(0);
  for (size_t k = 0; k < pieces; k++) {
    if (k + 1 < pieces) start(k + 1);  // piece k - 1, the buffer's last, has been copied out
    wait_event(st.ev[k & 1]);
    memcpy(buf + k * kPiece, st.host[k & 1], bytes_of(k));
  }
}

}  // namespace opsmi
