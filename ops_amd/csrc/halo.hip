// Multi-block halo exchange behind ops_halo_transfer
// (ops/c/include/ops_lib_core.h:888-911; semantics of the host path
// ops/c/src/sequential/ops_host_singlenode.cpp:172-446).
//
// A halo copies an iter_size box from one dat to another through a linear
// buffer.  Buffer dimension q has extent iter_size[q]; dat dimension i walks
// buffer dimension |dir[i]|-1, forwards when dir[i] > 0 and backwards when
// dir[i] < 0, so blocks may meet with permuted or flipped axes.  Values pass
// through the narrower of the two element types when a float and a double
// dat meet.  A halo whose source and target overlap goes through the buffer
// (one pack and one unpack kernel), as in the reference; the others of a
// group are copied straight from source to target, as many in one launch as
// leave each other's boxes alone (exchanges between neighbours do: they read
// interiors and write halos).
#include "engine.h"

using namespace opsmi;

namespace {

struct HaloSide {
  char *data;          // start of the dat's array (raw index 0)
  long size0, size1;   // raw extents of dims 0, 1
  long pstride;        // bytes between neighbouring points of one component
  long cstride;        // bytes between the components of a point
  int tsize;           // bytes per component
  int dim;             // components
  int first[3];        // raw index of the first box point per dat dimension
  int q[3];            // buffer dimension walked by each dat dimension
  int sgn[3];          // +1 forward, -1 backward
};

struct HaloBox {
  int ext[3];  // buffer extents
};

__device__ __forceinline__ long side_offset(const HaloSide &s, const int *b, const HaloBox &box, int d) {
  long r[3];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const int pos = b[s.q[i]];
    r[i] = s.sgn[i] > 0 ? s.first[i] + pos : s.first[i] + (box.ext[s.q[i]] - 1 - pos);
  }
  return (r[0] + r[1] * s.size0 + r[2] * s.size0 * s.size1) * s.pstride + (long)d * s.cstride;
}

// storage: 8 or 4 bytes per buffer value
template <bool PACK>
__global__ __launch_bounds__(256) void k_halo(HaloSide s, HaloBox box, char *buf, int storage) {
  const long n = (long)box.ext[0] * box.ext[1] * box.ext[2] * s.dim;
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) {
    const int d = (int)(t % s.dim);
    long rest = t / s.dim;
    int b[3];
    b[0] = (int)(rest % box.ext[0]);
    rest /= box.ext[0];
    b[1] = (int)(rest % box.ext[1]);
    b[2] = (int)(rest / box.ext[1]);
    char *p = s.data + side_offset(s, b, box, d);
    char *q = buf + t * storage;
    if (PACK) {
      if (storage == 8) {
        *(double *)q = s.tsize == 8 ? *(double *)p : (double)*(float *)p;
      } else {
        *(float *)q = s.tsize == 4 ? *(float *)p : (float)*(double *)p;
      }
    } else {
      if (s.tsize == 8) *(double *)p = storage == 8 ? *(double *)q : (double)*(float *)q;
      else *(float *)p = storage == 4 ? *(float *)q : (float)*(double *)q;
    }
  }
}

HaloSide make_side(ops_dat dat, const int *base, const int *dir, const int *iter) {
  HaloSide s;
  s.data = dat->data_d;
  s.size0 = dat->size[0];
  s.size1 = dat->size[1];
  // AoS: a point's components are adjacent; SoA (ops_set_soa): each
  // component is one array (ops/c/src/sequential/ops_host_singlenode.cpp:124-131)
  const DatView v = view_of(dat);
  s.pstride = v.sx * dat->type_size;
  s.cstride = v.cs * dat->type_size;
  s.tsize = dat->type_size;
  s.dim = dat->dim;
  const int nd = dat->block->dims;
  for (int i = 0; i < 3; i++) {
    if (i >= nd) {
      s.first[i] = 0;
      s.q[i] = i;
      s.sgn[i] = 1;
      continue;
    }
    int q = abs(dir[i]) - 1;
    if (q < 0 || q >= nd) fail(OPS_INVALID_ARGUMENT, cat("ops_halo_transfer: bad direction ", dir[i]));
    s.q[i] = q;
    s.sgn[i] = dir[i] > 0 ? 1 : -1;
    s.first[i] = base[i] - dat->d_m[i] - dat->base[i];
    if (s.first[i] < 0 || s.first[i] + iter[q] > dat->size[i])
      fail(OPS_INVALID_ARGUMENT, cat("ops_halo_transfer: halo box leaves dat ", dat->name, " in dimension ", i));
  }
  return s;
}

// ------------------------------------------------------------ many halos in one launch
// A side as base + sum of buffer position q times stride[q] (flips folded in)
struct CopySide {
  char *base;
  long stride[3], cstride;  // bytes
};
struct CopyHalo {
  CopySide from, to;
  unsigned ext0, ext1, n;  // buffer extents 0 and 1, values in total
  int dim;
};
// Descriptors travel as kernel arguments, so nothing is uploaded and a call
// keeps no table: pointers are the dats' at this call.  36 of 96 bytes, 3.4 KiB
// of the 4 a launch takes, leave room for the runtime's own arguments (some
// 256 bytes); a larger group takes another launch, 2.5 us.
constexpr int kHalosPerLaunch = 36;
struct CopyHalos {
  CopyHalo h[kHalosPerLaunch];
};
static_assert(sizeof(CopyHalos) + 256 <= 4096, "kernel arguments of a halo launch");

// Bounded by launches and latency, not bytes: twelve 250 x 181 blocks with
// two-point halos (0.2 MB in 34 halos) took 271 us in 68 launches, 6 us in
// one.  One row of workgroups per halo.
template <class F, class T>
__global__ __launch_bounds__(256) void k_halo_copy(CopyHalos all) {
  const CopyHalo &c = all.h[blockIdx.y];
  for (unsigned t = blockIdx.x * 256u + threadIdx.x; t < c.n; t += gridDim.x * 256u) {
    unsigned d = 0, rest = t;
    if (c.dim > 1) {
      d = t % (unsigned)c.dim;
      rest = t / (unsigned)c.dim;
    }
    const long b0 = rest % c.ext0;
    rest /= c.ext0;
    const long b1 = rest % c.ext1, b2 = rest / c.ext1;
    const F v = *(const F *)(c.from.base + b0 * c.from.stride[0] + b1 * c.from.stride[1] + b2 * c.from.stride[2] +
                             (long)d * c.from.cstride);
    *(T *)(c.to.base + b0 * c.to.stride[0] + b1 * c.to.stride[1] + b2 * c.to.stride[2] + (long)d * c.to.cstride) =
        (T)v;
  }
}

CopySide copy_side(const HaloSide &s, const HaloBox &box) {
  const long step[3] = {s.pstride, s.pstride * s.size0, s.pstride * s.size0 * s.size1};
  CopySide c;
  c.base = s.data;
  c.cstride = s.cstride;
  for (int i = 0; i < 3; i++) {
    c.base += step[i] * (s.sgn[i] > 0 ? s.first[i] : s.first[i] + box.ext[s.q[i]] - 1);
    c.stride[s.q[i]] = s.sgn[i] * step[i];
  }
  return c;
}

// the raw index box a side covers in its dat
struct Covered {
  ops_dat dat;
  int lo[3], hi[3];
};
Covered covered(ops_dat dat, const HaloSide &s, const HaloBox &box) {
  Covered c;
  c.dat = dat;
  for (int i = 0; i < 3; i++) {
    c.lo[i] = s.first[i];
    c.hi[i] = s.first[i] + box.ext[s.q[i]];
  }
  return c;
}
bool meet(const Covered &a, const Covered &b) {
  if (a.dat != b.dat) return false;
  for (int i = 0; i < 3; i++)
    if (a.lo[i] >= b.hi[i] || b.lo[i] >= a.hi[i]) return false;
  return true;
}

// halos waiting for their common launch: same element sizes, no target that
// meets another's source or target
struct Pending {
  CopyHalos halos;
  Covered from[kHalosPerLaunch], to[kHalosPerLaunch];
  int n = 0, fs = 0, ts = 0;
  double bytes = 0.0;

  bool takes(const Covered &f, const Covered &t, int fsize, int tsize) const {
    if (n == kHalosPerLaunch || (n > 0 && (fsize != fs || tsize != ts))) return false;
    for (int i = 0; i < n; i++)
      if (meet(to[i], f) || meet(to[i], t) || meet(from[i], t)) return false;
    return true;
  }
  void launch() {
    if (n == 0) return;
    unsigned most = 0;
    for (int i = 0; i < n; i++) most = std::max(most, halos.h[i].n);
    // up to four values a thread
    const unsigned gx = std::max(1u, std::min((most + 1023) / 1024, (unsigned)inst().num_cus * 8));
    const int count = n;
    n = 0;
    run_loop("ops_halo_transfer", bytes, [&](hipStream_t s) {
      const dim3 g(gx, (unsigned)count), b(256);
      if (fs == 8 && ts == 8) hipLaunchKernelGGL((k_halo_copy<double, double>), g, b, 0, s, halos);
      else if (fs == 4 && ts == 4) hipLaunchKernelGGL((k_halo_copy<float, float>), g, b, 0, s, halos);
      else if (fs == 8) hipLaunchKernelGGL((k_halo_copy<double, float>), g, b, 0, s, halos);
      else hipLaunchKernelGGL((k_halo_copy<float, double>), g, b, 0, s, halos);
    });
    bytes = 0.0;
  }
};

void *g_buf = nullptr;
size_t g_buf_bytes = 0;

// source and target overlap: through the buffer
void buffered(const HaloSide &sf, const HaloSide &st, const HaloBox &box, long n, int storage) {
  Instance &I = inst();
  const size_t need = (size_t)n * storage;
  if (need > g_buf_bytes) {
    if (g_buf) {
      OPSMI_HIP(hipStreamSynchronize(I.stream));
      OPSMI_HIP(hipFree(g_buf));
      g_buf = nullptr;
      g_buf_bytes = 0;
    }
    OPSMI_HIP(hipMalloc(&g_buf, need));
    g_buf_bytes = need;
  }
  const int nb = (int)std::min<long>((n + 255) / 256, (long)I.num_cus * 8);
  char *buf = (char *)g_buf;
  run_loop("ops_halo_transfer", 2.0 * n * storage, [&](hipStream_t s) {
    hipLaunchKernelGGL(k_halo<true>, dim3(nb), dim3(256), 0, s, sf, box, buf, storage);
    hipLaunchKernelGGL(k_halo<false>, dim3(nb), dim3(256), 0, s, st, box, buf, storage);
  });
}

void transfer(ops_halo halo, Pending &wait) {
  ops_dat from = halo->from, to = halo->to;
  if (from->dim != to->dim) fail(OPS_INVALID_ARGUMENT, "ops_halo_transfer: dats differ in components");
  DType df = dtype_of(from->type, from->type_size), dt = dtype_of(to->type, to->type_size);
  if (from->type_size != to->type_size && !((df == DT_F64 || df == DT_F32) && (dt == DT_F64 || dt == DT_F32)))
    fail(OPS_INVALID_ARGUMENT, "ops_halo_transfer: mixed exchange needs float/double dats");
  if ((from->type_size != 4 && from->type_size != 8) || (to->type_size != 4 && to->type_size != 8))
    fail(OPS_NOT_IMPLEMENTED, "ops_halo_transfer: element types of 4 or 8 bytes are supported");
  HaloBox box;
  const int nd = from->block->dims;
  for (int i = 0; i < 3; i++) box.ext[i] = i < nd ? halo->iter_size[i] : 1;
  const long n = (long)box.ext[0] * box.ext[1] * box.ext[2] * from->dim;
  if (n <= 0) return;
  const HaloSide sf = make_side(from, halo->from_base, halo->from_dir, box.ext);
  const HaloSide st = make_side(to, halo->to_base, halo->to_dir, box.ext);
  const int storage = std::min(from->type_size, to->type_size);
  sync_to_device(from);
  sync_to_device(to);
  const Covered cf = covered(from, sf, box), ct = covered(to, st, box);
  // permuted axes must be a permutation for the strides to add up
  const bool perm = sf.q[0] + sf.q[1] + sf.q[2] == 3 && sf.q[0] != sf.q[1] && sf.q[1] != sf.q[2] &&
                    st.q[0] + st.q[1] + st.q[2] == 3 && st.q[0] != st.q[1] && st.q[1] != st.q[2];
  if (!perm || meet(cf, ct) || n >= 1L << 31) {
    wait.launch();
    buffered(sf, st, box, n, storage);
  } else {
    if (!wait.takes(cf, ct, from->type_size, to->type_size)) wait.launch();
    wait.fs = from->type_size;
    wait.ts = to->type_size;
    wait.from[wait.n] = cf;
    wait.to[wait.n] = ct;
    wait.halos.h[wait.n++] = CopyHalo{copy_side(sf, box), copy_side(st, box), (unsigned)box.ext[0],
                                      (unsigned)box.ext[1], (unsigned)n, from->dim};
    wait.bytes += 2.0 * n * storage;
  }
  mark_device_dirty(to);
  note_external_write(to);
}

}  // namespace

extern "C" void ops_halo_transfer(ops_halo_group group) {
  OPSMI_API_BEGIN
  require_init();
  flush_all();
  if (!group) fail(OPS_INVALID_ARGUMENT, "ops_halo_transfer: NULL group");
  Pending wait;
  try {
    for (int h = 0; h < group->nhalos; h++) transfer(group->halos[h], wait);
  } catch (...) {
    wait.launch();  // the halos before the refused one
    throw;
  }
  wait.launch();
  OPSMI_API_END()
}
