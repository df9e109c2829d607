// Sum of slices along one leading dimension of the parts of a vector:  r[.., t, ..] (+)= sum over the sources s of target
// t of x[.., s, ..]  -- the message-passing step that feeds the products (core/Gpart.hpp:537-563; the loop itself is
// cnine::GatherSlices, which is not part of the reference tree).
//
// The map arrives target-major (row_ptr / sources), so every output element is written by exactly one thread, which
// adds its sources in the order of the map: no atomics, and the float sum is reproducible.
//
// What bounds it: the slices of a target's sources, 8 B per (pair, element), which come from the memory-side cache or from
// HBM in pieces of one slice (128 B to 1.2 KB), and 8 B written per output element.  The kernel keeps as many of those
// reads in flight as it can: a thread owns 16 bytes of a target's slice (8 where alignment or an odd length forbids
// more), the indices and then the slices of four sources are requested together, and consecutive threads walk along a
// slice, so a wave's accesses are whole runs of a slice.  One launch serves all parts of a vector: with one each, three
// parts of 50021 nodes cost three launches of 50 us a direction, and a zero-fill each.
// L = 2, 16 channels, 50021 nodes, 8 sources each, one direction: 152 us in three launches (8 bytes a thread, one source at a
// time, 64-bit divisions) -> 68 us, 461 MB of slices at 6.8 TB/s.
#include <algorithm>
#include <cstring>

#include "cg_common.h"
#include "gather_plan.h"

namespace gelib_hip {

namespace {

struct GatherPart {
  float2 *r;
  const float2 *x;
  GatherSlices s;
  unsigned first_block;
};

struct GatherVecArgs {
  GatherPart p[kGatherParts];
  const int *row_ptr;      // [targets + 1]
  const int *sources;      // [row_ptr[targets]]
  unsigned targets;
  int nparts, accumulate;
};

template <int VEC>
struct Cplx;
template <>
struct Cplx<1> {
  typedef float2 T;
  static __device__ __forceinline__ void add(T &a, const T &b) { a.x += b.x, a.y += b.y; }
};
template <>
struct Cplx<2> {
  typedef float4 T;
  static __device__ __forceinline__ void add(T &a, const T &b) { a.x += b.x, a.y += b.y, a.z += b.z, a.w += b.w; }
};

template <int VEC>
__device__ __forceinline__ void gather_one(const GatherVecArgs &a, const GatherPart &p, unsigned w) {
  typedef typename Cplx<VEC>::T T;
  const unsigned row = p.s.magic ? (unsigned)__umul64hi(p.s.magic, w) : w;   // outer * targets + t
  const unsigned q = w - row * p.s.per_target;
  const unsigned o = row < a.targets ? 0u : row / a.targets, t = row - o * a.targets;
  const float2 *xp = p.x + (long long)o * p.s.xo + gather_element(q, VEC);
  float2 *rp = p.r + (long long)o * p.s.ro + (long long)t * p.s.rt + gather_element(q, VEC);
  const int k0 = a.row_ptr[t], k1 = a.row_ptr[t + 1];
  T acc = {};
  if (a.accumulate) acc = *(const T *)rp;
  int k = k0;
  for (; k + 4 <= k1; k += 4) {
    int s[4];
    T v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) s[i] = a.sources[k + i];
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = *(const T *)(xp + (long long)s[i] * p.s.xt);
#pragma unroll
    for (int i = 0; i < 4; i++) Cplx<VEC>::add(acc, v[i]);
  }
  if (k < k1) {  // up to three more; the spare requests repeat the last source and are not added
    int s[3];
    T v[3];
#pragma unroll
    for (int i = 0; i < 3; i++) s[i] = a.sources[k + i < k1 ? k + i : k1 - 1];
#pragma unroll
    for (int i = 0; i < 3; i++) v[i] = *(const T *)(xp + (long long)s[i] * p.s.xt);
#pragma unroll
    for (int i = 0; i < 3; i++)
      if (k + i < k1) Cplx<VEC>::add(acc, v[i]);
  }
  *(T *)rp = acc;
}

__global__ void __launch_bounds__(256) gather_vec_kernel(const GatherVecArgs a) {
  GatherPart p = a.p[0];
#pragma unroll
  for (int k = 1; k < kGatherParts; k++)
    if (k < a.nparts && blockIdx.x >= a.p[k].first_block) p = a.p[k];
  const long long w = (long long)(blockIdx.x - p.first_block) * 256 + threadIdx.x;
  if (w >= p.s.total) return;
  if (p.s.vec == 2) gather_one<2>(a, p, (unsigned)w);
  else gather_one<1>(a, p, (unsigned)w);
}

struct GatherArgs {
  float2 *r;
  const float2 *x;
  long long rs[5], xs[5];  // strides in complex elements over (batch, grid0, grid1, m, channel)
  long long D[5];          // extents of r
  const int *row_ptr;      // [D[dim] + 1]
  const int *sources;      // [row_ptr[D[dim]]], each below the extent of x along dim
  int dim, accumulate;
};

// Any strides: one thread per element, the element index running fastest.
__global__ void __launch_bounds__(256) gather_kernel(const GatherArgs a) {
  // extents with the gathered dimension taken out: one thread per element of a target slice, the element index
  // running fastest, so a wave covers 64 consecutive elements of one target (or the end of one and the start of the next)
  long long E[5];
  for (int k = 0; k < 5; k++) E[k] = k == a.dim ? 1 : a.D[k];
  const long long per_target = E[0] * E[1] * E[2] * E[3] * E[4];
  const long long total = per_target * a.D[a.dim];
  for (long long w = (long long)blockIdx.x * blockDim.x + threadIdx.x; w < total; w += (long long)gridDim.x * blockDim.x) {
    const long long t = w / per_target;
    long long rem = w - t * per_target, ro = t * a.rs[a.dim], xo = 0;
    for (int k = 4; k >= 0; k--) {
      const long long i = rem % E[k];
      rem /= E[k];
      ro += k == a.dim ? 0 : i * a.rs[k];
      xo += i * a.xs[k];   // i = 0 along the gathered dimension
    }
    float2 acc = a.accumulate ? a.r[ro] : make_float2(0.f, 0.f);
    const int k0 = a.row_ptr[t], k1 = a.row_ptr[t + 1];
    for (int k = k0; k < k1; k++) {
      const float2 v = a.x[xo + (long long)a.sources[k] * a.xs[a.dim]];
      acc.x += v.x;
      acc.y += v.y;
    }
    a.r[ro] = acc;
  }
}

int launch_any(const GatherJob &j, int dim, const int *row_ptr, const int *sources, bool accumulate, hipStream_t s) {
  GatherArgs a;
  a.r = j.r;
  a.x = j.x;
  long long total = 1;
  for (int k = 0; k < 5; k++) {
    a.rs[k] = j.rs[k];
    a.xs[k] = j.xs[k];
    a.D[k] = j.D[k];
    total *= j.D[k];
  }
  a.dim = dim;
  a.row_ptr = row_ptr;
  a.sources = sources;
  a.accumulate = accumulate ? 1 : 0;
  const long long want = (total + 255) / 256;
  hipLaunchKernelGGL(gather_kernel, dim3((unsigned)std::min<long long>(want, 256LL * 64)), dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 10;
}

}  // namespace

int launch_gather(const std::vector<GatherJob> &jobs, int dim, const int *row_ptr, const int *sources, bool accumulate,
                  hipStream_t s) {
  GatherVecArgs a;
  std::memset(&a, 0, sizeof(a));
  a.row_ptr = row_ptr;
  a.sources = sources;
  a.accumulate = accumulate ? 1 : 0;
  unsigned blocks = 0;
  auto flush = [&]() {
    if (a.nparts == 0) return 0;
    hipLaunchKernelGGL(gather_vec_kernel, dim3(blocks), dim3(256), 0, s, a);
    a.nparts = 0;
    blocks = 0;
    return hipGetLastError() == hipSuccess ? 0 : 10;
  };
  for (auto &j : jobs) {
    GatherPart p;
    int rc = 0;
    if (!gather_slices(j.rs, j.xs, j.D, dim, (((uintptr_t)j.r | (uintptr_t)j.x) & 15) == 0, &p.s)) {
      if ((rc = launch_any(j, dim, row_ptr, sources, accumulate, s))) return rc;
      continue;
    }
    a.targets = (unsigned)j.D[dim];   // the same for every part: the map says it
    const unsigned nb = (unsigned)gather_blocks(p.s.total);
    if (!gather_shares_launch(a.nparts, blocks, nb) && (rc = flush())) return rc;
    p.r = j.r;
    p.x = j.x;
    p.first_block = blocks;
    blocks += nb;
    a.p[a.nparts++] = p;
  }
  return flush();
}

}  // namespace gelib_hip
