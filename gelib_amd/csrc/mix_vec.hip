// Channel mixing of all parts of a vector in one launch, and its two gradients: complex matrix products
//     C_k[m, n] = sum_k A_k[m, k] B_k[k, n]        (one per part)
// of any sizes.  mix.hip's kernels want an even number of channels and rows that are 16-byte aligned, and cost a launch for the
// re-packed matrix and one or two more per part and direction; a layer on a few hundred cells, or with few channels, is over
// sooner than its launches, and one with odd counts went to the library's complex matrix product, which is slow where one side
// is long and the others are short.  Layers, forward and backward: L = 4, 7 x 7 -> 26 channels, 3631 cells 14.6 -> 1.4 ms, 3 x 1 -> 17,
// 2910 cells 10.8 -> 0.63 ms, L = 3, 15 x 15 -> 7, 5897 cells 13.3 -> 2.8 ms.
//
// A block of 256 threads takes BM x BN of one part's result; 16 values of k at a time go through LDS, the next 16 on their way
// meanwhile.  A thread holds RT rows and OT columns: per k it reads RT + OT complex numbers from LDS and does 4 RT OT
// multiply-adds.  The 16 terms of a step are added by themselves and then to the thread's sum: a chain of thousands of
// channels or rows is sixteen times shorter.  Results with few tiles are cut along k (splits): the partial results go to the
// workspace and a second launch adds them in their order; no atomics.
// What bounds it: small calls the latency of the steps (about 1 us each), large ones the vector unit at a third of its rate
// (LDS reads and the address arithmetic beside the multiply-adds), the gradient of the product the stores.
#include <algorithm>
#include <cstdint>
#include <cstring>
#include <vector>

#include "mix_vec.h"

namespace gelib_hip {

namespace {

constexpr int kVMParts = 16;   // parts of one launch
constexpr int kVMK = 16;       // values of k per step
constexpr int kVMSplits = 64;  // most pieces of k
constexpr int kVMBlocks = 1024;  // blocks that a launch aims at when it cuts k (four per compute unit)

struct VMPart {
  const float2 *a, *b;
  float2 *c;
  float2 *part;             // [split][m][n], or nullptr: straight into c
  long long m, k, per;      // per: values of k of a split
  long long n;
  long long first;          // first block
  int mtiles, ntiles, splits;
};
struct VMArgs {
  VMPart p[kVMParts];
  int nparts;
  long long sum_first[kVMParts + 1];   // summing launch: first element of part k
};
typedef const __attribute__((address_space(4))) VMArgs *VMArgPtr;

template <int MODE, int OG, int OT, int RT>
__global__ void __launch_bounds__(256) vec_mix_kernel(const VMArgs) {
  constexpr int RG = 256 / OG, BM = RG * RT, BN = OG * OT, K = kVMK;
  constexpr int NA = BM * K / 256, NB = (BN * K + 255) / 256;
  __shared__ float2 as[K][BM + 1], bs[K][BN + 1];
  // the parts are read from the argument segment by a run-time index (scalar loads)
  const VMArgPtr args = (VMArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
  int pi = 0;
  while (pi + 1 < args->nparts && (long long)blockIdx.x >= args->p[pi + 1].first) pi++;
  const __attribute__((address_space(4))) VMPart &p = args->p[pi];
  const long long M = p.m, N = p.n, KK = p.k;
  long long at = (long long)blockIdx.x - p.first;
  const int nt = (int)(at % p.ntiles);
  at /= p.ntiles;
  const long long mt = at % p.mtiles;
  const int split = (int)(at / p.mtiles);
  const long long m0 = mt * BM, n0 = (long long)nt * BN;
  const long long kbegin = split * p.per, kend = kbegin + p.per < KK ? kbegin + p.per : KK;
  const float2 *A = p.a, *B = p.b;
  const int tid = threadIdx.x, og = tid % OG, rg = tid / OG;

  // element e of the tile of A: k runs along the lanes where it is contiguous in memory, m otherwise
  float2 ra[NA], rb[NB];
  auto fetch = [&](long long k0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NA; u++) {
      const int e = tid + 256 * u;
      const int mi = MODE == kVMGrad ? e % BM : e / K, ki = MODE == kVMGrad ? e / BM : e % K;
      const long long m = m0 + mi < M ? m0 + mi : M - 1, k = k0 + ki < kend ? k0 + ki : kend - 1;
      float2 v = MODE == kVMGrad ? A[k * M + m] : A[m * KK + k];
      if (MODE == kVMGrad) v.y = -v.y;
      if (k0 + ki >= kend) v = make_float2(0.f, 0.f);
      ra[u] = v;
    }
#pragma unroll
    for (int u = 0; u < NB; u++) {
      const int e = tid + 256 * u;
      const int ni = MODE == kVMAdjoint ? (e / K) % BN : e % BN, ki = MODE == kVMAdjoint ? e % K : (e / BN) % K;
      const long long n = n0 + ni < N ? n0 + ni : N - 1, k = k0 + ki < kend ? k0 + ki : kend - 1;
      float2 v = MODE == kVMAdjoint ? B[n * KK + k] : B[k * N + n];
      if (MODE == kVMAdjoint) v.y = -v.y;
      if (k0 + ki >= kend) v = make_float2(0.f, 0.f);
      rb[u] = v;
    }
  };
  auto stage = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NA; u++) {
      const int e = tid + 256 * u;
      if (MODE == kVMGrad) as[e / BM][e % BM] = ra[u];
      else as[e % K][e / K] = ra[u];
    }
#pragma unroll
    for (int u = 0; u < NB; u++) {
      const int e = tid + 256 * u;
      if (BN * K % 256 == 0 || e < BN * K) {
        if (MODE == kVMAdjoint) bs[e % K][e / K] = rb[u];
        else bs[e / BN][e % BN] = rb[u];
      }
    }
  };

  float2 sum[RT][OT];
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int o = 0; o < OT; o++) sum[r][o] = make_float2(0.f, 0.f);
  fetch(kbegin);
  for (long long k0 = kbegin; k0 < kend; k0 += K) {
    __syncthreads();   // the reads of the last step are over
    stage();
    __syncthreads();
    if (k0 + K < kend) fetch(k0 + K);   // uniform
    float2 acc[RT][OT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int o = 0; o < OT; o++) acc[r][o] = make_float2(0.f, 0.f);
#pragma unroll
    for (int k = 0; k < K; k++) {
      float2 x[RT], v[OT];
#pragma unroll
      for (int r = 0; r < RT; r++) x[r] = as[k][rg + RG * r];
#pragma unroll
      for (int o = 0; o < OT; o++) v[o] = bs[k][og + OG * o];
#pragma unroll
      for (int r = 0; r < RT; r++)
#pragma unroll
        for (int o = 0; o < OT; o++) {
          acc[r][o].x = fmaf(x[r].x, v[o].x, acc[r][o].x);
          acc[r][o].x = fmaf(-x[r].y, v[o].y, acc[r][o].x);
          acc[r][o].y = fmaf(x[r].x, v[o].y, acc[r][o].y);
          acc[r][o].y = fmaf(x[r].y, v[o].x, acc[r][o].y);
        }
    }
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int o = 0; o < OT; o++) sum[r][o].x += acc[r][o].x, sum[r][o].y += acc[r][o].y;
  }
  float2 *C = p.part ? p.part + (long long)split * M * N : p.c;
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int o = 0; o < OT; o++) {
      const long long m = m0 + rg + RG * r, n = n0 + og + OG * o;
      if (m < M && n < N) C[m * N + n] = sum[r][o];
    }
}

// c[e] = the splits' partial results, added in their order; a thread an element
__global__ void __launch_bounds__(256) vec_mix_sum_kernel(const VMArgs) {
  const VMArgPtr args = (VMArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= args->sum_first[args->nparts]) return;
  for (int k = 0; k < args->nparts; k++) {
    if (idx < args->sum_first[k] || idx >= args->sum_first[k + 1]) continue;
    const __attribute__((address_space(4))) VMPart &p = args->p[k];
    const long long e = idx - args->sum_first[k], all = p.m * p.n;
    const float2 *q = p.part + e;
    float2 s = make_float2(0.f, 0.f);
#pragma unroll 4
    for (int i = 0; i < p.splits; i++) {
      const float2 v = q[i * all];
      s.x += v.x;
      s.y += v.y;
    }
    p.c[e] = s;
  }
}

// The tile: columns for the widest part, and rows so that a thread holds four results where the columns are few.
struct VMShape {
  int og, ot, rt;
  int bm() const { return 256 / og * rt; }
  int bn() const { return og * ot; }
};
VMShape shape_of(const std::vector<VecMixPart> &parts) {
  long long n = 0;
  for (auto &p : parts) n = std::max(n, p.n);
  if (n <= 4) return {4, 1, 2};
  if (n <= 8) return {8, 1, 4};
  if (n <= 16) return {16, 1, 4};
  return {16, 2, 4};
}

// the launch's blocks and the pieces of k of every part, as many as their partial results have room for; false: too many blocks
bool plan(const std::vector<VecMixPart> &parts, const VMShape &sh, size_t room, std::vector<VMPart> *out, long long *blocks, size_t *bytes) {
  out->clear();
  long long tiles = 0;
  for (auto &p : parts) {
    VMPart q;
    std::memset(&q, 0, sizeof(q));
    q.a = p.a, q.b = p.b, q.c = p.c;
    q.m = p.m, q.n = p.n, q.k = p.k;
    const long long mt = (p.m + sh.bm() - 1) / sh.bm(), nt = (p.n + sh.bn() - 1) / sh.bn();
    if (mt > 0x3fffffff || nt > 0x3fffffff) return false;
    q.mtiles = (int)mt, q.ntiles = (int)nt;
    tiles += mt * nt;
    out->push_back(q);
  }
  // a split has at least eight steps, so that writing and adding its partial result stays small beside it
  long long first = 0;
  size_t off = 0;
  for (auto &q : *out) {
    const long long want = std::max<long long>(1, kVMBlocks / std::max<long long>(1, tiles));
    const size_t piece = (size_t)q.m * q.n * sizeof(float2);
    const long long fit = (long long)(((room - off) & ~(size_t)255) / piece);
    long long s = std::max<long long>(1, std::min<long long>({want, q.k / (8 * kVMK), (long long)kVMSplits, fit}));
    q.per = ((q.k + s - 1) / s + kVMK - 1) / kVMK * kVMK;
    s = (q.k + q.per - 1) / q.per;
    q.splits = (int)s;
    q.first = first;
    first += (long long)q.mtiles * q.ntiles * s;
    if (s > 1) {
      q.part = (float2 *)off;   // the offset for now
      off += (s * piece + 255) & ~(size_t)255;
    }
  }
  *blocks = first;
  *bytes = off;
  return first < (1LL << 24);   // fewer than 2^32 threads
}

template <int MODE>
void launch_mode(const VMShape &sh, const VMArgs &a, long long blocks, hipStream_t s) {
  const dim3 grid((unsigned)blocks), block(256);
  if (sh.og == 4) hipLaunchKernelGGL((vec_mix_kernel<MODE, 4, 1, 2>), grid, block, 0, s, a);
  else if (sh.og == 8) hipLaunchKernelGGL((vec_mix_kernel<MODE, 8, 1, 4>), grid, block, 0, s, a);
  else if (sh.ot == 1) hipLaunchKernelGGL((vec_mix_kernel<MODE, 16, 1, 4>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((vec_mix_kernel<MODE, 16, 2, 4>), grid, block, 0, s, a);
}

// parts with something to compute, kVMParts at a time
std::vector<std::vector<VecMixPart>> groups_of(const std::vector<VecMixPart> &parts) {
  std::vector<std::vector<VecMixPart>> g;
  for (auto &p : parts) {
    if (p.m == 0 || p.n == 0 || p.k == 0) continue;
    if (g.empty() || g.back().size() == kVMParts) g.emplace_back();
    g.back().push_back(p);
  }
  return g;
}

}  // namespace

size_t vec_mix_workspace_bytes(const std::vector<VecMixPart> &parts) {
  size_t most = 0;
  for (auto &g : groups_of(parts)) {
    std::vector<VMPart> q;
    long long blocks = 0;
    size_t bytes = 0;
    plan(g, shape_of(g), SIZE_MAX, &q, &blocks, &bytes);
    most = std::max(most, bytes);
  }
  return most;
}

int launch_vec_mix(const std::vector<VecMixPart> &parts, int mode, void *ws, size_t ws_bytes, bool fit, hipStream_t s) {
  for (auto &g : groups_of(parts)) {
    const VMShape sh = shape_of(g);
    std::vector<VMPart> q;
    long long blocks = 0;
    size_t bytes = 0;
    if (!plan(g, sh, fit ? ws_bytes : SIZE_MAX, &q, &blocks, &bytes)) return 11;
    if (bytes && (!ws || ((uintptr_t)ws & 15) || ws_bytes < bytes)) return 13;
    VMArgs a;
    std::memset(&a, 0, sizeof(a));
    a.nparts = (int)q.size();
    long long sums = 0;
    for (size_t k = 0; k < q.size(); k++) {
      if (q[k].splits > 1) q[k].part = (float2 *)((char *)ws + (size_t)q[k].part);
      a.p[k] = q[k];
      a.sum_first[k] = sums;
      if (q[k].splits > 1) sums += q[k].m * q[k].n;
    }
    a.sum_first[q.size()] = sums;
    if (mode == kVMForward) launch_mode<kVMForward>(sh, a, blocks, s);
    else if (mode == kVMAdjoint) launch_mode<kVMAdjoint>(sh, a, blocks, s);
    else launch_mode<kVMGrad>(sh, a, blocks, s);
    GELIB_HIP_TRY(hipGetLastError());
    if (sums) {
      hipLaunchKernelGGL(vec_mix_sum_kernel, dim3((unsigned)((sums + 255) / 256)), dim3(256), 0, s, a);
      GELIB_HIP_TRY(hipGetLastError());
    }
  }
  return GELIB_HIP_OK;
}

}  // namespace gelib_hip
