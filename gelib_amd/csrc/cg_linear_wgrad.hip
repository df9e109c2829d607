// Gradient of the weight matrices of SO3vec CGproduct -> channel mixing, without the product in memory:
//
//   wg_l[c, o] (+)= sum over cells and m of conj(P_l[cell, m, c]) g_l[cell, m, o],   P = CGproduct(x, y)
//
// A GEMM whose reduction runs over the rows (cell, m) of the product, with the product's element as its A operand, formed by
// the lane that feeds it.  v_mfma_f32_32x32x2_f32 computes D (32 x 32) += A (32 x 2) B (2 x 32); lane (i, h) supplies A[i][h]
// and B[h][i]:
//   rows of D  = 32 product channels c = (a, j) of one pair (l1, l2): lane (i, h) forms component h of P_l[cell, m, c];
//   the two k  = real and imaginary part of ONE row (cell, m);
//   columns    = (output channel, component): B = [[gr, gi], [gi, -gr]] for conj(P) g, read from the row of g as it lies in
//                LDS, the halves of the wave in swapped order and with the sign of the second.
// A wave keeps one 32 x 32 sum per l of its pair (16 to 80 registers) and walks along a range of cells; the four waves of a
// block take neighbouring channels of the same pair and share the operands and the rows of g of eight cells at a time in LDS.
// Per channel and cell the lane forms q(m1) = component h of x[m1, a] y[m - m1, j] once for every l of the pair (two
// operations), then one multiply-add per term and one matrix instruction per row (l, m).  The coefficients are the same for
// all lanes: scalar loads.  The sums of the ranges go to memory and a second kernel adds them in the order of the ranges:
// no atomics, the same bits every run.
// Sums in two levels: the matrix instructions add the 2 (2 l + 1) terms of each of eight cells, and those sums are added to a
// second set of registers.  One chain of matrix instructions over a range was up to twice as far from the exact result as
// forming the product and summing it in mix.hip, whose chains are at least 128 rows long (relative error for l = 0..4, one chain /
// two levels / mix.hip, in 1e-7: 8192 cells in chunks of 1024 of 16 x 16 -> 16 channels 2.0 3.0 3.8 4.4 4.9 / 1.4 1.7 2.0 2.2
// 2.5 / 2.3 2.3 2.3 2.4 2.6, all at once - / 1.6 1.9 2.2 2.4 2.6 / 2.3 3.4 4.7 5.7 6.0; 8 x 8 2.6 4.0 5.0 5.9 6.6 /
// 1.4 1.7 2.0 2.2 2.5 / 2.3 2.4 2.5 2.6 2.8; 16 cells of 16 x 16
// 1.2 1.8 2.3 2.8 3.1 / 0.9 1.4 1.7 2.0 2.2 / 1.0 1.4 1.7 2.0 2.3).  The second set takes the kernel from three waves per
// SIMD to two: 8192 cells of 16 x 16 channels 1755 -> 2090 us, 8 x 8 767 -> 920.
// What bounds it: matrix instructions (64 clocks a row and 32 channels) plus vector instructions (4 clocks each, about 2600
// a cell and 32 channels of the L = 4 product), which do not overlap within a wave; the operands come from L2.  Packed parts are
// staged as they lie, 16 bytes a thread: with a quotient by the row length and one by the channel count for every element
// staging was a third of the vector instructions (8192 cells of 16 x 16 channels 2000 -> 1665 us).
// Measured against forming the product, the matrix-gradient kernels of mix.hip on it and their sums (L = 4, 16 outputs,
// microseconds, before that): 8192 cells of 16 x 16 channels 2638 -> 1888 (in 1 GiB 4414 -> 2091), of 8 x 8 910 -> 885; 1024 cells
// 543 -> 263 and 192 -> 140; 64 cells of 16 x 16 153 -> 81.
#include <algorithm>
#include <cstring>
#include <vector>

#include "cg_diag6.h"
#include "cg_linear.h"
#include "cg_unrolled_dev.h"

namespace gelib_hip {

namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef const __attribute__((address_space(4))) float *CoeffPtr;

constexpr int kWNL = kLinL + 1;
constexpr double kWgradLeast = 0.6;      // share of a sum's 32 rows that are channels
// ... and of a block's 128, for this many cells at a time
constexpr double least_of_block(long long ncells) { return ncells <= 2048 ? 0.0 : (ncells <= 8192 ? 0.43 : (ncells <= 16384 ? 0.62 : 0.7)); }
constexpr long long kWgradCells = 16;    // fewer: mix.hip's chains are shorter than those of eight cells here
constexpr int kWPairs = kWNL * kWNL;
constexpr int kWTile = 8;                       // cells staged at a time
constexpr int kWRow = 16;                       // complex numbers of a staged row of g (columns beyond its channels are zero)
constexpr int kWOp = (2 * kLinL + 1) * kLinMaxN;  // complex numbers of one cell's largest operand part

struct LinWgradArgs {
  FastPart x[kWNL], y[kWNL], g[kWNL];  // by l; operands: ptr == nullptr when the part is absent
  float2 *wg[kWNL];                    // gradients of the matrices, by l
  int offs[kWNL][kWNL][kWNL];          // [l1][l2][l]: first channel of the triple's block in product part l
  long long base[kWNL + 1];            // first channel of part l among the channels of all parts; [kWNL]: their number
  const float *bank;                   // coefficient tables, table_off(l1, l2, l)
  float *partial;                      // [range][channel of all parts][32 floats]
  long long ncells, cells_per_range;
  int nranges, accumulate;
  int first[kWPairs + 1];              // pair k = (l1, l2) = (4 - k / 5, 4 - k % 5), the costly ones first: blocks of 128
                                       // channels first[k] .. first[k + 1]
};

// n complex numbers that follow each other, 16 bytes a thread
__device__ __forceinline__ void stage_packed(float2 *dst, const float2 *src, int n, int tid) {
#pragma unroll 2
  for (int e = tid; e < n / 2; e += 256) ((float4 *)dst)[e] = ((const float4 *)src)[e];
  if ((n & 1) && tid == 0) dst[n - 1] = src[n - 1];
}

// LDS: x and y as in memory, [cell of the tile][row][channel]; g per l, [l][cell of the tile][row][16 columns].
template <int L1, int L2, bool PACKED>
__device__ __forceinline__ void wgrad_pair(const LinWgradArgs &a, float2 *xs, float2 *ys, float2 *gs, int group, int range) {
  constexpr int lmin = iabs(L1 - L2), lmax = imin(L1 + L2, kLinL), NLP = lmax - lmin + 1;
  constexpr int R1 = 2 * L1 + 1, R2 = 2 * L2 + 1;
  const FastPart X = a.x[L1], Y = a.y[L2];
  const int n1 = X.n, n2 = Y.n, nch = n1 * n2;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = tid & 31, h = (tid >> 5) & 1;
  const int c0 = group * 128 + wave * 32;   // the wave's first channel of the block
  const bool busy = c0 < nch;               // uniform for the wave; idle waves only stage
  const int c = imin(c0 + i, nch - 1), ca = c / n2, cj = c - ca * n2;
  const float sign = (h && (i & 1)) ? -1.f : 1.f;
  f16v acc[NLP], sum[NLP];
#pragma unroll
  for (int k = 0; k < NLP; k++)
#pragma unroll
    for (int e = 0; e < 16; e++) acc[k][e] = sum[k][e] = 0.f;

  const long long first = (long long)range * a.cells_per_range;
  const long long last = first + a.cells_per_range < a.ncells ? first + a.cells_per_range : a.ncells;
  for (long long cell0 = first; cell0 < last; cell0 += kWTile) {
    const int cells = last - cell0 < kWTile ? (int)(last - cell0) : kWTile;
    __syncthreads();
    if constexpr (PACKED) {
      stage_packed(xs, X.ptr + cell0 * (R1 * n1), cells * R1 * n1, tid);
      stage_packed(ys, Y.ptr + cell0 * (R2 * n2), cells * R2 * n2, tid);
      static_for<NLP>([&](auto dc) __attribute__((always_inline)) {
        constexpr int l = lmin + decltype(dc)::value, first_row = kWTile * (l * l - lmin * lmin);
        const FastPart G = a.g[l];
        float2 *dst = gs + first_row * kWRow;
        const float2 *src = G.ptr + cell0 * ((2 * l + 1) * G.n);
        const int rows = cells * (2 * l + 1);
        if (G.n == kWRow) {
          stage_packed(dst, src, rows * kWRow, tid);
        } else {
#pragma unroll 2
          for (int e = tid; e < rows * kWRow; e += 256) {
            const int o = e & (kWRow - 1);
            dst[e] = o < G.n ? src[(e / kWRow) * G.n + o] : make_float2(0.f, 0.f);
          }
        }
      });
    } else {
      for (int e = tid; e < cells * R1 * n1; e += 256) {
        const int t = e / (R1 * n1), r = e - t * (R1 * n1), m = r / n1;
        xs[e] = X.ptr[(cell0 + t) * X.sb + (long long)m * X.sm + (r - m * n1)];
      }
      for (int e = tid; e < cells * R2 * n2; e += 256) {
        const int t = e / (R2 * n2), r = e - t * (R2 * n2), m = r / n2;
        ys[e] = Y.ptr[(cell0 + t) * Y.sb + (long long)m * Y.sm + (r - m * n2)];
      }
      static_for<NLP>([&](auto dc) __attribute__((always_inline)) {
        constexpr int l = lmin + decltype(dc)::value, first_row = kWTile * (l * l - lmin * lmin);
        const FastPart G = a.g[l];
        for (int e = tid; e < cells * (2 * l + 1) * kWRow; e += 256) {
          const int o = e & (kWRow - 1), tr = e / kWRow, t = tr / (2 * l + 1), m = tr - t * (2 * l + 1);
          gs[first_row * kWRow + e] = o < G.n ? G.ptr[(cell0 + t) * G.sb + (long long)m * G.sm + o] : make_float2(0.f, 0.f);
        }
      });
    }
    __syncthreads();
    if (!busy) continue;
    for (int t = 0; t < cells; t++) {
      // opaque per cell: hoisted out of the loop the coefficients fill the scalar registers many times over and are
      // spilled into vector-register lanes, one more vector instruction per term (8192 cells, 16 channels, sums in one
      // level: 2.48 ms instead of 1.97)
      unsigned long long bank = (unsigned long long)a.bank;
      asm volatile("" : "+s"(bank));
      const CoeffPtr C = (CoeffPtr)bank;
      float u[R1], v[R1];
      float2 yv[R2];
#pragma unroll
      for (int k = 0; k < R1; k++) {
        const float2 x = xs[(t * R1 + k) * n1 + ca];
        u[k] = h ? x.y : x.x;
        v[k] = h ? x.x : -x.y;
      }
#pragma unroll
      for (int k = 0; k < R2; k++) yv[k] = ys[(t * R2 + k) * n2 + cj];
      const float *gp = (const float *)gs + (i ^ h);
      static_for<2 * lmax + 1>([&](auto mc) __attribute__((always_inline)) {
        constexpr int m = decltype(mc)::value - lmax;
        float q[R1];
        static_for<R1>([&](auto kc) __attribute__((always_inline)) {
          constexpr int k = decltype(kc)::value, m2 = m - (k - L1);
          if constexpr (m2 >= -L2 && m2 <= L2) q[k] = __builtin_fmaf(v[k], yv[m2 + L2].y, u[k] * yv[m2 + L2].x);
        });
        static_for<NLP>([&](auto dc) __attribute__((always_inline)) {
          constexpr int l = lmin + decltype(dc)::value;
          if constexpr (iabs(m) <= l) {
            float P = 0.f;
            bool start = true;
            static_for<R1>([&](auto kc) __attribute__((always_inline)) {
              constexpr int k = decltype(kc)::value, m2 = m - (k - L1);
              if constexpr (m2 >= -L2 && m2 <= L2) {
                const float cf = C[table_off(L1, L2, l) + k * R2 + (m2 + L2)];
                P = start ? cf * q[k] : __builtin_fmaf(cf, q[k], P);
                start = false;
              }
            });
            const float B = sign * gp[(kWTile * (l * l - lmin * lmin) + t * (2 * l + 1) + l + m) * 2 * kWRow];
            acc[dc.value] = __builtin_amdgcn_mfma_f32_32x32x2f32(P, B, acc[dc.value], 0, 0, 0);
          }
        });
      });
    }
#pragma unroll
    for (int k = 0; k < NLP; k++)
#pragma unroll
      for (int e = 0; e < 16; e++) {
        sum[k][e] += acc[k][e];
        acc[k][e] = 0.f;
      }
  }
  if (!busy) return;
  // register e of a sum: channel 8 (e / 4) + 4 h + e % 4, column i
  static_for<NLP>([&](auto dc) __attribute__((always_inline)) {
    constexpr int l = lmin + decltype(dc)::value;
    float *out = a.partial + ((long long)range * a.base[kWNL] + a.base[l] + a.offs[L1][L2][l] + c0) * 32 + i;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const int row = 8 * (e / 4) + 4 * h + (e % 4);
      if (c0 + row < nch) out[row * 32] = sum[dc.value][e];
    }
  });
}

// PACKED: every part is packed, so a tile of cells is one piece of memory, and 16-byte aligned.
template <bool PACKED>
__global__ void __launch_bounds__(256, 2) linear_wgrad_kernel(const LinWgradArgs a) {
  __shared__ __align__(16) float2 xs[kWTile * kWOp], ys[kWTile * kWOp], gs[kWTile * kWPairs * kWRow];
  const int work = (int)blockIdx.x / a.nranges, range = (int)blockIdx.x - work * a.nranges;
  static_for<kWPairs>([&](auto kc) __attribute__((always_inline)) {
    constexpr int k = decltype(kc)::value, L1 = kLinL - k / kWNL, L2 = kLinL - k % kWNL;
    if (work >= a.first[k] && work < a.first[k + 1]) wgrad_pair<L1, L2, PACKED>(a, xs, ys, gs, work - a.first[k], range);
  });
}

// One channel's row of its matrix's gradient per block: 16 threads an element, each adding a sixteenth of the ranges, whose
// sums are then added in their order (one chain over all ranges, up to 768 of them, would be the longest sum of all).
__global__ void __launch_bounds__(256) linear_wgrad_sum_kernel(const LinWgradArgs a) {
  __shared__ float2 sums[16][16];
  const int o = (int)threadIdx.x & 15, part = (int)threadIdx.x >> 4;
  const long long ch = blockIdx.x, all = a.base[kWNL];
  const float2 *p = (const float2 *)a.partial + ch * 16 + o;
  float2 s = make_float2(0.f, 0.f);
#pragma unroll 4
  for (int r = a.nranges * part / 16; r < a.nranges * (part + 1) / 16; r++) {
    const float2 v = p[(long long)r * all * 16];
    s.x += v.x;
    s.y += v.y;
  }
  sums[part][o] = s;
  __syncthreads();
  if (part != 0) return;
#pragma unroll
  for (int k = 1; k < 16; k++) s.x += sums[k][o].x, s.y += sums[k][o].y;
  static_for<kWNL>([&](auto lc) __attribute__((always_inline)) {
    constexpr int l = decltype(lc)::value;
    if (ch >= a.base[l] && ch < a.base[l + 1] && o < a.g[l].n) {
      float2 *q = a.wg[l] + (ch - a.base[l]) * a.g[l].n + o;
      if (a.accumulate) {
        s.x += q->x;
        s.y += q->y;
      }
      *q = s;
    }
  });
}

}  // namespace

int cg_linear_wgrad(const VecPlan &plan, const std::vector<const gelib_part_desc *> &g,
                    const std::vector<const gelib_part_desc *> &x, const std::vector<const gelib_part_desc *> &y,
                    const std::vector<float2 *> &wg, const std::vector<long long> &tau, bool accumulate, bool force, void *ws,
                    size_t ws_bytes, hipStream_t s, int *used) {
  *used = 0;
  if (plan.diag || plan.triples.empty() || ((uintptr_t)ws & 15)) return GELIB_HIP_OK;
  std::vector<FastPart> fx, fy, fg;
  std::vector<std::pair<int, int>> lx, ly, lg;
  if (!lists_to_fast(x, plan.E, false, &fx, &lx) || !lists_to_fast(y, plan.E, false, &fy, &ly) ||
      !lists_to_fast(g, plan.E, false, &fg, &lg))
    return GELIB_HIP_OK;
  for (auto &p : lg)
    if (p.first > kLinL || p.second < 1 || p.second > kLinMaxOut) return GELIB_HIP_OK;
  for (auto *L : {&lx, &ly})
    for (auto &p : *L)
      if (p.first > kLinL || p.second < 1 || p.second > kLinMaxN) return GELIB_HIP_OK;
  LinWgradArgs a;
  std::memset(&a, 0, sizeof(a));
  for (size_t k = 0; k < fx.size(); k++) a.x[lx[k].first] = fx[k];
  for (size_t k = 0; k < fy.size(); k++) a.y[ly[k].first] = fy[k];
  long long channels[kWNL] = {0, 0, 0, 0, 0};
  for (size_t k = 0; k < fg.size(); k++) {
    a.g[lg[k].first] = fg[k];
    a.wg[lg[k].first] = wg[k];
    channels[lg[k].first] = tau[k];
  }
  for (int l = 0; l < kWNL; l++) a.base[l + 1] = a.base[l] + channels[l];
  for (auto &t : plan.triples) a.offs[t.l1][t.l2][t.l] = t.offs;
  // every pair reaches every l of its range up to kLinL, as the kernel assumes, and the channels of a matrix are those the
  // pairs feed
  double useful = 0, padded = 0, blocks = 0;
  for (auto &p : lx)
    for (auto &q : ly) {
      int have = 0;
      for (auto &t : plan.triples) have += (t.l1 == p.first && t.l2 == q.first);
      if (have != std::min(p.first + q.first, kLinL) - std::abs(p.first - q.first) + 1) return GELIB_HIP_OK;
      const long long n = (long long)p.second * q.second;
      const double rows = (2.0 * p.first + 1) * (2 * q.first + 1);
      useful += rows * (double)n;
      padded += rows * (double)((n + 31) / 32 * 32);
      blocks += rows * (double)((n + 127) / 128 * 128);
    }
  const long long ncells = plan.E[0] * plan.E[1] * plan.E[2];
  if (ncells < kWgradCells) return GELIB_HIP_OK;
  // Channels fill the 32 rows of a sum and the 128 of a block; with fewer than 19 channels a pair half the matrix work is
  // padding, and with fewer than 128 some waves of a block only stage.  The product of few channels is small enough to store
  // once there are cells enough to hide the launches that takes (with the gradients of x and y, 12 outputs, product stored /
  // not, microseconds: 256 cells, 32 channels a pair 263 / 193; 2048 cells, 32 channels 365 / 361, 40 channels 468 / 450;
  // 3072 cells, 32 channels 524 / 533; 4096 cells, 48 channels 888 / 896, 56 channels 1043 / 955; 8192 cells, 50 channels 1837 /
  // 1906, 56 channels 1729 / 1670, 132 channels 3672 / 3700; 16384 cells, 64 channels 3105 / 3262, 80 channels 4010 / 3876, 144
  // channels 6413 / 6908, 192 channels 8651 / 8297; 32768 cells, 80 channels 7428 / 7964, 96 channels 8905 / 8412, 156
  // channels 15.7 / 16.2 ms, 192 channels 17.3 / 16.6).
  if (!force && (useful < kWgradLeast * padded || useful < least_of_block(ncells) * blocks)) return GELIB_HIP_OK;
  int nwork = 0;
  for (int k = 0; k < kWPairs; k++) {
    const int l1 = kLinL - k / kWNL, l2 = kLinL - k % kWNL;
    a.first[k] = nwork;
    if (a.x[l1].ptr && a.y[l2].ptr) nwork += (a.x[l1].n * a.y[l2].n + 127) / 128;
  }
  a.first[kWPairs] = nwork;
  if (nwork == 0) return GELIB_HIP_OK;
  // ranges of cells: three blocks per place of the GPU (two blocks a compute unit: two waves per SIMD), at least two tiles of
  // cells each, as far as the memory for their sums goes
  const long long fit = (long long)(ws_bytes / ((size_t)a.base[kWNL] * 32 * sizeof(float)));
  long long nranges = std::min<long long>({(1536LL + nwork - 1) / nwork, (ncells + 2 * kWTile - 1) / (2 * kWTile), fit});
  if (nranges < 1) return GELIB_HIP_OK;
  a.cells_per_range = ((ncells + nranges - 1) / nranges + kWTile - 1) / kWTile * kWTile;
  nranges = (ncells + a.cells_per_range - 1) / a.cells_per_range;
  int rc = cg_table_bank(&a.bank);
  if (rc) return rc;
  a.partial = (float *)ws;
  bool all_packed = true;
  auto packed = [&](const std::vector<FastPart> &v, const std::vector<std::pair<int, int>> &ln) {
    for (size_t k = 0; k < v.size(); k++)
      if (v[k].sm != ln[k].second || v[k].sb != (long long)(2 * ln[k].first + 1) * ln[k].second || ((uintptr_t)v[k].ptr & 15)) all_packed = false;
  };
  packed(fx, lx), packed(fy, ly), packed(fg, lg);
  a.ncells = ncells;
  a.nranges = (int)nranges;
  a.accumulate = accumulate ? 1 : 0;
  if (all_packed) hipLaunchKernelGGL(linear_wgrad_kernel<true>, dim3((unsigned)(nwork * nranges)), dim3(256), 0, s, a);
  else hipLaunchKernelGGL(linear_wgrad_kernel<false>, dim3((unsigned)(nwork * nranges)), dim3(256), 0, s, a);
  GELIB_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(linear_wgrad_sum_kernel, dim3((unsigned)a.base[kWNL]), dim3(256), 0, s, a);
  GELIB_HIP_TRY(hipGetLastError());
  *used = 1;
  return GELIB_HIP_OK;
}

}  // namespace gelib_hip
