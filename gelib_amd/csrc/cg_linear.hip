// Host side and helper kernels of the fused SO3vec CGproduct -> channel mixing forward pass (the kernel itself:
// cg_linear_impl.h): the matrices re-packed for the matrix cores, the first operand transposed per group of cells, the
// two launches.
#include <algorithm>
#include <cstring>
#include <vector>

#include "cg_linear_impl.h"

namespace gelib_hip {

namespace {

// xt[group][e][slot] = x[cell 32 group + slot][e], e = row * n + channel; cells beyond the last repeat it.
__global__ void __launch_bounds__(256) transpose_cells_kernel(float2 *xt, const FastPart X, int elems, long long ncells) {
  __shared__ float2 tile[32][33];
  const long long g = blockIdx.x;
  const int e0 = blockIdx.y * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int c = ty; c < 32; c += 8) {
    long long cell = g * 32 + c;
    cell = cell < ncells ? cell : ncells - 1;
    const int e = e0 + tx;
    if (e < elems) tile[c][tx] = X.ptr[cell * X.sb + (long long)(e / X.n) * X.sm + (e % X.n)];
  }
  __syncthreads();
  for (int ee = ty; ee < 32; ee += 8) {
    const int e = e0 + ee;
    if (e < elems) xt[(g * elems + e) * 32 + tx] = tile[tx][ee];
  }
}

// wp[c][h][2 o + p]: the real 2 x 2 form of W[c, o] = wr + i wi, rows h = (real, imaginary) part of the product's
// element, columns p = (real, imaginary) part of the result: [[wr, wi], [-wi, wr]]; columns beyond n_out are zero.
__global__ void pack_linear_kernel(float *wp, const float2 *w, long long tau, int n_out) {
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (tau + kBAhead) * 64) return;
  const long long c = idx >> 6;
  const int hh = (idx >> 5) & 1, col = idx & 31, o = col >> 1, p = col & 1;
  float val = 0.f;
  if (c < tau && o < n_out) {
    const float2 e = w[c * n_out + o];
    val = hh == 0 ? (p ? e.y : e.x) : (p ? e.x : -e.y);
  }
  wp[idx] = val;
}

// out_l[cell, m, o] (+)= sum over the shares of partial[share][group][l^2 + l + m][cell of the group][2 o, 2 o + 1], in the
// order of the shares; one thread per complex number.  Memory-bound (8192 cells, 4 shares: 105 MB read, 26 MB written).
__global__ void __launch_bounds__(256) sum_shares_kernel(const LinArgs a, int shares, long long groups) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;   // (group, row, cell of the group, o)
  const int o = idx & 15, c = (idx >> 4) & 31;
  const long long gr = idx >> 9;
  const long long g = gr / kLinRows;
  if (g >= groups) return;
  const int lm = (int)(gr - g * kLinRows);
  const long long cell = g * kLinCells + c;
  if (cell >= a.ncells) return;
  static_for<kNL>([&](auto lc) __attribute__((always_inline)) {
    constexpr int l = decltype(lc)::value;
    if (lm >= l * l && lm < (l + 1) * (l + 1)) {
      const FastPart O = a.out[l];
      if (o < O.n) {
        const float2 *p = (const float2 *)a.partial + (gr * kLinCells + c) * 16 + o;
        float2 s = make_float2(0.f, 0.f);
        for (int k = 0; k < shares; k++) {
          const float2 v = p[(long long)k * groups * (kLinGroupFloats / 2)];
          s.x += v.x;
          s.y += v.y;
        }
        float2 *q = O.ptr + cell * O.sb + (long long)(lm - l * l) * O.sm + o;
        if (a.accumulate) {
          s.x += q->x;
          s.y += q->y;
        }
        *q = s;
      }
    }
  });
}

size_t packed_bytes(long long tau) { return (size_t)(tau + kBAhead) * 256; }  // padding behind the last channel

// Waves that share a group of cells: split_a shares of the channels of x, times kLinSets sets of parts of y.
// A wave takes most of a SIMD's registers, so a launch fills the GPU with 1024 waves, and one of G groups takes
// ceil(G * shares / 1024) rounds of what one wave has to do: the channels of its share, plus about 3 % of a whole group's
// work for the pairs' coefficients, plus the writing and summing of the partial results (a 50000th of a whole group's time
// per wave).  The cheapest choice is taken; with 1024 groups (32768 cells) that is one wave per group, as it is for whole
// multiples of it.  One wave per group / shared, microseconds: L=4, 16 x 16 -> 16 channels, 64 cells 5340 / 187,
// 1024 cells 5380 / 306, 5003 cells 5430 / 1210, 8192 cells 5440 / 1570, 20000 cells 5470 / 4100, 32768 cells 5570 / (not
// shared) 5610, 40000 cells 11340 / 8700; 7 x 3 -> 12 channels, 8192 cells 896 / 327.
struct LinSplit {
  int a = 1, l2 = 0;
  int shares() const { return a * (l2 ? kLinSets : 1); }
};
constexpr long long kLinWaves = 1024;       // waves that run at once
constexpr long long kLinMaxPartial = 4096;  // most (share, group) pairs: 420 MB of partial sums

LinSplit choose_split(long long groups, int nmax) {
  LinSplit best;
  double least = 0;
  for (int l2 = 0; l2 < 2; l2++)
    for (int sa = 1; sa <= nmax; sa++) {
      LinSplit t;
      t.a = sa;
      t.l2 = l2;
      const long long waves = groups * t.shares();
      if (t.shares() > 1 && waves > kLinMaxPartial) continue;
      const double mine = ((double)((nmax + sa - 1) / sa) / nmax + 0.03) * (l2 ? 0.27 : 1.0);
      const double cost = (double)((waves + kLinWaves - 1) / kLinWaves) * mine + (t.shares() > 1 ? 2e-5 * (double)waves : 0.0);
      if (t.shares() == 1 || cost < least) {
        least = cost;
        best = t;
      }
    }
  return best;
}

size_t plain_workspace_bytes(const long long tau[kLinL + 1], long long x_elems_per_cell, long long groups) {
  size_t total = 0;
  for (int l = 0; l <= kLinL; l++) total += packed_bytes(tau[l]);
  return total + (size_t)groups * kLinCells * (size_t)x_elems_per_cell * sizeof(float2);
}

size_t partial_bytes(const LinSplit &t, long long groups) {
  return t.shares() > 1 ? (size_t)t.shares() * groups * kLinGroupFloats * sizeof(float) : 0;
}

}  // namespace

size_t cg_linear_workspace_bytes(const long long tau[kLinL + 1], long long x_elems_per_cell, int x_channels, long long ncells) {
  const long long groups = (ncells + kLinCells - 1) / kLinCells;
  const size_t plain = plain_workspace_bytes(tau, x_elems_per_cell, groups);
  if (x_channels <= 0) return plain;
  return plain + partial_bytes(choose_split(groups, std::min(x_channels, kLinMaxN)), groups);
}

int cg_linear_fwd(const VecPlan &plan, const std::vector<const gelib_part_desc *> &r,
                  const std::vector<const gelib_part_desc *> &x, const std::vector<const gelib_part_desc *> &y,
                  const std::vector<const float2 *> &w, bool accumulate, void *ws, size_t ws_bytes, hipStream_t s,
                  int *used) {
  *used = 0;
  if (plan.diag) return GELIB_HIP_OK;
  std::vector<FastPart> fx, fy, fr;
  std::vector<std::pair<int, int>> lx, ly, lr;
  if (!lists_to_fast(x, plan.E, false, &fx, &lx) || !lists_to_fast(y, plan.E, false, &fy, &ly) ||
      !lists_to_fast(r, plan.E, true, &fr, &lr))
    return GELIB_HIP_OK;
  // every product part l = 0..kLinL, operands up to kLinL, narrow channels
  if ((int)lr.size() != kNL) return GELIB_HIP_OK;
  for (int l = 0; l < kNL; l++)
    if (lr[l].first != l || lr[l].second < 1 || lr[l].second > kLinMaxOut) return GELIB_HIP_OK;
  for (auto &p : lx)
    if (p.first > kLinL || p.second < 1 || p.second > kLinMaxN) return GELIB_HIP_OK;
  for (auto &p : ly)
    if (p.first > kLinL || p.second < 1 || p.second > kLinMaxN) return GELIB_HIP_OK;
  const long long ncells = plan.E[0] * plan.E[1] * plan.E[2];
  const long long nblocks = (ncells + kLinCells - 1) / kLinCells;
  if (nblocks > 0x7fffffffLL) return GELIB_HIP_OK;

  LinArgs a;
  std::memset(&a, 0, sizeof(a));
  for (size_t i = 0; i < fx.size(); i++) a.x[lx[i].first] = fx[i];
  for (size_t i = 0; i < fy.size(); i++) a.y[ly[i].first] = fy[i];
  for (int l = 0; l < kNL; l++) a.out[l] = fr[l];
  long long tau[kNL] = {0, 0, 0, 0, 0};
  for (auto &t : plan.triples) {
    a.offs[t.l1][t.l2][t.l] = t.offs;
    tau[t.l] = std::max(tau[t.l], (long long)t.offs + t.nout);
  }
  // a pair reaches every l of its range (every product part is there): the kernel relies on it
  for (auto &p : lx)
    for (auto &q : ly) {
      int have = 0;
      for (auto &t : plan.triples) have += (t.l1 == p.first && t.l2 == q.first);
      if (have != std::min(p.first + q.first, kLinL) - std::abs(p.first - q.first) + 1) return GELIB_HIP_OK;
    }
  long long x_elems = 0;
  int x_channels = 1;
  for (auto &p : lx) x_elems += (long long)(2 * p.first + 1) * p.second, x_channels = std::max(x_channels, p.second);
  const size_t plain = plain_workspace_bytes(tau, x_elems, nblocks);
  if (!ws || ((uintptr_t)ws & 15) || ws_bytes < plain) return GELIB_HIP_ERR_WORKSPACE;
  LinSplit split = choose_split(nblocks, x_channels);
  if (ws_bytes - plain < partial_bytes(split, nblocks)) split = LinSplit();   // no room for partial sums: one wave per group
  int rc = cg_table_bank(&a.bank);
  if (rc) return rc;
  a.ncells = ncells;
  a.accumulate = accumulate ? 1 : 0;
  char *cursor = (char *)ws;
  for (int l = 0; l < kNL; l++) {
    a.wp[l] = (const float *)cursor;
    const long long n = (tau[l] + kBAhead) * 64;
    pack_linear_kernel<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s>>>((float *)cursor, w[l], tau[l], lr[l].second);
    GELIB_HIP_TRY(hipGetLastError());
    cursor += packed_bytes(tau[l]);
  }
  for (size_t i = 0; i < fx.size(); i++) {
    const int l = lx[i].first, elems = (2 * l + 1) * lx[i].second;
    a.xt[l] = (const float2 *)cursor;
    transpose_cells_kernel<<<dim3((unsigned)nblocks, (unsigned)((elems + 31) / 32)), dim3(256), 0, s>>>((float2 *)cursor, fx[i], elems, ncells);
    GELIB_HIP_TRY(hipGetLastError());
    cursor += (size_t)nblocks * kLinCells * elems * sizeof(float2);
  }
  a.split_a = split.a;
  a.split_l2 = split.l2;
  a.partial = split.shares() > 1 ? (float *)cursor : nullptr;
  if ((rc = launch_cg_linear_pass0(a, nblocks, s))) return rc;
  if ((rc = launch_cg_linear_pass1(a, nblocks, s))) return rc;
  if (a.partial) {
    const long long threads = nblocks * kLinRows * kLinCells * 16;
    sum_shares_kernel<<<dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s>>>(a, split.shares(), nblocks);
    GELIB_HIP_TRY(hipGetLastError());
  }
  *used = 1;
  return GELIB_HIP_OK;
}

}  // namespace gelib_hip
