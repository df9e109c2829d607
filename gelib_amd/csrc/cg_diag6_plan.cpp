// Host side of the lane-per-channel Diag kernels: which products they take, the coefficient table with its fixed
// layout, the per-type offset table (both cached on the device), and the argument block.
#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "cg_diag6.h"

namespace gelib_hip {

namespace {

// ---- host side ---------------------------------------------------------------------------------------------------

std::mutex g_mutex;
std::map<int, float *> g_banks;                     // device -> coefficient table
std::map<std::pair<int, std::vector<int>>, int *> g_offs;  // (device, offsets) -> device copy
int g_enable = 1;
int g_l8_enable = 1;    // the kernels for products up to l = 8 of operands up to l = 4: 1 forward, 2 backward too
int g_sets_enable = 1;  // backward: the kernel with the waves' sets of l2 fixed at compile time, where it applies
int g_small_enable = 1;  // operands up to l = 2, and backward up to l = 4: the kernels that give a wave, not a block, a cell and
                         // channel group
int g_hi_enable = 1;    // the kernels for the part l = 7..12 of a product by itself
int g_tight = -1;        // (cell, channel) pairs without gaps between the cells: -1 where enough lanes would idle, 0 never, 1 always
int g_small4_fwd = -1;   // forward, operands up to l = 4: the kernel that gives a wave a cell and channel group (-1 = by the shape)
int g_stream = -1;       // forward: streaming stores (-1 = by the shape, 0 never, 1 always)
int g_once = -1;         // backward: streaming loads of g (-1 = by the shape, 0 never, 1 always)
int g_one_channel = 1;  // CGproduct with a one-channel operand runs here as the Diag product with the channel repeated

int device_bank(const float **out) {
  int dev = 0;
  GELIB_HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_mutex);
  auto it = g_banks.find(dev);
  if (it == g_banks.end()) {
    std::vector<float> h((size_t)kBankFloats + kZeroFloats, 0.f);
    for (int a = 0; a <= kL6; a++)
      for (int b = 0; b <= kL6; b++)
        for (int c = iabs(a - b); c <= a + b; c++) cg_matrix_host(a, b, c, h.data() + table_off(a, b, c));
    float *d = nullptr;
    GELIB_HIP_TRY(hipMalloc((void **)&d, h.size() * sizeof(float)));
    GELIB_HIP_TRY(hipMemcpy(d, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice));
    it = g_banks.emplace(dev, d).first;
  }
  *out = it->second;
  return GELIB_HIP_OK;
}

int device_offs(const std::vector<int> &h, const int **out) {
  int dev = 0;
  GELIB_HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_mutex);
  auto key = std::make_pair(dev, h);
  auto it = g_offs.find(key);
  if (it == g_offs.end()) {
    int *d = nullptr;
    GELIB_HIP_TRY(hipMalloc((void **)&d, h.size() * sizeof(int)));
    GELIB_HIP_TRY(hipMemcpy(d, h.data(), h.size() * sizeof(int), hipMemcpyHostToDevice));
    it = g_offs.emplace(key, d).first;
  }
  *out = it->second;
  return GELIB_HIP_OK;
}

// Fills the argument block; *ok = false when the product is not one this family takes.
int make_args(const VecPlan &plan, const std::vector<const gelib_part_desc *> &r,
              const std::vector<const gelib_part_desc *> &x, const std::vector<const gelib_part_desc *> &y,
              const std::vector<const gelib_part_desc *> *xg, const std::vector<const gelib_part_desc *> *yg,
              bool r_is_dest, Diag6Args *a, int *lcap, bool *ok, int *llo = nullptr) {
  *ok = false;
  if (!g_enable) return GELIB_HIP_OK;
  std::vector<FastPart> fx, fy, fr, fxg, fyg;
  std::vector<std::pair<int, int>> lx, ly, lr;
  if (!lists_to_fast(x, plan.E, false, &fx, &lx) || !lists_to_fast(y, plan.E, false, &fy, &ly) ||
      !lists_to_fast(r, plan.E, r_is_dest, &fr, &lr))
    return GELIB_HIP_OK;
  if (xg && !lists_to_fast(*xg, plan.E, true, &fxg, nullptr)) return GELIB_HIP_OK;
  if (yg && !lists_to_fast(*yg, plan.E, true, &fyg, nullptr)) return GELIB_HIP_OK;
  // A CGproduct in which every part of one operand has ONE channel is the Diag product with that channel repeated:
  // block channel i * 1 + 0 (resp. 0 * n + j) is the wide operand's own channel, and the blocks follow each other n
  // apart either way (core/Gvec.hpp:311-321 against :358-367).  Lanes then all read the one channel, and its gradient
  // is a sum over the lanes of a cell (one block per cell: up to 64 channels).
  bool xbc = false, ybc = false;
  if (!plan.diag) {
    if (!g_one_channel) return GELIB_HIP_OK;
    auto all_one = [](const std::vector<std::pair<int, int>> &v) {
      for (auto &p : v)
        if (p.second != 1) return false;
      return true;
    };
    ybc = all_one(ly);
    xbc = all_one(lx);
    if (xbc && ybc && !xg && !yg) {
      // one channel on both sides, forward: block channel 0 * 1 + 0 -- the Diag product of one channel, a cell per lane
      // (the gradients of such a product stay with the unrolled kernels, which are faster there)
      xbc = ybc = false;
    } else if (xbc == ybc) {
      return GELIB_HIP_OK;   // otherwise exactly one narrow side
    }
  }
  const int n = (xbc ? ly : lx)[0].second;
  if (n < 1 || n > kMaxChannels) return GELIB_HIP_OK;
  if ((xbc && xg && n > 64) || (ybc && yg && n > 64)) return GELIB_HIP_OK;
  for (auto &p : lx)
    if (p.first > kL6 || p.second != (xbc ? 1 : n)) return GELIB_HIP_OK;
  for (auto &p : ly)
    if (p.first > kL6 || p.second != (ybc ? 1 : n)) return GELIB_HIP_OK;
  for (auto &p : lr)
    if (p.first > 2 * kL6) return GELIB_HIP_OK;
  std::memset(a, 0, sizeof(*a));
  for (size_t i = 0; i < fx.size(); i++) a->x[lx[i].first] = fx[i];
  for (size_t i = 0; i < fy.size(); i++) a->y[ly[i].first] = fy[i];
  for (size_t i = 0; i < fr.size(); i++) a->r[lr[i].first] = fr[i];
  for (size_t i = 0; i < fxg.size(); i++) a->xg[lx[i].first] = fxg[i];
  for (size_t i = 0; i < fyg.size(); i++) a->yg[ly[i].first] = fyg[i];
  {
    // Deal the parts of y to the four waves of a backward block, heaviest first, each to the wave with the least work so
    // far, so that the waves finish every l1 at about the same time.  Work of a pair: two multiply-adds per term of each
    // of its triples (the contraction over l) and eight per (m1, m2).
    long long cost[kNP] = {0, 0, 0, 0, 0, 0, 0};
    bool pair_seen[kNP][kNP] = {};
    for (auto &t : plan.triples) {
      long long terms = 0;
      for (int m = -t.l; m <= t.l; m++) terms += std::min(t.l1, m + t.l2) - std::max(-t.l1, m - t.l2) + 1;
      cost[t.l2] += 2 * terms;
      if (!pair_seen[t.l1][t.l2]) {
        pair_seen[t.l1][t.l2] = true;
        cost[t.l2] += 8LL * (2 * t.l1 + 1) * (2 * t.l2 + 1);
      }
    }
    long long load[4] = {0, 0, 0, 0};
    bool dealt[kNP] = {};
    for (int n = 0; n < kNP; n++) {
      int best = -1;
      for (int l2 = 0; l2 < kNP; l2++)
        if (!dealt[l2] && (best < 0 || cost[l2] > cost[best])) best = l2;
      dealt[best] = true;
      int w = 0;
      for (int k = 1; k < 4; k++)
        if (load[k] < load[w]) w = k;
      a->owner[best] = w;
      load[w] += cost[best];
    }
  }
  std::vector<int> offs((size_t)kNP * kNP * kNR, -1);
  *lcap = 0;
  int lowest = 1 << 30;
  for (auto &t : plan.triples) {
    offs[((size_t)t.l1 * kNP + t.l2) * kNR + t.l] = t.offs;
    *lcap = std::max(*lcap, t.l);
    lowest = std::min(lowest, t.l);
  }
  if (llo) *llo = lowest;
  // An operand part that feeds nothing (harmonics above the cap) and gets no gradient is left out: what remains decides which
  // kernel takes the product (300 channels of l = 0 x harmonics up to l = 6, capped at 0, x-gradient: 1071 -> 42 us).
  int top_x = 0, top_y = 0;
  bool feeds_x[kNP] = {}, feeds_y[kNP] = {};
  for (auto &t : plan.triples) {
    feeds_x[t.l1] = feeds_y[t.l2] = true;
    top_x = std::max(top_x, t.l1), top_y = std::max(top_y, t.l2);
  }
  for (int l = 0; l < kNP; l++) {
    if (!xg && !feeds_x[l]) a->x[l].ptr = nullptr;
    if (!yg && !feeds_y[l]) a->y[l].ptr = nullptr;
  }
  int rc = device_offs(offs, &a->offs);
  if (rc) return rc;
  if ((rc = device_bank(&a->bank))) return rc;
  const long long ncells = plan.E[0] * plan.E[1] * plan.E[2];
  a->ncells = ncells;
  a->n = n;
  a->xbc = xbc ? 1 : 0;
  a->ybc = ybc ? 1 : 0;
  int lg = 0;
  while ((1 << lg) < n && lg < 6) lg++;
  a->lg_npad = lg;
  // Sums over the lanes of a cell (the gradient of a one-channel operand) need the cells in aligned groups of lanes.
  // Otherwise the cells follow each other without gaps where enough lanes would idle.  Time without gaps over time in aligned
  // groups, at 100 MB / 300 MB / 1 GB or more of operands and results, memory that other calls have pushed out of the caches:
  // Forward, whole 64-byte pieces: Diag L = 3, 72 channels .79 .70 .63, L = 4 .85 .79 .64, L = 6 .99 .88 .82, 24 channels L = 3 1.01
  // .96 .96, L = 6 1.00 1.00 .91, but L = 4 1.00 1.08 .98.  Rows that are no multiple of 64 bytes lie across more cache lines per store: 17
  // channels 1.19 1.07 1.02, 1.06 1.14 1.29; above 64 channels that pays at L = 3 and 4 (65 channels .93 .83 .79, 98
  // 1.01 .95 .87), not below (L = 1, 98 channels 1.04 1.08 1.08).  Features x harmonics up to l = 1: 24 to 48 channels 1.00 to 1.04.
  // Backward the wave count falls with the gaps, and a launch that does not fill the GPU gains nothing for its unaligned
  // rows: L = 4, 33 channels 1.07 (870 waves) .93 (2670) .79, 44 channels 1.04 1.07 (2000) .92 (10000); L = 6, 36 channels
  // 1.11 (230) 1.05 (700) .90 (3400); L = 3, 48 channels 1.00 1.01 (4200) .92 (21000), 20 channels 1.02 1.07 (5000) .89
  // (25000).  Capped products only up to 32 channels
  // (every l: L = 4, 17 channels 1.04 1.03 1.06); harmonics of l = 0 alone 1.0 to 1.1.
  const double busy = n <= 64 ? (double)n / (1 << lg) : (double)n / (64 * ((n + 63) / 64));
  const bool lane_sums = (xbc && xg) || (ybc && yg);
  const long long waves = lg < 6 ? ncells >> (6 - lg) : ncells * ((n + 63) / 64);   // of aligned groups
  const int lop = std::max(top_x, top_y);
  const int narrow = xbc ? top_x : (ybc ? top_y : kNP);   // largest l of a one-channel operand
  bool gaps;
  if (r_is_dest) gaps = busy < 0.79 && (n > 64 ? n % 8 == 0 || (n < 128 && lop >= 3 && lop <= 4)
                                               : n >= 16 && n % 8 == 0 && lop != 4 && (narrow >= 2 || lop <= 1));
  else gaps = n >= 16 && ((busy <= 0.63 && waves >= (lop == 3 ? 6000 : 2200)) || (busy <= 0.76 && waves >= 8192)) &&
              (n > 32 || *lcap <= lop) && (narrow >= 1 || lop <= 1);
  const bool want_tight = g_tight < 0 ? gaps : g_tight != 0 && busy < 1;
  bool tight = false;
  if (want_tight && !lane_sums) {
    const long long reach = (n + 62) / n;   // cells behind the wave's first that its lanes reach
    auto fits = [&](const std::vector<FastPart> &v) {
      for (auto &p : v)
        if (p.sb < 0 || (reach * p.sb + n) * 8 >= (1LL << 31)) return false;
      return true;
    };
    tight = fits(fx) && fits(fy) && fits(fr) && fits(fxg) && fits(fyg) && ncells < (1LL << 36);
  }
  if (tight) {
    a->lg_npad = kDiagTight;
    a->groups = 1;
    a->nwaves = (ncells * n + 63) / 64;
    a->magic64 = ~0ull / (unsigned long long)n + 1;
    a->magic32 = ~0u / (unsigned)n + 1;
  } else if (lg < 6) {
    // several cells per wave: the lane's offset from the wave's first cell must fit 32 bits in every part
    const long long cpw = 64 >> lg;
    auto fits = [&](const std::vector<FastPart> &v) {
      for (auto &p : v)
        if (p.sb < 0 || ((cpw - 1) * p.sb + n) * 8 >= (1LL << 31)) return false;
      return true;
    };
    if (!fits(fx) || !fits(fy) || !fits(fr) || !fits(fxg) || !fits(fyg)) return GELIB_HIP_OK;
    a->groups = 1;
    a->nwaves = (ncells + cpw - 1) / cpw;
  } else {
    a->groups = (n + 63) / 64;
    a->nwaves = ncells * a->groups;
  }
  if (a->nwaves > 0x7fffffffLL) return GELIB_HIP_OK;
  *ok = true;
  return GELIB_HIP_OK;
}

}  // namespace

int cg_table_bank(const float **out) { return device_bank(out); }

namespace {
// no operand part (and no gradient of one) above l = lmax
bool operands_up_to(const Diag6Args &a, int lmax) {
  for (int l = lmax + 1; l < kNP; l++)
    if (a.x[l].ptr || a.y[l].ptr || a.xg[l].ptr || a.yg[l].ptr) return false;
  return true;
}
}  // namespace

int diag6_vec_fwd(const VecPlan &plan, const std::vector<const gelib_part_desc *> &r,
                  const std::vector<const gelib_part_desc *> &x, const std::vector<const gelib_part_desc *> &y,
                  bool accumulate, hipStream_t s, int *used) {
  *used = 0;
  Diag6Args a;
  int lcap = 0, llo = 0;
  bool ok = false;
  int rc = make_args(plan, r, x, y, nullptr, nullptr, true, &a, &lcap, &ok, &llo);
  if (rc || !ok) return rc;
  // kernels are built for products capped at l = 6, for products up to l = 8 of operands up to l = 4, and for the part
  // l = 7..12 of a product by itself
  const bool hi = llo > kL6 && g_hi_enable;
  const bool l8 = lcap > kL6 && !hi;
  if (l8 && !(lcap <= 8 && operands_up_to(a, 4) && g_l8_enable)) return GELIB_HIP_OK;
  // A one-channel operand up to l = 2 (harmonics) leaves few pairs per part of the other one, and the block form's staging
  // and barrier cost more than its waves' neighbouring stores gain, from 24 channels on.  Wave / block form at 100 MB and 1 GB:
  // harmonics of l = 0, L = 3 .45 to .76 and .38 to .66; up to l = 1, L = 3, 24 channels .87 .80, 64 .86 .81, 72 .67 .54, L = 4 .85
  // .87, .98 .86, .66 .54; up to l = 2, L = 3 .98 .90, .93 .85, .73 .67.  Not for 17 to 23 channels (L = 4, up to l = 2: 1.01
  // 1.25; 22 .97 1.25) and 25 to 31 (28: L = 3 1.01 1.04, L = 4 1.05 1.17), nor for harmonics up to l = 2 at L = 4 (32 channels 1.12
  // .89, 48 1.11 .84, 96 1.08 .76) or above (L = 4, up to l = 3 1.1 to 1.5).
  int narrow_l = kNP, wide_l = 0;
  for (int l = 0; l < kNP; l++) {
    if ((a.xbc && a.x[l].ptr) || (a.ybc && a.y[l].ptr)) narrow_l = l;
    if ((a.xbc && a.y[l].ptr) || (a.ybc && a.x[l].ptr)) wide_l = l;
  }
  const bool few_pairs = narrow_l <= 1 || (narrow_l == 2 && wide_l <= 3);
  const bool small4 = g_small_enable && (g_small4_fwd < 0 ? few_pairs && (a.n > 32 || (a.n >= 24 && a.n % 8 == 0)) : g_small4_fwd != 0);
  // Streaming stores where rows are whole half-lines; other rows' pieces must meet in a cache before they go to memory.  Streaming /
  // ordinary at 40, 250 and 1500 MB of product written again and again | the largest, pushed out of the caches: Diag L=6 64 channels
  // .89 .88 .78 | .96, 24 .90 .82 .74 | .79, 17 .91 1.60 1.71 | 1.71, L=4 48 .92 .95 .75 | .98, 8 .90 .99 .79 | .96, 20 .91 1.40 1.37 |
  // 1.41, L=2 16 .92 .80 .97 | 1.05; features x harmonics up to l = 2, L=3, 24 channels .89 .94 .75 | .90, 16 .96 .80 .63 | 1.02, 20
  // 1.00 1.11 1.02 | .96, L=4 24 .92 .79 .56 | .97.  Not for the wave form from 32 channels on (L=3, up to l = 2, 64 channels .91 1.02
  // .85 | 1.13), nor 8 channels with harmonics up to l = 1 (L=3 .97 .65 1.03 | 1.07).  The rows have to start at half-lines, too: in parts
  // of 4 channels more, 1 more and 16 more from the second on, 1.2 GB: 64 channels L=6 .97 1.10 1.18, 24 1.33 1.50 1.55, L=4 48 1.12 1.27
  // 1.28, 16 1.52 1.91 1.88, 8 1.67 1.97 1.88, L=2 16 1.38 1.67 1.58; of 8 more .83 to 1.03.  Nor products that fit the memory-side cache.
  bool rows = true;
  long long bytes = 0;
  for (auto &t : plan.triples) {
    rows = rows && pieces_aligned(a.r[t.l], t.offs + a.offs_add, 8);
    bytes += 8 * a.ncells * (2 * t.l + 1) * a.n;
  }
  const bool stream = a.n % 8 == 0 && rows && bytes > kMemoryCache && !(small4 && a.n >= 32) && !(a.n == 8 && narrow_l <= 1 && wide_l >= 3);
  a.write = accumulate ? kWriteAdd : ((g_stream < 0 ? stream : g_stream != 0) ? kWriteStream : kWriteOver);
  t_streaming |= a.write == kWriteStream ? 1 : 0;
  if (g_small_enable && lcap <= 4 && operands_up_to(a, 2)) rc = launch_diag6_small_fwd(a, s);
  else if (small4 && lcap <= 6 && operands_up_to(a, 4)) rc = launch_diag6_small4_fwd(a, s);
  else if (hi) rc = a.lg_npad < 6 ? launch_diag6_fwd_hi_packed(a, s) : launch_diag6_fwd_hi(a, s);
  else if (l8) rc = a.lg_npad < 6 ? launch_diag6_fwd_l8_packed(a, s) : launch_diag6_fwd_l8(a, s);
  else rc = a.lg_npad < 6 ? launch_diag6_fwd_l6_packed(a, s) : launch_diag6_fwd_l6(a, s);
  if (rc) return rc;
  *used = 1;
  return GELIB_HIP_OK;
}

int diag6_vec_bwd(const VecPlan &plan, const std::vector<const gelib_part_desc *> &g,
                  const std::vector<const gelib_part_desc *> &x, const std::vector<const gelib_part_desc *> &y,
                  const std::vector<const gelib_part_desc *> &xg, const std::vector<const gelib_part_desc *> &yg,
                  bool accumulate, hipStream_t s, int *used) {
  *used = 0;
  if (xg.empty() && yg.empty()) return GELIB_HIP_OK;
  Diag6Args a;
  int lcap = 0, llo = 0;
  bool ok = false;
  int rc = make_args(plan, g, x, y, xg.empty() ? nullptr : &xg, yg.empty() ? nullptr : &yg, false, &a, &lcap, &ok, &llo);
  if (rc || !ok) return rc;
  // (backward, the one-launch kernel for products up to l = 8 is used on request only, diag6_l8 = 2: the wave that owns
  // y[4] then has the terms of l = 5..8 on top of the largest share, and L=4, 64 channels, 131072 cells takes 16.4 ms
  // against 14.4 ms for the split at l = 6)
  const bool hi = llo > kL6 && g_hi_enable;
  const bool l8 = lcap > kL6 && !hi;
  if (l8 && !(lcap <= 8 && operands_up_to(a, 4) && g_l8_enable >= 2)) return GELIB_HIP_OK;
  a.write = accumulate ? kWriteAdd : kWriteOver;
  // Streaming loads of g (the line is not kept) where a block's rows are whole cache lines, or nearly (operands above l = 4): what
  // an ordinary load leaves in the caches is never read again, and pushes out what is.  Rows that share lines with the next
  // block's must keep them.  Streaming / ordinary, 250 MB and 1.5 GB of g that other calls have pushed out of the caches: Diag L=6
  // 64 channels .77 .87, 24 .80 .88, 17 .82 1.27, L=4 64 .78 .96, 24 .82 1.14, 8 .92 1.28, 3 1.23 1.32, L=2 32 .78 .96, L=1 16 .92
  // .97; features x harmonics up to l = 2, L=4 32 .64 .90, L=3 16 .65 .91, 24 .79 1.14; capped at l = 1 with harmonics above it .89
  // 1.02, and 1.1 to 1.2 where g is still in the caches.  Written just before, 40 to 200 MB .94 to 1.09, 400 MB and more .89 to .99.  Operands
  // up to l = 4 want the rows to start at lines (1.2 GB, half a line and 8 bytes off: L=4 48 channels 1.14 1.14, 16 1.23 1.23, L=2
  // 16 1.32 1.31, x harmonics up to l = 2 L=3 16 1.36 1.36; 300 MB .86 to 1.12), those above do not mind (64 channels .92, 24 .95 1.01).
  int top = 0, narrow = kNP;
  for (int l = 0; l < kNP; l++) {
    if (a.x[l].ptr || a.y[l].ptr) top = l;
    if ((a.xbc && a.x[l].ptr) || (a.ybc && a.y[l].ptr)) narrow = l;
  }
  bool lines = top > 4 ? a.n % 8 == 0 && a.n >= 16 : a.n % 16 == 0;
  if (top <= 4)
    for (auto &t : plan.triples) lines = lines && pieces_aligned(a.r[t.l], t.offs + a.offs_add, 16);
  a.once = g_once < 0 ? lines && !(lcap <= 1 && narrow >= 2 && narrow < kNP) : g_once;
  t_streaming |= a.once ? 2 : 0;
  a.want_x = xg.empty() ? 0 : 1;
  a.want_y = yg.empty() ? 0 : 1;
  bool all_y = true;
  for (int l = 0; l < kNP; l++) all_y = all_y && a.y[l].ptr != nullptr;
  if (g_small_enable && lcap <= 4 && operands_up_to(a, 2)) rc = launch_diag6_small_bwd(a, s);
  else if (g_small_enable && hi && lcap <= 8 && operands_up_to(a, 4)) rc = launch_diag6_small4_hi_bwd(a, s);
  else if (g_small_enable && lcap <= 6 && operands_up_to(a, 4)) rc = launch_diag6_small4_bwd(a, s);
  else if (hi) rc = a.lg_npad < 6 ? launch_diag6_bwd_hi_packed(a, s) : launch_diag6_bwd_hi(a, s);
  else if (l8) rc = a.lg_npad < 6 ? launch_diag6_bwd_l8_packed(a, s) : launch_diag6_bwd_l8(a, s);
  else if (a.lg_npad < 6) rc = launch_diag6_bwd_l6_packed(a, s);
  else if (all_y && g_sets_enable) rc = launch_diag6_bwd_l6_sets(a, s);
  else rc = launch_diag6_bwd_l6(a, s);
  if (rc) return rc;
  *used = 1;
  return GELIB_HIP_OK;
}

// One triple (the part-level entry points).  kind 0: r += x * y; 1: the x-shaped tensor is the gradient wanted, r is the
// incoming gradient and the x operand does not exist; 2: likewise for y.  The missing operand is stood in for by the
// gradient's own descriptor: it only marks the part as present, the kernel never reads an operand whose gradient is
// not wanted.
int diag6_part(int kind, const long long E[3], const gelib_part_desc *r, const gelib_part_desc *x,
               const gelib_part_desc *y, int l1, int l2, int l, int offs, bool accumulate, hipStream_t s, int *used) {
  *used = 0;
  VecPlan plan;
  plan.diag = true;
  for (int k = 0; k < 3; k++) plan.E[k] = E[k];
  VecTriple t;
  t.xi = t.yi = t.ri = 0;
  t.l1 = l1;
  t.l2 = l2;
  t.l = l;
  t.offs = offs;
  t.nout = (int)x->dims[4];
  plan.triples.push_back(t);
  const std::vector<const gelib_part_desc *> R = {r}, X = {x}, Y = {y}, none;
  if (kind == 0) return diag6_vec_fwd(plan, R, X, Y, accumulate, s, used);
  return diag6_vec_bwd(plan, R, X, Y, kind == 1 ? X : none, kind == 2 ? Y : none, accumulate, s, used);
}

int diag6_set_option(const char *name, int value) {
  if (!std::strcmp(name, "diag6")) {
    g_enable = value;
    return GELIB_HIP_OK;
  }
  if (!std::strcmp(name, "diag6_tight")) {
    if (value < -1 || value > 1) return GELIB_HIP_ERR_ARG;
    g_tight = value;
    return GELIB_HIP_OK;
  }
  if (!std::strcmp(name, "diag6_stream")) {
    if (value < -1 || value > 1) return GELIB_HIP_ERR_ARG;
    g_stream = value;
    return GELIB_HIP_OK;
  }
  if (!std::strcmp(name, "diag6_once")) {
    if (value < -1 || value > 1) return GELIB_HIP_ERR_ARG;
    g_once = value;
    return GELIB_HIP_OK;
  }
  if (!std::strcmp(name, "diag6_small4_fwd")) {
    if (value < -1 || value > 1) return GELIB_HIP_ERR_ARG;
    g_small4_fwd = value;
    return GELIB_HIP_OK;
  }
  if (!std::strcmp(name, "diag6_small")) {
    g_small_enable = value;
    return GELIB_HIP_OK;
  }
  if (!std::strcmp(name, "diag6_hi")) {
    g_hi_enable = value;
    return GELIB_HIP_OK;
  }
  if (!std::strcmp(name, "diag6_l8")) {
    g_l8_enable = value;
    return GELIB_HIP_OK;
  }
  if (!std::strcmp(name, "diag6_one_channel")) {
    g_one_channel = value;
    return GELIB_HIP_OK;
  }
  if (!std::strcmp(name, "diag6_sets")) {
    g_sets_enable = value;
    return GELIB_HIP_OK;
  }
  return GELIB_HIP_ERR_ARG;
}

}  // namespace gelib_hip
