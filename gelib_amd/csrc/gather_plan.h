// Which parts the vector form of the gather takes and how its threads cover them: plain arithmetic, no device code.
#pragma once

namespace gelib_hip {

// A launch holds fewer than 2^32 threads in all (gridDim.x * blockDim.x), so this many blocks of 256.
constexpr long long kGatherMaxBlocks = (1LL << 24) - 1;
constexpr int kGatherParts = 8;   // parts of one launch; more parts take more launches

constexpr long long gather_blocks(long long threads) { return (threads + 255) / 256; }
// Does a part of `more` blocks go into a launch that holds `parts` parts of `blocks` blocks in all?
constexpr bool gather_shares_launch(int parts, long long blocks, long long more) {
  return parts < kGatherParts && blocks + more <= kGatherMaxBlocks;
}

struct GatherSlices {
  long long ro, xo;          // strides of the outer index (complex elements)
  long long rt, xt;          // strides of a target slice / a source slice
  unsigned per_target;       // threads per (outer, target): slice elements / vec
  unsigned long long magic;  // ceil(2^64 / per_target), 0 for per_target == 1
  int vec;                   // complex elements per thread: 2 (16 bytes) or 1
  long long total;           // threads
};

// First element of a slice's thread q.  64 bits: there are fewer than 2^32 threads, but a slice of 2^32 or more complex
// numbers has twice as many elements as threads.
constexpr long long gather_element(unsigned q, int vec) { return (long long)q * vec; }

// The part (strides in complex elements and extents of the result over (batch, grid0, grid1, m, channel), none 0) as the
// vector kernel sees it: what follows the gathered dimension is one contiguous slice in both tensors, what precedes it one
// index with one stride.  False: the kernel for any strides takes the part.
inline bool gather_slices(const long long rs[5], const long long xs[5], const long long D[5], int dim, bool aligned16,
                          GatherSlices *p) {
  long long slice = 1;
  for (int k = 4; k > dim; k--) {
    if (D[k] > 1 && (rs[k] != slice || xs[k] != slice)) return false;
    slice *= D[k];
  }
  long long outer = 1;
  p->ro = p->xo = 0;
  for (int k = dim - 1; k >= 0; k--) {   // the innermost of the outer dimensions first
    if (D[k] == 1) continue;
    if (outer > 1 && (rs[k] != p->ro * outer || xs[k] != p->xo * outer)) return false;
    if (outer == 1) p->ro = rs[k], p->xo = xs[k];
    outer *= D[k];
  }
  p->rt = rs[dim];
  p->xt = xs[dim];
  const bool wide = slice % 2 == 0 && aligned16 && p->rt % 2 == 0 && p->xt % 2 == 0 && p->ro % 2 == 0 && p->xo % 2 == 0;
  p->vec = wide ? 2 : 1;
  const long long per = slice / p->vec;
  p->total = outer * D[dim] * per;
  if (gather_blocks(p->total) > kGatherMaxBlocks) return false;   // (which also keeps the kernel's thread index below 2^32)
  p->per_target = (unsigned)per;
  // floor(w / per) = high half of w * ceil(2^64 / per): exact for every 32-bit w
  p->magic = per > 1 ? ~0ull / (unsigned long long)per + 1 : 0;
  return true;
}

}  // namespace gelib_hip
