// Channel mixing of all parts of a vector, any channel counts (internal interface; kernels in mix_vec.hip).
#pragma once

#include <vector>

#include "cg_common.h"

namespace gelib_hip {

// C (m, n) = A (m, k) B (k, n), all packed:
//   kVMForward  A = x (rows, channels),           B = w (channels, outputs)
//   kVMAdjoint  A = g (rows, outputs),            B = w^H, w (channels, outputs) in memory: n = channels, k = outputs
//   kVMGrad     A = x^H, x (rows, channels) in memory: m = channels, k = rows;  B = g (rows, outputs)
enum { kVMForward = 0, kVMAdjoint = 1, kVMGrad = 2 };
struct VecMixPart {
  const float2 *a, *b;
  float2 *c;
  long long m, n, k;
};

// Bytes for the partial results of parts with few tiles (pointers are not looked at).  Fewer rows can need more: fewer tiles are cut
// into more pieces.
size_t vec_mix_workspace_bytes(const std::vector<VecMixPart> &parts);
// 0, 10, 11 (more tiles than a launch holds) or 13 (workspace).  Parts with k = 0 are left to the caller.  fit: no more pieces than
// ws_bytes has room for, so that any size will do.
int launch_vec_mix(const std::vector<VecMixPart> &parts, int mode, void *ws, size_t ws_bytes, bool fit, hipStream_t s);

}  // namespace gelib_hip
