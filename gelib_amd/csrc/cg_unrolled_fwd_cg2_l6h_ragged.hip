// One instantiation of the unrolled forward kernel: the part of a CGproduct of operands up to l = 6 that lies
// above l = 6 (l = 7..12), 2 channels of the first operand per thread, the last one left out where the count is odd.
#include "cg_unrolled_fwd_impl.h"

namespace gelib_hip {

int launch_unrolled_fwd_cg2_l6h_ragged(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s) {
  return launch_fwd_variant<12, false, 2, 6, true, 7>(a, nblocks, lds_bytes, s);
}

}  // namespace gelib_hip
