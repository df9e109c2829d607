// One instantiation of the unrolled forward kernel: CGproduct, 2 channels of the first operand per thread, channel counts
// that 2 does not divide, product l up to 8.
#include "cg_unrolled_fwd_impl.h"

namespace gelib_hip {

int launch_unrolled_fwd_cg2_l8_ragged(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s) {
  return launch_fwd_variant<8, false, 2, kLT, true>(a, nblocks, lds_bytes, s);
}

}  // namespace gelib_hip
