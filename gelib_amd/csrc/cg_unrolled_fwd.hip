// Dispatch of the unrolled forward kernels; the instantiations live in cg_unrolled_fwd_*.hip so that they
// compile in parallel.
#include "cg_unrolled_dev.h"

namespace gelib_hip {

int launch_unrolled_fwd_cg1_l4(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg1_l8(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg2_l4(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg2_l8(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg4_l4(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg4_l8(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_diag_l4(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_diag_l8(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg4_l4_ragged(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg4_l8_ragged(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg2_l6l(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg2_l6h(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg2_l6l_stream(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg2_l6h_stream(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg2_l6l_ragged(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);
int launch_unrolled_fwd_cg2_l6h_ragged(const FwdArgs &a, int nblocks, size_t lds_bytes, hipStream_t s);

// Operands up to l = 4: every product, Diag or not.  Operands up to l = 6: CGproduct capped at l = 6, and what lies above
// l = 6 of one by itself (llo = the smallest l present), with two channels of the first operand per thread.  Both are bound by their
// stores: L=6, 8 channels, 4099 cells, every l (4.5 GB): up to l = 6 740 us with ordinary stores, 625 streaming; above 590 in the any-l
// kernel, 530 here.  Odd counts went to the any-l kernel as a whole: L=6, 5 channels, 60 MB 245 us, 105 here in two launches.
bool unrolled_fwd_takes(bool diag, int ti, int lcap, int lop, int llo) {
  if (lop <= kLT) return lcap <= 2 * kLT;
  return lop <= kLTMax && !diag && ti == 2 && (lcap <= kLTMax || (llo > kLTMax && lcap <= 2 * kLTMax));
}

// lcap: largest l present in the product; code for l above 4 is left out when the product is capped there
int launch_unrolled_fwd(const FwdArgs &a, bool diag, int ti, bool ragged, int lcap, int lop, int nblocks, size_t lds_bytes,
                        hipStream_t s) {
  if (nblocks <= 0) return GELIB_HIP_OK;
  if (lop > kLT) {
    const bool high = lcap > kLTMax;
    if (ragged) return high ? launch_unrolled_fwd_cg2_l6h_ragged(a, nblocks, lds_bytes, s) : launch_unrolled_fwd_cg2_l6l_ragged(a, nblocks, lds_bytes, s);
    if (a.write == kWriteStream) return high ? launch_unrolled_fwd_cg2_l6h_stream(a, nblocks, lds_bytes, s) : launch_unrolled_fwd_cg2_l6l_stream(a, nblocks, lds_bytes, s);
    return high ? launch_unrolled_fwd_cg2_l6h(a, nblocks, lds_bytes, s) : launch_unrolled_fwd_cg2_l6l(a, nblocks, lds_bytes, s);
  }
  if (ragged) {   // four channels per thread, operands up to l = 4
    return lcap <= kLT ? launch_unrolled_fwd_cg4_l4_ragged(a, nblocks, lds_bytes, s) : launch_unrolled_fwd_cg4_l8_ragged(a, nblocks, lds_bytes, s);
  }
  const bool small = lcap <= kLT;
  if (diag) return small ? launch_unrolled_fwd_diag_l4(a, nblocks, lds_bytes, s) : launch_unrolled_fwd_diag_l8(a, nblocks, lds_bytes, s);
  if (ti == 4) return small ? launch_unrolled_fwd_cg4_l4(a, nblocks, lds_bytes, s) : launch_unrolled_fwd_cg4_l8(a, nblocks, lds_bytes, s);
  if (ti == 2) return small ? launch_unrolled_fwd_cg2_l4(a, nblocks, lds_bytes, s) : launch_unrolled_fwd_cg2_l8(a, nblocks, lds_bytes, s);
  return small ? launch_unrolled_fwd_cg1_l4(a, nblocks, lds_bytes, s) : launch_unrolled_fwd_cg1_l8(a, nblocks, lds_bytes, s);
}

}  // namespace gelib_hip
