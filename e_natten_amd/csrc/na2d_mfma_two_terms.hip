// The kernels of na2d_mfma_bias.hip without a table: P and dS in two 16-bit terms, 1 / Z, values that are
// not finite stay in their windows.  For head dims between 32 and 64 with kernel_size 11 and 13, which the build
// in na2d_mfma_narrow.hip does not take (use_two_terms in enatten_capi.hip).  With a table of zeros instead the table is
// filled per tile and read per logit: forward and backward, us, B2 N8 128x128 d48 k13 414 -> 357, B1 N16 162x174
// k11 836 -> 614, float16 B3 N5 61x83 k13 190 -> 164.
#include "na2d_common.h"

namespace enatten {
namespace {
constexpr bool kNarrow = true;
constexpr bool kSub = false;
constexpr bool kBias = true;
constexpr bool kTable = false;
}
}  // namespace enatten

#include "na2d_mfma_kernels.h"

namespace enatten {

int launch_fwd_two_terms(const FwdArgs &a, int dtype, hipStream_t st) { return fwd_dispatch(a, dtype, st); }
int launch_bwd_two_terms(const BwdArgs &a, int dtype, hipStream_t st) { return bwd_dispatch(a, dtype, 0, st); }

}  // namespace enatten
