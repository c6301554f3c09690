// The kernels of na2d_mfma_kernels.h with a relative position bias, any head dim that is a
// multiple of 8 up to 128 (channels a tensor does not have as in na2d_mfma_narrow.hip), square
// centred windows.
//
// B8 N4 56x56 d32 k7 bf16, views of a projection: 68 + 103 + 171 us of general kernels and 61 us for
// the bias gradient before, 16 + 30 + 25 + 5 us here, under the profiler.  What the bias costs is LDS work:
// a table read per logit, 28 plane writes and 48 reads per lane and tile for the gradient; the second
// terms of P and dS double the second products.
#include "na2d_common.h"

namespace enatten {
namespace {
constexpr bool kNarrow = true;
constexpr bool kSub = false;
constexpr bool kBias = true;
constexpr bool kTable = true;
}
}  // namespace enatten

#include "na2d_mfma_kernels.h"

namespace enatten {

int launch_fwd_mfma_bias(const FwdArgs &a, int dtype, hipStream_t st) { return fwd_dispatch(a, dtype, st); }
int launch_bwd_mfma_bias(const BwdArgs &a, int dtype, hipStream_t st, bool rpb_typed) {
    return bwd_dispatch(a, dtype, rpb_typed ? kRpbTyped : 0, st);
}

}  // namespace enatten
