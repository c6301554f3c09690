// The kernels of na2d_mfma_kernels.h on the sub-grids of a dilated call, any head dim that is a
// multiple of 8 up to 128 (channels a tensor does not have as in na2d_mfma_narrow.hip).
//
// Sub-grids are small (14x14 pixels for a 56x56 image at dilation 4: four tiles), so one launch
// per sub-grid left most CUs without a tile, and dilation^2 launches of each kernel and as many
// calls through Python bounded the call.  One launch for all of one size: B8 N4 56x56 d32 k7
// dilation 4, views of a projection, forward and backward 1060 -> 70 us (16 launches each of 5 +
// 14 us of kernels and 1100 us of host time before; three kernels of 14 + 25 + 31 us).  Sub-grids
// that fit one workgroup's LDS go to na2d_mfma_small.hip, and those that fill the chip on their own to
// the kernels for undilated images (`alone` in enatten_capi.hip).
#include "na2d_common.h"

namespace enatten {
namespace {
constexpr bool kNarrow = true;
constexpr bool kSub = true;
constexpr bool kBias = false;
constexpr bool kTable = false;
}
}  // namespace enatten

#include "na2d_mfma_kernels.h"

namespace enatten {

static bool sub_ok(const View &v, int dil) {
    return layout_ok(v) && v.sh * dil < (1 << 22) && v.sw * dil < (1 << 22);  // 24-bit multiplies
}
bool sub_layout_ok(const FwdArgsSub &a) {
    return sub_ok(a.q, a.dil) && sub_ok(a.k, a.dil) && sub_ok(a.v, a.dil) && sub_ok(a.o, a.dil);
}
bool sub_layout_ok(const BwdArgsSub &a) {
    auto al = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    return sub_ok(a.q, a.dil) && sub_ok(a.k, a.dil) && sub_ok(a.v, a.dil) && sub_ok(a.o, a.dil) &&
           sub_ok(a.d_o, a.dil) && al(a.dq) && al(a.dk) && al(a.dv) &&
           a.gsb % 8 == 0 && a.gsn % 8 == 0 && a.gsh % 8 == 0 && a.gsw % 8 == 0 &&  // 16-byte stores
           a.s.H < 32768 && a.s.W < 32768;  // (the dK/dV pass keeps window starts in 16 bits)
}

int launch_fwd_mfma_sub(const FwdArgsSub &a, int dtype, hipStream_t st) {
    if (small_fwd_supported(a)) return launch_fwd_small(a, dtype, st);
    return fwd_dispatch(a, dtype, st);
}
int launch_bwd_mfma_sub(const BwdArgsSub &a, int dtype, hipStream_t st) {
    if (small_bwd_supported(a)) return launch_bwd_small(a, dtype, st);
    return bwd_dispatch(a, dtype, 0, st);
}

}  // namespace enatten
