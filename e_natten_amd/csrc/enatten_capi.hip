// C ABI of libenatten.so: argument validation and dispatch.  See enatten.h.

#include <stdarg.h>
#include <stdio.h>

#include <atomic>
#include <type_traits>

#include "na2d_common.h"

namespace enatten {

static thread_local char g_err[512] = "";
static std::atomic<int> g_path{0};

void set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

namespace {

int elem_size(int dtype) {
    switch (dtype) {
        case ENATTEN_F64: return 8;
        case ENATTEN_F32: return 4;
        case ENATTEN_BF16:
        case ENATTEN_F16: return 2;
    }
    return 0;
}

int check_shape(const char *fn, int B, int N, int H, int W, int D, int ks, int dtype) {
    if (elem_size(dtype) == 0) {
        set_error("%s: unknown dtype code %d (expected ENATTEN_F32/BF16/F16/F64)", fn, dtype);
        return ENATTEN_EINVAL;
    }
    if (B < 1 || N < 1 || H < 1 || W < 1 || D < 1) {
        set_error("%s: every dimension must be >= 1, got B=%d heads=%d H=%d W=%d D=%d", fn, B, N,
                  H, W, D);
        return ENATTEN_EINVAL;
    }
    if (ks < 1 || ks % 2 == 0) {
        set_error("%s: kernel_size must be odd and >= 1, got %d", fn, ks);
        return ENATTEN_EINVAL;
    }
    if (H < ks || W < ks) {
        set_error("%s: image %dx%d is smaller than kernel_size %d", fn, H, W, ks);
        return ENATTEN_EINVAL;
    }
    // elements of one tensor, checked factor by factor so that nothing overflows
    const int64_t limit = (int64_t)1 << 40;
    int64_t count = 1;
    for (const int f : {B, N, H, W, D}) {
        if (count > limit / f) {
            set_error("%s: tensor too large (more than 2^40 elements)", fn);
            return ENATTEN_EUNSUPPORTED;
        }
        count *= f;
    }
    return ENATTEN_OK;
}

int make_view(const char *fn, const char *name, const void *p, const int64_t *st, int N, int H,
              int W, int D, View *out) {
    if (!p) {
        set_error("%s: %s is NULL", fn, name);
        return ENATTEN_EINVAL;
    }
    out->ptr = p;
    if (st) {
        out->sb = st[0]; out->sn = st[1]; out->sh = st[2]; out->sw = st[3];
        if (out->sb < 0 || out->sn < 0 || out->sh < 0 || out->sw < 0) {
            set_error("%s: negative stride for %s", fn, name);
            return ENATTEN_EINVAL;
        }
    } else {
        out->sw = D;
        out->sh = (int64_t)W * D;
        out->sn = (int64_t)H * W * D;
        out->sb = (int64_t)N * H * W * D;
    }
    return ENATTEN_OK;
}

bool use_mfma(int D, int ks, int dtype) {
    return g_path.load() != ENATTEN_PATH_SIMT && mfma_supported(D, ks, dtype);
}
// Head dims between 32 and 64 with kernel_size 11 and 13: the kernels for a relative position bias, and
// without one their build without a table (two terms for P and dS, 1 / Z, values that are not finite stay in
// their windows).  bf16, forward and backward, us, general -> these: B1 N16 162x174 d48 k11 4050 -> 614, with a
// bias 5800 -> 768; B2 N8 128x128 d48 k13 3090 -> 357, with a bias 4570 -> 495.
bool use_two_terms(int D, int ks, int dtype) {
    return g_path.load() != ENATTEN_PATH_SIMT && (dtype == ENATTEN_BF16 || dtype == ENATTEN_F16) && D > 32 && D < 64 &&
           D % 8 == 0 && (ks == 11 || ks == 13);
}
bool use_mfma_f32(int D, int ks, int dtype) {
    return g_path.load() != ENATTEN_PATH_SIMT && mfma_f32_supported(D, ks, dtype);
}
// 1D windows of any length (H = 1): causal ones, and centred ones beyond what mfma1d_supported
// takes
template <typename ARGS>
bool use_band(const ARGS &a, int dtype) {
    return g_path.load() != ENATTEN_PATH_SIMT && band_supported(a, dtype);
}
// float32 per query of backward workspace: two for the general and the 16-bit kernels
// (delta and 1/Z), 2 * ks * ks for the float32 matrix-core kernels (P and dS), four for
// float64 tensors (two doubles: the log-sum-exp in double and delta)
size_t ws_floats_per_query(int D, int ks, int dtype) {
    if (dtype == ENATTEN_F64) return 4;
    return mfma_f32_supported(D, ks, dtype) ? mfma_f32_workspace_floats(ks) : 2;
}
// Layout of dq, dk, dv: contiguous [B, heads, H, W, D], or the caller's element strides on
// (batch, head, row, column) with unit stride on the channels.  Call after a->s is set.
int set_grad_layout(const char *fn, BwdArgs *a, const int64_t *st) {
    const Shape &s = a->s;
    if (st) {
        a->gsb = st[0]; a->gsn = st[1]; a->gsh = st[2]; a->gsw = st[3];
        if (a->gsb < 0 || a->gsn < 0 || a->gsh < 0 || a->gsw < s.D) {
            set_error("%s: gradient strides must be non-negative, and at least D between pixels", fn);
            return ENATTEN_EINVAL;
        }
    } else {
        a->gsw = s.D;
        a->gsh = (int64_t)s.W * s.D;
        a->gsn = (int64_t)s.H * s.W * s.D;
        a->gsb = (int64_t)s.N * s.H * s.W * s.D;
    }
    return ENATTEN_OK;
}
// float64 tensors: one kernel family (na2d_f64.hip), whatever the path setting
int bwd_f64(const char *fn, const BwdArgs &a, size_t ws_floats, hipStream_t st) {
    if (ws_floats < (size_t)4 * a.s.B * a.s.N * a.s.H * a.s.W) {
        set_error("%s: float64 tensors need 16 bytes of workspace per query", fn);
        return ENATTEN_EUNSUPPORTED;
    }
    return launch_bwd_f64(a, st);
}

// an undilated call as a dilated one with a single sub-grid
template <typename SUB, typename ARGS>
SUB whole(const ARGS &a) {
    SUB w;
    static_cast<ARGS &>(w) = a;
    w.sub_r = w.sub_c = w.dil = 1;
    return w;
}
// a square, centred, undilated window: the kernel family that serves the call
int run_fwd(const FwdArgs &a, int dtype, hipStream_t st) {
    const int D = a.s.D, ks = a.s.kh;
    if (dtype == ENATTEN_F64) return launch_fwd_f64(a, st);
    if (use_mfma(D, ks, dtype)) {
        const FwdArgsSub w = whole<FwdArgsSub>(a);
        if (g_path.load() == 0 && small_fwd_supported(w) && sub_layout_ok(w)) return launch_fwd_small(w, dtype, st);
        return launch_fwd_mfma(a, dtype, st);
    }
    if (use_mfma_f32(D, ks, dtype)) return launch_fwd_mfma_f32(a, st);
    if (use_two_terms(D, ks, dtype)) return launch_fwd_two_terms(a, dtype, st);
    return launch_fwd_simt(a, dtype, st);
}
int run_bwd(const char *fn, const BwdArgs &a, int dtype, size_t ws_floats, hipStream_t st) {
    const int D = a.s.D, ks = a.s.kh;
    if (dtype == ENATTEN_F64) return bwd_f64(fn, a, ws_floats, st);
    if (use_mfma(D, ks, dtype)) {
        const int path = g_path.load();
        const BwdArgsSub w = whole<BwdArgsSub>(a);
        if (path == 0 && small_bwd_supported(w) && sub_layout_ok(w)) return launch_bwd_small(w, dtype, st);
        return launch_bwd_mfma(a, dtype, path, st);
    }
    // the float32 matrix-core backward where the workspace at hand holds its P and dS (it
    // writes contiguous gradients only)
    if (use_mfma_f32(D, ks, dtype) && a.grads_contiguous() &&
        ws_floats >= (size_t)a.s.B * a.s.N * a.s.H * a.s.W * mfma_f32_workspace_floats(ks))
        return launch_bwd_mfma_f32(a, st);
    if (use_two_terms(D, ks, dtype)) return launch_bwd_two_terms(a, dtype, st);
    return launch_bwd_simt(a, dtype, st);
}

// The sub-grids of a dilated call (pixels of one residue class modulo the dilation on each
// axis) are images of at most two sizes per axis: H = dil * h + r gives r classes of h + 1 rows
// and dil - r of h.  One axis of one such group: the classes from `first` on, `count` of them,
// `extent` positions each.
struct SubAxis {
    int first, count, extent;
};
int split_axis(int L, int dil, SubAxis (&out)[2]) {
    const int r = L % dil, h = L / dil;
    int n = 0;
    if (r) out[n++] = SubAxis{0, r, h + 1};
    out[n++] = SubAxis{r, dil - r, h};
    return n;
}
// the same tensor from the group's first pixel on
View group_view(const View &v, int es, const SubAxis &r, const SubAxis &c) {
    View o = v;
    o.ptr = static_cast<const char *>(v.ptr) + (r.first * v.sh + c.first * v.sw) * es;
    return o;
}
// sub-grid (i, j) of a group as an image of its own
View one_sub(const View &v, int es, int dil, int i, int j) {
    View o = v;
    o.ptr = static_cast<const char *>(v.ptr) + (i * v.sh + j * v.sw) * es;
    o.sh = v.sh * dil; o.sw = v.sw * dil;
    return o;
}
// Sub-grids that fill the chip on their own run one after the other on the kernels for undilated
// images: these are built for head dims of exactly 32, 64 and 128 and have the fused backward, which
// the build for all sub-grids at once has not.  `tiles`: 8x8 tiles of one sub-grid over batch and heads.
// bf16, views of a projection, us, one after the other / all at once.
// Backward: d128 from 1024 tiles on (B4 N4 128x128 dilation 2 k3 158 / 188, k5 173 / 220, k9 394 / 414; k13
// already at 512, 224 / 363), d64 and d32 from 2048 (B8 N8 128x128 dilation 2 d64 k5 353 / 486, d32 k7 308 / 384; at
// 1024 d32 k7 119 / 99); at 512 and 1024 tiles where the tensors no longer fit the caches (B8 N8 128x128 dilation
// 4 d32 k7 374 / 419, d64 k9 1061 / 1116, B8 N4 d128 k5 470 / 560); head dims between the built ones from 4096
// (B4 N8 256x256 d48 k7 1149 / 1231, at 2048 294 / 254).
// Forward, which has one kernel either way: d32 and d64 at 4096 tiles k9 112 / 135 and 181 / 211, at 1024 k7 39 / 33;
// small windows only at dilation 2 (d64 k3 56 / 67; dilation 3, 4096 tiles, d32 k3 216 / 202: pixels far apart
// share lines with other sub-grids); d128 k13 at 1024 tiles 101 / 113, k3 at 1936 267 / 291, k7 at 4096 328 / 301.
bool exact_dim(int D) { return D == 32 || D == 64 || D == 128; }
template <typename ARGS>
bool alone(const ARGS &a) {
    const Shape &s = a.s;
    const int64_t subs = (int64_t)a.sub_r * a.sub_c;
    const int64_t tiles = (int64_t)s.B * s.N * ((s.H + 7) / 8) * ((s.W + 7) / 8);
    if constexpr (std::is_same_v<ARGS, FwdArgsSub>) {
        if (!exact_dim(s.D) || small_fwd_supported(a)) return false;
        if (subs == 1) return true;
        if (s.D == 128) return s.kh >= 11 ? tiles >= 1024 : s.kh <= 5 && tiles >= 1536;
        return tiles >= 2048 && (s.kh >= 7 || a.dil == 2);
    } else {
        if (small_bwd_supported(a)) return false;
        if (!exact_dim(s.D)) return tiles >= 4096;
        return subs == 1 || tiles >= (s.D == 128 ? (s.kh >= 11 ? 512 : 1024) : 2048) ||
               (tiles >= 512 && tiles * subs >= 8192);
    }
}
void *offset(void *p, int64_t elements, int es) { return static_cast<char *>(p) + elements * es; }

int check_dilation(const char *fn, int H, int W, int ks, int dil) {
    if (dil < 1) {
        set_error("%s: dilation must be >= 1, got %d", fn, dil);
        return ENATTEN_EINVAL;
    }
    if (H / dil < ks || W / dil < ks) {
        set_error("%s: image %dx%d is smaller than kernel_size * dilation = %lld", fn, H, W,
                  (long long)ks * dil);
        return ENATTEN_EINVAL;
    }
    return ENATTEN_OK;
}

}  // namespace
}  // namespace enatten

using namespace enatten;

extern "C" {
#pragma GCC visibility push(default)

int enatten_abi_version(void) { return ENATTEN_ABI_VERSION; }

const char *enatten_last_error(void) { return g_err; }

int enatten2d_kernel_path(int D, int kernel_size, int dtype) {
    if (elem_size(dtype) == 0 || D < 1 || D > 1024 || kernel_size < 1 || kernel_size % 2 == 0)
        return ENATTEN_PATH_NONE;
    return use_mfma(D, kernel_size, dtype) || use_mfma_f32(D, kernel_size, dtype) ? ENATTEN_PATH_MFMA
                                                                                  : ENATTEN_PATH_SIMT;
}

int enatten_set_path(int path) {
    if (path != 0 && path != ENATTEN_PATH_SIMT && path != ENATTEN_PATH_MFMA_FUSED &&
        path != ENATTEN_PATH_MFMA_SPLIT && path != ENATTEN_PATH_MFMA_SPLIT_QUEUE)
        return g_path.load();
    return g_path.exchange(path);
}

int enatten2d_fwd(const void *q, const void *k, const void *v, void *o, float *lse, int B,
                  int heads, int H, int W, int D, int kernel_size, int dtype,
                  const int64_t *q_strides, const int64_t *k_strides, const int64_t *v_strides,
                  const int64_t *o_strides, float scale, void *stream) {
    const char *fn = "enatten2d_fwd";
    int rc = check_shape(fn, B, heads, H, W, D, kernel_size, dtype);
    if (rc) return rc;
    FwdArgs a;
    if ((rc = make_view(fn, "q", q, q_strides, heads, H, W, D, &a.q))) return rc;
    if ((rc = make_view(fn, "k", k, k_strides, heads, H, W, D, &a.k))) return rc;
    if ((rc = make_view(fn, "v", v, v_strides, heads, H, W, D, &a.v))) return rc;
    if ((rc = make_view(fn, "o", o, o_strides, heads, H, W, D, &a.o))) return rc;
    a.lse = lse;
    a.s = Shape{B, heads, H, W, D, kernel_size, kernel_size, scale};
    return run_fwd(a, dtype, static_cast<hipStream_t>(stream));
}

size_t enatten2d_bwd_workspace_bytes(int B, int heads, int H, int W, int D, int kernel_size,
                                     int dtype) {
    if (B < 1 || heads < 1 || H < 1 || W < 1 || D < 1 || kernel_size < 1) return 0;
    return (size_t)B * heads * H * W * ws_floats_per_query(D, kernel_size, dtype) * sizeof(float);
}

// Shared body of the two backward entry points: `workspace` holds two float32 per query.
static int bwd2d(const char *fn, const void *q, const void *k, const void *v, const void *o,
                 const void *d_o, const float *lse, void *dq, void *dk, void *dv,
                 float *workspace, size_t ws_floats, int B, int heads, int H, int W, int D, int kernel_size,
                 int dtype, const int64_t *q_strides, const int64_t *k_strides,
                 const int64_t *v_strides, const int64_t *o_strides, const int64_t *do_strides,
                 float scale, void *stream, const int64_t *grad_strides = nullptr) {
    BwdArgs a;
    int rc;
    if ((rc = make_view(fn, "q", q, q_strides, heads, H, W, D, &a.q))) return rc;
    if ((rc = make_view(fn, "k", k, k_strides, heads, H, W, D, &a.k))) return rc;
    if ((rc = make_view(fn, "v", v, v_strides, heads, H, W, D, &a.v))) return rc;
    if ((rc = make_view(fn, "o", o, o_strides, heads, H, W, D, &a.o))) return rc;
    if ((rc = make_view(fn, "d_o", d_o, do_strides, heads, H, W, D, &a.d_o))) return rc;
    if (!lse || !dq || !dk || !dv) {
        set_error("%s: lse, dq, dk and dv must all be non-NULL", fn);
        return ENATTEN_EINVAL;
    }
    a.lse = lse;
    a.dq = dq; a.dk = dk; a.dv = dv;
    a.delta = workspace;
    a.zinv = a.delta + (size_t)B * heads * H * W;
    a.s = Shape{B, heads, H, W, D, kernel_size, kernel_size, scale};
    if ((rc = set_grad_layout(fn, &a, grad_strides))) return rc;
    return run_bwd(fn, a, dtype, ws_floats, static_cast<hipStream_t>(stream));
}

int enatten2d_bwd(const void *q, const void *k, const void *v, const void *o, const void *d_o,
                  const float *lse, void *dq, void *dk, void *dv, void *workspace, int B,
                  int heads, int H, int W, int D, int kernel_size, int dtype,
                  const int64_t *q_strides, const int64_t *k_strides, const int64_t *v_strides,
                  const int64_t *o_strides, const int64_t *do_strides, float scale,
                  void *stream) {
    const char *fn = "enatten2d_bwd";
    const int rc = check_shape(fn, B, heads, H, W, D, kernel_size, dtype);
    if (rc) return rc;
    if (!workspace) {
        set_error("%s: workspace is NULL", fn);
        return ENATTEN_EINVAL;
    }
    // the caller provides enatten2d_bwd_workspace_bytes() for this very call
    return bwd2d(fn, q, k, v, o, d_o, lse, dq, dk, dv, static_cast<float *>(workspace),
                 (size_t)B * heads * H * W * ws_floats_per_query(D, kernel_size, dtype), B, heads,
                 H, W, D, kernel_size, dtype, q_strides, k_strides, v_strides, o_strides,
                 do_strides, scale, stream);
}

int enatten2d_bwd_into(const void *q, const void *k, const void *v, const void *o,
                       const void *d_o, const float *lse, void *dq, void *dk, void *dv,
                       void *workspace, int B, int heads, int H, int W, int D, int kernel_size,
                       int dtype, const int64_t *q_strides, const int64_t *k_strides,
                       const int64_t *v_strides, const int64_t *o_strides,
                       const int64_t *do_strides, const int64_t *grad_strides, float scale,
                       void *stream) {
    const char *fn = "enatten2d_bwd_into";
    const int rc = check_shape(fn, B, heads, H, W, D, kernel_size, dtype);
    if (rc) return rc;
    if (!workspace) {
        set_error("%s: workspace is NULL", fn);
        return ENATTEN_EINVAL;
    }
    return bwd2d(fn, q, k, v, o, d_o, lse, dq, dk, dv, static_cast<float *>(workspace),
                 (size_t)B * heads * H * W * ws_floats_per_query(D, kernel_size, dtype), B, heads,
                 H, W, D, kernel_size, dtype, q_strides, k_strides, v_strides, o_strides,
                 do_strides, scale, stream, grad_strides);
}

// ---- backward without a caller-provided workspace ---------------------------
// The two float32 per query that the backward passes hand to each other live in a
// device array of this library instead.  Every GPU holds its own copy of the array at
// its own address; `scratch` below is only the host-side handle of the symbol, the
// address on the current device comes from hipGetSymbolAddress, once per device.
static __device__ __align__(256) float scratch[2 * (size_t)ENATTEN_STATIC_BWD_MAX_QUERIES];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<float *> g_scratch_ptr[kMaxDevices];

int scratch_of_current_device(const char *fn, float **out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        set_error("%s: no current HIP device (or a device number beyond %d)", fn, kMaxDevices - 1);
        return ENATTEN_ELAUNCH;
    }
    float *p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        // two threads may both ask; they get the same answer
        const hipError_t e = hipGetSymbolAddress(reinterpret_cast<void **>(&p), HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error("%s: hipGetSymbolAddress(scratch) failed: %s", fn, hipGetErrorString(e));
            return ENATTEN_ELAUNCH;
        }
        g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return ENATTEN_OK;
}
}  // namespace

int enatten2d_bwd_static(const void *q, const void *k, const void *v, const void *o,
                         const void *d_o, const float *lse, void *dq, void *dk, void *dv, int B,
                         int heads, int H, int W, int D, int kernel_size, int dtype,
                         const int64_t *q_strides, const int64_t *k_strides,
                         const int64_t *v_strides, const int64_t *o_strides,
                         const int64_t *do_strides, float scale, void *stream) {
    const char *fn = "enatten2d_bwd_static";
    int rc = check_shape(fn, B, heads, H, W, D, kernel_size, dtype);
    if (rc) return rc;
    if ((int64_t)B * heads * H * W > (int64_t)ENATTEN_STATIC_BWD_MAX_QUERIES) {
        set_error("%s: %lld queries exceed the %d that the built-in scratch holds; use "
                  "enatten2d_bwd with a workspace", fn, (long long)B * heads * H * W,
                  ENATTEN_STATIC_BWD_MAX_QUERIES);
        return ENATTEN_EUNSUPPORTED;
    }
    float *ws = nullptr;
    if ((rc = scratch_of_current_device(fn, &ws))) return rc;
    // Nothing in the scratch has to start at zero: the first pass writes both values of
    // every query before the second pass reads them.
    return bwd2d(fn, q, k, v, o, d_o, lse, dq, dk, dv, ws,
                 (size_t)2 * ENATTEN_STATIC_BWD_MAX_QUERIES, B, heads, H, W, D, kernel_size, dtype,
                 q_strides, k_strides, v_strides, o_strides, do_strides, scale, stream);
}

// ---- dilated neighborhoods --------------------------------------------------
// Sub-grids of one size run as one batch on the matrix-core kernels (up to four groups, one if
// the dilation divides both sides), and one after the other where they are large (`alone`) and on the
// other kernels.  The
// log-sum-exp and the workspace are laid out by group, within a group one [B, heads, h, w]
// block per sub-grid, whichever kernels serve the call, so that a backward that is routed
// differently from its forward (a misaligned upstream gradient) finds what it needs.
int enatten2d_fwd_dilated(const void *q, const void *k, const void *v, void *o, float *lse, int B,
                          int heads, int H, int W, int D, int kernel_size, int dilation, int dtype,
                          const int64_t *q_strides, const int64_t *k_strides,
                          const int64_t *v_strides, const int64_t *o_strides, float scale,
                          void *stream) {
    const char *fn = "enatten2d_fwd_dilated";
    int rc = check_shape(fn, B, heads, H, W, D, kernel_size, dtype);
    if (rc || (rc = check_dilation(fn, H, W, kernel_size, dilation))) return rc;
    FwdArgs full;
    if ((rc = make_view(fn, "q", q, q_strides, heads, H, W, D, &full.q))) return rc;
    if ((rc = make_view(fn, "k", k, k_strides, heads, H, W, D, &full.k))) return rc;
    if ((rc = make_view(fn, "v", v, v_strides, heads, H, W, D, &full.v))) return rc;
    if ((rc = make_view(fn, "o", o, o_strides, heads, H, W, D, &full.o))) return rc;
    const int es = elem_size(dtype);
    hipStream_t st = static_cast<hipStream_t>(stream);
    SubAxis rows[2], cols[2];
    const int nr = split_axis(H, dilation, rows), nc = split_axis(W, dilation, cols);
    for (int gi = 0; gi < nr; gi++)
        for (int gj = 0; gj < nc; gj++) {
            const SubAxis &r = rows[gi], &c = cols[gj];
            FwdArgsSub a;
            a.q = group_view(full.q, es, r, c);
            a.k = group_view(full.k, es, r, c);
            a.v = group_view(full.v, es, r, c);
            a.o = group_view(full.o, es, r, c);
            a.lse = lse;
            a.s = Shape{B, heads, r.extent, c.extent, D, kernel_size, kernel_size, scale};
            a.sub_r = r.count; a.sub_c = c.count; a.dil = dilation;
            const int64_t per_sub = (int64_t)B * heads * r.extent * c.extent;
            if (use_mfma(D, kernel_size, dtype) && sub_layout_ok(a) && !alone(a)) {
                if ((rc = launch_fwd_mfma_sub(a, dtype, st))) return rc;
            } else {
                for (int i = 0; i < r.count; i++)
                    for (int j = 0; j < c.count; j++) {
                        FwdArgs b = a;
                        b.q = one_sub(a.q, es, dilation, i, j);
                        b.k = one_sub(a.k, es, dilation, i, j);
                        b.v = one_sub(a.v, es, dilation, i, j);
                        b.o = one_sub(a.o, es, dilation, i, j);
                        if (lse) b.lse = lse + (i * c.count + j) * per_sub;
                        if ((rc = run_fwd(b, dtype, st))) return rc;
                    }
            }
            if (lse) lse += r.count * c.count * per_sub;
        }
    return ENATTEN_OK;
}

size_t enatten2d_bwd_dilated_workspace_bytes(int B, int heads, int H, int W, int dtype) {
    if (B < 1 || heads < 1 || H < 1 || W < 1) return 0;
    // two floats per query, four for float64; sub-grids that run one after the other share them
    return (size_t)B * heads * H * W * (dtype == ENATTEN_F64 ? 4 : 2) * sizeof(float);
}

int enatten2d_bwd_dilated(const void *q, const void *k, const void *v, const void *o,
                          const void *d_o, const float *lse, void *dq, void *dk, void *dv,
                          void *workspace, int B, int heads, int H, int W, int D, int kernel_size,
                          int dilation, int dtype, const int64_t *q_strides,
                          const int64_t *k_strides, const int64_t *v_strides,
                          const int64_t *o_strides, const int64_t *do_strides, float scale,
                          void *stream) {
    const char *fn = "enatten2d_bwd_dilated";
    int rc = check_shape(fn, B, heads, H, W, D, kernel_size, dtype);
    if (rc || (rc = check_dilation(fn, H, W, kernel_size, dilation))) return rc;
    BwdArgs full;
    if ((rc = make_view(fn, "q", q, q_strides, heads, H, W, D, &full.q))) return rc;
    if ((rc = make_view(fn, "k", k, k_strides, heads, H, W, D, &full.k))) return rc;
    if ((rc = make_view(fn, "v", v, v_strides, heads, H, W, D, &full.v))) return rc;
    if ((rc = make_view(fn, "o", o, o_strides, heads, H, W, D, &full.o))) return rc;
    if ((rc = make_view(fn, "d_o", d_o, do_strides, heads, H, W, D, &full.d_o))) return rc;
    if (!lse || !dq || !dk || !dv || !workspace) {
        set_error("%s: lse, dq, dk, dv and workspace must all be non-NULL", fn);
        return ENATTEN_EINVAL;
    }
    const int es = elem_size(dtype);
    const size_t ws_floats = (size_t)B * heads * H * W * (dtype == ENATTEN_F64 ? 4 : 2);
    hipStream_t st = static_cast<hipStream_t>(stream);
    SubAxis rows[2], cols[2];
    const int nr = split_axis(H, dilation, rows), nc = split_axis(W, dilation, cols);
    for (int gi = 0; gi < nr; gi++)
        for (int gj = 0; gj < nc; gj++) {
            const SubAxis &r = rows[gi], &c = cols[gj];
            BwdArgsSub a;
            a.q = group_view(full.q, es, r, c);
            a.k = group_view(full.k, es, r, c);
            a.v = group_view(full.v, es, r, c);
            a.o = group_view(full.o, es, r, c);
            a.d_o = group_view(full.d_o, es, r, c);
            a.lse = lse;
            a.s = Shape{B, heads, r.extent, c.extent, D, kernel_size, kernel_size, scale};
            // contiguous [B, heads, H, W, D] gradients
            const int64_t first = ((int64_t)r.first * W + c.first) * D;
            a.dq = offset(dq, first, es); a.dk = offset(dk, first, es); a.dv = offset(dv, first, es);
            a.gsw = D;
            a.gsh = (int64_t)W * D;
            a.gsn = (int64_t)H * W * D;
            a.gsb = (int64_t)heads * H * W * D;
            a.sub_r = r.count; a.sub_c = c.count; a.dil = dilation;
            const int64_t per_sub = (int64_t)B * heads * r.extent * c.extent;
            a.delta = static_cast<float *>(workspace);
            if (use_mfma(D, kernel_size, dtype) && sub_layout_ok(a) && !alone(a)) {
                a.zinv = a.delta + r.count * c.count * per_sub;
                if ((rc = launch_bwd_mfma_sub(a, dtype, st))) return rc;
            } else {
                for (int i = 0; i < r.count; i++)
                    for (int j = 0; j < c.count; j++) {
                        BwdArgs b = a;
                        b.q = one_sub(a.q, es, dilation, i, j);
                        b.k = one_sub(a.k, es, dilation, i, j);
                        b.v = one_sub(a.v, es, dilation, i, j);
                        b.o = one_sub(a.o, es, dilation, i, j);
                        b.d_o = one_sub(a.d_o, es, dilation, i, j);
                        const int64_t at = i * a.gsh + j * a.gsw;
                        b.dq = offset(a.dq, at, es); b.dk = offset(a.dk, at, es); b.dv = offset(a.dv, at, es);
                        b.gsh = a.gsh * dilation; b.gsw = a.gsw * dilation;
                        b.lse = lse + (i * c.count + j) * per_sub;
                        b.zinv = b.delta + per_sub;
                        if ((rc = run_bwd(fn, b, dtype, ws_floats, st))) return rc;
                    }
            }
            lse += r.count * c.count * per_sub;
        }
    return ENATTEN_OK;
}

// ---- rectangular and causal windows ----------------------------------------
// One axis of a window: extent k, causal or centred.
static int check_axis(const char *fn, const char *axis, int L, int k, int causal) {
    if (k < 1 || (!causal && k % 2 == 0)) {
        set_error("%s: kernel_%s must be >= 1, and odd unless that axis is causal, got %d", fn,
                  axis, k);
        return ENATTEN_EINVAL;
    }
    if (L < k) {
        set_error("%s: the image has %d positions along %s, fewer than kernel_%s = %d", fn, L, axis,
                  axis, k);
        return ENATTEN_EINVAL;
    }
    return ENATTEN_OK;
}

int enatten2d_fwd_window(const void *q, const void *k, const void *v, const void *rpb, void *o,
                         float *lse, int B, int heads, int H, int W, int D, int kernel_h,
                         int kernel_w, int causal_h, int causal_w, int dtype,
                         const int64_t *q_strides, const int64_t *k_strides,
                         const int64_t *v_strides, const int64_t *o_strides, float scale,
                         void *stream) {
    if (kernel_h == kernel_w && !causal_h && !causal_w && !rpb)
        return enatten2d_fwd(q, k, v, o, lse, B, heads, H, W, D, kernel_h, dtype, q_strides,
                             k_strides, v_strides, o_strides, scale, stream);
    const char *fn = "enatten2d_fwd_window";
    int rc = check_shape(fn, B, heads, H, W, D, 1, dtype);
    if (rc) return rc;
    if ((rc = check_axis(fn, "h", H, kernel_h, causal_h))) return rc;
    if ((rc = check_axis(fn, "w", W, kernel_w, causal_w))) return rc;
    if (rpb && (causal_h || causal_w)) {
        set_error("%s: a relative position bias goes with centred axes only", fn);
        return ENATTEN_EINVAL;
    }
    FwdArgs a;
    if ((rc = make_view(fn, "q", q, q_strides, heads, H, W, D, &a.q))) return rc;
    if ((rc = make_view(fn, "k", k, k_strides, heads, H, W, D, &a.k))) return rc;
    if ((rc = make_view(fn, "v", v, v_strides, heads, H, W, D, &a.v))) return rc;
    if ((rc = make_view(fn, "o", o, o_strides, heads, H, W, D, &a.o))) return rc;
    a.lse = lse;
    a.s = Shape{B, heads, H, W, D, kernel_h, kernel_w, scale, causal_h ? 1 : 0, causal_w ? 1 : 0};
    a.rpb = rpb;
    if (dtype == ENATTEN_F64) return launch_fwd_f64(a, static_cast<hipStream_t>(stream));
    if (use_band(a, dtype)) return launch_fwd_band(a, dtype, static_cast<hipStream_t>(stream));
    if (rpb && kernel_h == kernel_w && (use_mfma(D, kernel_h, dtype) || use_two_terms(D, kernel_h, dtype)))
        return launch_fwd_mfma_bias(a, dtype, static_cast<hipStream_t>(stream));
    return launch_fwd_simt(a, dtype, static_cast<hipStream_t>(stream));
}

size_t enatten2d_bwd_window_workspace_bytes(int B, int heads, int H, int W, int kernel_h,
                                            int kernel_w, int with_rpb) {
    if (B < 1 || heads < 1 || H < 1 || W < 1 || kernel_h < 1 || kernel_w < 1) return 0;
    // four floats per query (float64 tensors use all four), and with a bias dS of every
    // (query, window position)
    return (size_t)B * heads * H * W * (4 + (with_rpb ? (size_t)kernel_h * kernel_w : 0)) * sizeof(float);
}

static int bwd_window(const char *fn, const void *q, const void *k, const void *v, const void *rpb,
                      const void *o, const void *d_o, const float *lse, void *dq, void *dk,
                      void *dv, void *d_rpb, bool rpb_typed, void *workspace, int B, int heads, int H, int W,
                      int D, int kernel_h, int kernel_w, int causal_h, int causal_w, int dtype,
                      const int64_t *q_strides, const int64_t *k_strides,
                      const int64_t *v_strides, const int64_t *o_strides,
                      const int64_t *do_strides, float scale, void *stream) {
    const bool plain = kernel_h == kernel_w && !causal_h && !causal_w && !rpb;
    int rc = check_shape(fn, B, heads, H, W, D, plain ? kernel_h : 1, dtype);
    if (rc) return rc;
    if (!workspace) {
        set_error("%s: workspace is NULL", fn);
        return ENATTEN_EINVAL;
    }
    const size_t ws_floats = (size_t)B * heads * H * W * (dtype == ENATTEN_F64 ? 4 : 2);
    if (plain)  // the reference's window: every kernel family that two floats per query allow
        return bwd2d(fn, q, k, v, o, d_o, lse, dq, dk, dv, static_cast<float *>(workspace),
                     ws_floats, B, heads, H, W, D, kernel_h, dtype, q_strides, k_strides, v_strides,
                     o_strides, do_strides, scale, stream);
    if ((rc = check_axis(fn, "h", H, kernel_h, causal_h))) return rc;
    if ((rc = check_axis(fn, "w", W, kernel_w, causal_w))) return rc;
    if (rpb && (causal_h || causal_w)) {
        set_error("%s: a relative position bias goes with centred axes only", fn);
        return ENATTEN_EINVAL;
    }
    if (!rpb != !d_rpb) {
        set_error("%s: rpb and d_rpb come together", fn);
        return ENATTEN_EINVAL;
    }
    BwdArgs a;
    if ((rc = make_view(fn, "q", q, q_strides, heads, H, W, D, &a.q))) return rc;
    if ((rc = make_view(fn, "k", k, k_strides, heads, H, W, D, &a.k))) return rc;
    if ((rc = make_view(fn, "v", v, v_strides, heads, H, W, D, &a.v))) return rc;
    if ((rc = make_view(fn, "o", o, o_strides, heads, H, W, D, &a.o))) return rc;
    if ((rc = make_view(fn, "d_o", d_o, do_strides, heads, H, W, D, &a.d_o))) return rc;
    if (!lse || !dq || !dk || !dv) {
        set_error("%s: lse, dq, dk and dv must all be non-NULL", fn);
        return ENATTEN_EINVAL;
    }
    a.lse = lse;
    a.dq = dq; a.dk = dk; a.dv = dv;
    a.delta = static_cast<float *>(workspace);
    a.zinv = a.delta + (size_t)B * heads * H * W;
    a.s = Shape{B, heads, H, W, D, kernel_h, kernel_w, scale, causal_h ? 1 : 0, causal_w ? 1 : 0};
    if ((rc = set_grad_layout(fn, &a, nullptr))) return rc;
    a.rpb = rpb;
    a.d_rpb = d_rpb;
    a.ds_pairs = rpb ? a.delta + (size_t)4 * B * heads * H * W : nullptr;
    if (dtype == ENATTEN_F64) return bwd_f64(fn, a, ws_floats, static_cast<hipStream_t>(stream));
    if (use_band(a, dtype)) return launch_bwd_band(a, dtype, static_cast<hipStream_t>(stream));
    if (rpb && kernel_h == kernel_w && (use_mfma(D, kernel_h, dtype) || use_two_terms(D, kernel_h, dtype)))
        return launch_bwd_mfma_bias(a, dtype, static_cast<hipStream_t>(stream), rpb_typed);
    return launch_bwd_simt(a, dtype, static_cast<hipStream_t>(stream), rpb_typed);
}

int enatten2d_bwd_window(const void *q, const void *k, const void *v, const void *rpb,
                         const void *o, const void *d_o, const float *lse, void *dq, void *dk,
                         void *dv, float *d_rpb, void *workspace, int B, int heads, int H, int W,
                         int D, int kernel_h, int kernel_w, int causal_h, int causal_w, int dtype,
                         const int64_t *q_strides, const int64_t *k_strides,
                         const int64_t *v_strides, const int64_t *o_strides,
                         const int64_t *do_strides, float scale, void *stream) {
    return bwd_window("enatten2d_bwd_window", q, k, v, rpb, o, d_o, lse, dq, dk, dv, d_rpb, false, workspace, B, heads, H,
                      W, D, kernel_h, kernel_w, causal_h, causal_w, dtype, q_strides, k_strides, v_strides, o_strides,
                      do_strides, scale, stream);
}

int enatten2d_bwd_window_typed(const void *q, const void *k, const void *v, const void *rpb,
                               const void *o, const void *d_o, const float *lse, void *dq, void *dk,
                               void *dv, void *d_rpb, void *workspace, int B, int heads, int H, int W,
                               int D, int kernel_h, int kernel_w, int causal_h, int causal_w, int dtype,
                               const int64_t *q_strides, const int64_t *k_strides,
                               const int64_t *v_strides, const int64_t *o_strides,
                               const int64_t *do_strides, float scale, void *stream) {
    return bwd_window("enatten2d_bwd_window_typed", q, k, v, rpb, o, d_o, lse, dq, dk, dv, d_rpb, true, workspace, B,
                      heads, H, W, D, kernel_h, kernel_w, causal_h, causal_w, dtype, q_strides, k_strides, v_strides,
                      o_strides, do_strides, scale, stream);
}

static int view_1d(const char *fn, const char *name, const void *p, const int64_t *st, int N,
                   int T, int D, View *out) {
    if (!p) {
        set_error("%s: %s is NULL", fn, name);
        return ENATTEN_EINVAL;
    }
    out->ptr = p;
    out->sh = 0;
    if (st) {
        out->sb = st[0]; out->sn = st[1]; out->sw = st[2];
        if (out->sb < 0 || out->sn < 0 || out->sw < 0) {
            set_error("%s: negative stride for %s", fn, name);
            return ENATTEN_EINVAL;
        }
    } else {
        out->sw = D;
        out->sn = (int64_t)T * D;
        out->sb = (int64_t)N * T * D;
    }
    return ENATTEN_OK;
}

// A sequence is a 1 x T image with a 1 x k window: the size limit applies to
// B * heads * T * D elements.
static int check_shape_1d(const char *fn, int B, int N, int T, int D, int ks, int dtype) {
    if (ks >= 1 && ks % 2 == 1 && T >= 1 && T < ks) {
        set_error("%s: sequence length %d is smaller than kernel_size %d", fn, T, ks);
        return ENATTEN_EINVAL;
    }
    if (ks < 1 || ks % 2 == 0) return check_shape(fn, B, N, 1, T, D, ks, dtype);  // reports it
    return check_shape(fn, B, N, 1, T, D, 1, dtype);
}

int enatten1d_fwd(const void *q, const void *k, const void *v, void *o, float *lse, int B,
                  int heads, int T, int D, int kernel_size, int dtype, const int64_t *q_strides,
                  const int64_t *k_strides, const int64_t *v_strides, const int64_t *o_strides,
                  float scale, void *stream) {
    const char *fn = "enatten1d_fwd";
    int rc = check_shape_1d(fn, B, heads, T, D, kernel_size, dtype);
    if (rc) return rc;
    FwdArgs a;
    if ((rc = view_1d(fn, "q", q, q_strides, heads, T, D, &a.q))) return rc;
    if ((rc = view_1d(fn, "k", k, k_strides, heads, T, D, &a.k))) return rc;
    if ((rc = view_1d(fn, "v", v, v_strides, heads, T, D, &a.v))) return rc;
    if ((rc = view_1d(fn, "o", o, o_strides, heads, T, D, &a.o))) return rc;
    a.lse = lse;
    a.s = Shape{B, heads, 1, T, D, 1, kernel_size, scale};  // a 1 x k window on a 1 x T image
    if (dtype == ENATTEN_F64) return launch_fwd_f64(a, static_cast<hipStream_t>(stream));
    if (g_path.load() != ENATTEN_PATH_SIMT && mfma1d_supported(D, kernel_size, dtype))
        return launch_fwd1d_mfma(a, dtype, static_cast<hipStream_t>(stream));
    if (use_band(a, dtype)) return launch_fwd_band(a, dtype, static_cast<hipStream_t>(stream));
    return launch_fwd_simt(a, dtype, static_cast<hipStream_t>(stream));
}

size_t enatten1d_bwd_workspace_bytes(int B, int heads, int T) {
    if (B < 1 || heads < 1 || T < 1) return 0;
    return (size_t)B * heads * T * 4 * sizeof(float);  // float64 tensors use all four
}

int enatten1d_bwd(const void *q, const void *k, const void *v, const void *o, const void *d_o,
                  const float *lse, void *dq, void *dk, void *dv, void *workspace, int B,
                  int heads, int T, int D, int kernel_size, int dtype, const int64_t *q_strides,
                  const int64_t *k_strides, const int64_t *v_strides, const int64_t *o_strides,
                  const int64_t *do_strides, float scale, void *stream) {
    return enatten1d_bwd_into(q, k, v, o, d_o, lse, dq, dk, dv, workspace, B, heads, T, D, kernel_size,
                              dtype, q_strides, k_strides, v_strides, o_strides, do_strides, nullptr,
                              scale, stream);
}

int enatten1d_bwd_into(const void *q, const void *k, const void *v, const void *o, const void *d_o,
                       const float *lse, void *dq, void *dk, void *dv, void *workspace, int B,
                       int heads, int T, int D, int kernel_size, int dtype,
                       const int64_t *q_strides, const int64_t *k_strides, const int64_t *v_strides,
                       const int64_t *o_strides, const int64_t *do_strides,
                       const int64_t *grad_strides, float scale, void *stream) {
    const char *fn = grad_strides ? "enatten1d_bwd_into" : "enatten1d_bwd";
    int rc = check_shape_1d(fn, B, heads, T, D, kernel_size, dtype);
    if (rc) return rc;
    BwdArgs a;
    if ((rc = view_1d(fn, "q", q, q_strides, heads, T, D, &a.q))) return rc;
    if ((rc = view_1d(fn, "k", k, k_strides, heads, T, D, &a.k))) return rc;
    if ((rc = view_1d(fn, "v", v, v_strides, heads, T, D, &a.v))) return rc;
    if ((rc = view_1d(fn, "o", o, o_strides, heads, T, D, &a.o))) return rc;
    if ((rc = view_1d(fn, "d_o", d_o, do_strides, heads, T, D, &a.d_o))) return rc;
    if (!lse || !dq || !dk || !dv || !workspace) {
        set_error("%s: lse, dq, dk, dv and workspace must all be non-NULL", fn);
        return ENATTEN_EINVAL;
    }
    a.lse = lse;
    a.dq = dq; a.dk = dk; a.dv = dv;
    a.delta = static_cast<float *>(workspace);
    a.zinv = a.delta + (size_t)B * heads * T;
    a.s = Shape{B, heads, 1, T, D, 1, kernel_size, scale};
    {
        // (batch, head, position) strides -> the four of an image with one row
        const int64_t g4[4] = {grad_strides ? grad_strides[0] : 0, grad_strides ? grad_strides[1] : 0, 0,
                               grad_strides ? grad_strides[2] : 0};
        if ((rc = set_grad_layout(fn, &a, grad_strides ? g4 : nullptr))) return rc;
    }
    if (dtype == ENATTEN_F64)
        return bwd_f64(fn, a, (size_t)4 * B * heads * T, static_cast<hipStream_t>(stream));
    if (g_path.load() != ENATTEN_PATH_SIMT && mfma1d_supported(D, kernel_size, dtype))
        return launch_bwd1d_mfma(a, dtype, g_path.load(), static_cast<hipStream_t>(stream));
    if (use_band(a, dtype)) return launch_bwd_band(a, dtype, static_cast<hipStream_t>(stream));
    return launch_bwd_simt(a, dtype, static_cast<hipStream_t>(stream));
}

#pragma GCC visibility pop
}  // extern "C"
