// Images of at most 256 pixels, above all the sub-grids of a dilated call (14x14 for 56x56 at
// dilation 4): one workgroup per image, everything it needs in LDS at once.  bf16 / fp16, head dims that are
// multiples of 8 up to 64, any window.
//
// The tiled kernels of na2d_mfma_kernels.h cut such an image into four tiles that all touch the
// border, stage most of the image for each of them, and the dK/dV pass walks it block by block.
// Here the rows are staged once, tokens are the pixels in row order, and a wave takes 16 of them at
// a time: as queries against the run of tokens that their windows' rows span (forward, dQ), or as
// keys against the run of queries that see them (dK, dV), 32 tokens to a step, the window being a
// mask from a table of the tokens' places.  The backward is one kernel: five tensors read, three
// written, its jobs (16 queries' dQ, and behind a barrier 16 keys' dK and dV) dealt to the waves in
// turn, from both ends.
// A result that is not finite is computed again from its window alone, as in na1d_band_mfma.hip.
// Bound by the latency of the staging loads and the vector work on the logits (half of a step's
// pairs are inside a window at 14x14, k = 7).  B8 N4 56x56 d32 k7 dilation 4, forward and backward
// under the profiler: 70.1 us of three tiled kernels before, 13.4 + 26.1 here (1.8 TB/s of its 71 MB).
#include "na2d_mfma.h"

namespace enatten {
namespace {

constexpr int kNowhere = 20000;  // place of a row that is no token: outside every window
template <int D>
constexpr int kPitch = D + 8;

// Built for images of up to MAXP tokens and NW waves.  Smaller images get fewer waves (they have
// fewer blocks of 16 tokens to deal out) and less LDS, so that more of them share a CU: four, two
// and one workgroup of the backward at head_dim 32, for 96, 208 and 256 tokens.
template <int D_, int MAXP_, int NW_>
struct SGeo {
    static constexpr int D = D_, MAXP = MAXP_, NW = NW_, NT = 64 * NW;
    // a step of 32 tokens starts at a multiple of 16, so it may reach 16 past the last block of them
    static constexpr int ROWS = MAXP + 16;
    static constexpr int PITCH = kPitch<D>, CPR = D / 8, DS = D / 32, DT = D / 16;
    static constexpr int NL = (ROWS * CPR + NT - 1) / NT;
    static constexpr int WPS = D == 32 ? 4 : 2;  // waves per SIMD that the registers are budgeted for
    static_assert(MAXP % 16 == 0, "whole blocks");
};

struct Img {
    int bb, nn, ri, rj;
    int64_t tok;  // its first token in the log-sum-exp and the workspace
};
// Image of a workgroup: (batch, sub-grid row, sub-grid column, head), every XCD one contiguous run
// (neighbouring sub-grids and heads share lines).  false: no such image
template <typename ARGS>
__device__ __forceinline__ bool image_of(const ARGS &a, int nimages, Img &im) {
    int t = ((int)blockIdx.x & 7) * ((int)gridDim.x >> 3) + ((int)blockIdx.x >> 3);
    if (t >= nimages) return false;
    im.nn = t % a.s.N;
    t /= a.s.N;
    im.rj = t % a.sub_c;
    t /= a.sub_c;
    im.ri = t % a.sub_r;
    im.bb = t / a.sub_r;
    im.tok = ((((int64_t)im.ri * a.sub_c + im.rj) * a.s.B + im.bb) * a.s.N + im.nn) * a.s.H * a.s.W;
    return true;
}
__device__ __forceinline__ const short *img_ptr(const View &v, const Img &im) {
    return static_cast<const short *>(v.ptr) + im.bb * v.sb + im.nn * v.sn + im.ri * v.sh + im.rj * v.sw;
}
// element offset of pixel t
__device__ __forceinline__ int64_t pix(const View &v, int dil, int y, int x) { return y * v.sh * dil + x * v.sw * dil; }

// all rows of a tensor, zeros behind the last token and the tensor's channels
template <typename G>
struct Rows {
    u32x4 v[G::NL];
    __device__ __forceinline__ void fetch(const View &t, const Img &im, int dil, int W, int P, int dlim) {
        const short *base = img_ptr(t, im);
        const int c = (int)threadIdx.x % G::CPR;
#pragma unroll
        for (int i = 0; i < G::NL; i++) {
            const int r = ((int)threadIdx.x + i * G::NT) / G::CPR;
            v[i] = u32x4{0u, 0u, 0u, 0u};
            if (r < P && c * 8 < dlim)
                v[i] = *reinterpret_cast<const u32x4 *>(base + pix(t, dil, r / W, r % W) + c * 8);
        }
    }
    __device__ __forceinline__ void commit(short *lds) const {
        const int c = (int)threadIdx.x % G::CPR;
#pragma unroll
        for (int i = 0; i < G::NL; i++) {
            const int r = ((int)threadIdx.x + i * G::NT) / G::CPR;
            if (r < G::ROWS) *reinterpret_cast<u32x4 *>(lds + r * G::PITCH + c * 8) = v[i];
        }
    }
};
// places as (row, column << 16)
__device__ __forceinline__ int pack(int y, int x) { return y | x << 16; }
__device__ __forceinline__ bool inside(int pos, int win, int k) {
    return (unsigned)((pos & 0xffff) - (win & 0xffff)) < (unsigned)k && (unsigned)((pos >> 16) - (win >> 16)) < (unsigned)k;
}
// tables of every row: its place, and the start of its window
template <typename G>
__device__ __forceinline__ void fill_places(int *lds_pos, int *lds_win, const Shape &s, int P) {
    for (int t = threadIdx.x; t < G::ROWS; t += G::NT) {
        const int y = t / s.W, x = t % s.W;
        lds_pos[t] = t < P ? pack(y, x) : kNowhere;
        lds_win[t] = t < P ? pack(win_start(y, s.H, s.kh), win_start(x, s.W, s.kw)) : kNowhere;
    }
}
// the tokens of the rows that the windows of tokens [t0, t0 + 16) span: [lo, hi)
__device__ __forceinline__ void key_run(int t0, int P, const Shape &s, int &lo, int &hi) {
    lo = win_start(t0 / s.W, s.H, s.kh) * s.W;
    hi = (win_start(min(t0 + 15, P - 1) / s.W, s.H, s.kh) + s.kh) * s.W;
}
// the tokens of the rows whose queries may see tokens [t0, t0 + 16)
__device__ __forceinline__ void query_run(int t0, int P, const Shape &s, int &lo, int &hi) {
    lo = inv_lo(t0 / s.W, s.kh) * s.W;
    hi = inv_hi(min(t0 + 15, P - 1) / s.W, s.H, s.kh) * s.W;
}
template <int DS>
__device__ __forceinline__ void lds_row(s16x8 (&reg)[DS], const short *row, int g) {
#pragma unroll
    for (int ds = 0; ds < DS; ds++) reg[ds] = *reinterpret_cast<const s16x8 *>(row + ds * 32 + g * 8);
}
// c[h] = X rows t0 + 16 h .. of LDS times the wave's 16 columns
template <bool BF, int D>
__device__ __forceinline__ void first_product(f32x4 (&c)[2], const short *lds, int t0, int n, int g,
                                              const s16x8 (&reg)[D / 32]) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const short *p = lds + (t0 + h * 16 + n) * kPitch<D> + g * 8;
        c[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ds = 0; ds < D / 32; ds++) c[h] = mfma16<BF>(*reinterpret_cast<const s16x8 *>(p + ds * 32), reg[ds], c[h]);
    }
}
// acc += X^T w over 32 rows of LDS from t0 on
template <bool BF, int D>
__device__ __forceinline__ void second_product(f32x4 (&acc)[D / 16], const short *lds, int t0, int n, int g, s16x8 w) {
    const short *p = lds + (t0 + g * 4 + (n >> 2)) * kPitch<D> + (n & 3) * (D / 4);
#pragma unroll
    for (int t = 0; t < D / 16; t++)
        acc[t] = mfma16<BF>(cat(lds_read_tr(p + t * 4), lds_read_tr(p + 16 * kPitch<D> + t * 4)), w, acc[t]);
}
// ... and acc2 += X^T w2 with the same rows
template <bool BF, int D>
__device__ __forceinline__ void second_product(f32x4 (&acc)[D / 16], const short *lds, int t0, int n, int g, s16x8 w,
                                               f32x4 (&acc2)[D / 16], s16x8 w2) {
    const short *p = lds + (t0 + g * 4 + (n >> 2)) * kPitch<D> + (n & 3) * (D / 4);
#pragma unroll
    for (int t = 0; t < D / 16; t++) {
        const s16x8 x = cat(lds_read_tr(p + t * 4), lds_read_tr(p + 16 * kPitch<D> + t * 4));
        acc[t] = mfma16<BF>(x, w, acc[t]);
        acc2[t] = mfma16<BF>(x, w2, acc2[t]);
    }
}
// element e of a lane's eight: row t0 + (e >> 2) * 16 + g * 4 + (e & 3)
__device__ __forceinline__ void lane_places(int (&x)[8], const int *table, int t0, int g) {
    typedef int i32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const i32x4 r = *reinterpret_cast<const i32x4 *>(table + t0 + h * 16 + g * 4);
#pragma unroll
        for (int e = 0; e < 4; e++) x[h * 4 + e] = r[e];
    }
}

// channel l of a row, 0 beyond the channels
template <bool BF>
__device__ __forceinline__ float chan(const short *row, int l, int channels) {
    return l < channels ? cvt32<BF>(row[l]) : 0.f;
}

template <bool BF, typename G>
__global__ __launch_bounds__(G::NT, G::WPS) void fwd_small_mfma(FwdArgsSub a, int nimages) {
    constexpr int D = G::D;
    __shared__ __attribute__((aligned(16))) short lds_k[G::ROWS * G::PITCH], lds_v[G::ROWS * G::PITCH];
    __shared__ __attribute__((aligned(16))) int lds_pos[G::ROWS], lds_win[G::ROWS];
    const Shape &s = a.s;
    const int P = s.H * s.W, ks = s.kh;
    Img im;
    if (!image_of(a, nimages, im)) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const float sc2 = s.scale * kLog2e;
    {
        Rows<G> k, v;
        k.fetch(a.k, im, a.dil, s.W, P, s.D);
        v.fetch(a.v, im, a.dil, s.W, P, s.D);
        fill_places<G>(lds_pos, lds_win, s, P);
        k.commit(lds_k);
        v.commit(lds_v);
    }
    __syncthreads();
    const short *qimg = img_ptr(a.q, im);
    short *oimg = const_cast<short *>(img_ptr(a.o, im));
    for (int t0 = wave * 16; t0 < P; t0 += G::NW * 16) {
        const int qt = min(t0 + n, P - 1), qy = qt / s.W, qx = qt % s.W;
        s16x8 qreg[G::DS];
        load_row_chunks(qreg, qimg + pix(a.q, a.dil, qy, qx), g, s.D);
        const int win = lds_win[qt];
        int lo, hi;
        key_run(t0, P, s, lo, hi);
        f32x4 o[G::DT];
#pragma unroll
        for (int t = 0; t < G::DT; t++) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        float m = -__FLT_MAX__, sum = 0.f;
        for (int kk = lo & ~15; kk < hi; kk += 32) {
            f32x4 c[2];
            first_product<BF, D>(c, lds_k, kk, n, g, qreg);
            int pos[8];
            lane_places(pos, lds_pos, kk, g);
            float x[8], mx = -INFINITY;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                x[e] = inside(pos[e], win, ks) ? c[e >> 2][e & 3] * sc2 : -INFINITY;
                mx = fmaxf(mx, x[e]);
            }
            // (the maximum follows once a logit exceeds it by 2^8, as in na1d_band_mfma.hip)
            if (__any(mx > m + 8.f)) {
                const float mn = fmaxf(m, col_max(mx)), corr = __builtin_amdgcn_exp2f(m - mn);
                m = mn;
                sum *= corr;
#pragma unroll
                for (int t = 0; t < G::DT; t++) o[t] *= corr;
            }
            s16x8 p;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                x[e] = __builtin_amdgcn_exp2f(x[e] - m);
                sum += x[e];
                p[e] = cvt16<BF>(x[e]);
            }
            second_product<BF, D>(o, lds_v, kk, n, g, p);
        }
        const float total = col_sum(sum);
        unsigned bad = bad_columns(o, total);
        const bool live = t0 + n < P && !(bad >> n & 1);
        store_token<BF, D>(oimg + pix(a.o, a.dil, qy, qx), g, o, 1.f / total, live, s.D);
        if (a.lse && live && g == 0) a.lse[im.tok + qt] = (m + __builtin_amdgcn_logf(total)) * kLn2;
        for (; bad; bad &= bad - 1) {
            const int t = t0 + __builtin_ctz(bad);
            if (t >= P) break;
            const float q = chan<BF>(qimg + pix(a.q, a.dil, t / s.W, t % s.W), l, s.D);
            float acc = 0.f, mx = -INFINITY, z = 0.f;
            for (int j = 0; j < ks * ks; j++) {
                const int w = lds_win[t], key = ((w & 0xffff) + j / ks) * s.W + (w >> 16) + j % ks;
                const float x = wave_sum(q * chan<BF>(lds_k + key * G::PITCH, l, D)) * sc2;
                const float mn = x > mx ? x : mx, corr = __builtin_amdgcn_exp2f(mx - mn);
                const float p = __builtin_amdgcn_exp2f(x - mn);
                mx = mn;
                z = z * corr + p;
                acc = acc * corr + p * chan<BF>(lds_v + key * G::PITCH, l, D);
                if (z != z) break;  // nothing finite can come of it
            }
            if (l < s.D) oimg[pix(a.o, a.dil, t / s.W, t % s.W) + l] = cvt16<BF>(acc / z);
            if (a.lse && l == 0) a.lse[im.tok + t] = (mx + __builtin_amdgcn_logf(z)) * kLn2;
        }
    }
}

template <bool BF, typename G>
__global__ __launch_bounds__(G::NT, G::WPS) void bwd_small_mfma(BwdArgsSub a, int nimages) {
    constexpr int D = G::D;
    __shared__ __attribute__((aligned(16))) short lds_q[G::ROWS * G::PITCH], lds_k[G::ROWS * G::PITCH],
        lds_v[G::ROWS * G::PITCH], lds_g[G::ROWS * G::PITCH];
    __shared__ __attribute__((aligned(16))) int lds_pos[G::ROWS], lds_win[G::ROWS];
    __shared__ __attribute__((aligned(16))) float lds_lse[G::ROWS], lds_delta[G::ROWS];  // (lse * log2e)
    const Shape &s = a.s;
    const int P = s.H * s.W, ks = s.kh;
    Img im;
    if (!image_of(a, nimages, im)) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const float sc2 = s.scale * kLog2e;
    {
        Rows<G> x, go, o;
        go.fetch(a.d_o, im, a.dil, s.W, P, s.D);
        o.fetch(a.o, im, a.dil, s.W, P, s.D);
        x.fetch(a.q, im, a.dil, s.W, P, s.D);
        fill_places<G>(lds_pos, lds_win, s, P);
        for (int t = threadIdx.x; t < G::ROWS; t += G::NT) lds_lse[t] = t < P ? a.lse[im.tok + t] * kLog2e : 0.f;
        go.commit(lds_g);
#pragma unroll
        for (int i = 0; i < G::NL; i++) {
            const int r = ((int)threadIdx.x + i * G::NT) / G::CPR;
            const float d = group_sum<G::CPR>(dot8<BF>(go.v[i], o.v[i]));
            if (r < G::ROWS && threadIdx.x % G::CPR == 0) lds_delta[r] = d;
        }
        x.commit(lds_q);
        x.fetch(a.k, im, a.dil, s.W, P, s.D);
        go.fetch(a.v, im, a.dil, s.W, P, s.D);
        x.commit(lds_k);
        go.commit(lds_v);
    }
    __syncthreads();
    const int blocks = (P + 15) / 16;
    auto grad_pix = [&](int t) __attribute__((always_inline)) {
        return a.grad_at(im.bb, im.nn, im.ri + t / s.W * a.dil, im.rj + t % s.W * a.dil);
    };
    // dQ.  delta = dO . O is what O was rounded to away from the sum of P dP, an error that all keys
    // of a window share and that keys or values with a common component multiply.  So the residual
    // E = sum p (dP - delta) is summed beside the products, dQ = A - E sum p k, and the dK/dV jobs
    // find delta + E (sum p is 1 to what the log-sum-exp was rounded to; 14x14 d64 k9 bf16, k and v of
    // mean 2: dQ off by 4.4e-2 in 2-norm without, 4.1e-3 with).
    for (int t0 = wave * 16; t0 < P; t0 += G::NW * 16) {
        const int own = min(t0 + n, P - 1);
        s16x8 qreg[G::DS], greg[G::DS];
        lds_row(qreg, lds_q + own * G::PITCH, g);
        lds_row(greg, lds_g + own * G::PITCH, g);
        const int win = lds_win[own];
        const float lse2 = lds_lse[own], delta = lds_delta[own];
        int lo, hi;
        key_run(t0, P, s, lo, hi);
        f32x4 dq[G::DT], pk[G::DT];
        float esum = 0.f;
#pragma unroll
        for (int t = 0; t < G::DT; t++) {
            dq[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            pk[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        for (int kk = lo & ~15; kk < hi; kk += 32) {
            f32x4 c[2], cp[2];
            first_product<BF, D>(c, lds_k, kk, n, g, qreg);
            first_product<BF, D>(cp, lds_v, kk, n, g, greg);
            int pos[8];
            lane_places(pos, lds_pos, kk, g);
            s16x8 ph, ds;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float x = c[e >> 2][e & 3] * sc2 - lse2;
                const float p = __builtin_amdgcn_exp2f(inside(pos[e], win, ks) ? x : -INFINITY);
                const float y = p * (cp[e >> 2][e & 3] - delta);
                esum += y;
                ph[e] = cvt16<BF>(p);
                ds[e] = cvt16<BF>(y);
            }
            second_product<BF, D>(dq, lds_k, kk, n, g, ds, pk, ph);
        }
        const float shift = col_sum(esum);
#pragma unroll
        for (int t = 0; t < G::DT; t++) dq[t] -= shift * pk[t];
        unsigned bad = bad_columns(dq);
        const bool here = t0 + n < P && !(bad >> n & 1);
        store_token<BF, D>(static_cast<short *>(a.dq) + grad_pix(own), g, dq, s.scale, here, s.D);
        // (only the jobs behind the barrier read another block's)
        if (here && g == 0) lds_delta[own] = delta + shift;
        for (; bad; bad &= bad - 1) {
            const int t = t0 + __builtin_ctz(bad);
            if (t >= P) break;
            const float q = chan<BF>(lds_q + t * G::PITCH, l, D), go = chan<BF>(lds_g + t * G::PITCH, l, D);
            float acc = 0.f, accp = 0.f, z = 0.f, res = 0.f;
            const int w = lds_win[t];
            for (int j = 0; j < ks * ks; j++) {
                const int key = ((w & 0xffff) + j / ks) * s.W + (w >> 16) + j % ks;
                const float kr = chan<BF>(lds_k + key * G::PITCH, l, D);
                const float p = __builtin_amdgcn_exp2f(wave_sum(q * kr) * sc2 - lds_lse[t]);
                const float y = p * (wave_sum(go * chan<BF>(lds_v + key * G::PITCH, l, D)) - lds_delta[t]);
                z += p;
                res += y;
                acc += y * kr;
                accp += p * kr;
                if (z != z) break;  // nothing finite can come of it
            }
            if (l < s.D) static_cast<short *>(a.dq)[grad_pix(t) + l] = cvt16<BF>((acc - res / z * accp) * s.scale);
            if (l == 0) lds_delta[t] += res / z;
        }
    }
    __syncthreads();
    for (int t0 = (G::NW - 1 - wave) * 16; t0 < P; t0 += G::NW * 16) {
        const int own = min(t0 + n, P - 1);
        const int64_t at = grad_pix(own);
        s16x8 kreg[G::DS], vreg[G::DS];
        lds_row(kreg, lds_k + own * G::PITCH, g);
        lds_row(vreg, lds_v + own * G::PITCH, g);
        const int pos = lds_pos[own];
        int lo, hi;
        query_run(t0, P, s, lo, hi);
        f32x4 dk[G::DT], dv[G::DT];
#pragma unroll
        for (int t = 0; t < G::DT; t++) {
            dk[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            dv[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        for (int qq = lo & ~15; qq < hi; qq += 32) {
            f32x4 c[2], cp[2];
            first_product<BF, D>(c, lds_q, qq, n, g, kreg);
            first_product<BF, D>(cp, lds_g, qq, n, g, vreg);
            int win[8];
            lane_places(win, lds_win, qq, g);
            s16x8 ph, ds;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const f32x4 lse2 = *reinterpret_cast<const f32x4 *>(lds_lse + qq + h * 16 + g * 4);
                const f32x4 delta = *reinterpret_cast<const f32x4 *>(lds_delta + qq + h * 16 + g * 4);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float x = c[h][i] * sc2 - lse2[i];
                    const float p = __builtin_amdgcn_exp2f(inside(pos, win[h * 4 + i], ks) ? x : -INFINITY);
                    ph[h * 4 + i] = cvt16<BF>(p);
                    ds[h * 4 + i] = cvt16<BF>(p * (cp[h][i] - delta[i]));
                }
            }
            second_product<BF, D>(dv, lds_g, qq, n, g, ph);
            second_product<BF, D>(dk, lds_q, qq, n, g, ds);
        }
        unsigned bad = bad_columns(dk) | bad_columns(dv);
        const bool here = t0 + n < P && !(bad >> n & 1);
        store_token<BF, D>(static_cast<short *>(a.dk) + at, g, dk, s.scale, here, s.D);
        store_token<BF, D>(static_cast<short *>(a.dv) + at, g, dv, 1.f, here, s.D);
        for (; bad; bad &= bad - 1) {
            const int t = t0 + __builtin_ctz(bad);
            if (t >= P) break;
            const float kr = chan<BF>(lds_k + t * G::PITCH, l, D), vr = chan<BF>(lds_v + t * G::PITCH, l, D);
            float ak = 0.f, av = 0.f;
            query_run(t, t + 1, s, lo, hi);
            for (int q = lo; q < hi; q++) {
                if (!inside(lds_pos[t], lds_win[q], ks)) continue;
                const float qr = chan<BF>(lds_q + q * G::PITCH, l, D), gr = chan<BF>(lds_g + q * G::PITCH, l, D);
                const float p = __builtin_amdgcn_exp2f(wave_sum(qr * kr) * sc2 - lds_lse[q]);
                av += p * gr;
                ak += p * (wave_sum(gr * vr) - lds_delta[q]) * qr;
                if (p != p) break;  // nothing finite can come of it
            }
            if (l < s.D) {
                static_cast<short *>(a.dk)[grad_pix(t) + l] = cvt16<BF>(ak * s.scale);
                static_cast<short *>(a.dv)[grad_pix(t) + l] = cvt16<BF>(av);
            }
        }
    }
}

template <typename ARGS>
int64_t images_of(const ARGS &a) { return (int64_t)a.s.B * a.s.N * a.sub_r * a.sub_c; }
int small_grid(int64_t nimages) { return (int)((nimages + 7) / 8 * 8); }

template <bool BF, typename G>
int fwd_go(const FwdArgsSub &a, hipStream_t st) {
    const int64_t ni = images_of(a);
    {
        ProfScope prof(ENATTEN_KERNEL_FWD, "fwd_small_mfma", st);
        hipLaunchKernelGGL((fwd_small_mfma<BF, G>), dim3(small_grid(ni)), dim3(G::NT), 0, st, a, (int)ni);
    }
    return check_launch("fwd_small_mfma");
}
template <bool BF, typename G>
int bwd_go(const BwdArgsSub &a, hipStream_t st) {
    const int64_t ni = images_of(a);
    {
        ProfScope prof(ENATTEN_KERNEL_BWD_FUSED, "bwd_small_mfma", st);
        hipLaunchKernelGGL((bwd_small_mfma<BF, G>), dim3(small_grid(ni)), dim3(G::NT), 0, st, a, (int)ni);
    }
    return check_launch("bwd_small_mfma");
}
// (a launch holds fewer than 2^32 threads: more images are left to the tiled kernels, whose grid does
// not grow with them)
bool size_ok(const Shape &s, int64_t nimages, int max_tokens, int threads) {
    return s.D <= 64 && (int64_t)s.H * s.W <= max_tokens && nimages <= ((int64_t)1 << 32) / threads - 8;
}

// threads of the workgroups that fwd_size and bwd_size choose
int fwd_threads(const Shape &s) { return s.H * s.W <= 96 ? 256 : 512; }
int bwd_threads(const Shape &s) {
    const int P = s.H * s.W;
    return P <= 96 ? 256 : P <= 208 || s.D > 32 ? 512 : 1024;
}
template <bool BF, int D>
int fwd_size(const FwdArgsSub &a, hipStream_t st) {
    return a.s.H * a.s.W <= 96 ? fwd_go<BF, SGeo<D, 96, 4>>(a, st) : fwd_go<BF, SGeo<D, 208, 8>>(a, st);
}
template <bool BF, int D>
int bwd_size(const BwdArgsSub &a, hipStream_t st) {
    const int P = a.s.H * a.s.W;
    return P <= 96    ? bwd_go<BF, SGeo<D, 96, 4>>(a, st)
           : P <= 208 ? bwd_go<BF, SGeo<D, 208, 8>>(a, st) : bwd_go<BF, SGeo<D, 256, D == 32 ? 16 : 8>>(a, st);
}

}  // namespace

// Where an image is taken whole, tiled / whole in us, bf16.  The forward: where there are more
// images than CUs, since the tiled kernel spreads one over four workgroups (14x14 pixels d32 k7: 8
// images 5.3 / 8.3, 128 images 6.6 / 8.4, 512 images 14.2 / 11.7), and up to 208 pixels: at 16x16 the
// tiles are whole and level (8192 images d32 k5 211 / 215).  Undilated ones for k >= 7 from the second tile on
// (8x8 d32, 1024 images 7.1 / 7.5).
// The backward, one kernel in the place of two whose dK/dV pass walks the border: always for the smallest size
// (8x8 d32 k7, 16 to 256 images 8.4 to 9.0 / 6.3 to 6.8; 9x10 d64 k9, 8 images, dilated 16.0 / 13.0), and where the 8x8
// tiles are too many for two workgroups per CU (14x14 d32 k7 192 images 22.8 / 16.0, d64 k9 31.8 / 23.8, dilated 256
// images 44.2 / 26.7; 14x18 d48 k9 96 images 35.3 / 28.8; 16x16 d64 k13 128 dilated images 41.7 / 31.4), at head dims
// up to 32 a little before (14x14 d32 k7 96 images 15.9 / 15.5) and dilated for k >= 5 always (14x14 d32 k7, 8 images 17.0 /
// 15.2).  With fewer tiles the tiled kernels have the chip to themselves (64 images 14x14 d32 k7 12.9 / 15.3, d64
// k9 17.9 / 22.9, dilated 20.4 / 23.0, 14x14 d32 k3 dilated 11.6 / 12.6; 128 images 16x16 d32 k7 13.4 / 15.1).  Undilated
// images for k >= 7 only: at k = 3 and 5 the other passes have little border to walk (14x14 d64 k3, 128
// images 10.8 / 14.5).
bool small_fwd_supported(const FwdArgsSub &a) {
    return size_ok(a.s, images_of(a), 208, fwd_threads(a.s)) && images_of(a) > 256 &&
           (a.dil > 1 || (a.s.kh >= 7 && a.s.H * a.s.W > 64));
}
bool small_bwd_supported(const BwdArgsSub &a) {
    const Shape &s = a.s;
    const int64_t ni = images_of(a), tiles = ni * ((s.H + 7) / 8) * ((s.W + 7) / 8);
    if (!size_ok(s, ni, 256, bwd_threads(s))) return false;
    if (s.H * s.W <= 96) return a.dil > 1 || s.kh >= 7;
    if (a.dil > 1) return tiles >= 512 || (s.D <= 32 && s.kh >= 5);
    return s.kh >= 7 && (tiles > 512 || (s.D <= 32 && s.H * s.W <= 208 && tiles >= 384));
}
int launch_fwd_small(const FwdArgsSub &a, int dtype, hipStream_t st) {
    if (dtype == ENATTEN_BF16) return a.s.D <= 32 ? fwd_size<true, 32>(a, st) : fwd_size<true, 64>(a, st);
    return a.s.D <= 32 ? fwd_size<false, 32>(a, st) : fwd_size<false, 64>(a, st);
}
int launch_bwd_small(const BwdArgsSub &a, int dtype, hipStream_t st) {
    if (dtype == ENATTEN_BF16) return a.s.D <= 32 ? bwd_size<true, 32>(a, st) : bwd_size<true, 64>(a, st);
    return a.s.D <= 32 ? bwd_size<false, 32>(a, st) : bwd_size<false, 64>(a, st);
}

}  // namespace enatten
