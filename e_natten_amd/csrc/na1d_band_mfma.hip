// Matrix-core kernels for 1D windows of any length, centred or causal (sliding-window causal
// attention), bf16 / fp16, head dims that are multiples of 8 up to 128.
//
// The kernels of na1d_mfma_kernels.h stage all keys of a tile at once, which ends at a
// kernel_size of 49.  Here a workgroup of four waves owns a tile of queries and walks the keys
// that any of them sees, 64 (or 32) at a time, with an online softmax: K and V rows of a block are in
// LDS, the next block's are in flight into registers and go into a second buffer, one barrier
// per block.  A wave owns 16 queries (the columns of v_mfma_f32_16x16x32), or in the forward of long
// windows two groups of 16, where every operand that comes out of LDS feeds twice the matrix
// instructions.  It takes the keys 32 at a time, skips the steps its own queries do not reach, and masks only the steps that
// the band's edges cut.  Operand layouts are those of na2d_mfma_kernels.h (tokens as MFMA rows,
// the second product's other operand through the transposing LDS read).
//
// The running maximum is only raised when a logit exceeds it by more than 8 (in units of log2; the
// conditional rescaling published with FlashAttention-4):
// until then the probabilities are at most 2^8 times what they would be, which neither float32
// sums nor 16-bit operands lose anything by, and no cross-lane maximum is formed.
//
// Probabilities and dS enter the second products as the sum of two 16-bit terms (the value
// rounded, and what the rounding left): the products are exact to 16 (bf16) or 22 (fp16, down to
// 2^-25 of the largest) bits of them, as close as the results' own type can show to the float32
// probabilities of the general kernels.  float16 dS, and P in the dK/dV pass, are scaled by a power
// of two for that (DsScale; kPScale).
//
// The backward is renormalised as that of the general kernels: delta = dO . O carries what O was
// rounded to, and the recomputed probabilities what the log-sum-exp was.  The dQ pass sums
// Z = sum p and E = sum p (dP - delta) beside the products, dQ = (A - E / Z sum p k) / Z, and leaves
// delta + E / Z and 1 / Z for the dK/dV pass.  (k and v of mean 2, bf16, d64 k128 causal: dQ off by
// 4.7e-2 in 2-norm without, 1.7e-3 with.)
//
// What bounds it: at k = 128 the bytes (each key row is read by two or three workgroups of one
// XCD, out of its L2); from k of about 512 the matrix pipe and the LDS reads that feed it.
//
// Per-query math: e_natten/triton.py:65-222; the causal rule is not in the reference.

#include "na2d_mfma.h"

namespace enatten {
namespace {

// Rows of a staged block: keys in the forward and the dQ pass, queries in the dK/dV pass.  64, and
// 32 for the dK/dV pass at head_dim 64, where the smaller buffers let a third workgroup share the CU
// (B4 N16 T8192 k32 causal 101 -> 86 us), and for the forward at 128 (short_blocks); not for the
// forward at 64 (54.6 -> 57.1), not for the backward at head_dim 128, where the registers leave room for two
// workgroups (dK/dV B1 N16 T8192 k128 62 -> 68), nor at 32, where 32 rows are fewer than the 64 that a
// pass of all threads moves.
constexpr int kRowsQ = 64;
template <int D>
constexpr int kRowsK = D == 64 ? 32 : 64;

template <int D, int KB>
struct BGeo {
    static constexpr int PITCH = D + 8, CPR = D / 8, RPP = 256 / CPR, NL = KB / RPP;
    static_assert(KB % RPP == 0, "every thread moves the same number of chunks");
    static constexpr int DS = D / 32, DT = D / 16;
};

// KB rows of a sequence from p0 on, clamped to its last position (such rows only meet zero
// probabilities); channels at or beyond dlim are zero.
template <int D, int KB, bool NARROW>
struct Block {
    using G = BGeo<D, KB>;
    u32x4 v[G::NL];
    __device__ __forceinline__ void fetch(const short *sq, int64_t sw, int p0, int T, int dlim) {
        const int c = (int)threadIdx.x % G::CPR;
        if (NARROW && c * 8 >= dlim) {
#pragma unroll
            for (int i = 0; i < G::NL; i++) v[i] = u32x4{0u, 0u, 0u, 0u};
            return;
        }
        const int pb = min(p0, T - 1), rmax = T - 1 - pb;
        const char *base = reinterpret_cast<const char *>(sq + pb * sw);
        const unsigned sw2 = (unsigned)sw * 2u;
#pragma unroll
        for (int i = 0; i < G::NL; i++) {
            const int r = min((int)threadIdx.x / G::CPR + i * G::RPP, rmax);
            v[i] = *reinterpret_cast<const u32x4 *>(base + __umul24((unsigned)r, sw2) + (unsigned)c * 16u);
        }
    }
    __device__ __forceinline__ void commit(short *lds) const {
#pragma unroll
        for (int i = 0; i < G::NL; i++)
            *reinterpret_cast<u32x4 *>(lds + ((int)threadIdx.x / G::CPR + i * G::RPP) * G::PITCH +
                                       ((int)threadIdx.x % G::CPR) * 8) = v[i];
    }
};

struct BTile {
    int bb, nn, t0;
};
// Consecutive workgroup ids go round-robin to the 8 XCDs: each XCD gets one contiguous run of
// tiles, so that the tiles that share key rows meet in one L2.  false: no such tile.
__device__ __forceinline__ bool btile(int block, int nblocks, int ntiles, int tiles_t, int size, int N, BTile &tl) {
    const int t = (block & 7) * (nblocks >> 3) + (block >> 3);
    if (t >= ntiles) return false;
    tl.t0 = (t % tiles_t) * size;
    const int slab = t / tiles_t;
    tl.bb = slab / N;
    tl.nn = slab % N;
    return true;
}
__device__ __forceinline__ const short *bseq(const View &v, const BTile &tl) {
    return static_cast<const short *>(v.ptr) + tl.bb * v.sb + tl.nn * v.sn;
}
// window of position t: keys [band_lo, band_hi)
__device__ __forceinline__ int band_lo(int t, int T, int k, int causal) { return axis_start(t, T, k, causal); }
__device__ __forceinline__ int band_hi(int t, int T, int k, int causal) {
    return causal ? t + 1 : win_start(t, T, k) + k;
}
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// eight float32 values as the sum of two vectors of 16-bit ones
template <bool BF>
__device__ __forceinline__ void split16(const float (&x)[8], s16x8 &hi, s16x8 &lo) {
#pragma unroll
    for (int e = 0; e < 8; e++) {
        hi[e] = cvt16<BF>(x[e]);
        lo[e] = cvt16<BF>(x[e] - cvt32<BF>(hi[e]));
    }
}
// rows of an operand straight from global memory
template <int DS, bool NARROW>
__device__ __forceinline__ void load_row(s16x8 (&reg)[DS], const short *row, int g, int dlim) {
    if constexpr (NARROW) {
        load_row_chunks(reg, row, g, dlim);
    } else {
#pragma unroll
        for (int ds = 0; ds < DS; ds++) reg[ds] = *reinterpret_cast<const s16x8 *>(row + ds * 32 + g * 8);
    }
}

// ---- results that are not finite
// A matrix instruction multiplies every staged row by every weight, and zero times an infinity or
// a NaN is NaN: such a value in a position that a query does not see (the future of a causal
// sequence) would reach the query's result through its zero probability, and a dS beyond float16
// would as infinity minus infinity.  So each wave looks at its results before it stores them (one
// instruction per value, once a tile) and computes the tokens with a value that is not finite
// again, one after the other, from the rows in their windows alone, in float32.
// Queries whose logits lie beyond kFar take the same way: log2 and natural units do not convert
// into each other closely enough there for probabilities out of a log-sum-exp, so these are computed in
// natural units throughout, as by the general kernels.
constexpr float kFar = 1048576.f;
__device__ __forceinline__ bool far(float lse) { return !(fabsf(lse) <= kFar); }  // (also NaN)
__device__ __forceinline__ float exp_neg(float x) { return __builtin_amdgcn_exp2f(x * kLog2e); }
// ------------------------------------------------------------------ forward
// Blocks of 32 keys: 35 KB of LDS and, with half of the staging registers, 119 to 124 in all, so that four workgroups
// share a CU instead of two (145 registers, 70 KB).  The steps of 32 keys and their order are the same: so are the results.
template <bool BF, int D, int NQ, bool NARROW, int KB>
__global__ __launch_bounds__(256, (KB == 32 ? 4 : 2)) void fwd_band_mfma(FwdArgs a, int tiles_t, int ntiles) {
    using G = BGeo<D, KB>;
    __shared__ __attribute__((aligned(16))) short lds_k[2][KB * G::PITCH];
    __shared__ __attribute__((aligned(16))) short lds_v[2][KB * G::PITCH];
    const Shape &s = a.s;
    const int T = s.W, k = s.kw, causal = s.cw, dlim = NARROW ? s.D : D;
    BTile tl;
    if (!btile(blockIdx.x, gridDim.x, ntiles, tiles_t, 64 * NQ, s.N, tl)) return;
    const int wave = uni(threadIdx.x >> 6), l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const float sc2 = s.scale * kLog2e;

    const short *kseq = bseq(a.k, tl), *vseq = bseq(a.v, tl), *qseq = bseq(a.q, tl);
    const int ka = band_lo(tl.t0, T, k, causal), kb = band_hi(min(tl.t0 + 64 * NQ, T) - 1, T, k, causal);
    Block<D, KB, NARROW> kst, vst;
    kst.fetch(kseq, a.k.sw, ka, T, dlim);
    vst.fetch(vseq, a.v.sw, ka, T, dlim);

    // this wave's queries and the keys they see between them
    const int w0 = tl.t0 + wave * 16 * NQ;
    const bool on = w0 < T;
    const int wa = band_lo(min(w0, T - 1), T, k, causal), wb = band_hi(min(w0 + 16 * NQ, T) - 1, T, k, causal);
    s16x8 qreg[NQ][G::DS];
    int lo[NQ], cnt[NQ], in_lo[NQ], in_hi[NQ];  // this lane's window; the keys that all 16 queries see
    f32x4 o[NQ][G::DT];
    float m[NQ], sum[NQ];
#pragma unroll
    for (int u = 0; u < NQ; u++) {
        const int qt = min(w0 + u * 16 + n, T - 1);
        load_row<G::DS, NARROW>(qreg[u], qseq + qt * a.q.sw, g, dlim);
        lo[u] = band_lo(qt, T, k, causal);
        cnt[u] = band_hi(qt, T, k, causal) - lo[u];
        in_lo[u] = band_lo(min(w0 + u * 16 + 15, T - 1), T, k, causal);
        in_hi[u] = band_hi(min(w0 + u * 16, T - 1), T, k, causal);
#pragma unroll
        for (int t = 0; t < G::DT; t++) o[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        m[u] = -__FLT_MAX__;
        sum[u] = 0.f;
    }
    kst.commit(lds_k[0]);
    vst.commit(lds_v[0]);
    __syncthreads();

    for (int k0 = ka, buf = 0; k0 < kb; k0 += KB, buf ^= 1) {
        const bool more = k0 + KB < kb;
        if (more) {
            kst.fetch(kseq, a.k.sw, k0 + KB, T, dlim);
            vst.fetch(vseq, a.v.sw, k0 + KB, T, dlim);
        }
        const short *lk = lds_k[buf], *lv = lds_v[buf];
#pragma unroll
        for (int st = 0; st < KB / 32; st++) {
            const int kk = k0 + st * 32;
            if (!on || kk >= wb || kk + 32 <= wa) continue;  // (the same for the whole wave)
            f32x4 c[NQ][2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const short *kp = lk + (st * 32 + h * 16 + n) * G::PITCH + g * 8;
#pragma unroll
                for (int u = 0; u < NQ; u++) c[u][h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ds = 0; ds < G::DS; ds++) {
                    const s16x8 kr = *reinterpret_cast<const s16x8 *>(kp + ds * 32);
#pragma unroll
                    for (int u = 0; u < NQ; u++) c[u][h] = mfma16<BF>(kr, qreg[u][ds], c[u][h]);
                }
            }
            s16x8 ph[NQ], pl[NQ];
#pragma unroll
            for (int u = 0; u < NQ; u++) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; e++) x[e] = c[u][e >> 2][e & 3] * sc2;
                if (kk < in_lo[u] || kk + 32 > in_hi[u]) {
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const int key = kk + (e >> 2) * 16 + g * 4 + (e & 3);
                        x[e] = (unsigned)(key - lo[u]) < (unsigned)cnt[u] ? x[e] : -INFINITY;
                    }
                }
                const float mx = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])),
                                       fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
                if (__any(mx > m[u] + 8.f)) {
                    const float mn = fmaxf(m[u], col_max(mx)), corr = __builtin_amdgcn_exp2f(m[u] - mn);
                    m[u] = mn;
                    sum[u] *= corr;
#pragma unroll
                    for (int t = 0; t < G::DT; t++) o[u][t] *= corr;
                }
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    x[e] = __builtin_amdgcn_exp2f(x[e] - m[u]);
                    sum[u] += x[e];
                }
                split16<BF>(x, ph[u], pl[u]);
            }
            const short *vp[2];
#pragma unroll
            for (int h = 0; h < 2; h++)
                vp[h] = lv + (st * 32 + h * 16 + g * 4 + (n >> 2)) * G::PITCH + (n & 3) * (D / 4);
#pragma unroll
            for (int t = 0; t < G::DT; t++) {
                const s16x8 vt = cat(lds_read_tr(vp[0] + t * 4), lds_read_tr(vp[1] + t * 4));
#pragma unroll
                for (int u = 0; u < NQ; u++) {
                    o[u][t] = mfma16<BF>(vt, ph[u], o[u][t]);
                    o[u][t] = mfma16<BF>(vt, pl[u], o[u][t]);
                }
            }
        }
        if (more) {
            kst.commit(lds_k[buf ^ 1]);
            vst.commit(lds_v[buf ^ 1]);
        }
        __syncthreads();
    }
    if (!on) return;
    short *oseq = const_cast<short *>(bseq(a.o, tl));
#pragma unroll
    for (int u = 0; u < NQ; u++) {
        const int q0 = w0 + u * 16 + n, qt = min(q0, T - 1);
        const bool live = q0 < T;
        const float total = col_sum(sum[u]);
        unsigned bad = bad_columns(o[u], far(m[u]) ? INFINITY : total);
        const bool here = live && !(bad >> n & 1);
        store_token<BF, D, (D >= 64 && !NARROW)>(oseq + qt * a.o.sw, g, o[u], 1.f / total, here, dlim);
        if (a.lse && here && g == 0)
            a.lse[((int64_t)tl.bb * s.N + tl.nn) * T + qt] = (m[u] + __builtin_amdgcn_logf(total)) * kLn2;
        for (; bad; bad &= bad - 1) {
            const int t = w0 + u * 16 + __builtin_ctz(bad);
            if (t >= T) break;
            const Chan2 q = chan_load<BF>(qseq + t * a.q.sw, dlim);
            Chan2 acc{0.f, 0.f};
            float mx = -INFINITY, z = 0.f;
            for (int key = band_lo(t, T, k, causal); key < band_hi(t, T, k, causal); key++) {
                const float x = chan_dot(q, chan_load<BF>(kseq + key * a.k.sw, dlim)) * s.scale;
                const float mn = x > mx ? x : mx, corr = exp_neg(mx - mn), p = exp_neg(x - mn);
                mx = mn;
                z = z * corr + p;
                acc.a *= corr;
                acc.b *= corr;
                chan_add(acc, p, chan_load<BF>(vseq + key * a.v.sw, dlim));
                if (z != z) break;  // nothing finite can come of it
            }
            chan_store<BF>(oseq + t * a.o.sw, dlim, acc, 1.f / z);
            if (a.lse && l == 0)
                a.lse[((int64_t)tl.bb * s.N + tl.nn) * T + t] = mx + __builtin_amdgcn_logf(z) * kLn2;
        }
    }
}

// ------------------------------------------------------------------ dQ
// The forward's walk with P from the saved log-sum-exp, dP^T = V dO^T, dS = P (dP - delta),
// dQ^T += K^T dS^T, and the sums that correct delta = dO . O (see the top of the file).  sum p k
// takes P rounded to 16 bits: what it multiplies is of the size of O's rounding.
template <bool BF, int D, bool NARROW>
__global__ __launch_bounds__(256, 2) void bwd_band_dq_mfma(BwdArgs a, int tiles_t, int ntiles) {
    constexpr int KB = kRowsQ;
    using G = BGeo<D, KB>;
    __shared__ __attribute__((aligned(16))) short lds_k[2][KB * G::PITCH];
    __shared__ __attribute__((aligned(16))) short lds_v[2][KB * G::PITCH];
    const Shape &s = a.s;
    const int T = s.W, k = s.kw, causal = s.cw, dlim = NARROW ? s.D : D;
    BTile tl;
    if (!btile(blockIdx.x, gridDim.x, ntiles, tiles_t, 64, s.N, tl)) return;
    const int wave = uni(threadIdx.x >> 6), l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const float sc2 = s.scale * kLog2e;

    const short *kseq = bseq(a.k, tl), *vseq = bseq(a.v, tl);
    const int ka = band_lo(tl.t0, T, k, causal), kb = band_hi(min(tl.t0 + 64, T) - 1, T, k, causal);
    Block<D, KB, NARROW> kst, vst;
    kst.fetch(kseq, a.k.sw, ka, T, dlim);
    vst.fetch(vseq, a.v.sw, ka, T, dlim);

    const int w0 = tl.t0 + wave * 16;
    const bool on = w0 < T;
    const int wa = band_lo(min(w0, T - 1), T, k, causal), wb = band_hi(min(w0 + 16, T) - 1, T, k, causal);
    const int64_t tok0 = ((int64_t)tl.bb * s.N + tl.nn) * T;
    s16x8 qreg[G::DS], greg[G::DS];
    int lo, cnt, in_lo, in_hi;
    f32x4 dq[G::DT], pk[G::DT];
    float lse2, delta, zsum, esum;
    DsScale<BF> scl;
    const int qt = min(w0 + n, T - 1);
    load_row<G::DS, NARROW>(qreg, bseq(a.q, tl) + qt * a.q.sw, g, dlim);
    load_row<G::DS, NARROW>(greg, bseq(a.d_o, tl) + qt * a.d_o.sw, g, dlim);
    s16x8 orow[G::DS];
    load_row<G::DS, NARROW>(orow, bseq(a.o, tl) + qt * a.o.sw, g, dlim);
    const float lse = a.lse[tok0 + qt];
    lse2 = far(lse) ? NAN : lse * kLog2e;  // (the whole column is then computed again)
    zsum = esum = 0.f;
    lo = band_lo(qt, T, k, causal);
    cnt = band_hi(qt, T, k, causal) - lo;
    in_lo = band_lo(min(w0 + 15, T - 1), T, k, causal);
    in_hi = band_hi(min(w0, T - 1), T, k, causal);
    float d = 0.f;
#pragma unroll
    for (int ds = 0; ds < G::DS; ds++)
        d += dot8<BF>(__builtin_bit_cast(u32x4, greg[ds]), __builtin_bit_cast(u32x4, orow[ds]));
    delta = col_sum(d);
#pragma unroll
    for (int t = 0; t < G::DT; t++) {
        dq[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        pk[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    kst.commit(lds_k[0]);
    vst.commit(lds_v[0]);
    __syncthreads();

    for (int k0 = ka, buf = 0; k0 < kb; k0 += KB, buf ^= 1) {
        const bool more = k0 + KB < kb;
        if (more) {
            kst.fetch(kseq, a.k.sw, k0 + KB, T, dlim);
            vst.fetch(vseq, a.v.sw, k0 + KB, T, dlim);
        }
        const short *lk = lds_k[buf], *lv = lds_v[buf];
#pragma unroll
        for (int st = 0; st < KB / 32; st++) {
            const int kk = k0 + st * 32;
            if (!on || kk >= wb || kk + 32 <= wa) continue;
            f32x4 c[2], cp[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int row = (st * 32 + h * 16 + n) * G::PITCH + g * 8;
                c[h] = f32x4{0.f, 0.f, 0.f, 0.f};
                cp[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ds = 0; ds < G::DS; ds++) {
                    const s16x8 kr = *reinterpret_cast<const s16x8 *>(lk + row + ds * 32);
                    const s16x8 vr = *reinterpret_cast<const s16x8 *>(lv + row + ds * 32);
                    c[h] = mfma16<BF>(kr, qreg[ds], c[h]);
                    cp[h] = mfma16<BF>(vr, greg[ds], cp[h]);
                }
            }
            s16x8 sh, sl, ph;
            float x[8], mag = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = c[e >> 2][e & 3] * sc2 - lse2;
            if (kk < in_lo || kk + 32 > in_hi) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const int key = kk + (e >> 2) * 16 + g * 4 + (e & 3);
                    x[e] = (unsigned)(key - lo) < (unsigned)cnt ? x[e] : -INFINITY;
                }
            }
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float p = __builtin_amdgcn_exp2f(x[e]);
                x[e] = p * (cp[e >> 2][e & 3] - delta);
                zsum += p;
                esum += x[e];
                ph[e] = cvt16<BF>(p);
                if (!BF) mag = fmaxf(mag, fabsf(x[e]));
            }
            if constexpr (!BF) {
                scl.fit(mag, dq);
                const float f = scl.factor();
#pragma unroll
                for (int e = 0; e < 8; e++) x[e] *= f;
            }
            split16<BF>(x, sh, sl);
            const short *kp[2];
#pragma unroll
            for (int h = 0; h < 2; h++)
                kp[h] = lk + (st * 32 + h * 16 + g * 4 + (n >> 2)) * G::PITCH + (n & 3) * (D / 4);
#pragma unroll
            for (int t = 0; t < G::DT; t++) {
                const s16x8 kt = cat(lds_read_tr(kp[0] + t * 4), lds_read_tr(kp[1] + t * 4));
                dq[t] = mfma16<BF>(kt, sh, dq[t]);
                pk[t] = mfma16<BF>(kt, ph, pk[t]);
                dq[t] = mfma16<BF>(kt, sl, dq[t]);
            }
        }
        if (more) {
            kst.commit(lds_k[buf ^ 1]);
            vst.commit(lds_v[buf ^ 1]);
        }
        __syncthreads();
    }
    if (!on) return;
    const float zinv = 1.f / col_sum(zsum), shift = col_sum(esum) * zinv;
#pragma unroll
    for (int t = 0; t < G::DT; t++) dq[t] = dq[t] * scl.inverse() - shift * pk[t];
    unsigned bad = bad_columns(dq, zinv);
    const bool here = w0 + n < T && !(bad >> n & 1);
    store_token<BF, D, (D >= 64 && !NARROW)>(static_cast<short *>(a.dq) + a.grad_at(tl.bb, tl.nn, 0, qt), g,
                                             dq, s.scale * zinv, here, dlim);
    if (here && g == 0) {
        a.delta[tok0 + qt] = delta + shift;
        a.zinv[tok0 + qt] = zinv;
    }
    for (; bad; bad &= bad - 1) {
        const int col = __builtin_ctz(bad), t = w0 + col;
        if (t >= T) break;
        const Chan2 q = chan_load<BF>(bseq(a.q, tl) + t * a.q.sw, dlim);
        const Chan2 go = chan_load<BF>(bseq(a.d_o, tl) + t * a.d_o.sw, dlim);
        const float lse_t = a.lse[tok0 + t], delta_t = __shfl(delta, col, 64);
        Chan2 acc{0.f, 0.f}, accp{0.f, 0.f};
        float z = 0.f, res = 0.f;
        for (int key = band_lo(t, T, k, causal); key < band_hi(t, T, k, causal); key++) {
            const Chan2 kr = chan_load<BF>(kseq + key * a.k.sw, dlim);
            const float p = exp_neg(chan_dot(q, kr) * s.scale - lse_t);
            const float y = p * (chan_dot(go, chan_load<BF>(vseq + key * a.v.sw, dlim)) - delta_t);
            z += p;
            res += y;
            chan_add(acc, y, kr);
            chan_add(accp, p, kr);
            if (z != z) break;  // nothing finite can come of it
        }
        const float sh_t = res / z;
        chan_add(acc, -sh_t, accp);
        chan_store<BF>(static_cast<short *>(a.dq) + a.grad_at(tl.bb, tl.nn, 0, t), dlim, acc, s.scale / z);
        if (l == 0) {
            a.delta[tok0 + t] = delta_t + sh_t;
            a.zinv[tok0 + t] = 1.f / z;
        }
    }
}

// ------------------------------------------------------------------ dK, dV
// The tile is 64 keys, 16 per wave (columns), and the walk is over the queries
// that see any of them, the inverse neighbourhood (e_natten/pytorch.py:13-23), a block at a time: Q
// and dO rows, the log-sum-exp, delta and 1 / Z of a block in LDS.  dV^T += dO^T P, dK^T += Q^T dS.
// head_dim 64 takes 128 to 152 registers without a budget, four waves per SIMD have 128 (20 bytes of scratch in float16 below
// 64): causal, us, float16 B4 N8 T8192 d64 k64 54.3 -> 48.7, B2 N16 T4096 k256 52.1 -> 45.6; B4 N8 T8192 d48 k128 60.5 -> 52.5,
// float16 64.6 -> 57.3; bf16 d64 level.  The dQ pass spills in four (d48 k128 44.6 -> 54.6) or, in blocks of 32 keys, gains only in bf16
// on many tiles (43.7 -> 43.0; float16 36.8 -> 40.6).
template <bool BF, int D, bool NARROW, int WAVES = D == 64 ? 4 : 2>
__global__ __launch_bounds__(256, WAVES) void bwd_band_dkdv_mfma(BwdArgs a, int tiles_t, int ntiles) {
    constexpr int KB = kRowsK<D>;
    using G = BGeo<D, KB>;
    __shared__ __attribute__((aligned(16))) short lds_q[2][KB * G::PITCH];
    __shared__ __attribute__((aligned(16))) short lds_g[2][KB * G::PITCH];
    __shared__ __attribute__((aligned(16))) float lds_stat[2][3][KB];  // lse * log2e, delta, kPScale / Z
    const Shape &s = a.s;
    const int T = s.W, k = s.kw, causal = s.cw, dlim = NARROW ? s.D : D;
    BTile tl;
    if (!btile(blockIdx.x, gridDim.x, ntiles, tiles_t, 64, s.N, tl)) return;
    const int wave = uni(threadIdx.x >> 6), l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const float sc2 = s.scale * kLog2e;

    const short *qseq = bseq(a.q, tl), *gseq = bseq(a.d_o, tl);
    const int64_t tok0 = ((int64_t)tl.bb * s.N + tl.nn) * T;
    const int qa = axis_inv_lo(tl.t0, k, causal), qb = axis_inv_hi(min(tl.t0 + 64, T) - 1, T, k, causal);
    Block<D, KB, NARROW> qst, gst;
    float sst[3] = {0.f, 0.f, 0.f};
    auto fetch = [&](int p0) __attribute__((always_inline)) {
        qst.fetch(qseq, a.q.sw, p0, T, dlim);
        gst.fetch(gseq, a.d_o.sw, p0, T, dlim);
        if (threadIdx.x < KB) {
            const int64_t at = tok0 + min(p0 + (int)threadIdx.x, T - 1);
            const float lse = a.lse[at];
            sst[0] = far(lse) ? NAN : lse * kLog2e;  // (the keys that this query sees are then computed again)
            sst[1] = a.delta[at];
            sst[2] = a.zinv[at] * kPScale<BF>;
        }
    };
    auto commit = [&](int buf) __attribute__((always_inline)) {
        qst.commit(lds_q[buf]);
        gst.commit(lds_g[buf]);
        if (threadIdx.x < KB) {
#pragma unroll
            for (int j = 0; j < 3; j++) lds_stat[buf][j][threadIdx.x] = sst[j];
        }
    };
    fetch(qa);

    const int w0 = tl.t0 + wave * 16;
    const bool on = w0 < T;
    const int wa = axis_inv_lo(min(w0, T - 1), k, causal), wb = axis_inv_hi(min(w0 + 16, T) - 1, T, k, causal);
    s16x8 kreg[G::DS], vreg[G::DS];
    f32x4 dk[G::DT], dv[G::DT];
    DsScale<BF> scl;
    const int kt = min(w0 + n, T - 1);  // this lane's key
    load_row<G::DS, NARROW>(kreg, bseq(a.k, tl) + kt * a.k.sw, g, dlim);
    load_row<G::DS, NARROW>(vreg, bseq(a.v, tl) + kt * a.v.sw, g, dlim);
#pragma unroll
    for (int t = 0; t < G::DT; t++) {
        dk[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        dv[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    commit(0);
    __syncthreads();

    for (int p0 = qa, buf = 0; p0 < qb; p0 += KB, buf ^= 1) {
        const bool more = p0 + KB < qb;
        if (more) fetch(p0 + KB);
        const short *lq = lds_q[buf], *lg = lds_g[buf];
#pragma unroll
        for (int st = 0; st < KB / 32; st++) {
            const int qq = p0 + st * 32;
            if (!on || qq >= wb || qq + 32 <= wa) continue;
            f32x4 c[2], cp[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int row = (st * 32 + h * 16 + n) * G::PITCH + g * 8;
                c[h] = f32x4{0.f, 0.f, 0.f, 0.f};
                cp[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ds = 0; ds < G::DS; ds++) {
                    const s16x8 qr = *reinterpret_cast<const s16x8 *>(lq + row + ds * 32);
                    const s16x8 gr = *reinterpret_cast<const s16x8 *>(lg + row + ds * 32);
                    c[h] = mfma16<BF>(qr, kreg[ds], c[h]);
                    cp[h] = mfma16<BF>(gr, vreg[ds], cp[h]);
                }
            }
            f32x4 sv[3][2];
#pragma unroll
            for (int j = 0; j < 3; j++)
#pragma unroll
                for (int h = 0; h < 2; h++)
                    sv[j][h] = *reinterpret_cast<const f32x4 *>(&lds_stat[buf][j][st * 32 + h * 16 + g * 4]);
            // the keys that all 32 queries of the step see
            const int in_lo = band_lo(min(qq + 31, T - 1), T, k, causal), in_hi = band_hi(qq, T, k, causal);
            s16x8 ph, pl, sh, sl;
            float x[8], y[8], mag = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = c[e >> 2][e & 3] * sc2 - sv[0][e >> 2][e & 3];
            if (w0 < in_lo || w0 + 16 > in_hi || qq + 32 > T) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    // (causal: the key is one of the query and the k - 1 positions before it)
                    const int q = qq + (e >> 2) * 16 + g * 4 + (e & 3), key = w0 + n;
                    const unsigned at = causal ? q - key : key - win_start(q, T, k);
                    x[e] = at < (unsigned)k && q < T ? x[e] : -INFINITY;
                }
            }
#pragma unroll
            for (int e = 0; e < 8; e++) {
                x[e] = __builtin_amdgcn_exp2f(x[e]) * sv[2][e >> 2][e & 3];
                y[e] = x[e] * (cp[e >> 2][e & 3] - sv[1][e >> 2][e & 3]);
                if (!BF) mag = fmaxf(mag, fabsf(y[e]));
            }
            if constexpr (!BF) {
                scl.fit(mag, dk);
                const float f = scl.factor();
#pragma unroll
                for (int e = 0; e < 8; e++) y[e] *= f;
            }
            split16<BF>(x, ph, pl);
            split16<BF>(y, sh, sl);
            const short *qp[2], *gp[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int row = (st * 32 + h * 16 + g * 4 + (n >> 2)) * G::PITCH + (n & 3) * (D / 4);
                qp[h] = lq + row;
                gp[h] = lg + row;
            }
#pragma unroll
            for (int t = 0; t < G::DT; t++) {
                const s16x8 gt = cat(lds_read_tr(gp[0] + t * 4), lds_read_tr(gp[1] + t * 4));
                const s16x8 qt = cat(lds_read_tr(qp[0] + t * 4), lds_read_tr(qp[1] + t * 4));
                dv[t] = mfma16<BF>(gt, ph, dv[t]);
                dk[t] = mfma16<BF>(qt, sh, dk[t]);
                dv[t] = mfma16<BF>(gt, pl, dv[t]);
                dk[t] = mfma16<BF>(qt, sl, dk[t]);
            }
        }
        if (more) commit(buf ^ 1);
        __syncthreads();
    }
    if (!on) return;
    const float unscale = scl.inverse() / kPScale<BF>;  // (powers of two)
#pragma unroll
    for (int t = 0; t < G::DT; t++) dk[t] *= unscale;
    unsigned bad = bad_columns(dk) | bad_columns(dv);
    const bool live = w0 + n < T && !(bad >> n & 1);
    const int64_t at = a.grad_at(tl.bb, tl.nn, 0, kt);
    store_token<BF, D, (D >= 64 && !NARROW)>(static_cast<short *>(a.dk) + at, g, dk, s.scale, live, dlim);
    store_token<BF, D, (D >= 64 && !NARROW)>(static_cast<short *>(a.dv) + at, g, dv, 1.f / kPScale<BF>, live, dlim);
    for (; bad; bad &= bad - 1) {
        const int key = w0 + __builtin_ctz(bad);
        if (key >= T) break;
        const Chan2 kr = chan_load<BF>(bseq(a.k, tl) + key * a.k.sw, dlim);
        const Chan2 vr = chan_load<BF>(bseq(a.v, tl) + key * a.v.sw, dlim);
        Chan2 ak{0.f, 0.f}, av{0.f, 0.f};
        for (int q = axis_inv_lo(key, k, causal); q < axis_inv_hi(key, T, k, causal); q++) {
            if ((unsigned)(key - band_lo(q, T, k, causal)) >= (unsigned)k) continue;
            const Chan2 qr = chan_load<BF>(qseq + q * a.q.sw, dlim), gr = chan_load<BF>(gseq + q * a.d_o.sw, dlim);
            const float p = exp_neg(chan_dot(qr, kr) * s.scale - a.lse[tok0 + q]) * a.zinv[tok0 + q];
            chan_add(av, p, gr);
            chan_add(ak, p * (chan_dot(gr, vr) - a.delta[tok0 + q]), qr);
            if (p != p) break;  // nothing finite can come of it
        }
        const int64_t to = a.grad_at(tl.bb, tl.nn, 0, key);
        chan_store<BF>(static_cast<short *>(a.dk) + to, dlim, ak, s.scale);
        chan_store<BF>(static_cast<short *>(a.dv) + to, dlim, av, 1.f);
    }
}

// ------------------------------------------------------------------ dispatch
// Two groups of 16 queries per wave (forward) where the walk is long, a key row is 256 bytes, and
// tiles of that size still give every CU its two workgroups: the LDS reads of a step then feed twice the
// matrix instructions.  One group in blocks of 32 keys / two, us, causal, head_dim 128: B2 N32 T8192 k256 172 / 199, k512
// 268 / 272, k1024 463 / 441, k2500 956 / 863; B2 N8 T4096 k400 32.5 / 33.3, k512 38.6 / 37.4; B1 N16 T4096 k2000 114 / 103.
// head_dim 64 B2 N16 T4096 k256 25.7 / 33.5: there more waves count for more.  Not in the dQ pass: its third product takes the
// registers that a second group needs (with two, B2 N32 T8192 d128 k512 spills and its backward
// takes 1432 us instead of 1005), nor in the dK/dV pass (head_dim 64: 108 / 151).
bool two_groups(const Shape &s) {
    return s.D == 128 && s.kw >= 512 && (int64_t)s.B * s.N * ((s.W + 127) / 128) >= 512;
}
// The forward above head_dim 64 in blocks of 32 keys: where there are more tiles than the two workgroups per CU of
// the blocks of 64 take at once; fewer only pay for the barriers.  Blocks of 64 / 32, us: B1 N16 T8192 d128 k200 causal
// 46.7 / 42.0, k128 on views of one projection, the call, 42.4 / 36.8, k91 centred 35.9 / 33.1; B1 N16 T3000 k400 (752 tiles) 32.7 / 26.0;
// B3 N4 T3000 k20 (564) 11.8 / 9.1; B2 N8 T8192 d96 k512 77 / 67, B3 N7 T2500 d80 k20 12.1 / 9.0; B1 N16 T2000 k128 (512) 10.2 / 10.0,
// B1 N7 T3001 k250 (329) 12.4 / 13.6, B1 N4 T4096 k1024 (256) 26.0 / 27.4.
bool short_blocks(const Shape &s) { return (int64_t)s.B * s.N * ((s.W + 63) / 64) > 512; }
// The dK/dV pass of head dims 40 to 56 in float16, whose build for four waves per SIMD has 20 bytes of scratch: up to as many tiles as
// three workgroups on each of the 256 CUs take at once there is nothing to run in the fourth, and the build without that budget is
// ahead by 2% of the backward in the mean of 28 calls each of d40 and d56, 128 to 768 tiles, windows of 16 to 401 (B4 N8 T800 d40 k101
// 24.6 -> 24.0 us).  With 812 to 2970 tiles four are ahead by 5%.  Bf16 and head_dim 64 are level up to 768.
constexpr int64_t kThreePerCu = 768;
int band_grid(int64_t ntiles) { return (int)((ntiles + 7) / 8 * 8); }

template <bool BF, int D, int NQ, bool NARROW, int KB = kRowsQ>
int fwd_go(const FwdArgs &a, hipStream_t st) {
    const int tiles_t = (a.s.W + 64 * NQ - 1) / (64 * NQ);
    const int64_t nt = (int64_t)a.s.B * a.s.N * tiles_t;
    {
        ProfScope prof(ENATTEN_KERNEL_FWD, "fwd_band_mfma", st);
        hipLaunchKernelGGL((fwd_band_mfma<BF, D, NQ, NARROW, KB>), dim3(band_grid(nt)), dim3(256), 0, st, a, tiles_t,
                           (int)nt);
    }
    return check_launch("fwd_band_mfma");
}
template <bool BF, int D, bool NARROW>
int bwd_go(const BwdArgs &a, hipStream_t st) {
    const int tiles_t = (a.s.W + 63) / 64;
    const int64_t nt = (int64_t)a.s.B * a.s.N * tiles_t;
    {
        ProfScope prof(ENATTEN_KERNEL_BWD_DQ, "bwd_band_dq_mfma", st);
        hipLaunchKernelGGL((bwd_band_dq_mfma<BF, D, NARROW>), dim3(band_grid(nt)), dim3(256), 0, st, a, tiles_t,
                           (int)nt);
    }
    {
        ProfScope prof(ENATTEN_KERNEL_BWD_DKDV, "bwd_band_dkdv_mfma", st);
        const auto kernel = !BF && NARROW && D == 64 && nt <= kThreePerCu ? bwd_band_dkdv_mfma<BF, D, NARROW, 2>
                                                                          : bwd_band_dkdv_mfma<BF, D, NARROW>;
        hipLaunchKernelGGL(kernel, dim3(band_grid(nt)), dim3(256), 0, st, a, tiles_t, (int)nt);
    }
    return check_launch("bwd_band_mfma");
}

bool band_layout_ok(const View &v) {
    return reinterpret_cast<uintptr_t>(v.ptr) % 16 == 0 && v.sb % 8 == 0 && v.sn % 8 == 0 && v.sw % 8 == 0 &&
           v.sw < (1 << 22);
}
// The smallest window that is taken here.  A tile walks at least two blocks of 64 keys (three of 32), however few of them its
// windows hold, and narrow heads give the matrix instructions little to do.  us, general kernels / here, causal, B4 N8
// T16384 bf16, forward and backward: d8 k6 34 / 37, 80 / 106, k12 58 / 37, 131 / 104; d16 k4 32 / 36, 81 / 107, k8 46 / 36,
// 109 / 107; d24 k4 40 / 53, 116 / 141, k8 59 / 53, 163 / 141; d32 k3 36 / 37, 110 / 116, k4 40 / 37, 123 / 117; d48 k2 52 / 77,
// 193 / 208, k4 70 / 77, 247 / 207, k6 87 / 77; d64 k2 61 / 50, 238 / 158.
// (Not windows of one key, whose probability is 1: dP - delta must cancel to an exact zero, which
// takes the two sums in one order, as in the general kernels.)
int least_window(int D, bool backward) {
    if (D >= 64) return 2;
    if (D > 32) return backward ? 3 : 6;
    if (D == 32) return 4;
    return D <= 8 ? (backward ? 12 : 8) : D <= 16 ? (backward ? 8 : 6) : 8;
}
bool band_shape_ok(const Shape &s, int dtype, bool backward) {
    return (dtype == ENATTEN_BF16 || dtype == ENATTEN_F16) && s.D >= 8 && s.D <= 128 && s.D % 8 == 0 &&
           s.kw >= least_window(s.D, backward) && s.H == 1 && s.kh == 1 &&
           (int64_t)s.B * s.N * ((s.W + 63) / 64) <= ((int64_t)1 << 32) / 256 - 8;  // (threads of a launch)
}

}  // namespace

bool band_supported(const FwdArgs &a, int dtype) {
    return band_shape_ok(a.s, dtype, false) && !a.rpb && band_layout_ok(a.q) && band_layout_ok(a.k) &&
           band_layout_ok(a.v) && band_layout_ok(a.o);
}
bool band_supported(const BwdArgs &a, int dtype) {
    auto al = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    return band_shape_ok(a.s, dtype, true) && !a.rpb && band_layout_ok(a.q) && band_layout_ok(a.k) &&
           band_layout_ok(a.v) && band_layout_ok(a.o) && band_layout_ok(a.d_o) && al(a.dq) && al(a.dk) &&
           al(a.dv) && a.gsb % 8 == 0 && a.gsn % 8 == 0 && a.gsw % 8 == 0;
}
template <bool BF>
int fwd_dim(const FwdArgs &a, hipStream_t st) {
    switch (a.s.D) {
        case 32: return fwd_go<BF, 32, 1, false>(a, st);
        case 64: return fwd_go<BF, 64, 1, false>(a, st);
        case 128:
            return two_groups(a.s)    ? fwd_go<BF, 128, 2, false>(a, st)
                   : short_blocks(a.s) ? fwd_go<BF, 128, 1, false, 32>(a, st) : fwd_go<BF, 128, 1, false>(a, st);
    }
    return a.s.D < 32   ? fwd_go<BF, 32, 1, true>(a, st)
           : a.s.D < 64 ? fwd_go<BF, 64, 1, true>(a, st)
           : short_blocks(a.s) ? fwd_go<BF, 128, 1, true, 32>(a, st) : fwd_go<BF, 128, 1, true>(a, st);
}
template <bool BF>
int bwd_dim(const BwdArgs &a, hipStream_t st) {
    switch (a.s.D) {
        case 32: return bwd_go<BF, 32, false>(a, st);
        case 64: return bwd_go<BF, 64, false>(a, st);
        case 128: return bwd_go<BF, 128, false>(a, st);
    }
    return a.s.D < 32 ? bwd_go<BF, 32, true>(a, st) : a.s.D < 64 ? bwd_go<BF, 64, true>(a, st) : bwd_go<BF, 128, true>(a, st);
}
int launch_fwd_band(const FwdArgs &a, int dtype, hipStream_t st) {
    return dtype == ENATTEN_BF16 ? fwd_dim<true>(a, st) : fwd_dim<false>(a, st);
}
int launch_bwd_band(const BwdArgs &a, int dtype, hipStream_t st) {
    return dtype == ENATTEN_BF16 ? bwd_dim<true>(a, st) : bwd_dim<false>(a, st);
}

}  // namespace enatten
