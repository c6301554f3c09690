// Matrix-core (MFMA) kernels for 2D neighborhood attention on gfx950.
//
// Geometry shared by all three kernels: a workgroup of four waves owns an 8x8
// tile of pixels of one (batch, head) image; each wave owns a 4x4 block of it.
// The 16 pixels of a wave are the N dimension of v_mfma_f32_16x16x32; the
// (4+k-1)^2 pixels of the block's halo are the other token dimension.  With the
// tokens of the halo as MFMA rows, every lane holds the logits of ONE query
// (column l%16) for several keys, so the softmax statistics need no transposes
// and the probabilities feed the second MFMA straight from the accumulators:
// the reduction index of the second product is enumerated in the order the
// accumulators hold it (slot e of lane group g <-> halo token 32*ks + 16*(e/4) +
// 4*g + e%4), and the other operand is fetched from LDS in that same order.
// That operand (V for O, K for dQ, dO/Q for dV/dK) is needed token-major while
// LDS holds it channel-major; ds_read_b64_tr_b16 does the transpose on the way
// out of LDS.  Output channels are likewise permuted (MFMA row g*4+i <-> channel
// g*D/4 + mt*4 + i) so that each lane ends up with D/4 contiguous channels of its
// query and writes them with 16-byte stores.
//
// Scheduling: the kernels are persistent.  Each workgroup walks a strided list
// of tiles and, while it computes one tile out of LDS, the global loads of the
// next tile's halo are already in flight into registers; they are written to LDS
// after the barrier that ends the current tile.  HBM latency is thus hidden
// behind compute even when LDS only admits one or two workgroups per CU.
//
// Forward follows e_natten/triton.py:242-302 per query (window start, mask,
// softmax, P.V); the log-sum-exp is kept for the backward.
//
// This file is compiled twice, by na2d_mfma.hip and by na2d_mfma_narrow.hip, each of
// which defines `enatten::(anonymous)::kNarrow` before including it.  false: the tensors'
// head dim IS the D a kernel is built for (32, 64, 128), and nothing below costs an
// instruction.  true: the head dim is any multiple of 8 up to D; the channels a tensor
// does not have are zero in LDS and in the operand registers and are left out of the
// stores (zero_row, HaloPlan::on, load_row_chunks, store_token in na2d_mfma.h).  One
// build serving both was measured 5-40% slower on the exact head dims (the predicates
// cost the large-halo kernels the registers they do not have).
//
// na2d_mfma_dilated.hip compiles it a third time with `kSub` true: the images are then the
// sub-grids of a dilated call (pixels of one residue class modulo the dilation on each axis,
// between which no query sees a key), all of one size, numbered batch, sub-grid row, sub-grid
// column, head.  The heads are innermost because in the layout of a projection they lie side by
// side in memory: a workgroup and its neighbours then read the same lines.  `kSub` false folds
// every one of these helpers to what it is without sub-grids.
//
// `kBias`: P and dS in two 16-bit terms, 1 / Z, results that are not finite computed again from their
// windows; with `kTable` (na2d_mfma_bias.hip) there is a relative position bias, without it
// (na2d_mfma_two_terms.hip) none.

#include <algorithm>

#include "na2d_mfma.h"

namespace enatten {
namespace {

// Whole-line stores (store_token's LINES) where a kernel runs at least two workgroups per CU
// on tensors of head_dim 128 or 64 itself (a token is then two aligned lines, or one).
// Measured, us, without -> with: d = 128 see store_token; d = 64 B4 N8 128x128 k5 forward 65.4 ->
// 61.4, dQ 67.8 -> 65.5, dK/dV 83.7 -> 76.1; B4 N4 256x256 k5 473 -> 427 per forward+backward;
// k7 284 -> 282; from k = 9 on the times do not change (343 -> 347, 281.4 -> 280.9 at k13: the
// kernels do not wait for their stores there), but the bytes do (dQ pass at d64 k13: 54.5 MB
// written for 34.6), so it is used at every kernel size.
// The dK/dV pass's inner tiles have no token outside the image, so their whole-line stores
// need no predicates (store_token's ALL), and without the branches that predicates put between
// the stores they pay at one workgroup per CU as well: dK/dV pass d128 k7 157.5 -> 154.6 us, k5
// 91.1 -> 88.7, d64 k5 82.1 -> 76.3, equal from k = 9 on.
template <int D>
constexpr bool kInnerLines = (D == 128 || D == 64) && !kNarrow;
template <int D, int KS, int WGS>
constexpr bool kLineStores = (D == 128 || D == 64) && !kNarrow && WGS >= 2;

// ------------------------------------------------------------------ images
using FArgs = std::conditional_t<kSub, FwdArgsSub, FwdArgs>;
using BArgs = std::conditional_t<kSub, BwdArgsSub, BwdArgs>;
struct SubTile : Tile {
    int ri, rj;  // sub-grid
};
using ATile = std::conditional_t<kSub, SubTile, Tile>;

// two tiles in one column of one image, the sub-grid included: a walk that hops from segment to
// segment may meet the same place of another sub-grid next
template <typename TL>
__device__ __forceinline__ bool same_column(const TL &x, const TL &y) {
    bool same = x.bb == y.bb && x.nn == y.nn && x.c0 == y.c0;
    if constexpr (kSub) same = same && x.ri == y.ri && x.rj == y.rj;
    return same;
}

// Images (one batch entry, head and sub-grid each) of a launch
template <typename ARGS>
int64_t images_of(const ARGS &a) {
    if constexpr (kSub) return (int64_t)a.s.B * a.s.N * a.sub_r * a.sub_c;
    else return (int64_t)a.s.B * a.s.N;
}
// tile_of and its like split an image number into (what is before the heads, head); with
// sub-grids the former is (batch, sub-grid row, sub-grid column)
template <typename ARGS, typename TL>
__device__ __forceinline__ void sub_grid(TL &tl, const ARGS &a) {
    tl.rj = tl.bb % a.sub_c; tl.bb /= a.sub_c;
    tl.ri = tl.bb % a.sub_r; tl.bb /= a.sub_r;
}
template <typename ARGS>
__device__ __forceinline__ ATile in_sub(Tile t, const ARGS &a) {
    ATile tl;
    static_cast<Tile &>(tl) = t;
    if constexpr (kSub) sub_grid(tl, a);
    return tl;
}
template <typename ARGS, typename TL>
__device__ __forceinline__ const short *image_at(const ARGS &a, const View &v, const TL &tl) {
    const short *p = image<short>(v, tl);
    if constexpr (kSub) p += tl.ri * v.sh + tl.rj * v.sw;
    return p;
}
// elements between pixels of an image that are one row / one column apart
template <typename ARGS>
__device__ __forceinline__ int64_t row_step(const ARGS &a, const View &v) {
    if constexpr (kSub) return v.sh * a.dil;
    else return v.sh;
}
template <typename ARGS>
__device__ __forceinline__ int64_t col_step(const ARGS &a, const View &v) {
    if constexpr (kSub) return v.sw * a.dil;
    else return v.sw;
}
template <typename ARGS, typename TL>
__device__ __forceinline__ int64_t grad_of(const ARGS &a, const TL &tl, int y, int x) {
    if constexpr (kSub) return a.grad_at(tl.bb, tl.nn, tl.ri + y * a.dil, tl.rj + x * a.dil);
    else return a.grad_at(tl.bb, tl.nn, y, x);
}
// place of an image's first query in the log-sum-exp and in the workspace
template <typename ARGS, typename TL>
__device__ __forceinline__ int64_t image_token(const ARGS &a, const TL &tl) {
    const Shape &s = a.s;
    int64_t b = tl.bb;
    if constexpr (kSub) b += (int64_t)(tl.ri * a.sub_c + tl.rj) * s.B;
    return (b * s.N + tl.nn) * s.H * (int64_t)s.W;
}
template <int KS, typename ARGS, typename TL>
__device__ __forceinline__ LaneQ lane_at(const ARGS &a, const TL &tl, int wave, int n) {
    LaneQ q = lane_query<KS>(tl, a.s, wave, n);
    if constexpr (kSub) q.tok = image_token(a, tl) + (int64_t)q.qr * a.s.W + q.qc;
    return q;
}

// ------------------------------------------------------------------ units of the logits
// Units of log2: one multiply less per logit.  With a bias natural units, as in the general kernels:
// a bias may be as low as its type goes (entries that are masked out), and there a log-sum-exp that goes
// through log2 and back is another number than the logits that it came from.
constexpr float kUnit = kBias ? 1.f : kLog2e;
__device__ __forceinline__ float exp_unit(float x) { return __builtin_amdgcn_exp2f(kBias ? x * kLog2e : x); }
__device__ __forceinline__ float lse_of(float mx, float sum) {
    if constexpr (kBias) return mx + __builtin_amdgcn_logf(sum) * kLn2;
    else return (mx + __builtin_amdgcn_logf(sum)) * kLn2;
}
// With a bias the backward is renormalised as in the general kernels: 1 / sum p of the recomputed
// probabilities per query, left by the dQ pass behind the block that holds its counter (a.zinv);
// without a table there is no counter, and the block itself has them.
constexpr bool kCounter = !kBias || kTable;
template <typename ARGS>
__device__ __forceinline__ float *row_zinv(const ARGS &a) {
    return a.zinv + (kCounter ? (int64_t)a.s.B * a.s.N * a.s.H * a.s.W : 0);
}
// (P in the float16 dK/dV pass, which 1 / Z brings along, as in na1d_band_mfma.hip: see DsScale)
template <bool BF>
constexpr float kPUnit = kBias ? kPScale<BF> : 1.f;
// what the dK/dV pass stages per query: the log-sum-exp in the logits' unit, delta, kPUnit / Z
using QStat = std::conditional_t<kBias, float4, float2>;
template <bool BF, bool BIAS = kBias>
__device__ __forceinline__ std::conditional_t<BIAS, float4, float2> load_qstat(const BArgs &a, int64_t qt) {
    if constexpr (BIAS) return make_float4(a.lse[qt], a.delta[qt], row_zinv(a)[qt] * kPUnit<BF>, 0.f);
    else return make_float2(a.lse[qt] * kLog2e, a.delta[qt]);
}
__device__ __forceinline__ float zinv_of(const float4 &st) { return st.z; }
__device__ __forceinline__ float zinv_of(const float2 &) { return 1.f; }

// ------------------------------------------------------------------ operands of the second products
// Eight probabilities (or dS) of a lane as an operand: rounded to 16 bits, or, with a bias, as the
// sum of two 16-bit terms (the value rounded, and what that left).  Calls with a bias used to run
// with float32 probabilities on the general kernels; two terms keep what they had (bf16: 16 bits
// of every probability, against the 8 bits of the results; float16: 22, for dS by DsScale).
struct TwoTerms {
    s16x8 hi, lo;
};
using Op8 = std::conditional_t<kBias, TwoTerms, s16x8>;
template <bool BF, typename OP>
__device__ __forceinline__ void put(OP &o, int e, float x) {
    if constexpr (std::is_same_v<OP, TwoTerms>) {
        o.hi[e] = cvt16<BF>(x);
        o.lo[e] = cvt16<BF>(x - cvt32<BF>(o.hi[e]));
    } else {
        o[e] = cvt16<BF>(x);
    }
}
template <bool BF, typename OP>
__device__ __forceinline__ float get(const OP &o, int e) {
    if constexpr (std::is_same_v<OP, TwoTerms>) return cvt32<BF>(o.hi[e]) + cvt32<BF>(o.lo[e]);
    else return cvt32<BF>(o[e]);
}
template <bool BF, typename OP>
__device__ __forceinline__ f32x4 mfma_op(s16x8 a, const OP &b, f32x4 c) {
    if constexpr (std::is_same_v<OP, TwoTerms>) return mfma16<BF>(a, b.lo, mfma16<BF>(a, b.hi, c));
    else return mfma16<BF>(a, b, c);
}

// eight dS of a lane, the largest magnitude of which is `mag`, as an operand; acc: the sums they go into
template <bool BF, int DT>
__device__ __forceinline__ void put_scaled(Op8 &o, const float (&y)[8], float mag, DsScale<BF> &scl, f32x4 (&acc)[DT]) {
    scl.fit(mag, acc);
    const float f = scl.factor();
#pragma unroll
    for (int e = 0; e < 8; e++) put<BF>(o, e, y[e] * f);
}
// dK and dV of a tile in their own units again
template <bool BF, int DT>
__device__ __forceinline__ void unscale(f32x4 (&dk)[DT], f32x4 (&dv)[DT], const DsScale<BF> &scl) {
    if constexpr (!BF) {
        const float f = scl.inverse() / kPUnit<BF>;
#pragma unroll
        for (int t = 0; t < DT; t++) {
            dk[t] *= f;
            dv[t] *= 1.f / kPUnit<BF>;
        }
    }
}

// ------------------------------------------------------------------ relative position bias
// The head's [2k-1, 2k-1] table in LDS, in float32, with a margin of 3 rows and columns: entry (key - query + k - 1)
// per axis lies at (.. + 3), so that every (token of a 4x4 block's halo, pixel of the block) pair has an entry, in its
// window or not, and the place of a token's entry is a lane constant plus (token row) * TB + (token column), which folds
// into the LDS read's offset.
template <int KS>
struct Bias {
    using G = Geo<32, KS>;  // (the numbering of the halo tokens depends on KS alone)
    static constexpr int TB = 2 * KS + 5, SPAN = 2 * KS - 1, E = SPAN * SPAN;
    // 16-token tiles that hold tokens at all, and the largest row that their numbers stand for
    static constexpr int W2 = G::W1 ? G::SW - G::W1 : 1, A_TILES = G::W1 ? G::SW * G::W1 / 16 : 0;
    static constexpr int USED = G::W1 ? A_TILES + (G::SW * W2 + 15) / 16 : (G::NK + 15) / 16;
    static constexpr int MAXR = G::W1 ? ((USED - A_TILES) * 16 - 1) / W2 : (USED * 16 - 1) / G::SWC;
    static constexpr int WORDS = (MAXR + KS + 3) * TB + 16;
    // (token row) * TB + (token column) of token tile * 16 + x; 0 for tiles without tokens
    static __device__ __forceinline__ int token(int tile, int x) {
        if (tile >= USED) return 0;
        int r, c;
        G::tok_rc(tile, x, r, c);
        return r * TB + c;
    }
    // lane constant of a query whose halo starts at (sr0, sc0): the entry of its token is query() + token()
    static __device__ __forceinline__ int query(const LaneQ &q) {
        return (q.hr0 + q.orow - q.qr + KS + 2) * TB + (q.hc0 + q.ocol - q.qc + KS + 2);
    }
};
// A thread's share of the table on its way to LDS
template <bool BF, int KS, int NT>
struct BiasRegs {
    using T = Bias<KS>;
    static constexpr int NB = (T::E + NT - 1) / NT;
    short v[NB];
    __device__ __forceinline__ void fetch(const void *rpb, int head) {
        const short *p = static_cast<const short *>(rpb) + (int64_t)head * T::E;
        // Never taken.  The branch only keeps the compiler from moving these loads' arithmetic through the kernels
        // of the largest windows, which then spill (forward B2 N8 128x128 d64 k11 90 -> 76 us with it; below 11x11 it
        // costs: forward B8 N4 56x56 d32 k7 15.7 -> 17.7).
        if (KS >= 11 && rpb == nullptr) {
#pragma unroll
            for (int i = 0; i < NB; i++) v[i] = 0;
            return;
        }
#pragma unroll
        for (int i = 0; i < NB; i++) v[i] = p[min((int)threadIdx.x + i * NT, T::E - 1)];
    }
    __device__ __forceinline__ void commit(float *lds) const {
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const int e = min((int)threadIdx.x + i * NT, T::E - 1);  // (the same value twice at the end)
            lds[(e / T::SPAN + 3) * T::TB + e % T::SPAN + 3] = cvt32<BF>(v[i]);
        }
    }
};
// Gradient of the bias.  A tile's dS is turned through LDS, wave by wave, one row of the block's four
// rows of queries at a time: the four queries' dS each in a plane of their own that is laid out
// like the wave's halo, with a margin of zeros.  A lane then owns displacements (t, u) = (token row -
// query row, token column - query column) and sums them over the planes with constant offsets.  The waves' sums
// of a tile are added in a fixed order and left in the workspace, one row of E floats per tile;
// rpb_tile_reduce sums the rows.  No atomics.  (Adding every dS to a table with ds_add_f32, in an order that
// was fixed too, took 76 cycles an instruction: dQ pass at B8 N8 112x112 d32 k7 309 us.)
template <int KS>
struct BiasGrad {
    using T = Bias<KS>;
    using G = typename T::G;
    static constexpr int P = (G::SW + 7 + 3) / 4 * 4;          // columns of a plane: c + 4, 16-byte aligned
    static constexpr int PLANE = (G::SW + 6) * P + 4;          // rows r + 3
    static constexpr int SIDE = G::SW + 3;                     // displacements per axis: -3 .. SW - 1
    static constexpr int SUMS = SIDE * SIDE, PASSES = (SUMS + 63) / 64;
    static constexpr int WORDS = 4 * PLANE + (SUMS + 3) / 4 * 4;  // per wave: planes, sums
    template <int NT>
    static __device__ __forceinline__ void clear(float *lds) {
        for (int i = threadIdx.x; i < NT / 64 * WORDS; i += NT) lds[i] = 0.f;
    }
    // ds[tile][i]: this lane's accumulator layout (token tile * 16 + 4 g + i, query n), zero where
    // the pair is not in the window or the query does not exist
    static __device__ __forceinline__ void sum(float *wave_lds, const f32x4 (&ds)[T::USED], int n, int g) {
        const int l = n + 16 * g;
        float *plane = wave_lds + (n & 3) * PLANE + 3 * P + 4;
        int at[PASSES];
        float acc[PASSES];
#pragma unroll
        for (int j = 0; j < PASSES; j++) {
            const int pos = min(j * 64 + l, SUMS - 1);
            at[j] = pos / SIDE * P + pos % SIDE + 1;
            acc[j] = 0.f;
        }
#pragma unroll
        for (int qr = 0; qr < 4; qr++) {
            if ((n >> 2) == qr) {
#pragma unroll
                for (int t = 0; t < T::USED; t++) {
                    int r, c;
                    G::tok_rc(t, g * 4, r, c);
                    if constexpr (G::SW == 6) {
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if (G::tok_rc(t, g * 4 + i, r, c)) plane[r * P + c] = ds[t][i];
                    } else if constexpr (T::W2 == 2) {
                        typedef float f32x2 __attribute__((ext_vector_type(2)));
                        if (t < T::A_TILES) {
                            *reinterpret_cast<f32x4 *>(plane + r * P + c) = ds[t];
                        } else if (r < G::SW) {  // two tokens of row r, two of row r + 1
                            *reinterpret_cast<f32x2 *>(plane + r * P + c) = f32x2{ds[t][0], ds[t][1]};
                            *reinterpret_cast<f32x2 *>(plane + (r + 1) * P + c) = f32x2{ds[t][2], ds[t][3]};
                        }
                    } else if (r < G::SW) {
                        *reinterpret_cast<f32x4 *>(plane + r * P + c) = ds[t];
                    }
                }
            }
            wave_fence();
#pragma unroll
            for (int j = 0; j < PASSES; j++)
#pragma unroll
                for (int qc = 0; qc < 4; qc++) acc[j] += wave_lds[at[j] + qc * PLANE + qr * P + qc];
            wave_fence();
        }
#pragma unroll
        for (int j = 0; j < PASSES; j++)
            if (j * 64 + l < SUMS) wave_lds[4 * PLANE + j * 64 + l] = acc[j];
    }
    // (LDS operations of one wave complete in program order: only the compiler has to be told that lanes read
    // what other lanes wrote)
    static __device__ __forceinline__ void wave_fence() {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    // the waves' sums to a tile's row of the workspace
    template <int NW>
    static __device__ __forceinline__ void flush(const float *lds, float *row, const Tile &tl, const Shape &s) {
        for (int e = threadIdx.x; e < T::E; e += 64 * NW) {
            const int dy = e / T::SPAN - (KS - 1), dx = e % T::SPAN - (KS - 1);
            float x = 0.f;
#pragma unroll
            for (int w = 0; w < NW; w++) {
                const int wr0 = tl.r0 + (w >> 1) * 4, wc0 = tl.c0 + (w & 1) * 4;
                const int t = dy + wr0 - win_start(min(wr0, s.H - 1), s.H, KS) + 3;
                const int u = dx + wc0 - win_start(min(wc0, s.W - 1), s.W, KS) + 3;
                const bool in = wr0 < s.H && wc0 < s.W && (unsigned)t < (unsigned)SIDE && (unsigned)u < (unsigned)SIDE;
                const float v = lds[w * WORDS + 4 * PLANE + (in ? t * SIDE + u : 0)];
                x += in ? v : 0.f;
            }
            row[e] = x;
        }
    }
};
// dS of a lane's halo tokens as operands of dQ's product (zero in tiles without tokens), and, times 1 / Z (0 for a
// lane without a query, or with one that again_dq computes), as terms of the bias gradient
template <bool BF, int KS, int STEPS>
__device__ __forceinline__ void operand_and_sums(Op8 (&dsb)[STEPS], f32x4 (&ds)[Bias<KS>::USED], DsScale<BF> &scl,
                                                 float zinv) {
    if constexpr (!BF) {
        float mag = 0.f;
#pragma unroll
        for (int mt = 0; mt < Bias<KS>::USED; mt++)
#pragma unroll
            for (int i = 0; i < 4; i++) mag = fmaxf(mag, fabsf(ds[mt][i]));
        scl.set(mag);
    }
    const float f = scl.factor();
#pragma unroll
    for (int mt = 0; mt < Bias<KS>::USED; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            put<BF>(dsb[mt >> 1], (mt & 1) * 4 + i, ds[mt][i] * f);
            ds[mt][i] = zinv != 0.f ? ds[mt][i] * zinv : 0.f;
        }
#pragma unroll
    for (int mt = Bias<KS>::USED; mt < 2 * STEPS; mt++)
#pragma unroll
        for (int i = 0; i < 4; i++) put<BF>(dsb[mt >> 1], (mt & 1) * 4 + i, 0.f);
}
// d_rpb[head][entry] = the sum over batch entries and tiles of the rows that the dQ pass left, in a
// fixed order: a workgroup takes 16 entries of a head, 64 threads a strided share of the rows each.  Bound by the
// latency of those loads, so the place of the next row comes without a branch or a loop: the steps back over whole images, one
// by one, were up to 64 a row (backward, us, B512 N4 d32: 8x8 k7 74.0 -> 60.6, 14x14 k7 274.6 -> 260.0; float16 12x7 k5 N3 90.5 -> 74.6).
// TYPED: the sum leaves in the tensors' type, which saves the caller a conversion kernel and
// its launch (B8 N4 56x56 d32 k7 forward and backward: 3.8 us of 80 on the device).
template <bool BIAS, bool BF, bool TYPED>
__global__ __launch_bounds__(1024) void rpb_tile_reduce(const float *rows, void *d_rpb, int B, int N, int tiles,
                                                        int E) {
    __shared__ float part[1024];
    const int n = blockIdx.x, e = blockIdx.y * 16 + threadIdx.x % 16;
    float acc = 0.f;
    if (e < E) {
        // row t of a batch entry, its place, and what 64 rows further are
        const int first = threadIdx.x / 16, dt = 64 % tiles;
        int t = first % tiles;
        const float *at = rows + ((int64_t)(first / tiles * N + n) * tiles + t) * E + e;
        const int64_t step = ((int64_t)(64 / tiles) * N * tiles + dt) * E, wrap = (int64_t)(N - 1) * tiles * E;
#pragma unroll 4
        for (int r = first; r < B * tiles; r += 64) {
            acc += *at;
            t += dt;
            at += step + (t >= tiles ? wrap : 0);
            t -= t >= tiles ? tiles : 0;
        }
    }
    part[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 512; w >= 16; w >>= 1) {
        if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < 16 && e < E) {
        if constexpr (TYPED) static_cast<short *>(d_rpb)[(int64_t)n * E + e] = cvt16<BF>(part[threadIdx.x]);
        else static_cast<float *>(d_rpb)[(int64_t)n * E + e] = part[threadIdx.x];
    }
}

// ------------------------------------------------------------------ results that are not finite
// With a bias: a result that is not finite is computed again from its window alone, as in
// na1d_band_mfma.hip (the general kernels, which used to serve these calls, read nothing else).
// A query's window, with the bias of every key: f(key row, key column, bias) until it returns false
template <bool BF, int KS, typename F>
__device__ __forceinline__ void walk_window(const Shape &s, const void *rpb, int head, int qr, int qc, F f) {
    constexpr int SPAN = 2 * KS - 1;
    const int r0 = win_start(qr, s.H, KS), c0 = win_start(qc, s.W, KS);
    const short *b = static_cast<const short *>(rpb) + ((int64_t)head * SPAN + r0 - qr + KS - 1) * SPAN + c0 - qc + KS - 1;
    for (int i = 0; i < KS * KS; i++)
        if (!f(r0 + i / KS, c0 + i % KS, kTable ? cvt32<BF>(b[i / KS * SPAN + i % KS]) : 0.f)) return;
}
template <typename ARGS>
__device__ __forceinline__ const short *pixel(const ARGS &a, const View &v, const ATile &tl, int r, int c) {
    return image_at(a, v, tl) + r * row_step(a, v) + c * col_step(a, v);
}
template <bool BF, int KS>
__device__ __forceinline__ void again_fwd(const FArgs &a, const ATile &tl, const LaneQ &lq, unsigned bad, int dlim) {
    const Shape &s = a.s;
    for (; bad; bad &= bad - 1) {
        const int col = __builtin_ctz(bad), qr = __shfl(lq.qr, col, 64), qc = __shfl(lq.qc, col, 64);
        if (!__shfl((int)lq.live, col, 64)) continue;
        const Chan2 q = chan_load<BF>(pixel(a, a.q, tl, qr, qc), dlim);
        Chan2 acc{0.f, 0.f};
        float mx = -INFINITY, z = 0.f;
        walk_window<BF, KS>(s, a.rpb, tl.nn, qr, qc, [&](int r, int c, float bias) {
            const float x = chan_dot(q, chan_load<BF>(pixel(a, a.k, tl, r, c), dlim)) * s.scale + bias;
            const float mn = x > mx ? x : mx, corr = exp_unit(mx - mn), p = exp_unit(x - mn);
            mx = mn;
            z = z * corr + p;
            acc.a *= corr;
            acc.b *= corr;
            chan_add(acc, p, chan_load<BF>(pixel(a, a.v, tl, r, c), dlim));
            return z == z;  // (else nothing finite can come of it)
        });
        chan_store<BF>(const_cast<short *>(pixel(a, a.o, tl, qr, qc)), dlim, acc, 1.f / z);
        if (a.lse && (threadIdx.x & 63) == 0) a.lse[image_token(a, tl) + (int64_t)qr * s.W + qc] = lse_of(mx, z);
    }
}
// sums: the wave's share of the bias gradient, without the queries whose delta is not finite
template <bool BF, int KS>
__device__ __forceinline__ void again_dq(const BArgs &a, const ATile &tl, const LaneQ &lq, unsigned bad, float lse,
                                         float delta, int wave, float *sums, int dlim) {
    const Shape &s = a.s;
    const int wr = tl.r0 + (wave >> 1) * 4 - lq.hr0 - lq.orow + 3, wc = tl.c0 + (wave & 1) * 4 - lq.hc0 - lq.ocol + 3;
    for (; bad; bad &= bad - 1) {
        const int col = __builtin_ctz(bad), qr = __shfl(lq.qr, col, 64), qc = __shfl(lq.qc, col, 64);
        if (!__shfl((int)lq.live, col, 64)) continue;
        const float lse_q = __shfl(lse, col, 64), delta_q = __shfl(delta, col, 64);
        const Chan2 q = chan_load<BF>(pixel(a, a.q, tl, qr, qc), dlim), go = chan_load<BF>(pixel(a, a.d_o, tl, qr, qc), dlim);
        float z = 0.f, d = 0.f;
        walk_window<BF, KS>(s, a.rpb, tl.nn, qr, qc, [&](int r, int c, float bias) {
            const float p = exp_unit(chan_dot(q, chan_load<BF>(pixel(a, a.k, tl, r, c), dlim)) * s.scale + bias - lse_q);
            z += p;
            d += p * chan_dot(go, chan_load<BF>(pixel(a, a.v, tl, r, c), dlim));
            return z == z;
        });
        d /= z;
        Chan2 acc{0.f, 0.f};
        if (d != d) {  // every dS of the window is NaN
            float *at = sums + (win_start(qr, s.H, KS) - qr + wr) * BiasGrad<KS>::SIDE + win_start(qc, s.W, KS) - qc + wc;
            for (int i = threadIdx.x & 63; kTable && i < KS * KS; i += 64) at[i / KS * BiasGrad<KS>::SIDE + i % KS] = d;
            acc = Chan2{d, d};
        } else {
            walk_window<BF, KS>(s, a.rpb, tl.nn, qr, qc, [&](int r, int c, float bias) {
                const Chan2 k = chan_load<BF>(pixel(a, a.k, tl, r, c), dlim);
                const float p = exp_unit(chan_dot(q, k) * s.scale + bias - lse_q) / z;
                const float ds = p * (chan_dot(go, chan_load<BF>(pixel(a, a.v, tl, r, c), dlim)) - d);
                chan_add(acc, ds, k);
                if (kTable && (threadIdx.x & 63) == 0 && !(delta_q * 0.f == 0.f))
                    sums[(r - qr + wr) * BiasGrad<KS>::SIDE + c - qc + wc] += ds;
                return true;
            });
        }
        chan_store<BF>(static_cast<short *>(a.dq) + grad_of(a, tl, qr, qc), dlim, acc, s.scale);
        if ((threadIdx.x & 63) == 0) {
            const int64_t tok = image_token(a, tl) + (int64_t)qr * s.W + qc;
            a.delta[tok] = d;
            row_zinv(a)[tok] = 1.f / z;
        }
    }
}
// kr, kc: this lane's key
template <bool BF, int KS>
__device__ __forceinline__ void again_keys(const BArgs &a, const ATile &tl, int kr_, int kc_, bool live, unsigned bad,
                                           int dlim) {
    constexpr int SPAN = 2 * KS - 1;
    const Shape &s = a.s;
    for (; bad; bad &= bad - 1) {
        const int col = __builtin_ctz(bad), kr = __shfl(kr_, col, 64), kc = __shfl(kc_, col, 64);
        if (!__shfl((int)live, col, 64)) continue;
        const Chan2 k = chan_load<BF>(pixel(a, a.k, tl, kr, kc), dlim), v = chan_load<BF>(pixel(a, a.v, tl, kr, kc), dlim);
        Chan2 ak{0.f, 0.f}, av{0.f, 0.f};
        bool open = true;
        for (int r = inv_lo(kr, KS); open && r < inv_hi(kr, s.H, KS); r++)
            for (int c = inv_lo(kc, KS); open && c < inv_hi(kc, s.W, KS); c++) {
                if ((unsigned)(kr - win_start(r, s.H, KS)) >= (unsigned)KS ||
                    (unsigned)(kc - win_start(c, s.W, KS)) >= (unsigned)KS)
                    continue;
                const int64_t tok = image_token(a, tl) + (int64_t)r * s.W + c;
                const int64_t at = ((int64_t)tl.nn * SPAN + kr - r + KS - 1) * SPAN + kc - c + KS - 1;
                const float bias = kTable ? cvt32<BF>(static_cast<const short *>(a.rpb)[at]) : 0.f;
                const Chan2 q = chan_load<BF>(pixel(a, a.q, tl, r, c), dlim), go = chan_load<BF>(pixel(a, a.d_o, tl, r, c), dlim);
                const float p = exp_unit(chan_dot(q, k) * s.scale + bias - a.lse[tok]) * row_zinv(a)[tok];
                chan_add(av, p, go);
                chan_add(ak, p * (chan_dot(go, v) - a.delta[tok]), q);
                open = p == p;
            }
        const int64_t to = grad_of(a, tl, kr, kc);
        chan_store<BF>(static_cast<short *>(a.dk) + to, dlim, ak, s.scale);
        chan_store<BF>(static_cast<short *>(a.dv) + to, dlim, av, 1.f);
    }
}

// ------------------------------------------------------------------ forward
// ROLL: walk down the columns of an image and keep the halo rows that consecutive
// tiles share in LDS (see make_runs); otherwise a strided walk over row-major tiles
// with the whole halo staged per tile.
// FULL: the image sides are multiples of the tile sides, so every lane's pixel exists: no
// wave is switched off and no store is predicated.  The compiler then knows how many stores
// a tile issues, and the wait for the next tile's staged rows (older than those stores) does
// not wait for the stores as well.  With a branch around the stores, even a uniform one with
// an explicit wait on its other side, it falls back to waiting for everything outstanding
// (B4 N4 128x128 d128 k5: 58.8 -> 56.7 us, 256x256: 198.2 -> 189.3, d64 k5: 60.4 -> 58.5).
// With a bias the head_dim 32 forward takes 169 to 175 registers (k = 7 and 9), one more than three
// waves per SIMD have: budgeted for three, B8 N8 112x112 k7 114.8 -> 97.8 us.  At k = 5 four (three at
// head_dim 64) take a register or two too many without a budget (B8 N4 56x56 d64 k5 16.6 us with two).
// Without one the compiler left alone takes 146 registers at head_dim 32, k = 7, where four waves per SIMD fit without a
// spill: B6 N9 91x128 49.4 -> 47.3 us, B1 N16 69x69 8.0 -> 6.8; k = 9 spills there, and k = 5, which runs four without a budget,
// loses by the order of instructions that one leads to (B2 N12 234x210 67.2 -> 69.5, B5 N5 126x126 21.4 -> 22.4).
template <int D, int KS, int NW>
constexpr int kFwdWaves = D == 32 && (kBias ? KS == 5 : !kNarrow && KS == 7) ? 4
                          : kBias && ((D == 32 && KS <= 9) || (D == 64 && KS == 5)) ? 3 : Geo<D, KS, NW>::WAVES;
// How the staging threads of the builds for narrow heads, sub-grids and a bias fetch (HaloPlan).  A branch around the loads of a thread
// without channels (SKIP) keeps them together, ahead of the tile's arithmetic; without one the compiler places them among it,
// which takes fewer registers.  Where a build has the registers the branch is level or ahead, elsewhere it costs up to 16%;
// where the places of the chunks are formed anew (not KEEP), the additions cost up to 9% at head_dim 128.  The rules follow the
// means of 6 to 24 calls of each build and window.  Forward, us, loads among the arithmetic, places of one period -> as here: bias d128 k3
// B4 N11 118x78 d96 82.9 -> 76.2, k5 B8 N4 56x56 23.7 -> 22.4, k11 58.9 -> 55.3, k13 bf16 65.7 -> 58.4 (float16 91.8, with the
// branch 95.4), d64 k9 25.3 -> 24.9; dilation 2 d32 k11 +11% -> level, d64 k11 +9% -> level, d128 k3 up to +6% -> level; narrow
// d120 k7 +4% -> level, d24 k11 +7% -> level.  Without the branch: bias d32 k7 -4%, d128 k9 -8%, dilation 2 d64 k5 -10%, d32 k9 -10%.
template <int D, int KS>
constexpr bool kFwdKeep = D == 128 && (kTable ? KS <= 5 || KS == 11 : kSub && KS == 3);
template <bool BF, int D, int KS>
constexpr bool kFwdSkip = kFwdKeep<D, KS> ||
    (kTable ? (D == 64 ? KS >= 9 && (BF || KS != 11) : D == 128 && KS == 13 && BF)
     : kSub ? D <= 64 && KS == 11 : KS <= 11 || D == 32);
template <bool BF, int D, int KS, bool ROLL, int NW = 4, bool FULL = false>
__global__ __launch_bounds__((Geo<D, KS, NW>::NT), (kFwdWaves<D, KS, NW>)) void fwd_mfma(FArgs a, int tiles_r, int tiles_c, int ntiles, Runs rp) {
    using G = Geo<D, KS, NW>;
    __shared__ __attribute__((aligned(16))) short lds_k[G::ROWS * G::PITCH];
    __shared__ __attribute__((aligned(16))) short lds_v[G::ROWS * G::PITCH];
    __shared__ float lds_bias[kTable ? Bias<KS>::WORDS : 1];

    const Shape &s = a.s;
    const int dlim = kNarrow ? s.D : D;  // head dim of the tensors: D, or less in the build for narrow dims
    Sched sc = ROLL ? make_runs(ntiles, blockIdx.x, gridDim.x, rp) : make_sched(ntiles, blockIdx.x, gridDim.x);
    if (sc.t >= sc.t_end) return;
    zero_row<D, KS, NW>(lds_k, dlim);
    zero_row<D, KS, NW>(lds_v, dlim);

    const int wave = FULL ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
    const int l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const float sc2 = s.scale * kUnit;

    // registers that carry the next tile while the current one is computed
    const auto plan = make_plan<D, KS, NW, 1, kFwdKeep<D, KS>>(dlim, kFwdSkip<BF, D, KS>);
    HaloRegs<D, KS, NW> kst, vst;
    s16x8 qnext[G::DS];
    BiasRegs<BF, KS, G::NT> bst;
    // rows [y0, y0 + nr) of the halo are what LDS does not hold yet
    auto prefetch = [&](const ATile &tl, const LaneQ &lq, int y0, int nr) __attribute__((always_inline)) {
        if constexpr (ROLL) {
            halo_fetch_rows<D, KS>(kst, plan, image_at(a, a.k, tl), row_step(a, a.k), col_step(a, a.k), y0, lq.hc0, nr, s.H, s.W);
            halo_fetch_rows<D, KS>(vst, plan, image_at(a, a.v, tl), row_step(a, a.v), col_step(a, a.v), y0, lq.hc0, nr, s.H, s.W);
        } else {
            halo_fetch<D, KS>(kst, plan, image_at(a, a.k, tl), row_step(a, a.k), col_step(a, a.k), lq.hr0, lq.hc0, s.H, s.W);
            halo_fetch<D, KS>(vst, plan, image_at(a, a.v, tl), row_step(a, a.v), col_step(a, a.v), lq.hr0, lq.hc0, s.H, s.W);
        }
        load_row_chunks(qnext, image_at(a, a.q, tl) + lq.qr * row_step(a, a.q) + lq.qc * col_step(a, a.q), g, dlim);
        if constexpr (kTable) bst.fetch(a.rpb, tl.nn);
    };

    auto pick = [&](int t) __attribute__((always_inline)) {
        return in_sub(ROLL ? tile_of_cm(t, tiles_r, tiles_c, s.N) : tile_of(t, tiles_r, tiles_c, s.N, G::TH), a);
    };
    ATile cur = pick(sc.t);
    LaneQ lq = lane_at<KS>(a, cur, wave, n);
    int y0 = lq.hr0, nr = G::HR;
    prefetch(cur, lq, y0, nr);
    s16x8 qreg[G::DS];
    // FULL: the staged rows go to LDS at the END of a tile's pass through the loop, after its
    // stores, not at the top of the next: there the compiler has to merge the first pass (where
    // these loads are the youngest memory operations) with the later ones, and waits for
    // everything outstanding, the tile's own stores included.
    auto commit = [&]() __attribute__((always_inline)) {
        if constexpr (ROLL) {
            halo_commit_rows<D, KS>(lds_k, plan, kst, y0, nr);
            halo_commit_rows<D, KS>(lds_v, plan, vst, y0, nr);
        } else {
            halo_commit<D, KS>(lds_k, plan, kst);
            halo_commit<D, KS>(lds_v, plan, vst);
        }
        if constexpr (kTable) bst.commit(lds_bias);
#pragma unroll
        for (int ds = 0; ds < G::DS; ds++) qreg[ds] = qnext[ds];
    };
    if constexpr (FULL) commit();
    for (;;) {
        if constexpr (!FULL) commit();
        __syncthreads();

        const int tn = sched_peek(sc);
        const bool more = tn < sc.t_end;
        ATile nxt = cur;
        LaneQ lqn = lq;
        if (more) {
            nxt = pick(tn);
            lqn = lane_at<KS>(a, nxt, wave, n);
            // the tile below in the same image keeps the rows the two halos share
            const bool below = ROLL && same_column(nxt, cur) &&
                               nxt.r0 > cur.r0 && lqn.hr0 < lq.hr0 + G::HR;
            y0 = below ? lq.hr0 + G::HR : lqn.hr0;
            nr = below ? lqn.hr0 - lq.hr0 : G::HR;
            prefetch(nxt, lqn, y0, nr);
        } else {
            // (the last tile of the walk: nothing is loaded, and the explicit wait says so to
            // the compiler, which does not know that this path leaves the loop below)
            if constexpr (FULL) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        }
        const int rot = ROLL ? lq.hr0 % G::HR : 0;
        auto trow = [&](int tile, int x) __attribute__((always_inline)) {
            return ROLL ? G::token_row_rot(tile, x, lq.orow, lq.ocol, rot) : G::token_row(tile, x, lq.orow, lq.ocol);
        };

        if (FULL || lq.wave_on) {
            // logits^T [halo token][query], masked
            const int bq = kTable ? Bias<KS>::query(lq) : 0;
            f32x4 acc[G::MT];
            float mx = -INFINITY;
#pragma unroll
            for (int mt = 0; mt < G::MT; mt++) {
                const typename G::ARow kp = G::a_row(lds_k, trow(mt, n), g);
                f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ds = 0; ds < G::DS; ds++)
                    c = mfma16<BF>(*reinterpret_cast<const s16x8 *>(G::a_at(kp, ds)), qreg[ds], c);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const bool ok = G::template tok_in<KS>(mt, g * 4 + i, lq.dr, lq.dc);
                    float x = c[i] * sc2;
                    if constexpr (kTable) x += lds_bias[bq + Bias<KS>::token(mt, g * 4 + i)];
                    c[i] = ok ? x : -INFINITY;
                    mx = fmaxf(mx, c[i]);
                }
                acc[mt] = c;
            }
            mx = col_max(mx);
            float sum = 0.f;
            Op8 pb[G::KSTEPS];
#pragma unroll
            for (int mt = 0; mt < G::MT; mt++) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float p = exp_unit(acc[mt][i] - mx);
                    sum += p;
                    put<BF>(pb[mt >> 1], (mt & 1) * 4 + i, p);
                }
            }
            sum = col_sum(sum);

            // O^T [channel][query] = V^T P^T over the halo tokens
            f32x4 o[G::DT];
#pragma unroll
            for (int mt = 0; mt < G::DT; mt++) o[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < G::KSTEPS; ks++) {
                typename G::TRow vp[2];
#pragma unroll
                for (int h = 0; h < 2; h++)
                    vp[h] = G::t_row(lds_v, trow(ks * 2 + h, g * 4 + (n >> 2)), n);
#pragma unroll
                for (int mt = 0; mt < G::DT; mt++)
                    o[mt] = mfma_op<BF>(cat(lds_read_tr(G::t_at(vp[0], mt)), lds_read_tr(G::t_at(vp[1], mt))), pb[ks],
                        o[mt]);
            }

            const unsigned bad = kBias ? bad_columns(o, sum) : 0u;
            const bool here = lq.live && !(bad >> n & 1);
            store_token<BF, D, kLineStores<D, KS, G::WAVES>, FULL>(const_cast<short *>(image_at(a, a.o, cur)) + lq.qr * row_step(a, a.o) + lq.qc * col_step(a, a.o),
                               g, o, 1.f / sum, here, dlim);
            // (FULL: all four lanes of a token write its log-sum-exp, the same value, so that
            // this store is not predicated either)
            if (a.lse && (FULL || (here && g == 0)))
                a.lse[lq.tok] = lse_of(mx, sum);
            if constexpr (kBias)
                if (__builtin_expect(bad != 0, 0)) again_fwd<BF, KS>(a, cur, lq, bad, dlim);
        }

        if (!more) {
            if constexpr (FULL) __builtin_amdgcn_s_waitcnt(0x0F70);  // (as above: this path shares its last block with the other)
            break;
        }
        __syncthreads();  // every wave is done with this tile's LDS
        if constexpr (FULL) commit();
        cur = nxt;
        lq = lqn;
        sched_advance(sc, tn);
    }
}

// Two halos of an 8x8 tile fit LDS (the kernels that keep K and V, or Q and dO, side by side)
template <int D, int KS>
constexpr bool fits() {
    return Geo<D, KS>::LDS_BYTES <= 160 * 1024;
}
// Workgroups per CU of the kernels that keep ONE halo in LDS at a time: two where that halo
// fits twice, one for the largest halos (head_dim 128 with kernel_size 11 and 13: 88 and
// 109 KB), where these kernels are the only matrix-core ones that fit at all.
template <int D, int KS>
constexpr int kOneHaloWgs = 2 * (Geo<D, KS>::ROWS * Geo<D, KS>::PITCH * 2 + 1024) <= 160 * 1024 ? 2 : 1;
template <int D, int KS>
constexpr bool kOneHaloFits = Geo<D, KS>::ROWS * Geo<D, KS>::PITCH * 2 + 1024 <= 160 * 1024;

// ------------------------------------------------------------------ forward, one halo in LDS at a time
// The forward for halos of which LDS holds two only once per CU (head_dim 128 with
// kernel_size 7 and 9) or not at all (kernel_size 11 and 13), like bwd_dq2_mfma: K rows first
// (logits, softmax; P stays in registers as 16-bit values) while the tile's V rows are in
// flight, V over K behind a barrier, then O^T = V^T P^T while the next tile's K rows are in
// flight.  Two workgroups per CU (one at kernel_size 11 and 13), four barriers per tile; 8x8
// tiles, no column walk.
// FULL: as in fwd_mfma.
template <bool BF, int D, int KS, int NW = 4, bool FULL = false>
__global__ __launch_bounds__((Geo<D, KS, NW>::NT), (NW == 4 ? kOneHaloWgs<D, KS> : 1)) void fwd2_mfma(FArgs a, int tiles_r, int tiles_c, int ntiles) {
    using G = Geo<D, KS, NW>;
    __shared__ __attribute__((aligned(16))) short lds_x[G::ROWS * G::PITCH];
    __shared__ float lds_bias[kTable ? Bias<KS>::WORDS : 1];
    const Shape &s = a.s;
    const int dlim = kNarrow ? s.D : D;  // head dim of the tensors: D, or less in the build for narrow dims
    Sched sc = make_sched(ntiles, blockIdx.x, gridDim.x);
    if (sc.t >= sc.t_end) return;
    zero_row<D, KS, NW>(lds_x, dlim);

    const int wave = FULL ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
    const int l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const float sc2 = s.scale * kUnit;
    const auto plan = make_plan<D, KS, NW, 1, kFwdKeep<D, KS>>(dlim, kFwdSkip<BF, D, KS>);
    HaloRegs<D, KS, NW> st;
    s16x8 qnext[G::DS];
    BiasRegs<BF, KS, G::NT> bst;
    auto fetch_rows = [&](const View &vw, const ATile &tl, const LaneQ &lq) __attribute__((always_inline)) {
        halo_fetch<D, KS>(st, plan, image_at(a, vw, tl), row_step(a, vw), col_step(a, vw), lq.hr0, lq.hc0, s.H, s.W);
    };
    auto fetch_q = [&](const ATile &tl, const LaneQ &lq) __attribute__((always_inline)) {
        load_row_chunks(qnext, image_at(a, a.q, tl) + lq.qr * row_step(a, a.q) + lq.qc * col_step(a, a.q), g, dlim);
        if constexpr (kTable) bst.fetch(a.rpb, tl.nn);
    };
    ATile cur = in_sub(tile_of(sc.t, tiles_r, tiles_c, s.N, G::TH), a);
    LaneQ lq = lane_at<KS>(a, cur, wave, n);
    fetch_rows(a.k, cur, lq);
    fetch_q(cur, lq);
    s16x8 qreg[G::DS];
    // (K rows and the query row at the end of a tile's pass through the loop, after its stores:
    // see fwd_mfma)
    auto commit_k = [&]() __attribute__((always_inline)) {
        halo_commit<D, KS>(lds_x, plan, st);
        if constexpr (kTable) bst.commit(lds_bias);
#pragma unroll
        for (int ds = 0; ds < G::DS; ds++) qreg[ds] = qnext[ds];
    };
    if constexpr (FULL) commit_k();
    for (;;) {
        if constexpr (!FULL) commit_k();
        __syncthreads();
        fetch_rows(a.v, cur, lq);
        auto trow = [&](int tile, int x) __attribute__((always_inline)) { return G::token_row(tile, x, lq.orow, lq.ocol); };
        Op8 pb[G::KSTEPS];
        float mx = -INFINITY, sum = 0.f;
        if (FULL || lq.wave_on) {
            const int bq = kTable ? Bias<KS>::query(lq) : 0;
            f32x4 acc[G::MT];
#pragma unroll
            for (int mt = 0; mt < G::MT; mt++) {
                const typename G::ARow kp = G::a_row(lds_x, trow(mt, n), g);
                f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ds = 0; ds < G::DS; ds++)
                    c = mfma16<BF>(*reinterpret_cast<const s16x8 *>(G::a_at(kp, ds)), qreg[ds], c);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const bool ok = G::template tok_in<KS>(mt, g * 4 + i, lq.dr, lq.dc);
                    float x = c[i] * sc2;
                    if constexpr (kTable) x += lds_bias[bq + Bias<KS>::token(mt, g * 4 + i)];
                    c[i] = ok ? x : -INFINITY;
                    mx = fmaxf(mx, c[i]);
                }
                acc[mt] = c;
            }
            mx = col_max(mx);
#pragma unroll
            for (int mt = 0; mt < G::MT; mt++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float p = exp_unit(acc[mt][i] - mx);
                    sum += p;
                    put<BF>(pb[mt >> 1], (mt & 1) * 4 + i, p);
                }
            sum = col_sum(sum);
        }
        __syncthreads();                      // every wave has read K
        halo_commit<D, KS>(lds_x, plan, st);  // V
        __syncthreads();

        const int tn = sched_peek(sc);
        const bool more = tn < sc.t_end;
        ATile nxt = cur;
        LaneQ lqn = lq;
        if (more) {
            nxt = in_sub(tile_of(tn, tiles_r, tiles_c, s.N, G::TH), a);
            lqn = lane_at<KS>(a, nxt, wave, n);
            fetch_rows(a.k, nxt, lqn);
            fetch_q(nxt, lqn);
        } else {
            if constexpr (FULL) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the last tile, nothing is loaded (see fwd_mfma)
        }
        if (FULL || lq.wave_on) {
            f32x4 o[G::DT];
#pragma unroll
            for (int mt = 0; mt < G::DT; mt++) o[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < G::KSTEPS; ks++) {
                typename G::TRow vp[2];
#pragma unroll
                for (int h = 0; h < 2; h++)
                    vp[h] = G::t_row(lds_x, trow(ks * 2 + h, g * 4 + (n >> 2)), n);
#pragma unroll
                for (int mt = 0; mt < G::DT; mt++)
                    o[mt] = mfma_op<BF>(cat(lds_read_tr(G::t_at(vp[0], mt)), lds_read_tr(G::t_at(vp[1], mt))), pb[ks],
                        o[mt]);
            }
            const unsigned bad = kBias ? bad_columns(o, sum) : 0u;
            const bool here = lq.live && !(bad >> n & 1);
            store_token<BF, D, kLineStores<D, KS, (NW == 4 ? kOneHaloWgs<D, KS> : 1)>, FULL>(const_cast<short *>(image_at(a, a.o, cur)) + lq.qr * row_step(a, a.o) + lq.qc * col_step(a, a.o),
                               g, o, 1.f / sum, here, dlim);
            if (a.lse && (FULL || (here && g == 0)))
                a.lse[lq.tok] = lse_of(mx, sum);
            if constexpr (kBias)
                if (__builtin_expect(bad != 0, 0)) again_fwd<BF, KS>(a, cur, lq, bad, dlim);
        }
        if (!more) {
            if constexpr (FULL) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), see fwd_mfma
            break;
        }
        __syncthreads();  // every wave has read V
        if constexpr (FULL) commit_k();
        cur = nxt;
        lq = lqn;
        sched_advance(sc, tn);
    }
}

// ------------------------------------------------------------------ dQ
// Query-centric like the forward: recompute P from the saved log-sum-exp, form
// dP^T = V dO^T on the same halo, dS = P * (dP - delta) with delta = sum_j P_j dP_j
// (equal to dO . O, so the forward output is never read), and dQ^T = K^T dS^T with
// K read back from LDS transposed.  Also writes delta for the dK/dV pass.
// Per-query math: e_natten/triton.py:383-398.
// FRAME: walk only the tiles of the frame of `ts` (the inner tiles are served by
// the fused backward).
// head_dim 32 with kernel_size 7 and 9: the dQ pass fits the 168 registers of three waves
// per SIMD (LDS admits three workgroups per CU and more); B8 N2 112x112 k = 7: 27.8 -> 24.4
// us, B4 N4 128x128 k = 9: 37.1 -> 35.0 (with a bias it spills 55 there).  The forward is as fast or faster compiled for two
// (it then takes about 150 registers and runs three per SIMD anyway).
// (not the sub-grids of a dilated call: 80 bytes of scratch in three at k = 7, B8 N4 112x112 dilation 2 67.4 -> 56.3 us in two;
// nor k = 9 there and in the build for narrow heads: B4 N4 128x128 d24 35.8 -> 34.0)
// k = 3 and 5 took one or two registers more than four waves per SIMD have (head_dim 64, k = 3: one more than
// three): B8 N16 63x93 d32 k5 54.0 -> 48.6 us, B8 N2 112x112 k3 15.1 -> 13.3, B4 N4 128x128 d64 k3 28.7 -> 27.4.
template <int D, int KS, int NW>
constexpr int kDqWaves = kBias || NW != 4 ? Geo<D, KS, NW>::WAVES
                         : !kNarrow && D == 32 && KS <= 5 ? 4
                         : (D == 32 && ((KS == 7 && !kSub) || (KS == 9 && !kNarrow))) || (!kNarrow && D == 64 && KS == 3) ? 3 : Geo<D, KS, NW>::WAVES;
// SKIP of the dQ pass (kFwdSkip).  Time without the branch: k = 3 up to 10% more at d48, 9% at d80 and d96, 7% on the
// sub-grids of d32; k = 5 6% more there, and 3 to 17% less at d48.  From k = 7 on the builds that spill with the branch are
// up to 48% faster without (d96 k11), the others level.
template <int D, int KS>
constexpr bool kDqSkip = !kTable && (KS == 3 || (D != 64 && KS == 5));
// FULL: as in fwd_mfma (no wave switched off, no store predicated, the staged rows go to LDS at
// the end of a tile's pass through the loop).
template <bool BF, int D, int KS, bool FRAME, bool ROLL, int NW = 4, bool FULL = false>
__global__ __launch_bounds__((Geo<D, KS, NW>::NT), (kDqWaves<D, KS, NW>)) void bwd_dq_mfma(BArgs a, TileSet ts, int ntiles, Runs rp) {
    // (the dK/dV pass that follows on the stream counts its frame tiles here, from zero)
    if (blockIdx.x == 0 && threadIdx.x == 0 && a.zinv && kCounter) *reinterpret_cast<int *>(a.zinv) = 0;
    using G = Geo<D, KS, NW>;
    __shared__ __attribute__((aligned(16))) short lds_k[G::ROWS * G::PITCH];
    __shared__ __attribute__((aligned(16))) short lds_v[G::ROWS * G::PITCH];
    __shared__ float lds_bias[kTable ? Bias<KS>::WORDS : 1];
    __shared__ __attribute__((aligned(16))) float lds_dbias[kTable ? NW * BiasGrad<KS>::WORDS : 1];

    const Shape &s = a.s;
    const int dlim = kNarrow ? s.D : D;  // head dim of the tensors: D, or less in the build for narrow dims
    static_assert(!(FRAME && ROLL), "the frame is not walked by columns");
    Sched sc = ROLL ? make_runs(ntiles, blockIdx.x, gridDim.x, rp) : make_sched(ntiles, blockIdx.x, gridDim.x);
    if (sc.t >= sc.t_end) return;
    zero_row<D, KS, NW>(lds_k, dlim);
    zero_row<D, KS, NW>(lds_v, dlim);

    const int wave = FULL ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
    const int l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const float sc2 = s.scale * kUnit;
    auto pick = [&](int t) __attribute__((always_inline)) {
        if constexpr (FRAME) return in_sub(frame_tile(t, ts, s.N), a);
        else if constexpr (ROLL) return in_sub(tile_of_cm(t, ts.tiles_r, ts.tiles_c, s.N), a);
        else return in_sub(tile_of(t, ts.tiles_r, ts.tiles_c, s.N, G::TH), a);
    };

    const HaloPlan<D, KS, NW> plan = make_plan<D, KS, NW>(dlim, kDqSkip<D, KS>);
    HaloRegs<D, KS, NW> kst, vst;
    s16x8 qnext[G::DS], gnext[G::DS];
    float lse_next = 0.f;
    BiasRegs<BF, KS, G::NT> bst;
    if constexpr (kTable) BiasGrad<KS>::template clear<G::NT>(lds_dbias);
    // rows [y0, y0 + nr) of the halo are what LDS does not hold yet
    auto prefetch = [&](const ATile &tl, const LaneQ &lq, int y0, int nr) __attribute__((always_inline)) {
        if constexpr (ROLL) {
            halo_fetch_rows<D, KS>(kst, plan, image_at(a, a.k, tl), row_step(a, a.k), col_step(a, a.k), y0, lq.hc0, nr, s.H, s.W);
            halo_fetch_rows<D, KS>(vst, plan, image_at(a, a.v, tl), row_step(a, a.v), col_step(a, a.v), y0, lq.hc0, nr, s.H, s.W);
        } else {
            halo_fetch<D, KS>(kst, plan, image_at(a, a.k, tl), row_step(a, a.k), col_step(a, a.k), lq.hr0, lq.hc0, s.H, s.W);
            halo_fetch<D, KS>(vst, plan, image_at(a, a.v, tl), row_step(a, a.v), col_step(a, a.v), lq.hr0, lq.hc0, s.H, s.W);
        }
        load_row_chunks(qnext, image_at(a, a.q, tl) + lq.qr * row_step(a, a.q) + lq.qc * col_step(a, a.q), g, dlim);
        load_row_chunks(gnext, image_at(a, a.d_o, tl) + lq.qr * row_step(a, a.d_o) + lq.qc * col_step(a, a.d_o), g, dlim);
        lse_next = a.lse[lq.tok];
        if constexpr (kTable) bst.fetch(a.rpb, tl.nn);
    };

    ATile cur = pick(sc.t);
    LaneQ lq = lane_at<KS>(a, cur, wave, n);
    int y0 = lq.hr0, nr = G::HR;
    prefetch(cur, lq, y0, nr);
    s16x8 qreg[G::DS], greg[G::DS];
    float lse2;
    // (at the end of a tile's pass through the loop, after its stores: see fwd_mfma)
    auto commit = [&]() __attribute__((always_inline)) {
        if constexpr (ROLL) {
            halo_commit_rows<D, KS>(lds_k, plan, kst, y0, nr);
            halo_commit_rows<D, KS>(lds_v, plan, vst, y0, nr);
        } else {
            halo_commit<D, KS>(lds_k, plan, kst);
            halo_commit<D, KS>(lds_v, plan, vst);
        }
#pragma unroll
        for (int ds = 0; ds < G::DS; ds++) {
            qreg[ds] = qnext[ds];
            greg[ds] = gnext[ds];
        }
        lse2 = lse_next * kUnit;
        if constexpr (kTable) bst.commit(lds_bias);
    };
    if constexpr (FULL) commit();
    for (;;) {
        if constexpr (!FULL) commit();
        __syncthreads();

        const int tn = sched_peek(sc);
        const bool more = tn < sc.t_end;
        ATile nxt = cur;
        LaneQ lqn = lq;
        if (more) {
            nxt = pick(tn);
            lqn = lane_at<KS>(a, nxt, wave, n);
            // the tile below in the same image keeps the rows the two halos share
            const bool below = ROLL && same_column(nxt, cur) &&
                               nxt.r0 > cur.r0 && lqn.hr0 < lq.hr0 + G::HR;
            y0 = below ? lq.hr0 + G::HR : lqn.hr0;
            nr = below ? lqn.hr0 - lq.hr0 : G::HR;
            prefetch(nxt, lqn, y0, nr);
        } else {
            if constexpr (FULL) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the last tile, nothing is loaded (see fwd_mfma)
        }
        const int rot = ROLL ? lq.hr0 % G::HR : 0;
        auto trow = [&](int tile, int x) __attribute__((always_inline)) {
            return ROLL ? G::token_row_rot(tile, x, lq.orow, lq.ocol, rot) : G::token_row(tile, x, lq.orow, lq.ocol);
        };

        if (FULL || lq.wave_on) {
            // P^T and dP^T on the halo; delta = sum_j P_j dP_j (= dO . O) comes from
            // the same values that form dS, so sum_j dS_j vanishes to rounding
            // P is kept rounded to 16 bits (it is about to be rounded into dS
            // anyway) in the registers that will hold dS; with a bias and in two terms, where
            // dS is not rounded to 16 bits, in float32.  dP stays float32; with
            // the largest halos it is not kept but formed a second time once delta
            // is known (measured faster there: the matrix cores are idle, the
            // registers are not).
            const int bq = kTable ? Bias<KS>::query(lq) : 0;
            constexpr bool kKeepDp = !(G::WAVES == 1 && G::MT >= 16);
            f32x4 dp[kKeepDp ? G::MT : 1];
            Op8 dsb[G::KSTEPS];
            f32x4 ds_all[kBias ? Bias<KS>::USED : 1];  // with a bias: P, then dS, in float32
            float dpart = 0.f, zsum = 0.f;
#pragma unroll
            for (int mt = 0; mt < G::MT; mt++) {
                const int row = trow(mt, n);
                const typename G::ARow kp = G::a_row(lds_k, row, g), vp = G::a_row(lds_v, row, g);
                f32x4 cs = {0.f, 0.f, 0.f, 0.f}, cp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ds = 0; ds < G::DS; ds++) {
                    cs = mfma16<BF>(*reinterpret_cast<const s16x8 *>(G::a_at(kp, ds)), qreg[ds], cs);
                    cp = mfma16<BF>(*reinterpret_cast<const s16x8 *>(G::a_at(vp, ds)), greg[ds], cp);
                }
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const bool ok = G::template tok_in<KS>(mt, g * 4 + i, lq.dr, lq.dc);
                    float x;
                    if constexpr (kTable) x = cs[i] * sc2 + lds_bias[bq + Bias<KS>::token(mt, g * 4 + i)] - lse2;
                    else x = cs[i] * sc2 - lse2;
                    cs[i] = exp_unit(ok ? x : -INFINITY);
                    if constexpr (kBias) zsum += cs[i];
                    dpart = fmaf(cs[i], cp[i], dpart);
                    if constexpr (!kBias) put<BF>(dsb[mt >> 1], (mt & 1) * 4 + i, cs[i]);
                }
                if constexpr (kBias)
                    if (mt < Bias<KS>::USED) ds_all[mt] = cs;
                if constexpr (kKeepDp) dp[mt] = cp;
            }
            const float zinv = kBias ? 1.f / col_sum(zsum) : 1.f, delta = col_sum(dpart) * zinv;
#pragma unroll
            for (int mt = 0; mt < G::MT; mt++) {
                f32x4 cp;
                if constexpr (kKeepDp) {
                    cp = dp[mt];
                } else {
                    const typename G::ARow vp = G::a_row(lds_v, trow(mt, n), g);
                    cp = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int ds = 0; ds < G::DS; ds++)
                        cp = mfma16<BF>(*reinterpret_cast<const s16x8 *>(G::a_at(vp, ds)), greg[ds], cp);
                }
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if constexpr (!kBias) {
                        const float p = get<BF>(dsb[mt >> 1], (mt & 1) * 4 + i);
                        put<BF>(dsb[mt >> 1], (mt & 1) * 4 + i, p * (cp[i] - delta));
                    } else if (mt < Bias<KS>::USED) {
                        ds_all[mt][i] *= cp[i] - delta;
                    }
                }
            }

            DsScale<BF> scl;
            if constexpr (kBias) {
                operand_and_sums<BF, KS>(dsb, ds_all, scl, lq.live && delta * 0.f == 0.f ? zinv : 0.f);
                if constexpr (kTable) BiasGrad<KS>::sum(lds_dbias + wave * BiasGrad<KS>::WORDS, ds_all, n, g);
            }
            f32x4 dq[G::DT];
#pragma unroll
            for (int mt = 0; mt < G::DT; mt++) dq[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < G::KSTEPS; ks++) {
                typename G::TRow kp[2];
#pragma unroll
                for (int h = 0; h < 2; h++)
                    kp[h] = G::t_row(lds_k, trow(ks * 2 + h, g * 4 + (n >> 2)), n);
#pragma unroll
                for (int mt = 0; mt < G::DT; mt++)
                    dq[mt] = mfma_op<BF>(cat(lds_read_tr(G::t_at(kp[0], mt)), lds_read_tr(G::t_at(kp[1], mt))), dsb[ks],
                        dq[mt]);
            }

            const unsigned bad = kBias ? bad_columns(dq, delta) : 0u;
            store_token<BF, D, kLineStores<D, KS, G::WAVES>, FULL>(static_cast<short *>(a.dq) + grad_of(a, cur, lq.qr, lq.qc), g, dq, s.scale * (kBias ? zinv * scl.inverse() : 1.f), lq.live && !(bad >> n & 1), dlim);
            if constexpr (kBias)
                if (__builtin_expect(bad != 0, 0)) {
                    BiasGrad<KS>::wave_fence();
                    again_dq<BF, KS>(a, cur, lq, bad, lse2, delta, wave,
                                     kTable ? lds_dbias + wave * BiasGrad<KS>::WORDS + 4 * BiasGrad<KS>::PLANE : nullptr, dlim);
                }
            if (FULL || (lq.live && g == 0 && !(bad >> n & 1))) {
                a.delta[lq.tok] = delta;
                if constexpr (kBias) row_zinv(a)[lq.tok] = zinv;
            }
        }
        if constexpr (kTable) {
            __syncthreads();
            BiasGrad<KS>::template flush<NW>(lds_dbias, a.ds_pairs + (int64_t)sc.t * Bias<KS>::E, cur, s);
        }

        if (!more) {
            if constexpr (FULL) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), see fwd_mfma
            break;
        }
        __syncthreads();
        if constexpr (FULL) commit();
        cur = nxt;
        lq = lqn;
        sched_advance(sc, tn);
    }
}

// ------------------------------------------------------------------ dQ, one halo in LDS at a time
// The dQ pass for halos of which LDS holds two only once per CU (head_dim 64 with
// kernel_size 13): a tile is done in two phases over ONE LDS
// buffer, so that two workgroups share a CU and each SIMD has two independent waves.
//   phase 1  V rows in LDS: dP^T = V dO^T for the wave's whole halo, kept in registers;
//            the tile's K rows are in flight meanwhile and replace V behind a barrier;
//   phase 2  K rows in LDS: P from the saved log-sum-exp, delta, dS, dQ^T = K^T dS^T;
//            the next tile's V rows are in flight meanwhile.
// Four barriers per tile instead of two; 8x8 tiles, no column walk.
// Chunks of a halo that bwd_dq2_mfma loads behind the arithmetic of a phase (see fetch_tail in
// the kernel).  With 16x8 tiles at head_dim 128, kernel_size 13 a thread stages 18 chunks (72
// registers) and the kernel spilled 70 registers, freshly loaded chunks among them, each spill
// behind a wait for its load: B4 N4 128x128 167 us; with 8 chunks behind the arithmetic 125 us,
// with 12 115.5, with 15 113.4 (5 registers spilled).  kernel_size 11: 16 chunks, 36 registers
// spilled; with 8 chunks behind the arithmetic 110.6 us, with 13 107.5.
template <int D, int KS, int NW>
constexpr int kDq2Tail = D == 128 && NW == 8 ? (KS == 13 ? 15 : KS == 11 ? 13 : 0) : 0;
// Head dims between 32 and 64 with kernel_size 11 and 13 used to run with float32 P and dS on the general
// kernels.  A window's dS sum to zero, so what its keys have in common cancels in dQ, but only as far as the terms
// and delta hold (keys and values of mean 32 and deviation 1: dQ 3.9 times as far from float64 as its rounding in
// bfloat16, 30 times in float16).  So delta's own rounding error is found from the sum that it leaves (`rest`), and
// what the terms sum to is taken out of dQ with the query's own pixel in the place of every key: within 1% of the
// rounding for means up to 32, as the general kernels are.  B2 N8 128x128 d48 k13 118 -> 131 us.
// (BALANCED; head_dim 64 itself, with a bias, is built without: float16 k13 214 us, 226 with it.)
template <int D, int KS>
constexpr bool kBalanced = kBias && D == 64 && KS >= 11;
// Workgroups per CU that the registers are budgeted for: one in two terms (and float32 dS beside them),
// which spills 150 to 340 registers otherwise.  dQ pass with a bias, 16x8 tiles of eight waves, which spill too, -> 8x8
// tiles: B2 N8 128x128 d64 k11 265 -> 193 us, float16 B3 N5 61x83 91 -> 78.
template <int D, int KS, int NW>
constexpr int kDq2Wgs = NW == 4 && !(kBias && D == 64) ? kOneHaloWgs<D, KS> : 1;
// FULL: as in fwd_mfma.
template <bool BF, int D, int KS, int NW = 4, bool FULL = false, bool BALANCED = kBalanced<D, KS> && !kTable>
__global__ __launch_bounds__((Geo<D, KS, NW>::NT), (kDq2Wgs<D, KS, NW>)) void bwd_dq2_mfma(BArgs a, TileSet ts, int ntiles) {
    // (the dK/dV pass that follows on the stream counts its frame tiles here, from zero)
    if (blockIdx.x == 0 && threadIdx.x == 0 && a.zinv && kCounter) *reinterpret_cast<int *>(a.zinv) = 0;
    using G = Geo<D, KS, NW>;
    __shared__ __attribute__((aligned(16))) short lds_x[G::ROWS * G::PITCH];
    __shared__ float lds_bias[kTable ? Bias<KS>::WORDS : 1];
    __shared__ __attribute__((aligned(16))) float lds_dbias[kTable ? NW * BiasGrad<KS>::WORDS : 1];
    const Shape &s = a.s;
    const int dlim = kNarrow ? s.D : D;  // head dim of the tensors: D, or less in the build for narrow dims
    Sched sc = make_sched(ntiles, blockIdx.x, gridDim.x);
    if (sc.t >= sc.t_end) return;
    zero_row<D, KS, NW>(lds_x, dlim);  // (a commit only writes the halo's own rows)

    const int wave = FULL ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
    const int l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const float sc2 = s.scale * kUnit;
    const HaloPlan<D, KS, NW> plan = make_plan<D, KS, NW>(dlim);
    HaloRegs<D, KS, NW> st;
    // This lane's dO row is loaded a phase ahead of phase 1, its q row and log-sum-exp a
    // phase ahead of phase 2: one spare set of row registers instead of two.
    s16x8 qreg[G::DS], gnext[G::DS];
    float lse_cur = 0.f;
    BiasRegs<BF, KS, G::NT> bst;
    if constexpr (kTable) BiasGrad<KS>::template clear<G::NT>(lds_dbias);
    // The last TAIL chunks of a halo are loaded when the arithmetic of the phase is over
    // (fetch_tail): where the registers do not hold a whole halo beside it.
    constexpr int TAIL = kDq2Tail<D, KS, NW>, HEAD = G::NL - TAIL;
    auto fetch_rows = [&](const View &vw, const ATile &tl, const LaneQ &lq) __attribute__((always_inline)) {
        halo_fetch<D, KS, NW, 1, 0, HEAD>(st, plan, image_at(a, vw, tl), row_step(a, vw), col_step(a, vw), lq.hr0, lq.hc0, s.H, s.W);
    };
    auto fetch_tail = [&](const View &vw, const ATile &tl, const LaneQ &lq) __attribute__((always_inline)) {
        if constexpr (TAIL > 0)
            halo_fetch<D, KS, NW, 1, HEAD, G::NL>(st, plan, image_at(a, vw, tl), row_step(a, vw), col_step(a, vw), lq.hr0, lq.hc0, s.H, s.W);
    };
    auto fetch_do = [&](const ATile &tl, const LaneQ &lq) __attribute__((always_inline)) {
        load_row_chunks(gnext, image_at(a, a.d_o, tl) + lq.qr * row_step(a, a.d_o) + lq.qc * col_step(a, a.d_o), g, dlim);
    };
    auto fetch_q = [&](const ATile &tl, const LaneQ &lq) __attribute__((always_inline)) {
        load_row_chunks(qreg, image_at(a, a.q, tl) + lq.qr * row_step(a, a.q) + lq.qc * col_step(a, a.q), g, dlim);
        lse_cur = a.lse[lq.tok];
        if constexpr (kTable) bst.fetch(a.rpb, tl.nn);
    };

    ATile cur = in_sub(tile_of(sc.t, ts.tiles_r, ts.tiles_c, s.N, G::TH), a);
    LaneQ lq = lane_at<KS>(a, cur, wave, n);
    fetch_rows(a.v, cur, lq);
    fetch_tail(a.v, cur, lq);
    fetch_do(cur, lq);
    s16x8 greg[G::DS];
    // (V rows and the dO row at the end of a tile's pass through the loop, after its stores:
    // see fwd_mfma)
    auto commit_v = [&]() __attribute__((always_inline)) {
        halo_commit<D, KS>(lds_x, plan, st);
#pragma unroll
        for (int ds = 0; ds < G::DS; ds++) greg[ds] = gnext[ds];
    };
    if constexpr (FULL) commit_v();
    for (;;) {
        if constexpr (!FULL) commit_v();
        __syncthreads();
        fetch_rows(a.k, cur, lq);
        fetch_q(cur, lq);
        auto trow = [&](int tile, int x) __attribute__((always_inline)) { return G::token_row(tile, x, lq.orow, lq.ocol); };

        f32x4 dp[G::MT];
        if (FULL || lq.wave_on) {
#pragma unroll
            for (int mt = 0; mt < G::MT; mt++) {
                const typename G::ARow vp = G::a_row(lds_x, trow(mt, n), g);
                f32x4 cp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ds = 0; ds < G::DS; ds++)
                    cp = mfma16<BF>(*reinterpret_cast<const s16x8 *>(G::a_at(vp, ds)), greg[ds], cp);
                dp[mt] = cp;
            }
        }
        fetch_tail(a.k, cur, lq);
        __syncthreads();                      // every wave has read V
        halo_commit<D, KS>(lds_x, plan, st);  // K
        if constexpr (kTable) bst.commit(lds_bias);
        __syncthreads();

        const int tn = sched_peek(sc);
        const bool more = tn < sc.t_end;
        ATile nxt = cur;
        LaneQ lqn = lq;
        if (more) {
            nxt = in_sub(tile_of(tn, ts.tiles_r, ts.tiles_c, s.N, G::TH), a);
            lqn = lane_at<KS>(a, nxt, wave, n);
            fetch_rows(a.v, nxt, lqn);
            fetch_do(nxt, lqn);
        } else {
            if constexpr (FULL) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the last tile, nothing is loaded (see fwd_mfma)
        }
        const float lse2 = lse_cur * kUnit;
        if (FULL || lq.wave_on) {
            const int bq = kTable ? Bias<KS>::query(lq) : 0;
            Op8 dsb[G::KSTEPS];
            f32x4 ds_all[kBias ? Bias<KS>::USED : 1];  // with a bias: P, then dS, in float32
            float dpart = 0.f, zsum = 0.f;
#pragma unroll
            for (int mt = 0; mt < G::MT; mt++) {
                const typename G::ARow kp = G::a_row(lds_x, trow(mt, n), g);
                f32x4 cs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ds = 0; ds < G::DS; ds++)
                    cs = mfma16<BF>(*reinterpret_cast<const s16x8 *>(G::a_at(kp, ds)), qreg[ds], cs);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const bool ok = G::template tok_in<KS>(mt, g * 4 + i, lq.dr, lq.dc);
                    float x;
                    if constexpr (kTable) x = cs[i] * sc2 + lds_bias[bq + Bias<KS>::token(mt, g * 4 + i)] - lse2;
                    else x = cs[i] * sc2 - lse2;
                    const float p = exp_unit(ok ? x : -INFINITY);
                    if constexpr (kBias) zsum += p;
                    dpart = fmaf(p, dp[mt][i], dpart);
                    if constexpr (!kBias) put<BF>(dsb[mt >> 1], (mt & 1) * 4 + i, p);
                    else if (mt < Bias<KS>::USED) ds_all[mt][i] = p;
                }
            }
            const float zinv = kBias ? 1.f / col_sum(zsum) : 1.f;
            const float most = col_sum(dpart) * zinv;
            float rest = 0.f;  // delta = most + rest
            if constexpr (BALANCED) {
                float e = 0.f;
#pragma unroll
                for (int mt = 0; mt < Bias<KS>::USED; mt++)
#pragma unroll
                    for (int i = 0; i < 4; i++) e = fmaf(ds_all[mt][i], dp[mt][i] - most, e);
                rest = col_sum(e) * zinv;
            }
            const float delta = BALANCED ? most + rest : most;
#pragma unroll
            for (int mt = 0; mt < G::MT; mt++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if constexpr (!kBias) {
                        const float p = get<BF>(dsb[mt >> 1], (mt & 1) * 4 + i);
                        put<BF>(dsb[mt >> 1], (mt & 1) * 4 + i, p * (dp[mt][i] - most));
                    } else if (mt < Bias<KS>::USED) {
                        ds_all[mt][i] *= dp[mt][i] - most - rest;
                    }
                }
            DsScale<BF> scl;
            if constexpr (kBias) {
                operand_and_sums<BF, KS>(dsb, ds_all, scl, lq.live && delta * 0.f == 0.f ? zinv : 0.f);
                if constexpr (kTable) BiasGrad<KS>::sum(lds_dbias + wave * BiasGrad<KS>::WORDS, ds_all, n, g);
            }
            f32x4 dq[G::DT];
#pragma unroll
            for (int mt = 0; mt < G::DT; mt++) dq[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (BALANCED) {
                const short one = cvt16<BF>(1.f);
                f32x4 sum = {0.f, 0.f, 0.f, 0.f};  // (every row is the column's sum)
#pragma unroll
                for (int ks = 0; ks < G::KSTEPS; ks++) sum = mfma_op<BF>(s16x8{one, one, one, one, one, one, one, one}, dsb[ks], sum);
                // this lane's channels of the query's own pixel
                const short *own = lds_x + ((lq.qr - lq.hr0) * G::HC + lq.qc - lq.hc0) * G::PITCH + g * (D / 4);
                static_assert(!G::SWZ);
#pragma unroll
                for (int h = 0; h < G::DT / 2; h++) {
                    const s16x8 k8 = *reinterpret_cast<const s16x8 *>(own + 8 * h);
#pragma unroll
                    for (int i = 0; i < 8; i++) dq[2 * h + i / 4][i % 4] = -sum[0] * cvt32<BF>(k8[i]);
                }
            }
#pragma unroll
            for (int ks = 0; ks < G::KSTEPS; ks++) {
                typename G::TRow kp[2];
#pragma unroll
                for (int h = 0; h < 2; h++)
                    kp[h] = G::t_row(lds_x, trow(ks * 2 + h, g * 4 + (n >> 2)), n);
#pragma unroll
                for (int mt = 0; mt < G::DT; mt++)
                    dq[mt] = mfma_op<BF>(cat(lds_read_tr(G::t_at(kp[0], mt)), lds_read_tr(G::t_at(kp[1], mt))), dsb[ks],
                        dq[mt]);
            }
            const unsigned bad = kBias ? bad_columns(dq, delta) : 0u;
            store_token<BF, D, kLineStores<D, KS, kDq2Wgs<D, KS, NW>>, FULL>(static_cast<short *>(a.dq) + grad_of(a, cur, lq.qr, lq.qc), g, dq, s.scale * (kBias ? zinv * scl.inverse() : 1.f), lq.live && !(bad >> n & 1), dlim);
            if constexpr (kBias)
                if (__builtin_expect(bad != 0, 0)) {
                    BiasGrad<KS>::wave_fence();
                    again_dq<BF, KS>(a, cur, lq, bad, lse2, delta, wave,
                                     kTable ? lds_dbias + wave * BiasGrad<KS>::WORDS + 4 * BiasGrad<KS>::PLANE : nullptr, dlim);
                }
            if (FULL || (lq.live && g == 0 && !(bad >> n & 1))) {
                a.delta[lq.tok] = delta;
                if constexpr (kBias) row_zinv(a)[lq.tok] = zinv;
            }
        }
        if constexpr (kTable) {
            __syncthreads();
            BiasGrad<KS>::template flush<NW>(lds_dbias, a.ds_pairs + (int64_t)sc.t * Bias<KS>::E, cur, s);
        }
        if (more) fetch_tail(a.v, nxt, lqn);
        if (!more) {
            if constexpr (FULL) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), see fwd_mfma
            break;
        }
        __syncthreads();  // every wave has read K
        if constexpr (FULL) commit_v();
        cur = nxt;
        lq = lqn;
        sched_advance(sc, tn);
    }
}

// ------------------------------------------------------------------ dK, dV
// Key-centric: the workgroup owns an 8x8 tile of keys and stages Q, dO, the
// log-sum-exp and delta of the queries that attend to them, i.e. the union of the
// keys' inverse neighbourhoods (e_natten/pytorch.py:13-23, :261-270).  That union
// is (8+k-1)^2 queries in the interior and larger beside an image edge (the
// clamped windows of the k//2 border queries all reach k pixels in), so it is
// walked in blocks of at most (8+k-1)^2 queries; a block is the unit that is
// staged in LDS and prefetched.  Each wave owns 4x4 keys (MFMA columns) and walks
// the queries of the block that can attend to them, 32 at a time:
//   S = Q K^T, dP = dO V^T           (query rows from LDS, key columns in registers)
//   P = exp(S - lse), dS = P (dP - delta), masked to the query's own window
//   dV^T += dO^T P, dK^T += Q^T dS    (dO, Q read back from LDS transposed)
struct KeyBlock {
    int t;                // tile
    ATile tl;
    int qa, qb, ca, cb;   // queries that attend to any key of the tile
    int br, bc;           // origin of the staged block of queries
    bool first, last;     // first / last block of its tile
};
// Next block of the same tile, or false when the tile is finished.
template <int HR, int HC>
__device__ __forceinline__ bool next_block(KeyBlock &b) {
    if (b.last) return false;
    b.first = false;
    b.bc += HC;
    if (b.bc >= b.cb) {
        b.bc = b.ca;
        b.br += HR;
    }
    b.last = b.br + HR >= b.qb && b.bc + HC >= b.cb;
    return true;
}


// One step of the dK/dV pass: 32 queries (two 16-token tiles) against the wave's 16 keys.
// AHEAD says how the reads are ordered, with scheduling barriers: -1 and 0 as the compiler likes (-1: each in
// the place where it is needed, for the bias, whose inner body has no registers to spare), 1 all
// operands and statistics of a tile before its matrix instructions, 2 those of both tiles.  Left
// alone in the frame body's rolled loop the compiler reads the statistics of one query after the
// other, each behind a wait of its own for LDS, 16 round trips in a row per step at 2 waves per
// SIMD; the inner body is unrolled and has the next step's arithmetic to put between, so there 1
// and 2 only cost registers (d128 k5 with its column walk spills with them, 107 -> 222 us; not tried at
// head_dim 64), but for head_dim 32, where 2 is ahead (B4 N4 128x128 k9 51.6 -> 48.8 us).
// With a bias at head_dim 32 the 7x7 and 9x9 windows run at two waves per SIMD anyway (kDkdvWaves), which leaves
// registers for both tiles in both bodies: B8 N4 56x56 d32 k7 28.9 -> 27.6 us, B8 N2 112x112 k9 66.9 -> 66.5.
// In the build for head dims 72 to 120 the bodies with blocks of 5x5 windows (k = 3, 5, and 11 and 13, whose tiles are all
// walked by such blocks) spill 130 to 200 bytes ahead and 50 to 170 with -1: B4 N2 70x94 d96 k11 78.7 -> 62.8 us, k3 18.6 ->
// 16.4, B2 N5 128x160 k5 71 -> 60; k = 7 and 9 lose (37.3 -> 42.0).  With a bias the border tiles of d128 k3 alone gain (B8 N4 56x56
// 49.4 -> 44.0).
//   a_of(h), t_of(h): this lane's row of tile h for the direct and for the transposing reads
//   stat(h, i), at(h, i, st), in(h, i, st): statistics of query 4 g + i of tile h, the place of its
//   bias in the table, and whether it attends to this lane's key
template <int D, int KS>
constexpr bool kWideNarrow = kNarrow && !kBias && D == 128 && KS != 7 && KS != 9;
template <int D, int KS>
constexpr int kInnerAhead = (kBias && (D > 32 || KS < 7 || KS > 9)) || kWideNarrow<D, KS> ? -1 : D == 32 ? 2 : 0;
template <int D, int KS>
constexpr int kFrameAhead = kBias && D == 32 && (KS == 7 || KS == 9) ? 2 : kWideNarrow<D, KS> || (kBias && D == 128 && KS == 3) ? -1 : 1;
// FRAME: a run of four reaches up to three queries past the wave's own, whose delta may be anything: what
// no window connects with a key is left out of dS, where P = 0 times a delta that is not finite would
// be NaN.  (With a bias such keys are computed again, again_keys.)
template <bool BF, typename G, int AHEAD, bool FRAME, typename AROW, typename TROW, typename STAT, typename AT, typename IN>
__device__ __forceinline__ void dkdv_step(const short *lds_q, const short *lds_g, const float *lds_bias, int n, int g,
                                          float sc2, const s16x8 (&kreg)[G::DS], const s16x8 (&vreg)[G::DS],
                                          f32x4 (&dk)[G::DT], f32x4 (&dv)[G::DT], DsScale<BF> &scl, AROW a_of,
                                          TROW t_of, STAT stat, AT at, IN in) {
    using ST = decltype(stat(0, 0));
    constexpr bool LAZY = AHEAD < 0;  // (four floats a query: no registers to hold eight of them)
    Op8 pb, dsb;
    float dsv[8], mag = 0.f;  // (float16 with a bias)
    s16x8 qa[2][G::DS], ga[2][G::DS];
    ST st[2][4];
    auto chunk = [&](const typename G::ARow &row, int ds) __attribute__((always_inline)) {
        return *reinterpret_cast<const s16x8 *>(G::a_at(row, ds));
    };
    auto read = [&](int h) __attribute__((always_inline)) {
        if constexpr (LAZY) return;
        const int row = a_of(h);
        const typename G::ARow qp = G::a_row(lds_q, row, g), gp = G::a_row(lds_g, row, g);
#pragma unroll
        for (int ds = 0; ds < G::DS; ds++) {
            qa[h][ds] = chunk(qp, ds);
            ga[h][ds] = chunk(gp, ds);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) st[h][i] = stat(h, i);
    };
    f32x4 cs[2], cp[2];
    auto first = [&](int h) __attribute__((always_inline)) {
        const int row = LAZY ? a_of(h) : 0;
        const typename G::ARow qp = G::a_row(lds_q, row, g), gp = G::a_row(lds_g, row, g);
        cs[h] = f32x4{0.f, 0.f, 0.f, 0.f};
        cp[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ds = 0; ds < G::DS; ds++) {
            cs[h] = mfma16<BF>(LAZY ? chunk(qp, ds) : qa[h][ds], kreg[ds], cs[h]);
            cp[h] = mfma16<BF>(LAZY ? chunk(gp, ds) : ga[h][ds], vreg[ds], cp[h]);
        }
    };
    auto weights = [&](int h) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const ST q = LAZY ? stat(h, i) : st[h][i];
            const bool ok = in(h, i, q);
            float x;
            if constexpr (kTable) x = cs[h][i] * sc2 + lds_bias[ok ? at(h, i, q) : 0] - q.x;
            else x = cs[h][i] * sc2 - q.x;
            float p = exp_unit(ok ? x : -INFINITY);
            if constexpr (kBias) p *= zinv_of(q);
            put<BF>(pb, h * 4 + i, p);
            if constexpr (kBias && !BF) {
                dsv[h * 4 + i] = p * (cp[h][i] - q.y);
                mag = fmaxf(mag, fabsf(dsv[h * 4 + i]));
            } else {
                const float ds = p * (cp[h][i] - q.y);
                put<BF>(dsb, h * 4 + i, kBias || !FRAME || ok ? ds : 0.f);
            }
        }
    };
    typename G::TRow qt[2], gt[2];
    auto turn_rows = [&](int h) __attribute__((always_inline)) {
        const int row = t_of(h);
        qt[h] = G::t_row(lds_q, row, n);
        gt[h] = G::t_row(lds_g, row, n);
    };
    auto fence = [&]() __attribute__((always_inline)) {
        if constexpr (AHEAD > 0) __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (AHEAD >= 2) {
        read(0);
        read(1);
        fence();
        first(0);
        first(1);
        turn_rows(0);
        turn_rows(1);
        fence();
        weights(0);
        weights(1);
    } else {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            read(h);
            fence();
            first(h);
            if constexpr (!LAZY) turn_rows(h);
            fence();
            weights(h);
        }
#pragma unroll
        for (int h = 0; h < 2 && LAZY; h++) turn_rows(h);
    }
    if constexpr (kBias) {  // (no registers for more rows than the next product needs)
        if constexpr (!BF) put_scaled<BF>(dsb, dsv, mag, scl, dk);
#pragma unroll
        for (int mt = 0; mt < G::DT; mt++) {
            dv[mt] = mfma_op<BF>(cat(lds_read_tr(G::t_at(gt[0], mt)), lds_read_tr(G::t_at(gt[1], mt))), pb, dv[mt]);
            dk[mt] = mfma_op<BF>(cat(lds_read_tr(G::t_at(qt[0], mt)), lds_read_tr(G::t_at(qt[1], mt))), dsb, dk[mt]);
        }
    } else {
        s16x8 gr[G::DT], qr[G::DT];
#pragma unroll
        for (int mt = 0; mt < G::DT; mt++) gr[mt] = cat(lds_read_tr(G::t_at(gt[0], mt)), lds_read_tr(G::t_at(gt[1], mt)));
#pragma unroll
        for (int mt = 0; mt < G::DT; mt++) qr[mt] = cat(lds_read_tr(G::t_at(qt[0], mt)), lds_read_tr(G::t_at(qt[1], mt)));
#pragma unroll
        for (int mt = 0; mt < G::DT; mt++) dv[mt] = mfma_op<BF>(gr[mt], pb, dv[mt]);
#pragma unroll
        for (int mt = 0; mt < G::DT; mt++) dk[mt] = mfma_op<BF>(qr[mt], dsb, dk[mt]);
    }
}

// Inner tiles.  Every key is attended by exactly the queries within k//2 of it
// and all windows are centred, so the picture is the forward's with the roles of
// queries and keys exchanged: the staged block is the tile's (8+k-1)^2 halo of
// queries, a wave's queries are the (4+k-1)^2 halo of its 4x4 keys at a fixed
// place in it, and the mask depends on the lane only.
// SKIP of the dK/dV pass, as in the forward (kFwdSkip): the bodies of large windows with a bias spill less with the branch, but for
// float16 in two shares of the queries.  Pass, us, without -> with: d32 k13 B5 N6 103x86 float16 149.3 -> 140.9, B2 N5 74x91 bf16 50.5 ->
// 49.7; bf16 d64 k11 B8 N4 56x56 69.3 -> 67.3, k13 B2 N5 74x91 80.9 -> 78.1 (float16 77.5 -> 78.9).
template <bool BF, int D, int KS, int SP>
constexpr bool kDkdvSkip = kTable && (SP == 2 ? BF : D == 32 && KS == 13);
template <bool BF, int D, int KS, bool ROLL, int SP, int PART>
__device__ __forceinline__ void dkdv_inner(const BArgs &a, const TileSet &ts, int ntiles, Runs rp,
                                           int block, int nblocks, short *lds_q, short *lds_g,
                                           QStat *lds_stat, f32x4 *lds_red, float *lds_bias) {
    using G = Geo<D, KS, 4, SP>;
    const Shape &s = a.s;
    const int dlim = kNarrow ? s.D : D;  // head dim of the tensors: D, or less in the build for narrow dims
    Sched sc = ROLL ? make_runs(ntiles, block, nblocks, rp) : make_sched(ntiles, block, nblocks);
    if (sc.t >= sc.t_end) return;
    zero_row<D, KS, 4, SP>(lds_q, dlim);
    zero_row<D, KS, 4, SP>(lds_g, dlim);
    if (threadIdx.x == 0) lds_stat[G::ZROW] = QStat{};

    // wave = block of 4x4 keys (0..3) + 4 * PART; part p takes reduction steps
    // K0 = p * CH .. K1 - 1 (compile-time, so that every token's place in the halo and its
    // mask fold to constants)
    const int wave = SP == 1 ? threadIdx.x >> 6 : (threadIdx.x >> 6) & 3;
    constexpr int part = PART;
    constexpr int CH = (G::KSTEPS + SP - 1) / SP;
    constexpr int K0 = PART * CH, K1 = K0 + CH < G::KSTEPS ? K0 + CH : G::KSTEPS;
    const int l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const float sc2 = s.scale * kUnit;
    const int orow = (wave >> 1) * 4, ocol = (wave & 1) * 4;
    int rot = 0;  // ROLL: (first image row of the staged block) % HR
    auto row_of = [&](int tile, int x) __attribute__((always_inline)) {
        return ROLL ? G::token_row_rot(tile, x, orow, ocol, rot) : G::token_row(tile, x, orow, ocol);
    };
    auto pick = [&](int t) __attribute__((always_inline)) {
        return in_sub(ROLL ? inner_tile_cm(t, ts, s.N) : inner_tile(t, ts, s.N), a);
    };

    const HaloPlan<D, KS, 4, SP> plan = make_plan<D, KS, 4, SP>(dlim, kDkdvSkip<BF, D, KS, SP>);
    HaloRegs<D, KS, 4, SP> qst, gst;
    QStat sst[G::NST];
    BiasRegs<BF, KS, G::NT> bst;
    // ROLL: rows [y0, y0 + nr) of the block are what LDS does not hold yet
    auto prefetch = [&](const ATile &tl, int y0, int nr) __attribute__((always_inline)) {
        const int64_t img_tok = kSub ? image_token(a, tl) : ((int64_t)tl.bb * s.N + tl.nn) * s.H * (int64_t)s.W;
        const int br = tl.r0 - KS / 2, bc = tl.c0 - KS / 2;
        if constexpr (ROLL) {
            halo_fetch_rows<D, KS>(qst, plan, image_at(a, a.q, tl), row_step(a, a.q), col_step(a, a.q), y0, bc, nr, s.H, s.W);
            halo_fetch_rows<D, KS>(gst, plan, image_at(a, a.d_o, tl), row_step(a, a.d_o), col_step(a, a.d_o), y0, bc, nr, s.H, s.W);
        } else {
            halo_fetch<D, KS>(qst, plan, image_at(a, a.q, tl), row_step(a, a.q), col_step(a, a.q), br, bc, s.H, s.W);
            halo_fetch<D, KS>(gst, plan, image_at(a, a.d_o, tl), row_step(a, a.d_o), col_step(a, a.d_o), br, bc, s.H, s.W);
        }
#pragma unroll
        for (int i = 0; i < G::NST; i++) {
            const int id = min((int)threadIdx.x + i * G::NT, G::ZROW - 1);
            const int pr = id / G::HC, pc = id % G::HC;
            if (!ROLL || pr < nr) {
                const int64_t qt = img_tok + (int64_t)((ROLL ? y0 : br) + pr) * s.W + bc + pc;
                sst[i] = load_qstat<BF>(a, qt);
            }
        }
        if constexpr (kTable) bst.fetch(a.rpb, tl.nn);
    };
    auto commit = [&](int y0, int nr) __attribute__((always_inline)) {
        if constexpr (ROLL) {
            halo_commit_rows<D, KS>(lds_q, plan, qst, y0, nr);
            halo_commit_rows<D, KS>(lds_g, plan, gst, y0, nr);
            const int r0m = y0 % G::HR;
#pragma unroll
            for (int i = 0; i < G::NST; i++) {
                const int id = threadIdx.x + i * G::NT;
                const int pr = id / G::HC, pc = id % G::HC;
                if (id < G::ZROW && pr < nr) {
                    int slot = r0m + pr;
                    slot = slot >= G::HR ? slot - G::HR : slot;
                    lds_stat[slot * G::HC + pc] = sst[i];
                }
            }
        } else {
            halo_commit<D, KS>(lds_q, plan, qst);
            halo_commit<D, KS>(lds_g, plan, gst);
#pragma unroll
            for (int i = 0; i < G::NST; i++) {
                const int id = threadIdx.x + i * G::NT;
                if (id < G::ZROW) lds_stat[id] = sst[i];
            }
        }
        if constexpr (kTable) bst.commit(lds_bias);
    };
    // (entry of this lane's key and a token of its halo: bk - token, see Bias)
    const int bk = kTable ? ((n >> 2) + KS / 2 + KS + 2) * Bias<KS>::TB + (n & 3) + KS / 2 + KS + 2 : 0;
    // B operands of a tile: this lane's key, channels ds*32 + g*8 ..  Loaded when
    // the previous tile's math is over (they would not fit beside it) and complete
    // before the barrier below, i.e. before any newer load is in flight.
    s16x8 kreg[G::DS], vreg[G::DS];
    auto load_keys = [&](const ATile &tl) __attribute__((always_inline)) {
        const int kr = tl.r0 + orow + (n >> 2), kc = tl.c0 + ocol + (n & 3);
        load_row_chunks(kreg, image_at(a, a.k, tl) + kr * row_step(a, a.k) + kc * col_step(a, a.k), g, dlim);
        load_row_chunks(vreg, image_at(a, a.v, tl) + kr * row_step(a, a.v) + kc * col_step(a, a.v), g, dlim);
    };

    ATile cur = pick(sc.t);
    int y0 = cur.r0 - KS / 2, nr = G::HR;
    prefetch(cur, y0, nr);
    load_keys(cur);
    for (;;) {
        commit(y0, nr);
#pragma unroll
        for (int ds = 0; ds < G::DS; ds++) asm volatile("" : "+v"(kreg[ds]), "+v"(vreg[ds]));
        __syncthreads();

        const int tn = sched_peek(sc);
        const bool more = tn < sc.t_end;
        ATile nxt = cur;
        if (ROLL) rot = (cur.r0 - KS / 2) % G::HR;
        if (more) {
            nxt = pick(tn);
            // the tile below in the same image keeps the rows the two blocks share
            const bool below = ROLL && same_column(nxt, cur) &&
                               nxt.r0 > cur.r0 && nxt.r0 - cur.r0 < G::HR;
            y0 = below ? cur.r0 - KS / 2 + G::HR : nxt.r0 - KS / 2;
            nr = below ? nxt.r0 - cur.r0 : G::HR;
            prefetch(nxt, y0, nr);
        }

        f32x4 dk[G::DT], dv[G::DT];
        DsScale<BF> scl;
#pragma unroll
        for (int mt = 0; mt < G::DT; mt++) {
            dk[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
            dv[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int ks = K0; ks < K1; ks++)
            dkdv_step<BF, G, kInnerAhead<D, KS>, false>(
                lds_q, lds_g, lds_bias, n, g, sc2, kreg, vreg, dk, dv, scl,
                [&](int h) __attribute__((always_inline)) { return row_of(ks * 2 + h, n); },
                [&](int h) __attribute__((always_inline)) { return row_of(ks * 2 + h, g * 4 + (n >> 2)); },
                // query of accumulator row g*4+i
                [&](int h, int i) __attribute__((always_inline)) { return lds_stat[row_of(ks * 2 + h, g * 4 + i)]; },
                [&](int h, int i, const QStat &) __attribute__((always_inline)) {
                    return bk - Bias<KS>::token(ks * 2 + h, g * 4 + i);
                },
                [&](int h, int i, const QStat &) __attribute__((always_inline)) {
                    return G::template tok_in<KS>(ks * 2 + h, g * 4 + i, n >> 2, n & 3);
                });

        if constexpr (kBias) unscale<BF>(dk, dv, scl);
        const int kr = cur.r0 + orow + (n >> 2), kc = cur.c0 + ocol + (n & 3);
        auto store = [&]() __attribute__((always_inline)) {
            const int64_t goff = grad_of(a, cur, kr, kc);
            const unsigned bad = kBias ? bad_columns(dk) | bad_columns(dv) : 0u;
            const bool here = !(bad >> n & 1);
            store_token<BF, D, kInnerLines<D>, !kBias>(static_cast<short *>(a.dk) + goff, g, dk, s.scale, here, dlim);
            store_token<BF, D, kInnerLines<D>, !kBias>(static_cast<short *>(a.dv) + goff, g, dv, 1.f, here, dlim);
            if constexpr (kBias)
                if (__builtin_expect(bad != 0, 0)) again_keys<BF, KS>(a, cur, kr, kc, true, bad, dlim);
        };
        if constexpr (SP == 1) {
            store();
            if (!more) break;
            load_keys(nxt);
            __syncthreads();
        } else {
            // the second part hands its sums to the first through LDS; the first adds
            // and stores them once the barrier that ends the tile has passed (the
            // second part writes again only after the next tile's first barrier)
            static_assert(SP <= 2, "two parts");
            f32x4 *red = lds_red + wave * 64 + l;
            if (part == 1) {
#pragma unroll
                for (int mt = 0; mt < G::DT; mt++) {
                    red[mt * 256] = dk[mt];
                    red[(G::DT + mt) * 256] = dv[mt];
                }
            }
            if (more) load_keys(nxt);
            __syncthreads();
            if (part == 0) {
#pragma unroll
                for (int mt = 0; mt < G::DT; mt++) {
                    dk[mt] += red[mt * 256];
                    dv[mt] += red[(G::DT + mt) * 256];
                }
                store();
            }
            if (!more) break;
        }
        cur = nxt;
        sched_advance(sc, tn);
    }
}

// Frame tiles: the general case, walked block by block (see above).  KSG sets the size of a
// staged block, (8 + KSG - 1)^2 queries: KS, or more (kFrameKS) so that the queries of a
// tile in the second ring from the border, up to 16 + k/2 rows and columns of them, are
// one block instead of up to four.  `lds_red` then lies over the staged rows (RED_OVER):
// the partial sums are exchanged when a tile's last block has been read by every wave.
template <typename G>
struct FrameStat {
    static constexpr int PITCH = G::HC + 3, NONE = G::HR * PITCH, WORDS = NONE + 4;
};
template <bool BF, int D, int KS, int SP, int KSG, bool RED_OVER>
__device__ __forceinline__ void dkdv_frame(const BArgs &a, const TileSet &ts, int ntiles,
                                           int block, int nblocks, short *lds_q, short *lds_g,
                                           float4 *lds_stat, f32x4 *lds_red, int *tile_ctr, int *lds_tile,
                                           float *lds_bias) {
    using G = Geo<D, KSG, 4, SP>;
    const Shape &s = a.s;
    const int dlim = kNarrow ? s.D : D;  // head dim of the tensors: D, or less in the build for narrow dims
    // Tiles: a strided share of the XCD's run (make_sched), or, with a counter in device memory
    // that is zero when the kernel starts (`tile_ctr`), whatever tile is next when the workgroup
    // is free.  A workgroup then knows its tile and the one after it, and asks for the tile after
    // those while it works on a tile's first block, so the answer never holds it up.
    const bool dyn = tile_ctr != nullptr;
    Sched sc = make_sched(ntiles, block, nblocks);
    int t_next = sc.t + sc.step;
    if (dyn) {
        if (threadIdx.x == 0) {
            lds_tile[0] = atomicAdd(tile_ctr, 1);
            lds_tile[1] = atomicAdd(tile_ctr, 1);
        }
        __syncthreads();
        sc.t = lds_tile[0];
        t_next = lds_tile[1];
        sc.t_end = ntiles;
    }
    if (sc.t >= sc.t_end) return;
    zero_row<D, KSG, 4, SP>(lds_q, dlim);
    zero_row<D, KSG, 4, SP>(lds_g, dlim);
    // The statistics' rows are STP apart: a run of four may reach up to three columns past the
    // block, and a run past the end of the rectangle reads the four from STNO on.  The windows of
    // those are nowhere, so no key is in them.
    constexpr int STP = FrameStat<G>::PITCH, STNO = FrameStat<G>::NONE, SPARE = G::HR * 3;
    for (int id = threadIdx.x; id < SPARE + 4; id += G::NT)
        lds_stat[id < SPARE ? id / 3 * STP + G::HC + id % 3 : STNO + id - SPARE] =
            kBias ? make_float4(0.f, 0.f, 0.f, __int_as_float(0xffff0000))
                  : make_float4(0.f, 0.f, __int_as_float(0x7fff7fff), 0.f);

    // wave = block of 4x4 keys (0..3) + 4 * (its part of the block's queries)
    const int wave = (threadIdx.x >> 6) & 3, part = threadIdx.x >> 8;
    const int l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const float sc2 = s.scale * kUnit;

    const HaloPlan<D, KSG, 4, SP> plan = make_plan<D, KSG, 4, SP>(dlim);
    HaloRegs<D, KSG, 4, SP> qst, gst;
    QStat sst[G::NST];
    BiasRegs<BF, KS, G::NT> bst;
    // the wave's 4x4 keys of a tile: this lane's key pixel (clamped into the image)
    auto key_of = [&](const ATile &tl, int &kr, int &kc) __attribute__((always_inline)) {
        kr = min(tl.r0 + (wave >> 1) * 4 + (n >> 2), s.H - 1);
        kc = min(tl.c0 + (wave & 1) * 4 + (n & 3), s.W - 1);
    };
    auto stage = [&](const KeyBlock &b) __attribute__((always_inline)) {
        // (image_token without sub-grids, written out: through the function the register allocation of the
        // narrow build comes out another way, 61x83 d48 k9 float16 B3 N5 83.9 us for 83.5)
        const int64_t img_tok = kSub ? image_token(a, b.tl) : ((int64_t)b.tl.bb * s.N + b.tl.nn) * s.H * (int64_t)s.W;
        if (!kDkdvSkip<BF, D, KS, SP> || plan.on) {
            halo_fetch<D, KSG>(qst, plan, image_at(a, a.q, b.tl), row_step(a, a.q), col_step(a, a.q), b.br, b.bc, b.qb, b.cb);
            halo_fetch<D, KSG>(gst, plan, image_at(a, a.d_o, b.tl), row_step(a, a.d_o), col_step(a, a.d_o), b.br, b.bc, b.qb, b.cb);
        }
#pragma unroll
        for (int i = 0; i < G::NST; i++) {
            const int id = threadIdx.x + i * G::NT;
            const int r = min(b.br + id / G::HC, b.qb - 1), c = min(b.bc + id % G::HC, b.cb - 1);
            const int64_t qt = img_tok + (int64_t)r * s.W + c;
            sst[i] = load_qstat<BF>(a, qt);
        }
        if constexpr (kTable) bst.fetch(a.rpb, b.tl.nn);
    };
    // B operands of the tile: this lane's key, channels ds*32 + g*8 ..
    s16x8 kreg[G::DS], vreg[G::DS];
    auto load_keys = [&](const ATile &tl) __attribute__((always_inline)) {
        int kr, kc;
        key_of(tl, kr, kc);
        load_row_chunks(kreg, image_at(a, a.k, tl) + kr * row_step(a, a.k) + kc * col_step(a, a.k), g, dlim);
        load_row_chunks(vreg, image_at(a, a.v, tl) + kr * row_step(a, a.v) + kc * col_step(a, a.v), g, dlim);
    };
    auto first_of = [&](int t) __attribute__((always_inline)) {
        KeyBlock b;
        b.t = t;
        b.tl = in_sub(frame_tile(t, ts, s.N), a);
        b.qa = inv_lo(b.tl.r0, KS);
        b.qb = inv_hi(min(b.tl.r0 + 8, s.H) - 1, s.H, KS);
        b.ca = inv_lo(b.tl.c0, KS);
        b.cb = inv_hi(min(b.tl.c0 + 8, s.W) - 1, s.W, KS);
        b.br = b.qa;
        b.bc = b.ca;
        b.first = true;
        b.last = b.br + G::HR >= b.qb && b.bc + G::HC >= b.cb;
        return b;
    };

    f32x4 dk[G::DT], dv[G::DT];
    DsScale<BF> scl;
    KeyBlock cur = first_of(sc.t);
    // With one part per block (SP == 1) the loads of a block are issued when the previous
    // block's math is over and the other workgroup on the CU covers their latency
    // (keeping them in flight across the math would need registers that the two
    // accumulators do not leave).  With two parts a thread stages half as much, and the
    // next block's loads are in flight while this one is computed.
    stage(cur);
    load_keys(cur.tl);
    for (;;) {
        int fetched = 0;
        if (dyn && cur.first && threadIdx.x == 0) fetched = atomicAdd(tile_ctr, 1);
        halo_commit<D, KSG>(lds_q, plan, qst);
        halo_commit<D, KSG>(lds_g, plan, gst);
#pragma unroll
        for (int i = 0; i < G::NST; i++) {
            const int id = threadIdx.x + i * G::NT;
            // per staged query: lse * log2e, delta, and where its window starts (row in the low,
            // column in the high half of a word), so that the mask of a logit is two differences
            const int r = min(cur.br + id / G::HC, cur.qb - 1), c = min(cur.bc + id % G::HC, cur.cb - 1);
            // (columns past the tile's queries are copies of the last one: nowhere, like what lies past the block)
            const bool none = cur.bc + id % G::HC >= cur.cb;
            const int ws = none ? 0x7fff7fff : win_start(r, s.H, KS) | (win_start(c, s.W, KS) << 16);
            const int to = id / G::HC * STP + id % G::HC;
            if constexpr (kBias) {
                // (1 / Z too, and in the word of the window the query's place in a table with TB columns,
                // all from the block's origin: a window starts at most 12 rows before it)
                const int at = (id / G::HC) * Bias<KS>::TB + id % G::HC;
                const unsigned w = none ? 0xffff0000u
                                        : (unsigned)at | (unsigned)((ws & 0xffff) - cur.br + 64) << 16 |
                                              (unsigned)((ws >> 16) - cur.bc + 64) << 24;
                if (id < G::ZROW) lds_stat[to] = make_float4(sst[i].x, sst[i].y, zinv_of(sst[i]), __uint_as_float(w));
            } else {
                if (id < G::ZROW) lds_stat[to] = make_float4(sst[i].x, sst[i].y, __int_as_float(ws), 0.f);
            }
        }
        if constexpr (kTable) bst.commit(lds_bias);
        if (cur.first) {
#pragma unroll
            for (int mt = 0; mt < G::DT; mt++) {
                dk[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
                dv[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
            scl = DsScale<BF>();
        }
        __syncthreads();

        KeyBlock nxt = cur;
        bool more = next_block<G::HR, G::HC>(nxt);
        if (!more && t_next < sc.t_end) {
            nxt = first_of(t_next);
            more = true;
        }
        if constexpr (SP > 1) {
            if (more) stage(nxt);
        }
        const int wr0 = cur.tl.r0 + (wave >> 1) * 4, wc0 = cur.tl.c0 + (wave & 1) * 4;
        const bool wave_on = wr0 < s.H && wc0 < s.W;
        int kr, kc;
        key_of(cur.tl, kr, kc);
        const int bk = kTable ? (kr - cur.br + KS + 2) * Bias<KS>::TB + (kc - cur.bc + KS + 2) : 0;
        if (wave_on) {
            // this wave's queries inside the staged block: those that attend to any
            // of its 4x4 keys, numbered row-major over their rectangle
            const int ra = max(inv_lo(wr0, KS), cur.br);
            const int rb = min(inv_hi(min(wr0 + 4, s.H) - 1, s.H, KS), cur.br + G::HR);
            const int cc = max(inv_lo(wc0, KS), cur.bc);
            const int cd = min(inv_hi(min(wc0 + 4, s.W) - 1, s.W, KS), cur.bc + G::HC);
            // The rectangle is walked in runs of four queries side by side, `runs` of them per row,
            // 8 runs per step: a run has one row, so its four statistics lie side by side in LDS
            // and share the row of their windows, and one division serves all of it.
            const int wcols = cd - cc, runs = (wcols + 3) >> 2;
            const int nu = (rb > ra && cd > cc) ? (rb - ra) * runs : 0;
            // u * magic >> 16 == u / runs for u < 2048, runs <= 8
            const int magic = wcols > 0 ? (65536 + runs - 1) / runs : 0;
            const int row0 = (ra - cur.br) * G::HC + cc - cur.bc, stat0 = (ra - cur.br) * STP + cc - cur.bc;
            // staged row of query x of run u (the zero row past the end of the rectangle)
            auto row_of = [&](int u, int x) __attribute__((always_inline)) {
                const int r = (u * magic) >> 16, c = (u - r * runs) * 4 + x;
                return ((u < nu) & (c < wcols)) ? row0 + r * G::HC + c : (int)G::ZROW;
            };
            for (int u0 = part * 8; u0 < nu; u0 += 8 * SP) {
                int at_run[2];
                bool row_in[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int u = u0 + h * 4 + g, r = (u * magic) >> 16;
                    at_run[h] = u < nu ? stat0 + r * STP + (u - r * runs) * 4 : (int)STNO;
                }
                dkdv_step<BF, G, kFrameAhead<D, KS>, true>(
                    lds_q, lds_g, lds_bias, n, g, sc2, kreg, vreg, dk, dv, scl,
                    [&](int h) __attribute__((always_inline)) { return row_of(u0 + h * 4 + (n >> 2), n & 3); },
                    [&](int h) __attribute__((always_inline)) { return row_of(u0 + h * 4 + g, n >> 2); },
                    [&](int h, int i) __attribute__((always_inline)) { return lds_stat[at_run[h] + i]; },
                    [&](int, int, const float4 &st) __attribute__((always_inline)) {
                        return bk - (int)(__float_as_uint(st.w) & 0xffffu);
                    },
                    [&](int h, int i, const float4 &st) __attribute__((always_inline)) {
                        const unsigned w = __float_as_uint(kBias ? st.w : st.z);
                        if constexpr (kBias) {
                            if (i == 0) row_in[h] = (unsigned)(kr - cur.br + 64) - (w >> 16 & 0xffu) < (unsigned)KS;
                            return row_in[h] & ((unsigned)(kc - cur.bc + 64) - (w >> 24) < (unsigned)KS);
                        } else {
                            if (i == 0) row_in[h] = (unsigned)(kr - (int)(w & 0xffffu)) < (unsigned)KS;
                            return row_in[h] & ((unsigned)(kc - ((int)w >> 16)) < (unsigned)KS);
                        }
                    });
            }
        }

        // (read below, behind the barrier that ends this block; the first block of the next tile
        // writes it again behind the barrier that opens its arithmetic)
        if (dyn && cur.first && threadIdx.x == 0) lds_tile[0] = fetched;
        const bool live = (wr0 + (n >> 2) < s.H) && (wc0 + (n & 3) < s.W);
        if constexpr (kBias)
            if (cur.last) unscale<BF>(dk, dv, scl);
        auto store = [&]() __attribute__((always_inline)) {
            const int64_t goff = grad_of(a, cur.tl, kr, kc);
            const unsigned bad = kBias ? bad_columns(dk) | bad_columns(dv) : 0u;
            const bool here = live && !(bad >> n & 1);
            store_token<BF, D, kLineStores<D, KS, fits<D, KS>() ? Geo<D, KS, 4, SP>::WAVES : 1>>(static_cast<short *>(a.dk) + goff, g, dk, s.scale, here, dlim);
            store_token<BF, D, kLineStores<D, KS, fits<D, KS>() ? Geo<D, KS, 4, SP>::WAVES : 1>>(static_cast<short *>(a.dv) + goff, g, dv, 1.f, here, dlim);
            if constexpr (kBias)
                if (__builtin_expect(bad != 0, 0)) again_keys<BF, KS>(a, cur.tl, kr, kc, live, bad, dlim);
        };
        if constexpr (SP == 1) {
            if (cur.last) store();
            if (!more) break;
            stage(nxt);
            if (nxt.first) load_keys(nxt.tl);
            __syncthreads();
        } else {
            // the second part's sums reach the first through LDS (see dkdv_inner)
            f32x4 *red = lds_red + wave * 64 + l;
            if (RED_OVER && cur.last) __syncthreads();  // every wave has read the block
            if (cur.last && part == 1) {
#pragma unroll
                for (int mt = 0; mt < G::DT; mt++) {
                    red[mt * 256] = dk[mt];
                    red[(G::DT + mt) * 256] = dv[mt];
                }
            }
            if (more && nxt.first) load_keys(nxt.tl);
            __syncthreads();
            if (cur.last && part == 0) {
#pragma unroll
                for (int mt = 0; mt < G::DT; mt++) {
                    dk[mt] += red[mt * 256];
                    dv[mt] += red[(G::DT + mt) * 256];
                }
                store();
            }
            if (!more) break;
            if (RED_OVER && cur.last) __syncthreads();  // the sums are read: the next block may land
            // (the channels that the tensors do not have are zero again in the rows the sums lay over)
            if (kNarrow && RED_OVER && cur.last && dlim < D) zero_row<D, KSG, 4, SP>(lds_q, dlim);
        }
        if (nxt.first) t_next = dyn ? lds_tile[0] : nxt.t + sc.step;  // the tile after the next one
        cur = nxt;
    }
}

// One launch for the whole dK/dV pass: the first `inner_blocks` workgroups sweep
// the inner tiles, the rest the frame tiles, so the two kinds of work overlap on
// every CU and end together.
// SP = 2: eight waves, two per 4x4 block of keys (see Geo), for halos that leave LDS for
// one workgroup per CU.
// Waves per SIMD that the dK/dV pass budgets its registers for: three where LDS admits
// three workgroups per CU (head_dim <= 64 with small halos; it fits 168 registers there,
// measured 35 -> 32 us at B8 N2 112x112 d32 k7 and 67 -> 60 us at B4 N4 128x128 d32 k9;
// the forward and the dQ pass spill under that budget and get slower).  With a bias this pass
// spills too, at head_dim 64 and from kernel_size 7 on: two and three waves B8 N8 64x64 d64 k5 60
// us and 84, B8 N4 56x56 d32 k7 28.6 and 34.4, but B8 N2 112x112 d32 k5 34.1 and 27.1.
// Size of the frame body's blocks as a kernel size (see dkdv_frame): larger than KS where the
// pass has one workgroup per CU anyway (two parts per block) and LDS has the room.
// Where not even one workgroup's Q and dO halos fit LDS (head_dim 128 with kernel_size 11 and
// 13), the pass has no inner body: EVERY tile is walked by the frame body in blocks of 12x12
// queries (78 KB for both tensors, two workgroups per CU), four to nine blocks per tile.
template <int D, int KS>
constexpr bool kDkdvFrameOnly = !fits<D, KS>();
template <int D, int KS, int SP>
constexpr int kFrameKS = kDkdvFrameOnly<D, KS> ? 5 : SP == 2 && KS >= 9 ? 9 + KS / 2 : KS;
// In the builds for narrow heads
// and sub-grids head_dim 64, k = 3 spills 100 to 148 bytes in three and runs in two: d48 B4 N4 128x128 42.2 -> 35.5 us, 61x83
// float16 16.9 -> 12.9; k = 5 (148 bytes) 44.7 -> 36.5 and 22.8 -> 16.1.
template <int D, int KS, int SP>
constexpr int kDkdvWaves =
    kDkdvFrameOnly<D, KS> ? 2 : kNarrow && !kBias && D == 64 && KS <= 5 ? 2 :
    SP == 1 && D <= (kBias ? KS <= 5 ? 32 : 0 : 64) && 3 * (Geo<D, KS>::LDS_BYTES + 2048) <= 160 * 1024 ? 3 : Geo<D, KS, 4, SP>::WAVES;
// head_dim 32, k = 5: a second build for four waves per SIMD (12 bytes of scratch) where there are more tiles than its four workgroups
// per CU take at once, with the workgroups shared out by share_inner at weight 2.6, from the times of every split of 54 calls:
// 8% faster in the mean (B8 N16 63x93 66.6 -> 57.9 us, B4 N8 128x128 40.7 -> 36.3, B8 N2 112x112 16.4 -> 16.1).  In proportion they
// lost where both sides come to whole tiles unevenly (B8 N2 112x112 16.8, B7 N5 127x115 43.5 -> 45.3), and fewer tiles lose to the
// scratch alone (B3 N16 21x32 6.9 -> 7.2).  At k = 7 they spill (B8 N2 112x112 22.4 -> 26.8).
template <int D, int KS>
constexpr bool kFourWaves = !kNarrow && D == 32 && KS == 5;
template <bool BF, int D, int KS, bool ROLL, int SP = 1, int WAVES = kDkdvWaves<D, KS, SP>>
__global__ __launch_bounds__((Geo<D, KS, 4, SP>::NT), WAVES) void bwd_dkdv_mfma(
    BArgs a, TileSet ts, int n_inner, int n_frame, int inner_blocks, Runs rp, int dyn) {
    using G = Geo<D, KS, 4, SP>;
    using FG = Geo<D, kFrameKS<D, KS, SP>, 4, SP>;  // blocks of the frame body
    // One LDS buffer, laid out by each body for itself: staged Q rows, staged dO rows,
    // (lse * log2e, delta) per staged query, and with two parts per block the second part's
    // partial dK and dV.  Where the frame body stages larger blocks, its partial sums lie
    // over its Q rows.
    constexpr bool FRAME_ONLY = kDkdvFrameOnly<D, KS>;
    constexpr bool RED_OVER = !std::is_same<FG, G>::value && !FRAME_ONLY;
    constexpr size_t RED = SP > 1 ? (size_t)2 * G::DT * 256 * sizeof(f32x4) : 0;
    constexpr size_t I_ROWS = FRAME_ONLY ? 0 : (size_t)G::ROWS * G::PITCH * sizeof(short);
    constexpr size_t F_ROWS = (size_t)FG::ROWS * FG::PITCH * sizeof(short);
    constexpr size_t I_STAT = FRAME_ONLY ? 0 : (G::ROWS * sizeof(QStat) + 15) / 16 * 16;
    constexpr size_t F_STAT = FrameStat<FG>::WORDS * sizeof(float4);
    constexpr size_t I_ALL = 2 * I_ROWS + I_STAT + RED;
    constexpr size_t F_ALL = 2 * F_ROWS + F_STAT + (RED_OVER ? 0 : RED);
    static_assert(RED <= F_ROWS || !RED_OVER, "the partial sums lie over the staged Q rows");
    __shared__ __attribute__((aligned(16))) char lds_raw[I_ALL > F_ALL ? I_ALL : F_ALL];
    static_assert(sizeof(lds_raw) <= 160 * 1024, "LDS");
    // dyn: the frame tiles are dealt out as workgroups become free, the inner workgroups joining
    // when their walk is over; the counter lies where the general kernels keep 1 / Z per query,
    // and the dQ pass, which runs before this one on the stream, has cleared it.
    __shared__ int lds_tile[2];
    __shared__ float lds_bias[kTable ? Bias<KS>::WORDS : 1];
    int *tile_ctr = dyn ? reinterpret_cast<int *>(a.zinv) : nullptr;
    if constexpr (!FRAME_ONLY) {
        if ((int)blockIdx.x < inner_blocks) {
            short *lds_q = reinterpret_cast<short *>(lds_raw);
            short *lds_g = reinterpret_cast<short *>(lds_raw + I_ROWS);
            QStat *lds_stat = reinterpret_cast<QStat *>(lds_raw + 2 * I_ROWS);
            f32x4 *lds_red = reinterpret_cast<f32x4 *>(lds_raw + 2 * I_ROWS + I_STAT);
            if (SP == 1 || threadIdx.x < 256)
                dkdv_inner<BF, D, KS, ROLL, SP, 0>(a, ts, n_inner, rp, blockIdx.x, inner_blocks, lds_q,
                                                   lds_g, lds_stat, lds_red, lds_bias);
            else  // the same number of barriers as the first part
                dkdv_inner<BF, D, KS, ROLL, SP, SP - 1>(a, ts, n_inner, rp, blockIdx.x, inner_blocks,
                                                        lds_q, lds_g, lds_stat, lds_red, lds_bias);
            if (!dyn) return;
            __syncthreads();
        }
    }
    {
        short *lds_q = reinterpret_cast<short *>(lds_raw);
        short *lds_g = reinterpret_cast<short *>(lds_raw + F_ROWS);
        float4 *lds_stat = reinterpret_cast<float4 *>(lds_raw + 2 * F_ROWS);
        f32x4 *lds_red = reinterpret_cast<f32x4 *>(RED_OVER ? lds_raw : lds_raw + 2 * F_ROWS + F_STAT);
        dkdv_frame<BF, D, KS, SP, kFrameKS<D, KS, SP>, RED_OVER>(
            a, ts, n_frame, dyn ? blockIdx.x : blockIdx.x - inner_blocks,
            dyn ? gridDim.x : gridDim.x - inner_blocks, lds_q, lds_g, lds_stat, lds_red, tile_ctr, lds_tile, lds_bias);
    }
}

// ------------------------------------------------------------------ dispatch

// Keeping shared halo rows in LDS pays where the kernels are bound by the bytes
// they pull through the CU's memory pipeline (d = 128) and a workgroup walks at
// least a few tiles down a column; elsewhere its extra address arithmetic costs
// more than the loads it saves (measured), so it is only built for d = 128.
template <int D>
constexpr bool kRollBuilt = D == 128;
template <int D>
bool roll_pays(int64_t ntiles, int grid) {
    return kRollBuilt<D> && ntiles >= (int64_t)4 * grid;
}

// Eight waves on a 16x8 tile instead of four on an 8x8 tile, for head_dim 64 with
// kernel_size >= 7 where the taller tile's halo fits LDS: a fifth to a third less halo
// per pixel, and at k = 11 and 13, where the halo of an 8x8 tile leaves LDS for one
// workgroup per CU, two waves per SIMD instead of one.  Measured at B4 N4 128x128
// (8x8 -> 16x8, us): forward 40 -> 39 (k=7), 76 -> 53 (k=11), 82 -> 55 (k=13); dQ pass
// 59 -> 48 (k=7), 82 -> 59 (k=9).  Not used where it was measured slower or no faster:
// k <= 5, head_dim 32, and the dQ pass at k = 11 and 13, where the pass with one halo in
// LDS at a time (bwd_dq2_mfma) is faster (k = 11: 87 us against 75; at k = 13 the 16x8
// tiles spill).
template <int D, int KS>
constexpr bool kTallBuilt =
    D == 64 && KS >= 7 &&
    (size_t)2 * Geo<D, KS, 8>::ROWS * Geo<D, KS, 8>::PITCH * sizeof(short) +
            (kTable ? Bias<KS>::WORDS * sizeof(float) : 0) <= 160 * 1024;
template <int D, int KS>
constexpr bool kTallDqBuilt = kTallBuilt<D, KS> && KS <= (kBias ? 7 : 9);  // (a bias's planes take LDS too)

// The dQ pass with one halo in LDS at a time (bwd_dq2_mfma): where two halos leave LDS for
// one workgroup per CU, one halo fits twice, and the 16x8 tiles are not used.  head_dim 64
// (kernel_size 11 and 13): 96 -> 79 us at B2 N8 128x128 k = 13; k = 11, against the 16x8
// tiles: 87.3 -> 75.2 us at B4 N4 128x128, 380 -> 296 at 256x256, 27.0 -> 23.1 at B2 N8 64x64.  head_dim 128 (kernel_size 7 and 9), B4 N4
// 128x128: 110.6 -> 72.2 us and 123.8 -> 80.3; B8 N8: 431 -> 302; B2 N2 64x64: 10.9 -> 10.1.
template <int D, int KS>
constexpr bool kDq2Built = (D == 64 || D == 128) && Geo<D, KS>::WAVES == 1 && !kTallDqBuilt<D, KS> &&
                           kOneHaloFits<D, KS>;

// The forward with one halo in LDS at a time (fwd2_mfma), for head_dim 128 where two halos
// leave LDS for one workgroup per CU (kernel_size 7 and 9).  Launched where the tiles give
// every CU its two workgroups (us, fwd_mfma -> fwd2_mfma, bf16, 128x128 images): k = 7
// B1 N2 14.1 -> 12.5, B1 N4 26.3 -> 20.3, B4 N4 91.8 -> 60.5, B8 N8 364 -> 245; k = 9
// B1 N4 28.0 -> 22.4, B4 N4 106.6 -> 68.5.  With fewer tiles fwd_mfma's single workgroup
// per CU is faster (B2 N2 64x64: 9.3 us against 9.9).  At head_dim 64 (kernel_size 11, 13)
// the 16x8 tiles of fwd_mfma are faster (57.8 us against 59.3, 61.6 against 69.5).
// 16x8 tiles with eight waves for the one-halo kernels where an 8x8 tile's halo leaves LDS for one
// workgroup of four waves per CU (head_dim 128, kernel_size 11 and 13) and the taller halo still
// fits (128 and 153 KB): two waves per SIMD instead of one, and a quarter less halo per pixel.
// B4 N4 128x128, us, 8x8 -> 16x8: forward k13 137.8 -> 104.5 (B8 N8: 526 -> 385), k11 143.4 -> 130.4;
// dQ pass k13 179.7 -> 167.7 (B8 N8: 736 -> 642), k11 185.2 -> 190.4 while it spilled 70 and 36
// registers there; with the last chunks of a halo loaded behind the arithmetic (kDq2Tail) it
// does not, and the tall tiles take k13 to 113 us and k11 to 107.5 (174 with 8x8 tiles; B8 N8:
// 700 -> 426).
template <int D, int KS>
constexpr bool kFwd2TallBuilt = D == 128 && kOneHaloWgs<D, KS> == 1 && kOneHaloFits<D, KS> &&
                                (size_t)Geo<D, KS, 8>::ROWS * Geo<D, KS, 8>::PITCH * 2 + 1024 <= 160 * 1024;
// At head_dim 64 (kernel_size 11 and 13, where one halo of an 8x8 tile fits LDS twice) the one-halo dQ
// pass takes the 16x8 tiles too: one workgroup of eight waves instead of two of four, a quarter less halo
// per pixel.  (Not in two terms: the 8x8 tiles have one workgroup per CU and all its registers there.)
// B2 N8 128x128 k13 81.5 -> 76.2 us, B4 N8 256x256 626 -> 606, B4 N4 128x128 k11 77.1 -> 76.3.
template <int D, int KS>
constexpr bool kDq2TallBuilt = !kBias && (kFwd2TallBuilt<D, KS> || (D == 64 && KS >= 11));
template <int D, int KS>
constexpr bool kFwd2Built = D == 128 && Geo<D, KS>::WAVES == 1 && kOneHaloFits<D, KS>;
// Built at all: two halos fit, or the one-halo kernels serve the forward and the dQ pass and
// the frame body in small blocks the dK/dV pass
template <int D, int KS>
constexpr bool kBuilt = kBias && !kTable ? D == 64 && KS >= 11 : fits<D, KS>() || (kFwd2Built<D, KS> && kDq2Built<D, KS>);

// A frame tile's time in inner tiles in the dK/dV pass, as the choice of the split takes it (bwd_launch).  At
// head_dim 128 the walks of the inner side are a staircase, and so are the times: with weights 1.0 to 2.0 over
// ten image sizes from 56x56 to 256x256, with a bias and without, these lose no size 3% against any other that gains on most.
// k9 2.0 -> 1.9: B4 N4 128x128 173 -> 158 us, 112x112 142 -> 120, B4 N8 96x96 215 -> 183, with a bias 277 -> 250, 224 ->
// 189, 342 -> 293, others level; (1.7 and 1.8 gain there too and lose B1 N4 90x140 20%).  k3 1.3 -> 1.4: B3 N5 61x83 23.3 ->
// 21.6, with a bias 49 -> 40; k5 1.45 -> 1.5: 75x75 20.2 -> 16.8; others level.
template <int KS>
constexpr double kFrameCost128 = KS >= 9 ? 1.9 : KS == 7 ? 1.3 : KS == 5 ? 1.5 : 1.4;
// ... and below that, measured by timing every split at eleven image sizes from 40x40 to 256x256, batch times
// heads 4 to 64.  Without a bias 2 at head_dim 64 (1.68 with the frame body's larger blocks) and 2.5 at head_dim 32
// are within 2% of the best weight in the mean.  With a bias an inner tile is dearer against a frame tile: dK/dV pass with the
// weights below and share_inner against 2, 1.68 and 2.5 in proportion, in the mean over the sizes, bf16 / float16, head_dim
// 64 k3 -6 / -6%, k5 -3 / -5, k7 -6 / -5, k9 -10 / -11, k11 -5 / -3, k13 -3 / 0, head_dim 32 k3 -2, k5 -2 / -2, k7 -8 / -7,
// k11 -10 / -10, k13 -13 / -10; the size that loses most 7% (B4 N4 96x96 d64 k5).  (k9 at head_dim 32: every other weight loses some size
// 6 to 13%.)
template <bool BF, int D, int KS>
constexpr double kFrameCostBias = D == 64 ? (KS == 13 && (!BF || !kTable) ? 1.75 : 1.5)
                                          : KS == 3 ? 2.1 : KS == 5 ? 2.3 : KS == 7 ? 2.0 : KS == 9 ? 2.5 : 1.9;
template <bool BF, int D, int KS, bool LARGE>
constexpr double kFrameCost = D >= 128 ? kFrameCost128<KS>
                              : kBias ? kFrameCostBias<BF, D, KS>
                              : LARGE ? 1.68 : D == 32 ? 2.5 : 2.0;
// With a bias, of `grid` workgroups those on inner tiles.  A workgroup has whole tiles, so a share in proportion may
// leave one side a tile longer than the other; whole tiles alone would not count that workgroups which end early
// leave the CU to the others.  So it is the split whose longer side is the shortest by the mean of both: level with the
// proportion at head_dim 64, 2% faster in the mean at head_dim 32 (B8 N4 56x56 d32 k7 26.4 -> 21.4 us).
inline int share_inner(int64_t n_inner, int64_t n_frame, int grid, double cost) {
    const int64_t per_i = (n_inner + 7) / 8, per_f = (n_frame + 7) / 8;
    double best = 1e30;
    int inner = 8;
    for (int ib = 8; ib <= grid - 8 && ib <= per_i * 8; ib += 8) {
        auto side = [](int64_t tiles, int64_t slots) { return (double)tiles / slots + (double)((tiles + slots - 1) / slots); };
        const double i = side(per_i, ib / 8), f = cost * side(per_f, (grid - ib) / 8), t = i > f ? i : f;
        if (t < best) {
            best = t;
            inner = ib;
        }
    }
    return inner;
}
template <int D, int KS>
constexpr int kDkdvSplit = D == 64 && Geo<D, KS>::WAVES == 1 ? 2 : 1;

template <bool BF, int D, int KS>
int fwd_launch(const FArgs &a, hipStream_t st) {
    if constexpr (kBuilt<D, KS>) {
        using G = Geo<D, KS>;
        const int tiles_r = (a.s.H + G::TH - 1) / G::TH, tiles_c = (a.s.W + G::TW - 1) / G::TW;
        const int64_t nb = images_of(a) * tiles_r * tiles_c;
        if constexpr (kTallBuilt<D, KS>) {
            using G8 = Geo<D, KS, 8>;
            const int tall_r = (a.s.H + G8::TH - 1) / G8::TH;
            const int64_t nb8 = images_of(a) * tall_r * tiles_c;
            if (nb8 >= 512) {  // enough tall tiles for every CU to have a few
                const int grid = persistent_grid<fwd_mfma<BF, D, KS, false, 8>>(nb8, G8::NT);
                ProfScope prof(ENATTEN_KERNEL_FWD, "fwd_mfma", st);
                if (!kNarrow && a.s.H % G8::TH == 0 && a.s.W % G8::TW == 0)
                    hipLaunchKernelGGL((fwd_mfma<BF, D, KS, false, 8, !kNarrow>), dim3(grid), dim3(G8::NT), 0,
                                       st, a, tall_r, tiles_c, (int)nb8, Runs{0, 0});
                else
                    hipLaunchKernelGGL((fwd_mfma<BF, D, KS, false, 8>), dim3(grid), dim3(G8::NT), 0, st, a,
                                       tall_r, tiles_c, (int)nb8, Runs{0, 0});
                return check_launch("enatten2d_fwd");
            }
        }
        if constexpr (kFwd2TallBuilt<D, KS>) {
            using G8 = Geo<D, KS, 8>;
            const int tall_r = (a.s.H + G8::TH - 1) / G8::TH;
            const int64_t nb8 = images_of(a) * tall_r * tiles_c;
            if (nb8 >= 256) {  // a tile for every CU
                const int grid = persistent_grid<fwd2_mfma<BF, D, KS, 8>>(nb8, G8::NT);
                ProfScope prof(ENATTEN_KERNEL_FWD, "fwd2_mfma", st);
                if (!kNarrow && a.s.H % G8::TH == 0 && a.s.W % G8::TW == 0)
                    hipLaunchKernelGGL((fwd2_mfma<BF, D, KS, 8, !kNarrow>), dim3(grid), dim3(G8::NT), 0, st, a,
                                       tall_r, tiles_c, (int)nb8);
                else
                    hipLaunchKernelGGL((fwd2_mfma<BF, D, KS, 8>), dim3(grid), dim3(G8::NT), 0, st, a, tall_r,
                                       tiles_c, (int)nb8);
                return check_launch("enatten2d_fwd");
            }
        }
        if constexpr (kFwd2Built<D, KS>) {
            const int grid = persistent_grid<fwd2_mfma<BF, D, KS>>(nb);
            if (nb >= 2 * 256 || !fits<D, KS>()) {  // two workgroups for each of the 256 CUs
                ProfScope prof(ENATTEN_KERNEL_FWD, "fwd2_mfma", st);
                if (!kNarrow && a.s.H % G::TH == 0 && a.s.W % G::TW == 0)
                    hipLaunchKernelGGL((fwd2_mfma<BF, D, KS, 4, !kNarrow>), dim3(grid), dim3(256), 0, st, a,
                                       tiles_r, tiles_c, (int)nb);
                else
                    hipLaunchKernelGGL((fwd2_mfma<BF, D, KS>), dim3(grid), dim3(256), 0, st, a, tiles_r,
                                       tiles_c, (int)nb);
                return check_launch("enatten2d_fwd");
            }
        }
        if constexpr (fits<D, KS>()) {
            const int grid = persistent_grid<fwd_mfma<BF, D, KS, false>>(nb);
            ProfScope prof(ENATTEN_KERNEL_FWD, "fwd_mfma", st);
            const bool full = !kNarrow && a.s.H % G::TH == 0 && a.s.W % G::TW == 0;
            if (roll_pays<D>(nb, grid)) {
                if (full)
                    hipLaunchKernelGGL((fwd_mfma<BF, D, KS, kRollBuilt<D>, 4, !kNarrow>), dim3(grid), dim3(256),
                                       0, st, a, tiles_r, tiles_c, (int)nb, plan_runs(nb, grid, tiles_r));
                else
                    hipLaunchKernelGGL((fwd_mfma<BF, D, KS, kRollBuilt<D>>), dim3(grid), dim3(256), 0,
                                       st, a, tiles_r, tiles_c, (int)nb, plan_runs(nb, grid, tiles_r));
            } else if (full) {
                hipLaunchKernelGGL((fwd_mfma<BF, D, KS, false, 4, !kNarrow>), dim3(grid), dim3(256), 0, st, a,
                                   tiles_r, tiles_c, (int)nb, Runs{0, 0});
            } else {
                hipLaunchKernelGGL((fwd_mfma<BF, D, KS, false>), dim3(grid), dim3(256), 0, st, a,
                                   tiles_r, tiles_c, (int)nb, Runs{0, 0});
            }
        }
        return check_launch("enatten2d_fwd");
    } else {
        set_error("no matrix-core kernel for head_dim %d, kernel_size %d", D, KS);
        return ENATTEN_EUNSUPPORTED;
    }
}

// Where the FULL form of bwd_dq2_mfma is used: at head_dim 128 it was measured faster with
// kernel_size 7 and 11 (B4 N4 128x128: 76.7 -> 68.2 and 184.7 -> 173.2 us) and slower with 9
// and 13 (82.4 -> 84.4, and 167.5 -> 214.7 with the 16x8 tiles: what those two spill moves
// into their inner loops); at head_dim 64 faster (k11 76.2 -> 73.9, k13 76.2 -> 75.6).
template <int D, int KS>
constexpr bool kDq2Full = !kNarrow && (D != 128 || KS == 7 || KS == 11);

// bwd_launch's `path` of a call with a bias whose gradient is of the tensors' type (else 0)
constexpr int kRpbTyped = 1 << 8;
template <bool BF, int D, int KS>
int bwd_launch(const BArgs &a, int path, hipStream_t st) {
    if constexpr (kBuilt<D, KS>) {
        using G = Geo<D, KS>;
        const int tiles_r = (a.s.H + G::TH - 1) / G::TH, tiles_c = (a.s.W + G::TW - 1) / G::TW;
        const int64_t nb = images_of(a) * tiles_r * tiles_c;
        // inner tiles (no key or query within reach of the border) and frame
        TileSet ts;
        ts.tiles_r = tiles_r; ts.tiles_c = tiles_c;
        // (tile row tr, keys 8 tr .. 8 tr + 7, is inner when no query with a clamped window
        // attends to its keys: the queries of rows 0 .. k/2 - 1 reach the keys of rows 0 .. k - 1,
        // so 8 tr >= k, and 8 tr + 7 <= H - 1 - k at the other end)
        ts.ir0 = (KS + 7) / 8; ts.ic0 = (KS + 7) / 8;
        ts.ni_r = (a.s.H - KS) / 8 - ts.ir0; ts.ni_c = (a.s.W - KS) / 8 - ts.ic0;
        if (ts.ni_r <= 0 || ts.ni_c <= 0 || kDkdvFrameOnly<D, KS>) {
            ts.ir0 = tiles_r; ts.ic0 = 0; ts.ni_r = 0; ts.ni_c = 0;
        }
        const int64_t slabs = images_of(a);
        const int64_t n_inner = slabs * ts.ni_r * ts.ni_c, n_frame = nb - n_inner;

        // The fused backward wherever it is built (fused_bwd_supported): 5-25% faster than the
        // two passes at every size measured, from B64 N16 8x8 (45.7 against 47.3 us) and B4 N4
        // 32x32 (14.8 against 24.1) to B16 N8 128x128 (938 against 1174).
        if (!kSub && !kBias && !split_forced(path) && fused_bwd_supported(a)) {
            const int rc = launch_bwd_fused(a, BF, ts, nb, st);
            return rc ? rc : check_launch("enatten2d_bwd");
        }

        // The one-pass backward (head_dim 32, and 64 with kernel_size 3; na2d_mfma_onepass.hip).
        // At these head dims the passes are bound by per-tile latency, not by HBM, so reading
        // the inputs once only pays where the two passes are at their worst: images that are
        // (nearly) all border tiles, which the dK/dV pass walks block by block and the one-pass
        // kernel serves from its one staged block.  Measured on a settled GPU, backward kernels,
        // one pass vs two (us, bf16, head_dim 32, kernel_size 7): B8 N16 14x14 17.2 vs 13.2;
        // B8 N8 28x28 24.9 vs 24.8; B8 N4 40x40 22.0 vs 16.1 (9 of 25 tiles inner); B8 N4 56x56
        // 32.6 vs 26.4; B8 N2 112x112 51.4 vs 42.8.  The whole step replayed as a graph, where
        // one launch less counts: 14x14 30.3 vs 29.0, 28x28 39.2 vs 40.7, 40x40 37.8 vs 32.9,
        // 56x56 52.7 vs 49.0.  So it is the default only where at most one tile in eight is an
        // inner tile (level with the two passes there, one launch less);
        // ENATTEN_PATH_MFMA_FUSED forces it wherever it is built.
        if (!kSub && !kBias && !split_forced(path) && onepass_bwd_supported(a) &&
            (path == ENATTEN_PATH_MFMA_FUSED || 8 * n_inner <= nb)) {
            const int rc = launch_bwd_onepass(a, BF, ts, nb, st);
            return rc ? rc : check_launch("enatten2d_bwd");
        }

        bool dq_done = false;
        int dq_tiles = tiles_r * tiles_c;  // per image, of the dQ pass
        if constexpr (kDq2TallBuilt<D, KS>) {
            using G8 = Geo<D, KS, 8>;
            TileSet tall = ts;  // only the tile counts are used by this pass
            tall.tiles_r = (a.s.H + G8::TH - 1) / G8::TH;
            const int64_t nb8 = slabs * tall.tiles_r * tiles_c;
            if (nb8 >= 256) {
                const int grid = persistent_grid<bwd_dq2_mfma<BF, D, KS, 8>>(nb8, G8::NT);
                ProfScope prof(ENATTEN_KERNEL_BWD_DQ, "bwd_dq2_mfma", st);
                if (kDq2Full<D, KS> && a.s.H % G8::TH == 0 && a.s.W % G8::TW == 0)
                    hipLaunchKernelGGL((bwd_dq2_mfma<BF, D, KS, 8, kDq2Full<D, KS>>), dim3(grid), dim3(G8::NT), 0,
                                       st, a, tall, (int)nb8);
                else
                    hipLaunchKernelGGL((bwd_dq2_mfma<BF, D, KS, 8>), dim3(grid), dim3(G8::NT), 0, st, a, tall,
                                       (int)nb8);
                dq_done = true;
                dq_tiles = tall.tiles_r * tiles_c;
            }
        }
        if constexpr (kDq2Built<D, KS>) {
            if (!dq_done) {
                // (without a table only dims below D come here, and the default is that)
                const bool balanced = kBalanced<D, KS> && a.s.D < D;
                const int grid = balanced ? persistent_grid<bwd_dq2_mfma<BF, D, KS, 4, false, kBalanced<D, KS>>>(nb)
                                          : persistent_grid<bwd_dq2_mfma<BF, D, KS>>(nb);
                ProfScope prof(ENATTEN_KERNEL_BWD_DQ, "bwd_dq2_mfma", st);
                if (kDq2Full<D, KS> && a.s.H % G::TH == 0 && a.s.W % G::TW == 0)
                    hipLaunchKernelGGL((bwd_dq2_mfma<BF, D, KS, 4, kDq2Full<D, KS>>), dim3(grid), dim3(256), 0, st,
                                       a, ts, (int)nb);
                else if (balanced)
                    hipLaunchKernelGGL((bwd_dq2_mfma<BF, D, KS, 4, false, kBalanced<D, KS>>), dim3(grid),
                                       dim3(256), 0, st, a, ts, (int)nb);
                else
                    hipLaunchKernelGGL((bwd_dq2_mfma<BF, D, KS>), dim3(grid), dim3(256), 0, st, a, ts, (int)nb);
                dq_done = true;
            }
        } else if constexpr (kTallDqBuilt<D, KS>) {
            using G8 = Geo<D, KS, 8>;
            TileSet tall = ts;  // only the tile counts are used by this pass
            tall.tiles_r = (a.s.H + G8::TH - 1) / G8::TH;
            const int64_t nb8 = slabs * tall.tiles_r * tiles_c;
            if (nb8 >= 512) {
                const int grid = persistent_grid<bwd_dq_mfma<BF, D, KS, false, false, 8>>(nb8, G8::NT);
                ProfScope prof(ENATTEN_KERNEL_BWD_DQ, "bwd_dq_mfma", st);
                if (!kNarrow && a.s.H % G8::TH == 0 && a.s.W % G8::TW == 0)
                    hipLaunchKernelGGL((bwd_dq_mfma<BF, D, KS, false, false, 8, !kNarrow>), dim3(grid),
                                       dim3(G8::NT), 0, st, a, tall, (int)nb8, Runs{0, 0});
                else
                    hipLaunchKernelGGL((bwd_dq_mfma<BF, D, KS, false, false, 8>), dim3(grid), dim3(G8::NT),
                                       0, st, a, tall, (int)nb8, Runs{0, 0});
                dq_done = true;
                dq_tiles = tall.tiles_r * tiles_c;
            }
        }
        if constexpr (fits<D, KS>() && !kDq2Built<D, KS>) if (!dq_done) {
            const int grid = persistent_grid<bwd_dq_mfma<BF, D, KS, false, false>>(nb);
            ProfScope prof(ENATTEN_KERNEL_BWD_DQ, "bwd_dq_mfma", st);
            const bool full = !kNarrow && a.s.H % G::TH == 0 && a.s.W % G::TW == 0;
            if (roll_pays<D>(nb, grid)) {
                if (full)
                    hipLaunchKernelGGL((bwd_dq_mfma<BF, D, KS, false, kRollBuilt<D>, 4, !kNarrow>), dim3(grid),
                                       dim3(256), 0, st, a, ts, (int)nb, plan_runs(nb, grid, tiles_r));
                else
                    hipLaunchKernelGGL((bwd_dq_mfma<BF, D, KS, false, kRollBuilt<D>>), dim3(grid),
                                       dim3(256), 0, st, a, ts, (int)nb, plan_runs(nb, grid, tiles_r));
            } else if (full) {
                hipLaunchKernelGGL((bwd_dq_mfma<BF, D, KS, false, false, 4, !kNarrow>), dim3(grid), dim3(256), 0,
                                   st, a, ts, (int)nb, Runs{0, 0});
            } else {
                hipLaunchKernelGGL((bwd_dq_mfma<BF, D, KS, false, false>), dim3(grid), dim3(256), 0,
                                   st, a, ts, (int)nb, Runs{0, 0});
            }
        }
        {
            // Share the resident workgroups between the two bodies so that they end together.
            // `cost` is a frame tile's time in inner tiles (kFrameCost).
            constexpr int SP = kDkdvSplit<D, KS>, NT = Geo<D, KS, 4, SP>::NT;
            constexpr int MANY = kFourWaves<D, KS> ? 4 : kDkdvWaves<D, KS, SP>;
            const bool many = kFourWaves<D, KS> && nb > 1024;
            const double cost = many ? 2.6 : kFrameCost<BF, D, KS, kFrameKS<D, KS, SP> != KS>;
            const int grid = many ? persistent_grid<bwd_dkdv_mfma<BF, D, KS, false, SP, MANY>>(nb, NT)
                                  : persistent_grid<bwd_dkdv_mfma<BF, D, KS, false, SP>>(nb, NT);
            int inner_blocks = 0, dyn = 0;
            if (n_frame == 0) {
                inner_blocks = grid;
            } else if (n_inner > 0 && kRollBuilt<D>) {
                // With the column walk the busiest inner workgroup's walk is a staircase in the
                // number of inner workgroups (plan_runs), and a share in proportion to the work
                // lands anywhere on a step.  So every split is tried: the fewest inner
                // workgroups among those whose longer side is shortest.
                double best = 1e30;
                const int64_t per_f = (n_frame + 7) / 8, per_i = (n_inner + 7) / 8;
                for (int ib = 8; ib <= grid - 8 && ib <= per_i * 8; ib += 8) {
                    double walk;
                    if (roll_pays<D>(n_inner, ib)) {
                        plan_runs(n_inner, ib, ts.ni_r, &walk);
                    } else {
                        const int64_t slots_i = ib / 8;
                        walk = 2.0 * (double)((per_i + slots_i - 1) / slots_i);
                    }
                    const int64_t slots_f = (grid - ib) / 8;
                    const double frame = 2.0 * cost * (double)((per_f + slots_f - 1) / slots_f);
                    const double t = walk > frame ? walk : frame;
                    if (t < best) {
                        best = t;
                        inner_blocks = ib;
                    }
                }
                if (inner_blocks == 0) inner_blocks = 8;
                // The other way to share: every workgroup walks inner tiles (the shortest walk
                // there is) and then takes frame tiles from a counter as it becomes free.  The
                // frame tiles then run at the end, next to no inner tile and in no XCD's order,
                // which costs where the static split is already even; it is taken where the
                // staircase leaves the static split 7% or more behind (B4 N4 128x128 k7: 154.6 ->
                // 135.4 us; measured 4-9% slower at k9 and at 256x256 and 96x96 k7, where it is
                // not taken).
                if (a.zinv != nullptr && kCounter) {
                    int all = grid;
                    if (all > per_i * 8) all = (int)(per_i * 8);
                    double walk;
                    if (roll_pays<D>(n_inner, all)) {
                        plan_runs(n_inner, all, ts.ni_r, &walk);
                    } else {
                        const int64_t slots_i = all / 8;
                        walk = 2.0 * (double)((per_i + slots_i - 1) / slots_i);
                    }
                    const double t_dyn = walk + 2.0 * cost * ((double)n_frame / grid + 1.0);
                    if (t_dyn < 0.93 * best) {
                        dyn = 1;
                        inner_blocks = all;
                    }
                }
            } else if (n_inner > 0 && (many || (kBias && !(D == 32 && KS == 9)))) {
                inner_blocks = share_inner(n_inner, n_frame, grid, cost);
            } else if (n_inner > 0) {
                const double f = (double)n_inner / ((double)n_inner + cost * (double)n_frame);
                inner_blocks = (int)(f * grid / 8.0 + 0.5) * 8;
                if (inner_blocks < 8) inner_blocks = 8;
                if (inner_blocks > grid - 8) inner_blocks = grid - 8;
                if (inner_blocks > (n_inner + 7) / 8 * 8) inner_blocks = (int)((n_inner + 7) / 8 * 8);
            }
            if (path == ENATTEN_PATH_MFMA_SPLIT_QUEUE && a.zinv != nullptr && kCounter && n_frame > 0 && !dyn) {
                dyn = 1;
                const int64_t all = (n_inner + 7) / 8 * 8;
                inner_blocks = all < grid ? (int)all : grid;
            }
            // (the counter deals tiles in their plain order)
            if (n_frame > 0 && !dyn) ts.order = frame_order((int)(n_frame / slabs), (grid - inner_blocks) / 8, n_frame);
            ProfScope prof(ENATTEN_KERNEL_BWD_DKDV, "bwd_dkdv_mfma", st);
            if (inner_blocks > 0 && roll_pays<D>(n_inner, inner_blocks))
                hipLaunchKernelGGL((bwd_dkdv_mfma<BF, D, KS, kRollBuilt<D>, SP>), dim3(grid), dim3(NT),
                                   0, st, a, ts, (int)n_inner, (int)n_frame, inner_blocks,
                                   plan_runs(n_inner, inner_blocks, ts.ni_r), dyn);
            else
                hipLaunchKernelGGL((many ? bwd_dkdv_mfma<BF, D, KS, false, SP, MANY> : bwd_dkdv_mfma<BF, D, KS, false, SP>),
                                   dim3(grid), dim3(NT), 0, st, a, ts, (int)n_inner, (int)n_frame, inner_blocks,
                                   Runs{0, 0}, dyn);
        }
        if constexpr (kTable) {
            const auto reduce = path == kRpbTyped ? rpb_tile_reduce<kTable, BF, true> : rpb_tile_reduce<kTable, BF, false>;
            hipLaunchKernelGGL(reduce, dim3(a.s.N, (Bias<KS>::E + 15) / 16), dim3(1024), 0, st, a.ds_pairs, a.d_rpb,
                               a.s.B, a.s.N, dq_tiles, Bias<KS>::E);
        }
        return check_launch("enatten2d_bwd");
    } else {
        set_error("no matrix-core kernel for head_dim %d, kernel_size %d", D, KS);
        return ENATTEN_EUNSUPPORTED;
    }
}

#define ENATTEN_BY_KS(FN, BF, D, ARGS, ...)                      \
    switch ((ARGS).s.kh) {                                       \
        case 3: return FN<BF, D, 3>(ARGS, __VA_ARGS__);          \
        case 5: return FN<BF, D, 5>(ARGS, __VA_ARGS__);          \
        case 7: return FN<BF, D, 7>(ARGS, __VA_ARGS__);          \
        case 9: return FN<BF, D, 9>(ARGS, __VA_ARGS__);          \
        case 11: return FN<BF, D, 11>(ARGS, __VA_ARGS__);        \
        case 13: return FN<BF, D, 13>(ARGS, __VA_ARGS__);        \
    }

// A head dim that is a multiple of 8 runs on the kernels built for the next of 32, 64 and
// 128: their LDS rows carry zeros in the channels the tensor does not have (zero_row,
// HaloPlan::on, load_row_chunks) and the stores leave those channels out (store_token).
constexpr int built_dim(int D) { return D <= 32 ? 32 : D <= 64 ? 64 : 128; }

#define ENATTEN_BY_D(FN, BF, ARGS, ...)                                  \
    switch (built_dim((ARGS).s.D)) {                                     \
        case 32: ENATTEN_BY_KS(FN, BF, 32, ARGS, __VA_ARGS__) break;     \
        case 64: ENATTEN_BY_KS(FN, BF, 64, ARGS, __VA_ARGS__) break;     \
        case 128: ENATTEN_BY_KS(FN, BF, 128, ARGS, __VA_ARGS__) break;   \
    }

bool fits_rt(int D, int ks) {
    const int rows = (8 + ks - 1) * (8 + ks - 1) + 1;
    // two halos of an 8x8 tile, or (head_dim 128) one halo for the kernels that stage one at a time
    return (size_t)2 * rows * (D + 8) * 2 + (size_t)rows * 8 <= 160 * 1024 ||
           (D == 128 && (size_t)rows * (D + 8) * 2 + 1024 <= 160 * 1024);
}

// The launchers' common body: tensors whose rows the 16-byte loads cannot take go to the
// general kernels, everything else to the kernel built for its head dim and kernel size.
int fwd_dispatch(const FArgs &a, int dtype, hipStream_t st) {
    if (!layout_ok(a.q) || !layout_ok(a.k) || !layout_ok(a.v) || !layout_ok(a.o))
        return launch_fwd_simt(a, dtype, st);  // 16-byte loads need aligned rows
    if (dtype == ENATTEN_BF16) {
        ENATTEN_BY_D(fwd_launch, true, a, st)
    } else {
        ENATTEN_BY_D(fwd_launch, false, a, st)
    }
    set_error("no matrix-core kernel for head_dim %d, kernel_size %d", a.s.D, a.s.kh);
    return ENATTEN_EUNSUPPORTED;
}

int bwd_dispatch(const BArgs &a, int dtype, int path, hipStream_t st) {
    auto al = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    const bool grads_ok = a.gsb % 8 == 0 && a.gsn % 8 == 0 && a.gsh % 8 == 0 && a.gsw % 8 == 0;
    if (!layout_ok(a.q) || !layout_ok(a.k) || !layout_ok(a.v) || !layout_ok(a.o) ||
        !layout_ok(a.d_o) || !al(a.dq) || !al(a.dk) || !al(a.dv) || !grads_ok ||
        a.s.H >= 32768 || a.s.W >= 32768)  // (the dK/dV pass keeps window starts in 16 bits)
        return launch_bwd_simt(a, dtype, st, path == kRpbTyped);
    if (dtype == ENATTEN_BF16) {
        ENATTEN_BY_D(bwd_launch, true, a, path, st)
    } else {
        ENATTEN_BY_D(bwd_launch, false, a, path, st)
    }
    set_error("no matrix-core kernel for head_dim %d, kernel_size %d", a.s.D, a.s.kh);
    return ENATTEN_EUNSUPPORTED;
}

}  // namespace
}  // namespace enatten
