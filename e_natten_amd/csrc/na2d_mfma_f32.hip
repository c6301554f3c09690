// Matrix-core kernels for float32 2D neighborhood attention on gfx950.
//
// float32 tensors need more than float32 logits: with unscaled q.k of magnitude ~50
// (the reference's benchmark inputs, e_natten/triton.py:280 applies no scale) a float32
// dot product is good to ~1e-5, which exp() turns into a relative error of the
// probabilities and ~1e-4 absolute error of dQ and dK.  So the logits are formed with
// a float64 matrix instruction and every other product (P.V, dO.V, dS.K, P^T.dO, dS^T.Q)
// with a float32 one: true float32 products, no reduced-precision operands anywhere.
//
// Geometry.  A workgroup of four waves owns an 8x8 tile of pixels, a wave a 4x4 block of it as four blocks of
// 2x2.  The matrix instructions are those of four (float64) and sixteen (float32) independent 4x4 products,
// v_mfma_f64_4x4x4_4b_f64 and v_mfma_f32_4x4x1_16b_f32: each 2x2 block of queries meets the (k+1)^2 pixels that
// its own windows reach, where a 16-wide instruction has the whole 4x4 block meet (k+3)^2 and more: 36 tokens per
// query instead of 64 at kernel_size 5 (25 are in its window), 16 instead of 48 at 3, 64 instead of 112 at 7.
// Both shapes run at the rate of the 16-wide ones (16 and 32 products per cycle and SIMD: measured 17.0 and 9.3
// cycles against 66.1 and 33.0).  Forward, dQ and dK/dV pass, us, 4x4 blocks on the 16-wide instructions -> 2x2 blocks,
// B4 N4 128x128, launches queued behind each other: d128 k5 163 + 226 + 187 -> 137 + 182 + 148, d64 k3 64 + 89 + 66 -> 46 + 64 +
// 47, k7 132 + 237 + 175 -> 109 + 171 + 130, d32 k5 49 + 64 + 56 -> 40 + 53 + 34.  What bounds them at d128 k5: a tile's two
// staging phases, which issue no matrix instruction (a fifth of the wave cycles are waits; 3.5 TB/s of the 5.7 that HBM gives
// the 16-bit forward), and LDS reads of the second products, whose bank conflicts are 40% of the LDS cycles (0 to 14% with
// the 4x4 blocks).  One tensor's halo at a time is staged in LDS (float32 rows of D + 4 floats), so two
// workgroups share a CU; the other tensor's halo travels from HBM into registers meanwhile.
//
// Lanes.  A lane is (g, b, j) = (lane >> 4, lane >> 2 & 3, lane & 3): block b of the wave, pixel j of the
// block.  The (k+1)^2 tokens of a block are numbered in 2x2 patches: token i of patch t lies at a constant distance
// from the block's first one, so operand addresses are one register and immediate offsets.
// The float64 product takes channel g of four as its reduction index and leaves lane (g, b, j) with token g of
// every patch; the float32 products take g as a quarter of the channels, in the first product as a part of
// the reduction (summed over the lane groups afterwards), in the second one as rows of the result.
//
// Backward.  The dQ pass recomputes the logits once (float64), forms P, dP, dS and dQ,
// and leaves P and dS of every (query, window position) in the workspace, k*k float32
// each per query.  The dK/dV pass then has no logits, masks or exponentials left: per
// key tile it walks the queries that attend to the tile (e_natten/pytorch.py:13-23,
// :261-270) and accumulates dV = P^T dO and dK = dS^T Q with the matrix instruction,
// P and dS gathered from the workspace (zero where a query does not attend a key).
// No atomics; results are bit-reproducible.
//
// Per-query math: e_natten/triton.py:242-302 (forward), :383-423 (backward).

#include <numeric>
#include <utility>

#include "na2d_mfma.h"

namespace enatten {
namespace {

template <int D, int KS>
struct Geo32 {
    static constexpr int HR = 8 + KS - 1, HC = HR;   // halo of the 8x8 tile
    static constexpr int PW = (KS + 1) / 2;          // 2x2 patches on a side of a block's halo
    static constexpr int T = PW * PW;                // patches
    static constexpr int KK = KS * KS;
    static constexpr int PITCH = D + 4;              // floats between LDS rows
    static constexpr int ROWS = HR * HC;
    static constexpr int CPR = D / 4;                // 16-byte chunks per row
    static constexpr int NCH = HR * HC * CPR;
    static constexpr int NL = (NCH + 255) / 256;     // chunks per thread
    static constexpr int DQ = D / 4;                 // channels per lane group in the first products
    static constexpr int DT = D / 16;                // 16-channel pieces of the outputs
    static constexpr int STEPS = T * 4;              // tokens of a block: reduction steps of the second products
    static constexpr size_t LDS_BYTES = (size_t)ROWS * PITCH * sizeof(float);
    // floats from a block's first token to token i of patch t, and its row and column there
    static constexpr int row(int t, int i) { return 2 * (t / PW) + (i >> 1); }
    static constexpr int col(int t, int i) { return 2 * (t % PW) + (i & 1); }
    static constexpr int at(int t, int i) { return (row(t, i) * HC + col(t, i)) * PITCH; }
};

// Whole-line stores (store32's LINES) where LDS admits two workgroups per CU: like the 16-bit
// kernels, those with one workgroup per CU (head_dim 128 at kernel_size 7) do not gain from them.
template <int D, int KS>
constexpr bool kLines32 = 2 * Geo32<D, KS>::LDS_BYTES <= 160 * 1024;

// dV and dK in one launch where the staged rows of both dO and Q admit two workgroups per CU
// (head_dim 32, and 64 up to kernel_size 5): the places and bounds of the weights are formed once, a
// weight pair is one 8-byte load, and what a workgroup waits for (rows, weights, two barriers) it
// waits for once.  P and dS of a window position then lie side by side in the workspace, which makes
// the dQ pass's scattered stores half as many as well.  Backward, us, two launches -> one, measured with 4x4 blocks: B8 N7 46x46 d32 k7
// 174 -> 142 (dK/dV 105 -> 77), B2 N8 128x128 d64 k5 258 -> 234, k3 178 -> 164, d32 k3 99 -> 90.  At head_dim 128
// the same with 64 channels to a workgroup was level at k5 (dQ pass 256 -> 248, dK/dV 210 -> 219).
template <int D, int KS>
constexpr bool kPair32 = 4 * (Geo32<D, KS>::LDS_BYTES + 16) <= 160 * 1024;
// (the caller's workspace is aligned to its floats)
typedef float f32x2 __attribute__((ext_vector_type(2), aligned(4)));

struct Regs32 {
    // the largest halo served: kernel_size 7 at head_dim 128 is 196 pixels x 32 chunks
    u32x4 v[25];
};

// Pixel of chunk i of this thread in the halo.  Every PER chunks the threads' pixels are RPER whole rows further
// down, so a thread has PER columns and as many rows to keep instead of one for every chunk.
template <int D, int KS>
__device__ __forceinline__ void chunk_pixel(int i, unsigned &r, unsigned &c) {
    using G = Geo32<D, KS>;
    constexpr int STEP = 256 / G::CPR, PER = std::lcm(STEP, G::HC) / STEP, RPER = std::lcm(STEP, G::HC) / G::HC;
    const unsigned pix = threadIdx.x / G::CPR + i % PER * STEP;
    r = pix / G::HC + i / PER * RPER;
    c = pix % G::HC;
}
// One tensor's halo (origin (hr0, hc0), pixels at or beyond (rlim, clim) clamped) into
// registers, then into LDS, in PARTS slices, so that the loads can be issued a few at a time between
// matrix instructions (a wave that issues a whole halo at once is blocked for
// microseconds while the CU's memory queue takes the loads, and issues no matrix
// instruction meanwhile).
template <int D, int KS, int PARTS>
__device__ __forceinline__ void fetch32_part(Regs32 &reg, const float *img, int64_t sh, int64_t sw,
                                             int hr0, int hc0, int rlim, int clim, int part) {
    using G = Geo32<D, KS>;
    static_assert(G::NL <= 25, "staging registers");
    const char *base = reinterpret_cast<const char *>(img + hr0 * sh + hc0 * sw);
    const unsigned sh4 = (unsigned)sh * 4u, sw4 = (unsigned)sw * 4u;
    const unsigned rmax = rlim - 1 - hr0, cmax = clim - 1 - hc0;
#pragma unroll
    for (int i = 0; i < G::NL; i++) {
        if (i * PARTS / G::NL != part) continue;
        unsigned r, c;
        chunk_pixel<D, KS>(i, r, c);  // (beyond the last pixel: a row below the halo, clamped like the others)
        const unsigned off = __umul24(min(r, min(rmax, G::HR - 1u)), sh4) + __umul24(min(c, cmax), sw4) +
                             (threadIdx.x % G::CPR) * 16u;
        reg.v[i] = *reinterpret_cast<const u32x4 *>(base + off);
    }
}
template <int D, int KS>
__device__ __forceinline__ void fetch32(Regs32 &reg, const float *img, int64_t sh, int64_t sw,
                                        int hr0, int hc0, int rlim, int clim) {
    fetch32_part<D, KS, 1>(reg, img, sh, sw, hr0, hc0, rlim, clim, 0);
}
template <int D, int KS>
__device__ __forceinline__ void commit32(float *lds, const Regs32 &reg) {
    using G = Geo32<D, KS>;
#pragma unroll
    for (int i = 0; i < G::NL; i++) {
        const int pix = (int)threadIdx.x / G::CPR + i * (256 / G::CPR);
        if (pix < G::HR * G::HC)
            *reinterpret_cast<u32x4 *>(lds + pix * G::PITCH + ((int)threadIdx.x % G::CPR) * 4) = reg.v[i];
    }
}

// exp(x) for x <= 0 with a float64 argument through the hardware 2^y: the float32
// rounding of y = x * log2(e) is put back to first order, 2^(hi + lo) = 2^hi (1 + lo ln 2).
__device__ __forceinline__ float exp_neg64(double x) {
    const double y = fmax(x * 1.4426950408889634, -200.0);  // also maps -inf to an exact 0
    const float hi = (float)y;
    const float lo = (float)(y - (double)hi);
    const float e = __builtin_amdgcn_exp2f(hi);
    return fmaf(e, lo * kLn2, e);
}

// XCD-aware tile of a workgroup: every XCD takes one contiguous run of tiles.
__device__ __forceinline__ int tile_of_block(int ntiles) {
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int per = (ntiles + 7) >> 3;
    const int t = xcd * per + slot;
    return (slot < per && t < ntiles) ? t : -1;
}

// Odd rows of 16 lanes of a against even rows of b: a = (a0, b0, a2, b2), b = (a1, b1, a3, b3).
__device__ __forceinline__ void swap_rows(float &a, float &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
}
// The upper 32 lanes of a against the lower ones of b.
__device__ __forceinline__ void swap_halves(float &a, float &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]), b = __uint_as_float(r[1]);
}
// out[i]: row i of x in every row
__device__ __forceinline__ void spread_rows(float x, float (&out)[4]) {
    float a = x, b = x;
    swap_rows(a, b);
    out[0] = a, out[2] = a, out[1] = b, out[3] = b;
    swap_halves(out[0], out[2]);
    swap_halves(out[1], out[3]);
}

// This lane's place: block and pixel of the wave's 4x4 queries (or keys), lane group.
struct Lane {
    int g, b, j;
};
__device__ __forceinline__ Lane lane_place() {
    const int l = threadIdx.x & 63;
    return Lane{l >> 4, (l >> 2) & 3, l & 3};
}
// lane_query for these lanes: the halo is that of the lane's 2x2 block, (dr, dc) are 0 or 1.
template <int KS>
__device__ __forceinline__ LaneQ block_query(const Tile &tl, const Shape &s, int wave, const Lane &ln) {
    LaneQ q = lane_query<KS>(tl, s, wave, (2 * (ln.b >> 1) + (ln.j >> 1)) * 4 + 2 * (ln.b & 1) + (ln.j & 1));
    const int r0 = tl.r0 + (wave >> 1) * 4 + 2 * (ln.b >> 1), c0 = tl.c0 + (wave & 1) * 4 + 2 * (ln.b & 1);
    const int sr0 = win_start(min(r0, s.H - 1), s.H, KS), sc0 = win_start(min(c0, s.W - 1), s.W, KS);
    q.dr += q.hr0 + q.orow - sr0;
    q.dc += q.hc0 + q.ocol - sc0;
    q.orow = sr0 - q.hr0;
    q.ocol = sc0 - q.hc0;
    return q;
}

// this lane's share of one pixel's channels for the first products, channels 16 s + 4 g .. + 3
template <int D>
__device__ __forceinline__ void load_quarter(const float *row, int g, float *out) {
#pragma unroll
    for (int s = 0; s < D / 16; s++) {
        const f32x4 x = *reinterpret_cast<const f32x4 *>(row + 16 * s + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; e++) out[4 * s + e] = x[e];
    }
}
// LDS address of this lane's rows in the first products: token j of a patch, lane group's channels
template <int D, int KS>
__device__ __forceinline__ const float *first_base(const float *lds, const LaneQ &lq, const Lane &ln) {
    using G = Geo32<D, KS>;
    return lds + ((lq.orow + (ln.j >> 1)) * G::HC + lq.ocol + (ln.j & 1)) * G::PITCH + 4 * ln.g;
}

// f(0), f(1), ..: with the unrolling pragma the longest of these loops stay loops
template <typename F, int... I>
__device__ __forceinline__ void each_step(F f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}

// The steps of a first product: the patches of a group (a row of them; all four at kernel_size 3) against four
// channels per lane group, mul(t, e, x) for patch t and channel e.  A step's rows are read from LDS a step ahead;
// independent accumulators lie between two uses of one.  `hook(s)` runs before the instructions of channel
// group s of D/16 (used to issue global loads a few at a time).
template <int D, int KS, typename Hook, typename Mul>
__device__ __forceinline__ void first_steps(const float *base, Hook hook, Mul mul) {
    using G = Geo32<D, KS>;
    constexpr int GRP = KS == 3 ? 4 : G::PW, PER = G::T / GRP, STEPS = PER * G::DT;
    f32x4 x[2][GRP];
    auto fetch = [&](auto at) __attribute__((always_inline)) {
        constexpr int step = decltype(at)::value;
#pragma unroll
        for (int i = 0; i < GRP; i++)
            x[step & 1][i] = *reinterpret_cast<const f32x4 *>(base + G::at(step % PER * GRP + i, 0) + 16 * (step / PER));
    };
    fetch(std::integral_constant<int, 0>{});
    each_step([&](auto at) __attribute__((always_inline)) {
        constexpr int step = decltype(at)::value;
        if constexpr (step + 1 < STEPS) fetch(std::integral_constant<int, step + 1>{});
        if constexpr (step % PER == 0) hook(step / PER);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < GRP; i++) mul(step % PER * GRP + i, 4 * (step / PER) + e, x[step & 1][i][e]);
        __builtin_amdgcn_sched_barrier(0);
    }, std::make_integer_sequence<int, STEPS>{});
}

// Logits of this lane's query in float64: acc[t] is that of token g of patch t.  `qf` holds the query's channels
// (load_quarter).
template <int D, int KS, typename Hook>
__device__ __forceinline__ void logits64(const float *base, const float *qf, double *acc, Hook hook) {
    using G = Geo32<D, KS>;
#pragma unroll
    for (int t = 0; t < G::T; t++) acc[t] = 0.0;
    first_steps<D, KS>(base, hook, [&](int t, int c, float x) __attribute__((always_inline)) {
        acc[t] = __builtin_amdgcn_mfma_f64_4x4x4f64((double)x, (double)qf[c], acc[t], 0, 0, 0);
    });
}
// The same product in float32 (dP = V dO): out[t] is that of token g of patch t.
template <int D, int KS, typename Hook>
__device__ __forceinline__ void first32(const float *base, const float *qf, float *out, Hook hook) {
    using G = Geo32<D, KS>;
    f32x4 acc[G::T];  // this lane group's quarter of the channels; element i: token i of the patch
#pragma unroll
    for (int t = 0; t < G::T; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    first_steps<D, KS>(base, hook, [&](int t, int c, float x) __attribute__((always_inline)) {
        acc[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(x, qf[c], acc[t], 0, 0, 0);
    });
#pragma unroll
    for (int t = 0; t < G::T; t++) {  // the lane groups' sums; group g keeps token g
        float x = acc[t][0], y = acc[t][1], z = acc[t][2], w = acc[t][3];
        swap_halves(x, z);
        swap_halves(y, w);
        x += z;
        y += w;
        swap_rows(x, y);
        out[t] = x + y;
    }
}

// One token of the second products: rows x of the 2x2 blocks' tokens (D / 16 values per lane, second_fetch), w the
// token's weight for this lane's query (or key).
// Rows of the result are channels: with D >= 64 lane (g, b, j) reads channels 64 h + 16 g + 4 j + 0 .. 3 as one
// 16-byte word, and element i of acc[4 h + m] is channel 64 h + 16 g + 4 i + m; at head_dim 32 it reads
// channels 16 m + 4 g + j, and element i of acc[m] is channel 16 m + 4 g + i.  From head_dim 64 on every other
// block has its lane groups read channels 32 further on or back (second_flip): two neighbouring blocks' rows are
// two pixels apart, which alone would put half of their words on the same banks.
template <int D>
__device__ __forceinline__ int second_flip(const Lane &ln) { return D == 32 ? 0 : (ln.b & 1) * 32; }
template <int D>
__device__ __forceinline__ int second_channel(const Lane &ln) {
    return D == 32 ? 4 * ln.g + ln.j : (16 * ln.g + 4 * ln.j) ^ second_flip<D>(ln);
}
template <int D>
__device__ __forceinline__ void second_fetch(const float *row, float *x) {
    if constexpr (D == 32) {
#pragma unroll
        for (int m = 0; m < 2; m++) x[m] = row[16 * m];
    } else {
#pragma unroll
        for (int h = 0; h < D / 64; h++) {
            const f32x4 r = *reinterpret_cast<const f32x4 *>(row + 64 * h);
#pragma unroll
            for (int m = 0; m < 4; m++) x[4 * h + m] = r[m];
        }
    }
}
template <int D>
__device__ __forceinline__ void second_step(const float *x, float w, f32x4 *acc) {
#pragma unroll
    for (int m = 0; m < D / 16; m++) acc[m] = __builtin_amdgcn_mfma_f32_4x4x1f32(x[m], w, acc[m], 0, 0, 0);
}
// acc[m] -> channels (16 m + 4 g .. + 3) ^ second_flip, as store32 takes them: a 4x4 transpose over elements and lane
// groups
template <int D>
__device__ __forceinline__ void second_pieces(f32x4 *acc) {
    if constexpr (D > 32) {
#pragma unroll
        for (int h = 0; h < D / 64; h++) {
            float x[4][4];
#pragma unroll
            for (int m = 0; m < 4; m++) {
#pragma unroll
                for (int i = 0; i < 4; i++) x[m][i] = acc[4 * h + m][i];
                swap_rows(x[m][0], x[m][1]);
                swap_rows(x[m][2], x[m][3]);
                swap_halves(x[m][0], x[m][2]);
                swap_halves(x[m][1], x[m][3]);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) acc[4 * h + i] = f32x4{x[0][i], x[1][i], x[2][i], x[3][i]};
        }
    }
}

// out [channel][query] = X^T w over the tokens of the lane's block, X rows from LDS, as second_pieces leaves
// them.  w[t] belongs to token g of patch t.  `hook(step)` runs before the instructions of token `step` of T * 4.
template <int D, int KS, typename Hook>
__device__ __forceinline__ void second32(const float *lds_x, const float *w, const LaneQ &lq, const Lane &ln, f32x4 *acc,
                                         Hook hook) {
    using G = Geo32<D, KS>;
#pragma unroll
    for (int m = 0; m < G::DT; m++) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float *base = lds_x + (lq.orow * G::HC + lq.ocol) * G::PITCH + second_channel<D>(ln);
    // the operands are read from LDS a token ahead, so the instructions never wait for LDS
    float x[2][G::DT], wb[4];
    second_fetch<D>(base, x[0]);
    each_step([&](auto at) __attribute__((always_inline)) {
        constexpr int step = decltype(at)::value;
        if constexpr (step + 1 < G::STEPS) second_fetch<D>(base + G::at((step + 1) >> 2, (step + 1) & 3), x[(step + 1) & 1]);
        if ((step & 3) == 0) spread_rows(w[step >> 2], wb);
        hook(step);
        __builtin_amdgcn_sched_barrier(0);
        second_step<D>(x[step & 1], wb[step & 3], acc);
        __builtin_amdgcn_sched_barrier(0);
    }, std::make_integer_sequence<int, G::STEPS>{});
    second_pieces<D>(acc);
}

// Stores one token's D channels.  Piece m of lane group g is channels 16m + 4g .. +3, so the
// four lanes of a token would write 64 contiguous bytes per instruction: half a line, and
// non-temporal half lines reach memory in pieces (1.2-1.4x the bytes, at 3.1 TB/s against 5.3 for
// whole lines).  With LINES the lanes of tokens n and n^1 (adjacent lanes) exchange every other
// piece, and the eight lanes of the pair write one token's whole 128-byte line per instruction.
// Every lane of the wave must call this; `live`: this lane's token exists; `flip`: second_flip.  The values
// stored are acc * mul, or, with REST, acc * (mul + low) with one rounding of the product by mul; low > 0, so that an
// infinity stays one.
template <int D, bool LINES, bool REST = false>
__device__ __forceinline__ void store32(float *token, int g, const f32x4 *acc, int flip, float mul, bool live, float low = 0.f) {
    auto times = [&](const f32x4 &x) __attribute__((always_inline)) {
        f32x4 y;
#pragma unroll
        for (int c = 0; c < 4; c++)
            y[c] = REST ? fmaf(x[c], mul, x[c] * low) : x[c] * mul;
        return y;
    };
    if constexpr (LINES) {
        const bool odd = threadIdx.x & 1;
        auto xchg = [](unsigned x) __attribute__((always_inline)) {
            return (unsigned)__builtin_amdgcn_mov_dpp((int)x, 0xB1 /* quad_perm [1,0,3,2] */, 0xF, 0xF, true);
        };
        const uintptr_t own = reinterpret_cast<uintptr_t>(token);
        const uintptr_t nbr = (uintptr_t)xchg((unsigned)own) | ((uintptr_t)xchg((unsigned)(own >> 32)) << 32);
        // (as an offset from this lane's pointer, so that the stores stay global-memory instructions)
        float *other = reinterpret_cast<float *>(reinterpret_cast<char *>(token) + (ptrdiff_t)(nbr - own));
        const bool nlive = xchg(live ? 1u : 0u) != 0;
        float *tok_a = odd ? other : token, *tok_b = odd ? token : other;
        const bool live_a = odd ? nlive : live, live_b = odd ? live : nlive;
        const int off = (odd ? 16 : 0) + 4 * g;
#pragma unroll
        for (int k = 0; k < D / 32; k++) {
            const f32x4 lo = times(acc[2 * k]), hi = times(acc[2 * k + 1]);
            f32x4 sa, sb;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float r = __uint_as_float(xchg(__float_as_uint(odd ? lo[c] : hi[c])));
                sa[c] = odd ? r : lo[c];
                sb[c] = odd ? hi[c] : r;
            }
            if (live_a) __builtin_nontemporal_store(sa, reinterpret_cast<f32x4 *>(tok_a + (32 * k ^ flip) + off));
            if (live_b) __builtin_nontemporal_store(sb, reinterpret_cast<f32x4 *>(tok_b + (32 * k ^ flip) + off));
        }
    } else {
        if (!live) return;
#pragma unroll
        for (int m = 0; m < D / 16; m++)
            __builtin_nontemporal_store(times(acc[m]), reinterpret_cast<f32x4 *>(token + (16 * m ^ flip) + 4 * g));
    }
}

__device__ __forceinline__ const float *image32(const View &v, const Tile &tl) {
    return static_cast<const float *>(v.ptr) + tl.bb * v.sb + tl.nn * v.sn;
}

// Is halo token (r, c) inside the window of the query whose window starts at (dr, dc)?
template <int KS>
__device__ __forceinline__ bool in_window(int r, int c, int dr, int dc) {
    return (unsigned)(r - dr) < (unsigned)KS && (unsigned)(c - dc) < (unsigned)KS;
}

// ------------------------------------------------------------------ forward
// S^T = K Q^T (float64), masked softmax, O^T = V^T P^T (float32); writes O and the
// log-sum-exp.  Persistent: K's halo is in LDS while the logits are formed and V's halo
// is loaded, a few loads between the matrix instructions of each token tile; then V's
// halo takes K's place, and the next tile's K is loaded between the instructions of P.V.
template <int D, int KS>
__global__ __launch_bounds__(256, 2) void fwd_mfma_f32(FwdArgs a, int tiles_r, int tiles_c, int ntiles) {
    using G = Geo32<D, KS>;
    constexpr int STEPS = G::STEPS;
    __shared__ __attribute__((aligned(16))) float lds[G::ROWS * G::PITCH];
    Sched sc = make_sched(ntiles, blockIdx.x, gridDim.x);
    if (sc.t >= sc.t_end) return;
    const Shape &s = a.s;
    const int wave = threadIdx.x >> 6;
    const Lane ln = lane_place();
    const int g = ln.g;

    Tile cur = tile_of(sc.t, tiles_r, tiles_c, s.N);
    LaneQ lq = block_query<KS>(cur, s, wave, ln);
    Regs32 st;
    float qf[G::DQ];
    fetch32<D, KS>(st, image32(a.k, cur), a.k.sh, a.k.sw, lq.hr0, lq.hc0, s.H, s.W);
    load_quarter<D>(image32(a.q, cur) + lq.qr * a.q.sh + lq.qc * a.q.sw, g, qf);
    for (;;) {
        commit32<D, KS>(lds, st);
        __syncthreads();
        const int tn = sc.t + sc.step;
        const bool more = tn < sc.t_end;
        const Tile nxt = more ? tile_of(tn, tiles_r, tiles_c, s.N) : cur;
        const LaneQ lqn = block_query<KS>(nxt, s, wave, ln);
        const float *vimg = image32(a.v, cur), *kimg = image32(a.k, nxt);
        auto load_v = [&](int part) __attribute__((always_inline)) {
            fetch32_part<D, KS, G::DQ / 4>(st, vimg, a.v.sh, a.v.sw, lq.hr0, lq.hc0, s.H, s.W, part);
        };
        auto load_next = [&](int part) __attribute__((always_inline)) {
            if (more) {
                fetch32_part<D, KS, STEPS>(st, kimg, a.k.sh, a.k.sw, lqn.hr0, lqn.hc0, s.H, s.W, part);
                if (part == STEPS - 1)
                    load_quarter<D>(image32(a.q, nxt) + lqn.qr * a.q.sh + lqn.qc * a.q.sw, g, qf);
            }
        };

        float p[G::T];
        float lse = 0.f, inv = 0.f, inv_rest = 0.f;
        if (lq.wave_on) {
            double acc[G::T];
            logits64<D, KS>(first_base<D, KS>(lds, lq, ln), qf, acc, load_v);
            double mx = -INFINITY;
#pragma unroll
            for (int t = 0; t < G::T; t++) {
                const bool ok = in_window<KS>(G::row(t, 0) + (g >> 1), G::col(t, 0) + (g & 1), lq.dr, lq.dc);
                acc[t] = ok ? acc[t] * (double)s.scale : -INFINITY;
                mx = fmax(mx, acc[t]);
            }
            mx = fmax(mx, __shfl_xor(mx, 16, 64));
            mx = fmax(mx, __shfl_xor(mx, 32, 64));
            float sum = 0.f;
#pragma unroll
            for (int t = 0; t < G::T; t++) {
                p[t] = exp_neg64(acc[t] - mx);
                sum += p[t];
            }
            sum = col_sum(sum);
            inv = 1.f / sum;
            inv_rest = fmaf(-sum, inv, 1.f);  // what its rounding leaves
            if (inv_rest <= 0.f) {            // (from below, store32; not where the sum is NaN or zero)
                inv = __uint_as_float(__float_as_uint(inv) - 1u);
                inv_rest = fmaf(-sum, inv, 1.f);
            }
            lse = (float)(mx + (double)logf(sum));
        } else {
#pragma unroll
            for (int part = 0; part < G::DQ / 4; part++) load_v(part);
        }
        __syncthreads();  // every wave is done with K
        commit32<D, KS>(lds, st);
        __syncthreads();
        if (lq.wave_on) {
            f32x4 o[G::DT];
            second32<D, KS>(lds, p, lq, ln, o, load_next);
            float *op = const_cast<float *>(image32(a.o, cur)) + lq.qr * a.o.sh + lq.qc * a.o.sw;
            store32<D, kLines32<D, KS>, true>(op, g, o, second_flip<D>(ln), inv, lq.live, inv * inv_rest);
            if (lq.live && a.lse && g == 0) a.lse[lq.tok] = lse;
        } else {
#pragma unroll
            for (int part = 0; part < STEPS; part++) load_next(part);
        }
        if (!more) break;
        __syncthreads();  // every wave is done with V
        cur = nxt;
        lq = lqn;
        sc.t = tn;
    }
}

// ------------------------------------------------------------------ dQ (+ P, dS)
// dP^T = V dO^T (float32) on V's halo, then K's halo into the same rows: logits in
// float64, P renormalised over the window (which removes the rounding of the stored
// log-sum-exp), delta = sum_j P_j dP_j, dS = P (dP - delta), dQ^T = K^T dS^T.  P and dS
// go to the workspace, k*k values per query in window order, for the dK/dV pass.
// Persistent like the forward: K is loaded between the instructions of dP, the next
// tile's V between those of dQ.
template <int D, int KS>
__global__ __launch_bounds__(256, 2) void bwd_dq_mfma_f32(BwdArgs a, float *ws_p, float *ws_ds,
                                                          int tiles_r, int tiles_c, int ntiles) {
    using G = Geo32<D, KS>;
    constexpr int STEPS = G::STEPS;
    __shared__ __attribute__((aligned(16))) float lds[G::ROWS * G::PITCH];
    Sched sc = make_sched(ntiles, blockIdx.x, gridDim.x);
    if (sc.t >= sc.t_end) return;
    const Shape &s = a.s;
    const int wave = threadIdx.x >> 6;
    const Lane ln = lane_place();
    const int g = ln.g;

    Tile cur = tile_of(sc.t, tiles_r, tiles_c, s.N);
    LaneQ lq = block_query<KS>(cur, s, wave, ln);
    Regs32 st;
    float go[G::DQ];
    fetch32<D, KS>(st, image32(a.v, cur), a.v.sh, a.v.sw, lq.hr0, lq.hc0, s.H, s.W);
    load_quarter<D>(image32(a.d_o, cur) + lq.qr * a.d_o.sh + lq.qc * a.d_o.sw, g, go);
    for (;;) {
        commit32<D, KS>(lds, st);
        __syncthreads();
        const int tn = sc.t + sc.step;
        const bool more = tn < sc.t_end;
        const Tile nxt = more ? tile_of(tn, tiles_r, tiles_c, s.N) : cur;
        const LaneQ lqn = block_query<KS>(nxt, s, wave, ln);
        const float *kimg = image32(a.k, cur), *vimg = image32(a.v, nxt);
        // this tile's q and log-sum-exp arrive while dP is formed (their registers are
        // free until then: dO's are needed first, q's afterwards)
        float qf[G::DQ];
        float lse_f = 0.f;
        auto load_k = [&](int part) __attribute__((always_inline)) {
            fetch32_part<D, KS, G::DT>(st, kimg, a.k.sh, a.k.sw, lq.hr0, lq.hc0, s.H, s.W, part);
            if (part == G::DT - 1) {
                load_quarter<D>(image32(a.q, cur) + lq.qr * a.q.sh + lq.qc * a.q.sw, g, qf);
                lse_f = a.lse[lq.tok];
            }
        };

        float dp[G::T];
        if (lq.wave_on) {
            first32<D, KS>(first_base<D, KS>(lds, lq, ln), go, dp, load_k);
        } else {
#pragma unroll
            for (int part = 0; part < G::DT; part++) load_k(part);
        }
        const double lse = (double)lse_f;
        __syncthreads();  // every wave is done with V
        commit32<D, KS>(lds, st);
        __syncthreads();
        auto load_next = [&](int part) __attribute__((always_inline)) {
            if (more) {
                fetch32_part<D, KS, STEPS>(st, vimg, a.v.sh, a.v.sw, lqn.hr0, lqn.hc0, s.H, s.W, part);
                if (part == STEPS - 1)
                    load_quarter<D>(image32(a.d_o, nxt) + lqn.qr * a.d_o.sh + lqn.qc * a.d_o.sw, g, go);
            }
        };
        if (lq.wave_on) {
            float ds[G::T];
            {
                double acc[G::T];
                logits64<D, KS>(first_base<D, KS>(lds, lq, ln), qf, acc, [](int) {});
                float z = 0.f;
#pragma unroll
                for (int t = 0; t < G::T; t++) {
                    const bool ok = in_window<KS>(G::row(t, 0) + (g >> 1), G::col(t, 0) + (g & 1), lq.dr, lq.dc);
                    ds[t] = ok ? exp_neg64(fmin(acc[t] * (double)s.scale - lse, 0.0)) : 0.f;
                    z += ds[t];
                }
                z = col_sum(z);
                const float zinv = 1.f / z, zlow = zinv * fmaf(-z, zinv, 1.f);
                float dpart = 0.f;
#pragma unroll
                for (int t = 0; t < G::T; t++) {
                    ds[t] = fmaf(ds[t], zinv, ds[t] * zlow);  // P
                    dpart = fmaf(ds[t], dp[t], dpart);
                }
                const float delta = col_sum(dpart);
                float *pp = ws_p + lq.tok * G::KK * (kPair32<D, KS> ? 2 : 1), *dsp = ws_ds + lq.tok * G::KK;
#pragma unroll
                for (int t = 0; t < G::T; t++) {
                    const int r = G::row(t, 0) + (g >> 1), c = G::col(t, 0) + (g & 1);
                    const float pv = ds[t];
                    ds[t] = pv * (dp[t] - delta);        // dS
                    if (in_window<KS>(r, c, lq.dr, lq.dc) && lq.live) {
                        const int at = (r - lq.dr) * KS + (c - lq.dc);
                        if constexpr (kPair32<D, KS>) {
                            *reinterpret_cast<f32x2 *>(pp + 2 * at) = f32x2{pv, ds[t]};
                        } else {
                            pp[at] = pv;
                            dsp[at] = ds[t];
                        }
                    }
                }
            }
            f32x4 dq[G::DT];
            second32<D, KS>(lds, ds, lq, ln, dq, load_next);
            store32<D, kLines32<D, KS>>(static_cast<float *>(a.dq) + lq.tok * D, g, dq, second_flip<D>(ln), s.scale, lq.live);
        } else {
#pragma unroll
            for (int part = 0; part < STEPS; part++) load_next(part);
        }
        if (!more) break;
        __syncthreads();  // every wave is done with K
        cur = nxt;
        lq = lqn;
        sc.t = tn;
    }
}

// Operands of a query that is not met: zeros, moved there on a branch that few patches take (as a choice between two values
// they would cost every patch; the empty asm keeps the compiler from making one of the branch).
template <int N>
__device__ __forceinline__ void cut(float *x) {
#pragma unroll
    for (int m = 0; m < N; m++) {
        x[m] = 0.f;
        asm volatile("" : "+v"(x[m]));
    }
}

// ------------------------------------------------------------------ dK or dV
// Key-centric: the workgroup owns 8x8 keys, a wave 4x4 of them in blocks of 2x2.  The
// queries that attend to any key of the tile form a rectangle (the union of the keys'
// inverse neighbourhoods, e_natten/pytorch.py:13-23), walked in blocks of at most
// (8+k-1)^2 queries whose X rows (dO for dV, Q for dK) are staged in LDS.  In each, a block of keys meets the
// patches of 2x2 queries from the first that attends to one of its keys on, as many as the wave's widest
// block of keys needs.  The weights W (P for dV, dS for dK) come from the workspace; a query
// that does not attend to a key contributes an exact zero.
// One tile per workgroup: as a persistent kernel that loads the next tile's rows between the products of the
// current one it was slower (d128 k5 149 -> 205 us for the two launches below, d64 k3 33 -> 41).
// WIDE: images wider than 65536 pixels, where a weight's place in the rows of a block takes more than 32 bits: plain loads
// of the weights that there are; the sums are the same.
template <int D, int KS, bool WIDE>
__global__ __launch_bounds__(256, 2) void bwd_dkdv_mfma_f32(BwdArgs a, View x0, View x1, const float *ws_w,
                                                            float *out0, float *out1, float mul0, float mul1,
                                                            int tiles_r, int tiles_c, int ntiles) {
    using G = Geo32<D, KS>;
    // Two neighbouring keys are attended by at most k + k/2 + 1 rows of queries, and by up to 2k where both ends of
    // the axis clamp their windows, which an axis of at most 2k pixels has: it is walked in shorter blocks.
    constexpr int NP = (KS + KS / 2 + 2) / 2;       // patches on a side
    constexpr int NB = kPair32<D, KS> ? 2 : 1;      // results of this launch (one: x0 and out0)
    __shared__ __attribute__((aligned(16))) float lds[NB][(G::ROWS + 1) * G::PITCH];  // (the column behind the last)
    const int t = tile_of_block(ntiles);
    if (t < 0) return;
    const Shape &s = a.s;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Lane ln = lane_place();
    const int g = ln.g;
    const int rows = s.H > 2 * NP && s.H <= 2 * KS ? 2 * NP : G::HR, cols = s.W > 2 * NP && s.W <= 2 * KS ? 2 * NP : G::HC;

    // the tile's keys and the queries that attend to them, the wave's keys and this lane's
    const Tile tl = tile_of(t, tiles_r, tiles_c, s.N);
    const int qa = inv_lo(tl.r0, KS), qb = inv_hi(min(tl.r0 + 8, s.H) - 1, s.H, KS);
    const int ca = inv_lo(tl.c0, KS), cb = inv_hi(min(tl.c0 + 8, s.W) - 1, s.W, KS);
    const int wr0 = tl.r0 + (wave >> 1) * 4, wc0 = tl.c0 + (wave & 1) * 4;
    const int kr0 = wr0 + 2 * (ln.b >> 1) + (ln.j >> 1), kc0 = wc0 + 2 * (ln.b & 1) + (ln.j & 1);
    const int kr = min(kr0, s.H - 1), kc = min(kc0, s.W - 1);
    const bool live = kr0 < s.H && kc0 < s.W;
    const int64_t img_tok = ((int64_t)tl.bb * s.N + tl.nn) * s.H * (int64_t)s.W;
    Regs32 st[NB];
    auto fetch_rows = [&](int br, int bc) __attribute__((always_inline)) {
        fetch32<D, KS>(st[0], image32(x0, tl), x0.sh, x0.sw, br, bc, qb, cb);
        if constexpr (NB == 2) fetch32<D, KS>(st[1], image32(x1, tl), x1.sh, x1.sw, br, bc, qb, cb);
    };
    // Patches of a block that the wave's keys need (the same number for its blocks of keys), the rows and columns of
    // queries in them, this lane's first query there, and the weights of query g of every patch
    // for this lane's key.  Where it does not attend, or is not in the block, the weight's place is beyond the
    // buffer, which reads as zero: a place is one addition of its row's and its column's, without a mask or a branch
    // (d128 k5 176 -> 149 us for the two launches).
    // All patches lie within the queries that the wave's keys together need, a block that needs fewer moved up where
    // its last patch would leave them, and where they are an odd number the last patch is cut: every query is met once
    // and no other is, so that a value that is not finite reaches no key that does not see it but one beside such keys.
    int npr, npc, nr, nc, base;
    float w[NB][NP * NP];
    auto weights = [&](int br, int bc) __attribute__((always_inline)) {
        const int rend = min(br + rows, qb), cend = min(bc + cols, cb);
        // of the queries [lo, end), those that attend to one of the two keys from k0 on, and of the two keys behind them: the
        // first ones, the patches that the longer of both takes, and how many queries both are together
        auto span = [&](int k0, int L, int lo, int end, int (&first)[2], int &patches) __attribute__((always_inline)) {
            int last[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                first[i] = max(inv_lo(min(k0 + 2 * i, L - 1), KS), lo);
                last[i] = min(inv_hi(min(k0 + 2 * i + 1, L - 1), L, KS), end);
            }
            patches = (max(last[0] - first[0], last[1] - first[1]) + 1) >> 1;
            const int from = min(first[0], first[1]), all = max(last[0], last[1]) - from, most = max(all - 2 * patches, 0);
#pragma unroll
            for (int i = 0; i < 2; i++) first[i] = min(first[i], from + most);
            return min(all, 2 * patches);
        };
        int r0[2], c0[2];
        nr = span(wr0, s.H, br, rend, r0, npr);
        nc = span(wc0, s.W, bc, cend, c0, npc);
        if (wr0 >= s.H || wc0 >= s.W) npr = nr = 0;
        const int fr = ln.b >> 1 ? r0[1] : r0[0], fc = ln.b & 1 ? c0[1] : c0[0];
        base = ((fr - br) * G::HC + fc - bc) * G::PITCH + second_channel<D>(ln);
        // (at most 14 rows of an image of at most 2^16 columns, WIDE: below 2^30 bytes)
        constexpr unsigned kNone = 0x60000000u;
        const int64_t row0 = img_tok + (int64_t)br * s.W;
        const auto buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(ws_w + row0 * (G::KK * NB)), 0,
                                                           (rend - br) * s.W * (G::KK * NB * 4), 0x00027000);
        if constexpr (WIDE) {
#pragma unroll
            for (int pr = 0; pr < NP; pr++) {
                if (pr >= npr) break;
                const int qr = fr + 2 * pr + (g >> 1), ar = kr - win_start(qr, s.H, KS);
#pragma unroll
                for (int pc = 0; pc < NP; pc++) {
                    if (pc >= npc) break;
                    const int qc = fc + 2 * pc + (g & 1), ac = kc - win_start(qc, s.W, KS);
                    const bool ok = qr < rend && qc < cend && (unsigned)ar < (unsigned)KS && (unsigned)ac < (unsigned)KS;
                    const float *at = ws_w + ((img_tok + qr * (int64_t)s.W + qc) * G::KK + ar * KS + ac) * NB;
#pragma unroll
                    for (int b = 0; b < NB; b++) w[b][pr * NP + pc] = ok ? at[b] : 0.f;
                }
            }
            return;
        }
        unsigned col[NP];
#pragma unroll
        for (int pc = 0; pc < NP; pc++) {
            const int qc = fc + 2 * pc + (g & 1), at = kc - win_start(qc, s.W, KS);
            col[pc] = qc < cend && (unsigned)at < (unsigned)KS ? (unsigned)(qc * G::KK + at) * (4u * NB) : kNone;
        }
#pragma unroll
        for (int pr = 0; pr < NP; pr++) {
            if (pr >= npr) break;
            const int qr = fr + 2 * pr + (g >> 1), at = kr - win_start(qr, s.H, KS);
            const unsigned row = qr < rend && (unsigned)at < (unsigned)KS
                                     ? (unsigned)((qr - br) * s.W * G::KK + at * KS) * (4u * NB) : kNone;
#pragma unroll
            for (int pc = 0; pc < NP; pc++) {
                if (pc >= npc) break;
                if constexpr (NB == 2) {
                    const auto pair = __builtin_amdgcn_raw_buffer_load_b64(buf, row + col[pc], 0, 0);
                    w[0][pr * NP + pc] = __uint_as_float(pair[0]);
                    w[1][pr * NP + pc] = __uint_as_float(pair[1]);
                } else {
                    w[0][pr * NP + pc] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(buf, row + col[pc], 0, 0));
                }
            }
        }
    };

    f32x4 acc[NB][G::DT];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int m = 0; m < G::DT; m++) acc[b][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    int br = qa, bc = ca;
    fetch_rows(br, bc);
    weights(br, bc);
    for (;;) {
#pragma unroll
        for (int b = 0; b < NB; b++) commit32<D, KS>(lds[b], st[b]);
        __syncthreads();
        bc += cols;
        if (bc >= cb) bc = ca, br += rows;
        const bool more = br < qb;
        if (more) fetch_rows(br, bc);
        const float *xrow[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) xrow[b] = lds[b] + base;
        if ((KS > 3 || D < 128) && nr == KS + 1 && nc == KS + 1) {
            // The patches of an inner tile, without a branch between them: a token's operands are read a token ahead (B4 N4 96x96
            // d64 k7 85 -> 70 us, d128 k7 256 -> 181; the four patches of d128 k3 56 -> 62).
            float x[2][NB][G::DT], wb[NB][4];
#pragma unroll
            for (int b = 0; b < NB; b++) second_fetch<D>(xrow[b], x[0][b]);
            each_step([&](auto at) __attribute__((always_inline)) {
                constexpr int step = decltype(at)::value, next = step + 1;
                if constexpr (next < G::STEPS)
#pragma unroll
                    for (int b = 0; b < NB; b++) second_fetch<D>(xrow[b] + G::at(next >> 2, next & 3), x[next & 1][b]);
                if constexpr (step % 4 == 0)
#pragma unroll
                    for (int b = 0; b < NB; b++) spread_rows(w[b][step / 4 / G::PW * NP + step / 4 % G::PW], wb[b]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < NB; b++) second_step<D>(x[step & 1][b], wb[b][step & 3], acc[b]);
                __builtin_amdgcn_sched_barrier(0);
            }, std::make_integer_sequence<int, G::STEPS>{});
        } else {
#pragma unroll
            for (int pr = 0; pr < NP; pr++) {
                if (pr >= npr) break;
                const bool cut_row = 2 * pr + 1 >= nr;
                const int below = cut_row ? 0 : G::HC * G::PITCH;  // (a row cut off is not in the staged block, perhaps)
#pragma unroll
                for (int pc = 0; pc < NP; pc++) {
                    if (pc >= npc) break;
                    // A patch's operands are read from LDS ahead of its matrix instructions.
                    float x[4][NB][G::DT], wb[NB][4];
#pragma unroll
                    for (int i = 0; i < 4; i++)
#pragma unroll
                        for (int b = 0; b < NB; b++)
                            second_fetch<D>(xrow[b] + (i >> 1 ? below : 0) + (2 * pr * G::HC + 2 * pc + (i & 1)) * G::PITCH, x[i][b]);
#pragma unroll
                    for (int b = 0; b < NB; b++) spread_rows(w[b][pr * NP + pc], wb[b]);
                    if (cut_row)
#pragma unroll
                        for (int b = 0; b < NB; b++) cut<G::DT>(x[2][b]), cut<G::DT>(x[3][b]);
                    if (2 * pc + 1 >= nc)
#pragma unroll
                        for (int b = 0; b < NB; b++) cut<G::DT>(x[1][b]), cut<G::DT>(x[3][b]);
#pragma unroll
                    for (int i = 0; i < 4; i++)
#pragma unroll
                        for (int b = 0; b < NB; b++) second_step<D>(x[i][b], wb[b][i], acc[b]);
                }
            }
        }
        if (!more) break;
        weights(br, bc);
        __syncthreads();  // every wave is done with these rows
    }
    if (wr0 >= s.H || wc0 >= s.W) return;
    const int64_t tok = img_tok + (int64_t)kr * s.W + kc;
#pragma unroll
    for (int b = 0; b < NB; b++) {
        second_pieces<D>(acc[b]);
        store32<D, kLines32<D, KS>>((b ? out1 : out0) + tok * D, g, acc[b], second_flip<D>(ln), b ? mul1 : mul0, live);
    }
}

// ------------------------------------------------------------------ dispatch
template <int D, int KS>
int fwd32_launch(const FwdArgs &a, hipStream_t st) {
    const int tiles_r = (a.s.H + 7) / 8, tiles_c = (a.s.W + 7) / 8;
    const int64_t nt = (int64_t)a.s.B * a.s.N * tiles_r * tiles_c;
    const int grid = persistent_grid<fwd_mfma_f32<D, KS>>(nt);
    {
        ProfScope prof(ENATTEN_KERNEL_FWD, "fwd_mfma_f32", st);
        hipLaunchKernelGGL((fwd_mfma_f32<D, KS>), dim3(grid), dim3(256), 0, st, a, tiles_r, tiles_c, (int)nt);
    }
    return check_launch("enatten2d_fwd");
}

template <int D, int KS>
int bwd32_launch(const BwdArgs &a, hipStream_t st) {
    const int tiles_r = (a.s.H + 7) / 8, tiles_c = (a.s.W + 7) / 8;
    const int64_t nt = (int64_t)a.s.B * a.s.N * tiles_r * tiles_c;
    const int grid = (int)((nt + 7) / 8 * 8);
    const int64_t queries = (int64_t)a.s.B * a.s.N * a.s.H * a.s.W;
    float *ws_p = a.delta, *ws_ds = a.delta + queries * KS * KS;
    {
        ProfScope prof(ENATTEN_KERNEL_BWD_DQ, "bwd_dq_mfma_f32", st);
        hipLaunchKernelGGL((bwd_dq_mfma_f32<D, KS>), dim3(persistent_grid<bwd_dq_mfma_f32<D, KS>>(nt)),
                           dim3(256), 0, st, a, ws_p, ws_ds, tiles_r, tiles_c, (int)nt);
    }
    {
        // dV = P^T dO and dK = dS^T Q: in one launch, or one after the other
        ProfScope prof(ENATTEN_KERNEL_BWD_DKDV, "bwd_dkdv_mfma_f32", st);
        float *dv = static_cast<float *>(a.dv), *dk = static_cast<float *>(a.dk);
        const auto kernel = a.s.W > 65536 ? bwd_dkdv_mfma_f32<D, KS, true> : bwd_dkdv_mfma_f32<D, KS, false>;
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, st, a, a.d_o, a.q, ws_p, dv, dk, 1.f, a.s.scale, tiles_r,
                           tiles_c, (int)nt);
        if (!kPair32<D, KS>)
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, st, a, a.q, a.q, ws_ds, dk, dk, a.s.scale, 1.f,
                               tiles_r, tiles_c, (int)nt);
    }
    return check_launch("enatten2d_bwd");
}

#define ENATTEN_F32_BY_KS(FN, D, ARGS, ST)                 \
    switch ((ARGS).s.kh) {                                 \
        case 3: return FN<D, 3>(ARGS, ST);                 \
        case 5: return FN<D, 5>(ARGS, ST);                 \
        case 7: return FN<D, 7>(ARGS, ST);                 \
    }
#define ENATTEN_F32_BY_D(FN, ARGS, ST)                     \
    switch ((ARGS).s.D) {                                  \
        case 32: ENATTEN_F32_BY_KS(FN, 32, ARGS, ST) break;   \
        case 64: ENATTEN_F32_BY_KS(FN, 64, ARGS, ST) break;   \
        case 128: ENATTEN_F32_BY_KS(FN, 128, ARGS, ST) break; \
    }

// 16-byte loads of float rows: aligned base, strides that are multiples of 4 floats,
// row and pixel strides small enough for 24-bit multiplies of byte offsets
bool layout32_ok(const View &v) {
    return reinterpret_cast<uintptr_t>(v.ptr) % 16 == 0 && v.sb % 4 == 0 && v.sn % 4 == 0 &&
           v.sh % 4 == 0 && v.sw % 4 == 0 && v.sh < (1 << 21) && v.sw < (1 << 21);
}

}  // namespace

// float32 tensors, head_dim 32 / 64 / 128, kernel_size 3 / 5 / 7
bool mfma_f32_supported(int D, int ks, int dtype) {
    return dtype == ENATTEN_F32 && (D == 32 || D == 64 || D == 128) && (ks == 3 || ks == 5 || ks == 7);
}

// float32 per query that the backward of these kernels needs in the workspace
size_t mfma_f32_workspace_floats(int ks) { return (size_t)2 * ks * ks; }

int launch_fwd_mfma_f32(const FwdArgs &a, hipStream_t st) {
    if (!layout32_ok(a.q) || !layout32_ok(a.k) || !layout32_ok(a.v) || !layout32_ok(a.o))
        return launch_fwd_simt(a, ENATTEN_F32, st);
    ENATTEN_F32_BY_D(fwd32_launch, a, st)
    set_error("no float32 matrix-core kernel for head_dim %d, kernel_size %d", a.s.D, a.s.kh);
    return ENATTEN_EUNSUPPORTED;
}

int launch_bwd_mfma_f32(const BwdArgs &a, hipStream_t st) {
    auto al = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    if (!layout32_ok(a.q) || !layout32_ok(a.k) || !layout32_ok(a.v) || !layout32_ok(a.d_o) ||
        !al(a.dq) || !al(a.dk) || !al(a.dv))
        return launch_bwd_simt(a, ENATTEN_F32, st);
    ENATTEN_F32_BY_D(bwd32_launch, a, st)
    set_error("no float32 matrix-core kernel for head_dim %d, kernel_size %d", a.s.D, a.s.kh);
    return ENATTEN_EUNSUPPORTED;
}

}  // namespace enatten
