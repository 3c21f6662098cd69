// gemm_q8.hpp — int8 g64 rows times a block of tokens on the matrix cores:
//     Y[t][n] = Σ_g s[n][g]·(Σ_{k in g} q[n][k]·X[t][k]) + b[n][g]·(Σ_{k in g} X[t][k])
// in the decode kernels' factored form (gemv.hpp): the codes 0..255 are exact
// in fp16, so v_mfma_f32_16x16x32_f16 forms each group's Σ q·x and (with an
// operand of ones) Σ x with exact products and fp32 sums, and the scale and
// bias are applied to those sums in fp32. No weight is rounded to fp16. The
// gated form runs the same features' gate and up rows in one wavefront and
// stores act = fp16(gelu_tanh(gate)·up), both in fp32 until that rounding
// (shared_int8_gate_up_act_simd, S/Metal/Quant/dequant_int8.metal:99-154,
// over the rows of S/Kernels/Prefill/MoE/PrefillSharedExpert.swift:11-60).
//
// Block: 8 wavefronts over the same 16·RT weight rows and 16·NTT tokens,
// wave w taking an eighth of the groups (a split of K inside the block: the
// main loop has no barrier, and few rows still give many independent
// streams). A operand = 16 tokens, B operand = 16 weight rows, so in the D
// layout (column lane%16 = weight row, rows 4·(lane/16) + r = tokens) a lane
// has one row and applies one scale and bias per group. Lane quarter q takes
// codes 16q..16q+15 of a group: one 16-byte load per row tile, two k-steps.
// The eight partial tiles are added through LDS in wave order. From 65 tokens
// on, blocks of 64 tokens x 64 rows over the whole of K take over
// (gemm_q8_tile).
//
// Measured on MI355X, shared expert 2816 x 2112, gate/up + down launches: the
// decode kernels once per token took 17.4 us for 4 tokens, 53 for 16, 175 for
// 64 and 1463 for 512 (fp32 VALU dots, every weight converted again for every
// token); here 13.7 us for 16, 28 for 64 (strided operand reads bound it: see
// gemm_q8_tile), and the tile 34.6 us for 128, 62 for 512. The tile's 528
// gate/up blocks are 2.06 per CU: the 16 CUs with three set its time (27 us
// where no CU has more than two).
#pragma once

#include "moe_prefill.hpp"

namespace tfq {

constexpr uint32_t kQ8BlockThreads = 512;                 // 8 wavefronts
constexpr uint32_t kQ8BlockWaves = kQ8BlockThreads / 64;
constexpr uint32_t kQ8MaxK = 4096;                        // longest reduction (the int8 forms' limit)
constexpr int kQ8RedTokens = 2;                           // token tiles per LDS reduction round

// Token tiles of one reduction round.
constexpr int q8_round(int NTT) { return NTT < kQ8RedTokens ? NTT : kQ8RedTokens; }

// 8 byte codes (two words, element order) as exact fp16 values: each pair of
// bytes into the mantissas of two halves of exponent 2^10, minus base (1024
// for the codes 0..255 themselves).
__device__ __forceinline__ h8 q8_to_h8(uint32_t w0, uint32_t w1, _Float16 base = (_Float16)1024.0f) {
    const h2 m = {base, base};
    const h2 p[4] = {__builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w0, 0x04010400u)) - m,
                     __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w0, 0x04030402u)) - m,
                     __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w1, 0x04010400u)) - m,
                     __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w1, 0x04030402u)) - m};
    h8 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = p[i][0];
        v[2 * i + 1] = p[i][1];
    }
    return v;
}

// One group of a lane: its 16 codes of each row tile and its token's 16
// activations of each token tile.
template <int RT, int NTT>
struct Q8Stage {
    uint4 w[RT];
    uint4 x[NTT][2];
};

// GATED: row tiles 0..RT/2-1 are rows of m0 (gate), RT/2..RT-1 the same rows
// of m1 (up), and Y receives the activation; else every row tile is of m0.
// N rows; row t of X starts at X + t·ldx (16-byte aligned), of Y at Y + t·ldy.
template <int RT, int NTT, bool GATED>
__device__ __forceinline__ void gemm_q8_block(const Q8Mat& m0, const Q8Mat& m1, const uint16_t* __restrict__ X,
                                              uint16_t* __restrict__ Y, uint32_t M, uint32_t N, uint32_t K,
                                              uint32_t ldx, uint32_t ldy) {
    constexpr int NR = GATED ? RT / 2 : RT;               // row tiles of Y per block
    constexpr int RD = q8_round(NTT);
    static_assert(!GATED || RT % 2 == 0, "gate and up tiles in pairs");
    __shared__ f32x4 red[kQ8BlockWaves][RD][RT][64];
    __shared__ __attribute__((aligned(16))) uint32_t sb[16 * RT * (kQ8MaxK / 64)];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r16 = lane & 15u, q = lane >> 4;
    const uint32_t G = K >> 6;
    const uint32_t n0 = blockIdx.x * (16u * NR), t0 = blockIdx.y * (16u * NTT);
    // this wave's groups [g0, g1)
    const uint32_t g0 = wave * G / kQ8BlockWaves, g1 = (wave + 1) * G / kQ8BlockWaves;

    const uint8_t* wrow[RT];
    const uint32_t* sbt[RT];          // this lane's row of the scale/bias table
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const Q8Mat& m = GATED && i >= NR ? m1 : m0;
        const uint32_t r = n0 + 16u * (i % NR) + r16, rc = r < N ? r : N - 1;    // rows past N: clamped, not stored
        wrow[i] = m.w + (size_t)rc * K + 16u * q;
        sbt[i] = sb + (16u * NR * (i / NR) + rc - n0) * G;
    }
    // k-step u of a group: quarter q takes 16-byte piece 4u + {0,2,1,3}[q] of the token's 128 bytes
    const uint32_t piece = (q >> 1) | ((q & 1u) << 1);
    const uint16_t* xrow[NTT];
#pragma unroll
    for (int j = 0; j < NTT; ++j) {
        const uint32_t t = t0 + 16u * j + r16;
        xrow[j] = X + (size_t)(t < M ? t : M - 1) * ldx + 8u * piece;            // tokens past M: clamped, not stored
    }
    // unconditional: a group past the wave's last one re-reads that one (a
    // wave without groups reads the row's last group and uses none of it)
    auto load = [&](uint32_t g, Q8Stage<RT, NTT>& st) {
        const uint32_t gg = g < g1 ? g : (g1 > g0 ? g1 : G) - 1;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            st.w[i] = ldg16(wrow[i] + 64u * gg);
        }
#pragma unroll
        for (int j = 0; j < NTT; ++j)
#pragma unroll
            for (int u = 0; u < 2; ++u) st.x[j][u] = *reinterpret_cast<const uint4*>(xrow[j] + 64u * gg + 32u * u);
    };
    f32x4 acc[RT][NTT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NTT; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const h8 ones = {(_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f,
                     (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f};
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    auto compute = [&](uint32_t g, const Q8Stage<RT, NTT>& st) {
        h8 wv[RT][2];
        float sv[RT], bv[RT];
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            // the lane's codes are pieces 2q and 2q + 1 of the row's 64 (8
            // codes each): swapping the halves of the wavefront leaves pieces
            // {0,2,1,3}[q] and 4 + {0,2,1,3}[q], so that the activations of a
            // k-step are one 64-byte run of each token
            const auto p0 = __builtin_amdgcn_permlane32_swap(st.w[i].x, st.w[i].z, false, false);
            const auto p1 = __builtin_amdgcn_permlane32_swap(st.w[i].y, st.w[i].w, false, false);
            wv[i][0] = q8_to_h8((uint32_t)p0[0], (uint32_t)p1[0]);
            wv[i][1] = q8_to_h8((uint32_t)p0[1], (uint32_t)p1[1]);
            const uint32_t t = sbt[i][g];
            sv[i] = h2f((uint16_t)t);
            bv[i] = h2f((uint16_t)(t >> 16));
        }
#pragma unroll
        for (int j = 0; j < NTT; ++j) {
            const h8 x0 = __builtin_bit_cast(h8, st.x[j][0]), x1 = __builtin_bit_cast(h8, st.x[j][1]);
            f32x4 sx = __builtin_amdgcn_mfma_f32_16x16x32_f16(x0, ones, zero, 0, 0, 0);
            f32x4 d[RT];
#pragma unroll
            for (int i = 0; i < RT; ++i) d[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x0, wv[i][0], zero, 0, 0, 0);
            sx = __builtin_amdgcn_mfma_f32_16x16x32_f16(x1, ones, sx, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < RT; ++i) d[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x1, wv[i][1], d[i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc[i][j][r] = fmaf(bv[i], sx[r], fmaf(sv[i], d[i][r], acc[i][j][r]));
        }
    };
    Q8Stage<RT, NTT> sa, sc;
    load(g0, sa);
    {
        // scale | bias << 16 of the block's rows (contiguous in each matrix)
        const uint32_t cnt = (N - n0 < 16u * NR ? N - n0 : 16u * NR) * G;
        copy_sb_to_lds<kQ8BlockThreads, 1>(m0.s + (size_t)n0 * G, m0.b + (size_t)n0 * G, sb, cnt);
        if constexpr (GATED)
            copy_sb_to_lds<kQ8BlockThreads, 1>(m1.s + (size_t)n0 * G, m1.b + (size_t)n0 * G, sb + 16u * NR * G, cnt);
    }
    __syncthreads();
    uint32_t g = g0;
    for (; g + 2 <= g1; g += 2) {
        load(g + 1, sc);
        __builtin_amdgcn_sched_barrier(0);
        compute(g, sa);
        load(g + 2, sa);
        __builtin_amdgcn_sched_barrier(0);
        compute(g + 1, sc);
    }
    if (g < g1) compute(g, sa);

    // sum of the eight K-slices in wave order, kQ8RedTokens token tiles per
    // round: position p of a round is (token tile, row tile of Y, lane)
#pragma unroll
    for (int j0 = 0; j0 < NTT; j0 += RD) {
        if (j0) __syncthreads();
#pragma unroll
        for (int j = 0; j < RD; ++j)
#pragma unroll
            for (int i = 0; i < RT; ++i) red[wave][j][i][lane] = acc[i][j0 + j];
        __syncthreads();
        for (uint32_t p = tid; p < (uint32_t)(RD * NR) * 64u; p += kQ8BlockThreads) {
            const uint32_t l = p & 63u, i = (p >> 6) % NR, j = (p >> 6) / NR;
            f32x4 v = red[0][j][i][l];
#pragma unroll
            for (uint32_t w = 1; w < kQ8BlockWaves; ++w) v += red[w][j][i][l];
            if constexpr (GATED) {
                f32x4 u = red[0][j][NR + i][l];
#pragma unroll
                for (uint32_t w = 1; w < kQ8BlockWaves; ++w) u += red[w][j][NR + i][l];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = gelu_tanh(v[r]) * u[r];
            }
            const uint32_t n = n0 + 16u * i + (l & 15u), t = t0 + 16u * (j0 + j) + 4u * (l >> 4);
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r)
                if (n < N && t + r < M) Y[(size_t)(t + r) * ldy + n] = f2h(v[r]);
        }
    }
}

// ------------------------------------------------------ many-token tile ----

constexpr uint32_t kQ8TileTok = 64;          // tokens per block
constexpr uint32_t kQ8TileRows = 64;         // weight rows per block (gated: 32 features' gate and up rows)
constexpr uint32_t kQ8TileThreads = 256;     // four wavefronts, each 32 tokens x 32 rows

// LDS of the tile: two buffers of [64 tokens][64 halves] and [64 rows][64
// bytes], then the scale/bias table of its rows (K/64 words each).
constexpr uint32_t kQ8TileXBytes = kQ8TileTok * 128u, kQ8TileWBytes = kQ8TileRows * 64u;
constexpr uint32_t q8_tile_lds_bytes(uint32_t K) {
    return 2u * (kQ8TileXBytes + kQ8TileWBytes) + 4u * kQ8TileRows * (K / 64u);
}

// Block: 64 tokens x 64 weight rows, the whole of K, one group per step. Both
// operands pass through LDS, loaded in memory order (eight lanes per 128-byte
// run of a token, four per 64-byte run of a row). Read straight into the MFMA
// layout, where neighbouring lanes hold different rows, every 16-byte piece
// is a cache access of its own, and that rate bounds the kernel (the few-token
// form at 512 tokens: as long without its arithmetic as with it). A row's
// 16-byte pieces are stored at position piece ^ f(row), which spreads the 16
// rows of a quarter-wave read over all banks.
//
// Wave (wm, wn): tokens 32·wm.., rows 32·wn.. with v_mfma_f32_32x32x16_f16:
// lane (col = lane % 32, h = lane / 32) takes codes 32h + 8s..+7 of a group in
// k-step s. Σ q·x of a group starts from zero and is scaled into acc in fp32
// one step later (so that its four MFMAs have finished); b·Σ x is a second
// product with the bias itself (fp16, exact) as every weight of the group,
// summed over all groups on the matrix core in accb.
template <bool GATED>
__device__ __forceinline__ void gemm_q8_tile(const Q8Mat& m0, const Q8Mat& m1, const uint16_t* __restrict__ X,
                                             uint16_t* __restrict__ Y, uint32_t M, uint32_t N, uint32_t K,
                                             uint32_t ldx, uint32_t ldy) {
    extern __shared__ __attribute__((aligned(16))) uint8_t q8_lds[];
    constexpr uint32_t NR = GATED ? kQ8TileRows / 2 : kQ8TileRows;      // rows of Y per block
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t col = lane & 31u, h = lane >> 5, wm = wave & 1u, wn = wave >> 1;
    const uint32_t G = K >> 6;
    const uint32_t n0 = blockIdx.x * NR, t0 = blockIdx.y * kQ8TileTok;
    uint8_t* const xl = q8_lds;
    uint8_t* const wl = q8_lds + 2u * kQ8TileXBytes;
    uint32_t* const sb = reinterpret_cast<uint32_t*>(q8_lds + 2u * (kQ8TileXBytes + kQ8TileWBytes));

    // staging: token rows tid/8 and 32 + tid/8, piece tid%8; weight row tid/4, piece tid%4.
    // Gated LDS row 32·wn + c is feature 16·wn + c%16 of gate (c < 16) or up.
    const uint32_t xr = tid >> 3, xp = tid & 7u, wr = tid >> 2, wp = tid & 3u;
    const uint16_t* xsrc[2];
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t t = t0 + xr + 32u * i;
        xsrc[i] = X + (size_t)(t < M ? t : M - 1) * ldx + 8u * (xp ^ ((xr >> 1) & 7u));   // tokens past M: clamped, not stored
    }
    const uint32_t wf = GATED ? 16u * (wr >> 5) + (wr & 15u) : wr;
    const uint32_t wrow = n0 + wf < N ? n0 + wf : N - 1;                                  // rows past N: clamped, not stored
    const uint8_t* wsrc = (GATED && (wr & 16u) ? m1.w : m0.w) + (size_t)wrow * K + 16u * (wp ^ ((wr >> 2) & 3u));
    constexpr int DEPTH = 4;           // groups in flight per thread (register ring)
    u32x4 xa[DEPTH], xb[DEPTH], ws[DEPTH];
    auto load = [&](uint32_t g, auto sl) {
        constexpr int S = decltype(sl)::value;
        const uint32_t gg = g < G ? g : G - 1;
        xa[S] = *reinterpret_cast<const u32x4*>(xsrc[0] + 64u * gg);
        xb[S] = *reinterpret_cast<const u32x4*>(xsrc[1] + 64u * gg);
        ws[S] = *reinterpret_cast<const u32x4*>(wsrc + 64u * gg);
    };
    auto store = [&](auto sl, uint32_t b) {
        constexpr int S = decltype(sl)::value;
        u32x4* x = reinterpret_cast<u32x4*>(xl + b * kQ8TileXBytes);
        x[8u * xr + xp] = xa[S];
        x[8u * (xr + 32u) + xp] = xb[S];
        reinterpret_cast<u32x4*>(wl + b * kQ8TileWBytes)[4u * wr + wp] = ws[S];
    };
    // this lane's operand pieces: token row, weight row, table row
    const uint32_t ar = 32u * wm + col, br = 32u * wn + col;
    const uint32_t af = (ar >> 1) & 7u, bf = (br >> 2) & 3u;
    const uint32_t bfe = GATED ? 16u * wn + (col & 15u) : br;
    const uint32_t* const sbt = sb + (GATED && (col & 16u) ? NR * G : 0u) + (n0 + bfe < N ? bfe : N - 1 - n0) * G;

    f32x16 acc, accb, d[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = accb[r] = d[0][r] = d[1][r] = 0.0f;
    const f32x16 zero = acc;
    float sv[2] = {0.0f, 0.0f};
    // step g (ring slot ST = g % DEPTH): MFMAs of group g from buffer g % 2,
    // group g + 1 from its ring slot into the other buffer, group g + 1 + DEPTH
    // requested into that slot
    auto step = [&](uint32_t g, auto st_c) {
        constexpr int ST = decltype(st_c)::value, P = ST & 1, NS = (ST + 1) % DEPTH;
        const uint4* x = reinterpret_cast<const uint4*>(xl + P * kQ8TileXBytes) + 8u * ar;
        const uint4* w = reinterpret_cast<const uint4*>(wl + P * kQ8TileWBytes) + 4u * br;
        const uint32_t t = sbt[g];
        h8 a[4];
#pragma unroll
        for (uint32_t s = 0; s < 4; ++s) a[s] = __builtin_bit_cast(h8, x[(4u * h + s) ^ af]);
        const uint4 w0 = w[(2u * h) ^ bf], w1 = w[(2u * h + 1u) ^ bf];
        const h8 b[4] = {q8_to_h8(w0.x, w0.y), q8_to_h8(w0.z, w0.w), q8_to_h8(w1.x, w1.y), q8_to_h8(w1.z, w1.w)};
        const _Float16 bh = __builtin_bit_cast(_Float16, (uint16_t)(t >> 16));
        const h8 bv = {bh, bh, bh, bh, bh, bh, bh, bh};
        d[P] = zero;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            d[P] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[s], b[s], d[P], 0, 0, 0);
            accb = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[s], bv, accb, 0, 0, 0);
        }
        sv[P] = h2f((uint16_t)t);
        // the group before this one: its sum times its scale
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = fmaf(sv[P ^ 1], d[P ^ 1][r], acc[r]);
        store(std::integral_constant<int, NS>{}, P ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        load(g + 1 + DEPTH, std::integral_constant<int, NS>{});
        __syncthreads();
    };
    sfor_w<0, DEPTH>([&](auto c) { load((uint32_t)c.value, c); });
    const uint32_t cnt = (N - n0 < NR ? N - n0 : NR) * G;
    copy_sb_to_lds<kQ8TileThreads, 2>(m0.s + (size_t)n0 * G, m0.b + (size_t)n0 * G, sb, cnt);
    if constexpr (GATED) copy_sb_to_lds<kQ8TileThreads, 2>(m1.s + (size_t)n0 * G, m1.b + (size_t)n0 * G, sb + NR * G, cnt);
    store(std::integral_constant<int, 0>{}, 0);
    load(DEPTH, std::integral_constant<int, 0>{});
    __syncthreads();
    uint32_t g = 0;
    for (; g + DEPTH <= G; g += DEPTH) sfor_w<0, DEPTH>([&](auto c) { step(g + c.value, c); });
    sfor_while<0, DEPTH - 1>([&](auto c) {
        if (g + c.value >= G) return false;
        step(g + c.value, c);
        return true;
    });
    // the last group's sum
    if (G & 1u) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = fmaf(sv[0], d[0][r], acc[r]);
    } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = fmaf(sv[1], d[1][r], acc[r]);
    }
    acc += accb;
    // D layout: column = lane % 32, row = 8·(r/4) + 4·h + r%4
    if constexpr (GATED) {
        // gate of feature col % 16 in lanes col < 16, up 16 lanes on: both to
        // both, each half of the lanes storing half of the tokens
        const uint32_t n = n0 + 16u * wn + (col & 15u);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t v = __builtin_bit_cast(uint32_t, (float)acc[r]);
            const auto p = __builtin_amdgcn_permlane16_swap(v, v, false, false);
            const float ga = __builtin_bit_cast(float, (uint32_t)p[0]), up = __builtin_bit_cast(float, (uint32_t)p[1]);
            acc[r] = gelu_tanh(ga) * up;
        }
#pragma unroll
        for (uint32_t r = 0; r < 8; ++r) {
            const float v = (col & 16u) ? acc[8 + r] : acc[r];
            const uint32_t rr = r + ((col & 16u) ? 8u : 0u);
            const uint32_t t = t0 + 32u * wm + 8u * (rr >> 2) + 4u * h + (rr & 3u);
            if (n < N && t < M) Y[(size_t)t * ldy + n] = f2h(v);
        }
    } else {
        const uint32_t n = n0 + br;
#pragma unroll
        for (uint32_t r = 0; r < 16; ++r) {
            const uint32_t t = t0 + 32u * wm + 8u * (r >> 2) + 4u * h + (r & 3u);
            if (n < N && t < M) Y[(size_t)t * ldy + n] = f2h(acc[r]);
        }
    }
}

// ------------------------------------------------ router, many tokens ----

// Logits of a block of prompt tokens: logits[t][e] = Σ_g s·Σ q·x + b·Σ x over
// x = h[t] ⊙ eff, as router_logits (gemv.hpp) forms them, in another order of
// the fp32 sums. The product of two fp16 values has 22 significant bits, so
// x·2^k = hi + lo with two fp16 values, exactly (k scales the largest |x| of
// the wavefront's slice of the token to [2^14, 2^15): nothing overflows, and
// what lo loses to fp16's smallest step lies 2^38 below that largest value);
// both go through the matrix cores with exact products. A slice that holds an
// infinity takes k = -17, which keeps every finite x finite, and lo = 0 beside
// a non-finite hi: sums come out infinite or NaN where the scalar form's do.
//
// 512 tokens, 128 experts x 2816: 36.4 us once per token (fp32 VALU dots over
// the whole router for every token), 9.3 us here; relative error against 64
// bits 2.0e-7 and 1.15e-7.
//
// Block: 8 wavefronts, 16 experts x 16 tokens, wave w the groups CNT·w ..
// (CNT = ceil(K / 512), all loaded before the first use; groups past K take
// x = 0). Operand layout as in gemm_q8_block.
template <int CNT>
__device__ __forceinline__ void router_block(const Q8Mat& m, const uint16_t* __restrict__ h, uint32_t stride,
                                             const uint16_t* __restrict__ eff, float* __restrict__ logits, uint32_t T,
                                             uint32_t E, uint32_t K) {
    __shared__ f32x4 red[kQ8BlockWaves][64];
    __shared__ __attribute__((aligned(16))) uint32_t sb[16 * (kQ8MaxK / 64)];
    __shared__ __attribute__((aligned(16))) float inv[kQ8BlockWaves][16];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r16 = lane & 15u, q = lane >> 4;
    const uint32_t G = K >> 6, n0 = blockIdx.x * 16u, t0 = blockIdx.y * 16u, g0 = wave * CNT;
    const uint32_t row = n0 + r16 < E ? n0 + r16 : E - 1;               // experts past E: clamped, not stored
    const uint32_t t = t0 + r16 < T ? t0 + r16 : T - 1;                 // tokens past T: clamped, not stored
    const uint32_t piece = (q >> 1) | ((q & 1u) << 1);                  // as in gemm_q8_block
    const uint8_t* wrow = m.w + (size_t)row * K + 16u * q;
    const uint16_t* xrow = h + (size_t)t * stride + 8u * piece;
    const uint16_t* erow = (eff ? eff : h) + 8u * piece;
    h8 xv[CNT][2], ev[CNT][2];
    u32x4 w[CNT];
#pragma unroll
    for (int c = 0; c < CNT; ++c) {
        const uint32_t g = g0 + c < G ? g0 + c : G - 1;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            xv[c][u] = *reinterpret_cast<const h8*>(xrow + 64u * g + 32u * u);
            ev[c][u] = *reinterpret_cast<const h8*>(erow + 64u * g + 32u * u);
        }
    }
#pragma unroll
    for (int c = 0; c < CNT; ++c)
        w[c] = *reinterpret_cast<const u32x4*>(wrow + 64u * (g0 + c < G ? g0 + c : G - 1));
    copy_sb_to_lds<kQ8BlockThreads, 1>(m.s + (size_t)n0 * G, m.b + (size_t)n0 * G, sb, (E - n0 < 16u ? E - n0 : 16u) * G);
    // x = h ⊙ eff, and the largest |x| of the slice (NaN aside) over the four lanes of the token
    float x[CNT][2][8], top = 0.0f;
#pragma unroll
    for (int c = 0; c < CNT; ++c)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float v = (float)xv[c][u][i] * (eff ? (float)ev[c][u][i] : 1.0f);
                x[c][u][i] = g0 + c < G ? v : 0.0f;
                top = fmaxf(top, fabsf(x[c][u][i]));
            }
    top = rows_combine<true>(top);
    // 2^k, k = 14 - exponent of the largest (a normal fp32 value: |x| is 0 or at least 2^-48)
    const uint32_t ex = __builtin_bit_cast(uint32_t, top) >> 23;
    const uint32_t kb = ex == 0 ? 127u : ex == 255u ? 127u - 17u : 127u + 14u + 127u - ex;
    const float up = __builtin_bit_cast(float, kb << 23);
    if (q == 0) inv[wave][r16] = __builtin_bit_cast(float, (254u - kb) << 23);
    const uint32_t* sbt = sb + (row - n0) * G;
    __syncthreads();
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const h8 ones = {(_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f,
                     (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f};
    // The codes are centred, q - 128 with bias b + 128·s: the same sum from
    // terms that hardly cancel. INF: for tokens whose slice holds an infinity
    // they stay 0..255, so that infinities and NaN arise where they do in the
    // scalar form.
    auto sum = [&](auto inf_c) {
        constexpr bool INF = decltype(inf_c)::value;
        f32x4 acc = zero;
        const _Float16 base = (_Float16)(INF ? 1024.0f : 1152.0f);
#pragma unroll
        for (int c = 0; c < CNT; ++c) {
            const auto p0 = __builtin_amdgcn_permlane32_swap(w[c].x, w[c].z, false, false);
            const auto p1 = __builtin_amdgcn_permlane32_swap(w[c].y, w[c].w, false, false);
            const h8 wv[2] = {q8_to_h8((uint32_t)p0[0], (uint32_t)p1[0], base),
                              q8_to_h8((uint32_t)p0[1], (uint32_t)p1[1], base)};
            f32x4 d = zero, sx = zero;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                h8 hi, lo;
#pragma unroll
                for (int i = 0; i < 8; i += 2) {
                    // truncated to 11 bits each: the rest of a 22-bit value again has 11
                    const float v0 = x[c][u][i] * up, v1 = x[c][u][i + 1] * up;
                    const auto hp = __builtin_amdgcn_cvt_pkrtz(v0, v1);
                    hi[i] = __builtin_bit_cast(h2, hp)[0];
                    hi[i + 1] = __builtin_bit_cast(h2, hp)[1];
                    float r0 = v0 - (float)hi[i], r1 = v1 - (float)hi[i + 1];
                    if (INF) {
                        r0 = __builtin_isfinite(v0) ? r0 : 0.0f;
                        r1 = __builtin_isfinite(v1) ? r1 : 0.0f;
                    }
                    const auto lp = __builtin_amdgcn_cvt_pkrtz(r0, r1);
                    lo[i] = __builtin_bit_cast(h2, lp)[0];
                    lo[i + 1] = __builtin_bit_cast(h2, lp)[1];
                }
                d = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, wv[u], d, 0, 0, 0);
                sx = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, ones, sx, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, wv[u], d, 0, 0, 0);
                sx = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, ones, sx, 0, 0, 0);
            }
            const uint32_t tw = sbt[g0 + c < G ? g0 + c : G - 1];
            const float sv = h2f((uint16_t)tw), bv = fmaf(INF ? 0.0f : 128.0f, sv, h2f((uint16_t)(tw >> 16)));
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = fmaf(bv, sx[r], fmaf(sv, d[r], acc[r]));
        }
        return acc;
    };
    f32x4 acc = sum(std::false_type{});
    if (__any(ex == 255u)) {
        // opaque copies: nothing of the sum above is kept in registers for this rare one
#pragma unroll
        for (int c = 0; c < CNT; ++c) {
#pragma unroll
            for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(x[c][0][i]), "+v"(x[c][1][i]));
            asm volatile("" : "+v"(w[c]));
        }
        const f32x4 a = sum(std::true_type{});
        const uint64_t inf = __ballot(ex == 255u);        // bit t: token t (lanes 0..15)
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r)
            if ((inf >> (4u * q + r)) & 1u) acc[r] = a[r];
    }
    // back to the tokens' own scale, then the sum of the eight slices in wave order
    acc *= *reinterpret_cast<const f32x4*>(&inv[wave][4u * q]);
    red[wave][lane] = acc;
    __syncthreads();
    if (wave != 0) return;
    f32x4 v = red[0][lane];
#pragma unroll
    for (uint32_t i = 1; i < kQ8BlockWaves; ++i) v += red[i][lane];
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r)
        if (n0 + r16 < E && t0 + 4u * q + r < T) logits[(size_t)(t0 + 4u * q + r) * E + n0 + r16] = v[r];
}

}  // namespace tfq
