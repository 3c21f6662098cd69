// gemm_skinny.hpp — the prefill projection GEMM for a few tokens:
//     Y[t][n] = Σ_k X[t][k] · W[n][k],  t < M (small), W affine g64 (2/3/4-bit)
//
// The 64-token projection tile (gemm.hpp) gives every block 256 outputs and
// the whole K loop, so below a few hundred tokens most of the chip idles
// (N/256 blocks per token tile) and each block's per-group barriers set the
// pace. For few tokens the work is a weight stream instead: each weight is
// dequantised once and multiplied with at most 16 tokens, on the matrix
// cores with v_mfma_f32_16x16x32_f16 whose A operand is 16 weight rows and
// whose B operand is 16 tokens.
//
// Block: 8 wavefronts over the same 16·RT rows, wave w taking the 128-code
// tiles w, w+8, w+16, … of K (CNT = ceil(K/1024) tiles each) (a split of K
// inside the block, so a block's rows are finished in one pass over K/8 per
// wave and the grid has N/(16·RT) blocks of 8 independent streams). Both
// operands are loaded in memory order, four lanes per 64-byte run of a row or
// token (row lane/4, quarter lane%4), and handed to the operand lanes (row or
// token lane%16, quarter lane/16) with ds_bpermute. Read straight in operand
// order, neighbouring lanes hold different rows and every 16-byte piece is a
// cache access of its own: that rate bounded this kernel (2816 x 4096, 48 tokens: 20.6
// us, now 11.9; 8192 x 2816, 128 tokens: 39.9 and 26.8; 16 tokens: 8.1 and 5.8).
// k-step j of a tile covers its codes 32j..32j+31, quarter q 8q..8q+7 of them:
// the x of a step is one 64-byte run of a token, and a weight lane, which holds
// chunk q, gets word q of chunk j from a 4 x 4 transpose over the lane
// quarters (four permlane swaps per row tile). Scales and biases: lane l loads
// row l/4's two groups of tile l%4 of the wave's next four, one bpermute per
// group hands them out. The weights are dequantised exactly as in the
// projection tile (fp16(q·s + b), one rounding), so both paths multiply the
// same fp16 weights. Nothing is staged in LDS except the final sum of the
// eight K-slices (fixed wave order: deterministic).
//
// A handful of tokens is another matter: the lanes past the last token repeat
// it, so operand-order accesses of x fall together, and what the launch waits
// for is the chain from a load to its MFMA, which the hand-over lengthens (2
// tokens bf16, 8192 x 2816: 8.4 us against 7.3; 704 x 2816: 5.3 and 4.5). There
// (skinny_loads) x, and up to 3072 inputs the weights too, are loaded in operand
// order: k-step j is then word j of the lane's chunk 4T + q.
#pragma once

#include "gemm.hpp"

namespace tfq {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kSkinnyThreads = 512;   // 8 wavefronts per block
constexpr uint32_t kSkinnyWaves = kSkinnyThreads / 64;
constexpr uint32_t kSkinnyTok = 16;        // tokens per blockIdx.y (the MFMA's N)

// Order in which a block loads its operands: both in memory order, x in operand
// order, or both in operand order.
enum SkinnyLoads { kLoadsMemory, kLoadsXOperand, kLoadsOperand };
// The order for a handful of tokens. us with both in memory order, x and both in
// operand order, 2 tokens bf16: 2048 x 2816 5.6, 5.0, 4.8; 8192 x 2816 8.5, 7.8,
// 7.4; 2816 x 4096 7.1, 6.4, 6.5; 2816 x 8192 11.7, 10.5, 10.7 (8 tokens 11.8,
// 11.1, 12.7).
constexpr SkinnyLoads skinny_loads(int CNT) { return CNT <= 3 ? kLoadsOperand : kLoadsXOperand; }

// One 128-code tile of a lane as loaded: its chunk of each of the RT rows, its
// four pieces of 8 activations (one per k-step) and, with weights in operand
// order, the scale and bias of each row's chunk.
template <int RT, int BITS>
struct SkinnyStage {
    QChunk<BITS> w[RT];
    u32x4 x[4];
    uint32_t s[RT], b[RT];
};

__device__ __forceinline__ h8 mask_h8(h8 v, uint32_t mask) {
    return __builtin_bit_cast(h8, __builtin_bit_cast(u32x4, v) & mask);
}

// Lane l loads quarter load_quarter(l) of row l/4 (the upper half of the
// wavefront in swapped order, which gives the 32 operand lanes of a bpermute
// pass 32 distinct source lanes mod 32).
__device__ __forceinline__ uint32_t load_quarter(uint32_t lane) { return (lane & 3u) ^ ((lane >> 4) & 2u); }
// ds_bpermute address of the lane that loaded quarter q of row r16.
__device__ __forceinline__ uint32_t operand_source(uint32_t r16, uint32_t q) {
    return 4u * (4u * r16 + (q ^ ((r16 >> 2) & 2u)));
}
__device__ __forceinline__ uint32_t from_lane(uint32_t addr, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)addr, (int)v);
}

// t[j] of lane quarter q <-> t[q] of lane quarter j.
__device__ __forceinline__ void transpose_quarters(uint32_t (&t)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(t[0], t[2], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(t[1], t[3], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    t[0] = (uint32_t)c[0];
    t[1] = (uint32_t)c[1];
    t[2] = (uint32_t)d[0];
    t[3] = (uint32_t)d[1];
}

// The K loop of a block and the sum of its eight K-slices: in wavefront 0 (true
// is returned there) acc[i] is row tile i in the 16x16 D layout (column lane%16
// = token, rows 4·(lane/16) + r). wrow, srow, brow: the row lane/4 of each tile;
// xrow: the token row lane/4 (lane%16 where LOADS has them in operand order).
// CNT: 128-code tiles per wave, ceil(K / 1024) (a compile-time count, so the
// loop unrolls and every wait names exactly the tile it needs).
template <bool X_BF16, int RT, int BITS, int CNT, SkinnyLoads LOADS = kLoadsMemory>
__device__ __forceinline__ bool skinny_rows(const uint8_t* const (&wrow)[RT], const uint16_t* const (&srow)[RT],
                                            const uint16_t* const (&brow)[RT], const uint16_t* __restrict__ xrow,
                                            uint32_t K, f32x4 (&acc)[RT]) {
    constexpr bool W_OP = LOADS == kLoadsOperand, X_OP = LOADS != kLoadsMemory;
    __shared__ f32x4 red[kSkinnyWaves][RT][64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r16 = lane & 15u, q = lane >> 4;
    const uint32_t nch = K >> 5;                       // 32-code chunks per row
    const uint32_t G = K >> 6;
    const uint32_t lq = load_quarter(lane), from = operand_source(r16, q);
    const uint32_t ntile = (K + 127u) >> 7;

    const DequantConsts<BITS> dc = dequant_consts<BITS>();

    // tile m of this wave is tile wave + 8m of the row; a chunk or piece past
    // the row end (the half-filled last tile, or a wave with fewer tiles)
    // re-reads a valid one, and its k-steps are left out
    auto load = [&](uint32_t m, SkinnyStage<RT, BITS>& st) {
        const uint32_t tile = wave + kSkinnyWaves * m;
        const uint32_t c = 4u * tile + (W_OP ? q : lq), cc = c < nch ? c : nch - 1;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            st.w[i] = ldg_chunk<BITS, false>(wrow[i], cc);
            if constexpr (W_OP) {
                st.s[i] = srow[i][cc >> 1];
                st.b[i] = brow[i][cc >> 1];
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t k = 128u * tile + 32u * j;
            const uint16_t* xp = W_OP ? xrow + 32u * cc + 8u * j : xrow + (k < K ? k : 0u) + 8u * (X_OP ? q : lq);
            st.x[j] = *reinterpret_cast<const u32x4*>(xp);
        }
    };
    // scale | bias << 16 of both groups of tile 4h + lane%4 (h-th four of the wave's tiles)
    uint32_t sb[(CNT + 3) / 4][RT][2];
    uint32_t sraw[(CNT + 3) / 4][RT][2], braw[(CNT + 3) / 4][RT][2];
    if constexpr (!W_OP) {
#pragma unroll
        for (uint32_t h = 0; h < (CNT + 3) / 4; ++h)
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (uint32_t g = 0; g < 2; ++g) {
                    const uint32_t gr = 2u * (wave + kSkinnyWaves * (4u * h + (lane & 3u))) + g, gc = gr < G ? gr : G - 1;
                    sraw[h][i][g] = srow[i][gc];
                    braw[h][i][g] = brow[i][gc];
                }
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto compute = [&](uint32_t m, const SkinnyStage<RT, BITS>& st) {
        const uint32_t tile = wave + kSkinnyWaves * m;       // wave-uniform
        if constexpr (W_OP) {
            // a chunk past the row end adds nothing: masked, not skipped (a
            // branch per tile took 0.4 us more)
            const uint32_t mask = 4u * tile + q < nch ? 0xFFFFFFFFu : 0u;
            h8 a[RT][4];
#pragma unroll
            for (int i = 0; i < RT; ++i) dequant_chunk_sb<BITS>(st.w[i], st.s[i] | (st.b[i] << 16), dc, a[i]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const h8 xv = X_BF16 ? bf16x8_to_f16(__builtin_bit_cast(uint4, st.x[j])) : __builtin_bit_cast(h8, st.x[j]);
                const h8 b = mask_h8(unit_b_order<BITS>(xv), mask);
#pragma unroll
                for (int i = 0; i < RT; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(mask_h8(a[i][j], mask), b, acc[i], 0, 0, 0);
            }
            return;
        }
        if (tile >= ntile) return;
        uint32_t t[RT][4], sw[RT][2];
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            QChunk<BITS> w;
#pragma unroll
            for (int k = 0; k < BITS; ++k) w.w[k] = from_lane(from, st.w[i].w[k]);
#pragma unroll
            for (int j = 0; j < 4; ++j) t[i][j] = block_word<BITS>(w, j);
            transpose_quarters(t[i]);
#pragma unroll
            for (int g = 0; g < 2; ++g) sw[i][g] = from_lane(4u * (4u * r16 + (m & 3u)), sb[m >> 2][i][g]);
        }
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            if (j >= 2 && 128u * tile + 32u * j >= K) break;       // the half-filled last tile
            u32x4 xr;
#pragma unroll
            for (int e = 0; e < 4; ++e) xr[e] = X_OP ? st.x[j][e] : from_lane(from, st.x[j][e]);
            const h8 xv = X_BF16 ? bf16x8_to_f16(__builtin_bit_cast(uint4, xr)) : __builtin_bit_cast(h8, xr);
            const h8 b = unit_b_order<BITS>(xv);
#pragma unroll
            for (int i = 0; i < RT; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(dequant_block_sb<BITS>(t[i][j], sw[i][j >> 1], dc), b,
                                                                acc[i], 0, 0, 0);
        }
    };
    // up to four tiles in flight: tile m + D is requested as soon as tile m
    // has been consumed
    constexpr int D = CNT < 4 ? CNT : 4;
    SkinnyStage<RT, BITS> st[D];
#pragma unroll
    for (int m = 0; m < D; ++m) load(m, st[m]);
    // keep every load ahead of the first use (the scheduler would otherwise
    // sink later tiles' loads into the first tile's compute)
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!W_OP) {
#pragma unroll
        for (uint32_t h = 0; h < (CNT + 3) / 4; ++h)
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int g = 0; g < 2; ++g) sb[h][i][g] = sraw[h][i][g] | (braw[h][i][g] << 16);
    }
#pragma unroll
    for (int m = 0; m < CNT; ++m) {
        compute((uint32_t)m, st[m % D]);
        if (m + D < CNT) load(m + D, st[m % D]);
        __builtin_amdgcn_sched_barrier(0);
    }

    // sum of the eight K-slices, in wave order
#pragma unroll
    for (int i = 0; i < RT; ++i) red[wave][i][lane] = acc[i];
    __syncthreads();
    if (wave != 0) return false;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        acc[i] = red[0][i][lane];
#pragma unroll
        for (uint32_t w = 1; w < kSkinnyWaves; ++w) acc[i] += red[w][i][lane];
    }
    return true;
}

// RT: 16-row MFMA tiles per wave (1 or 2); X_BF16: X and Y in bf16 (else
// fp16); rows of X and Y ldx and ldy halves apart.
template <bool X_BF16, int RT, int BITS, int CNT, SkinnyLoads LOADS = kLoadsMemory>
__device__ __forceinline__ void gemm_skinny(const uint16_t* __restrict__ X, const uint8_t* __restrict__ W,
                                            const uint16_t* __restrict__ S, const uint16_t* __restrict__ B,
                                            uint16_t* __restrict__ Y, uint32_t M, uint32_t N, uint32_t K,
                                            uint32_t ldx, uint32_t ldy) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t G = K >> 6, row_bytes = (K >> 3) * BITS;
    const uint32_t n0 = blockIdx.x * (16u * RT);
    const uint32_t t0 = blockIdx.y * kSkinnyTok, t = t0 + (lane & 15u), q = lane >> 4;
    const uint32_t lrow = lane >> 2;
    const uint8_t* wrow[RT];
    const uint16_t* srow[RT];
    const uint16_t* brow[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const uint32_t r = n0 + 16u * i + (LOADS == kLoadsOperand ? lane & 15u : lrow), rc = r < N ? r : N - 1;    // rows past N: clamped, not stored
        wrow[i] = W + (size_t)rc * row_bytes;
        srow[i] = S + (size_t)rc * G;
        brow[i] = B + (size_t)rc * G;
    }
    const uint32_t tl = t0 + (LOADS == kLoadsMemory ? lrow : lane & 15u);
    const uint16_t* xrow = X + (size_t)(tl < M ? tl : M - 1) * ldx;      // tokens past M: clamped, not stored
    f32x4 acc[RT];
    if (!skinny_rows<X_BF16, RT, BITS, CNT, LOADS>(wrow, srow, brow, xrow, K, acc)) return;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t n = n0 + 16u * i + 4u * q + r;
            if (n < N && t < M)
                Y[(size_t)t * ldy + n] = X_BF16 ? __builtin_bit_cast(uint16_t, (__bf16)acc[i][r]) : f2h(acc[i][r]);
        }
}

}  // namespace tfq
