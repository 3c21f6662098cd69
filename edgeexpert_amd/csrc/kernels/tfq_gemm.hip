// tfq_gemm.hip — the prefill dequant-fused GEMM: the 64-token MFMA projection tile
// and the few-token weight stream, int4 and 3-bit, fp16 and bf16 activations; the
// int8 rows over a block of tokens (shared expert, router).
#include "entry_points.hpp"
#include "gemm_q8.hpp"

#define TFQ_GEMM(TAG, BITS, DT, X_BF16)                                                          \
    extern "C" __global__ __launch_bounds__(kProjGemmThreads) void tfq_gemm_##TAG##_##DT(        \
        const uint16_t* X, const uint8_t* W, const uint16_t* S, const uint16_t* B, uint16_t* Y,  \
        uint32_t M, uint32_t N, uint32_t K, uint32_t ldx, uint32_t ldy) {                          \
        gemm_q4_proj<X_BF16, BITS>(X, W, S, B, Y, M, N, K, ldx, ldy);                             \
    }
TFQ_GEMM(q4, 4, f16, false)
TFQ_GEMM(q4, 4, bf16, true)
TFQ_GEMM(q3, 3, f16, false)
TFQ_GEMM(q3, 3, bf16, true)

// Few-token form (gemm_skinny.hpp): RT 16-row MFMA tiles per wave, C = ceil(K/1024)
// 128-code tiles per wave; _few: the loads for a handful of tokens.
#define TFQ_SKINNY_FORM(NAME, BITS, X_BF16, RT, C, LOADS)                                        \
    extern "C" __global__ __launch_bounds__(kSkinnyThreads) void NAME(                            \
        const uint16_t* X, const uint8_t* W, const uint16_t* S, const uint16_t* B, uint16_t* Y,   \
        uint32_t M, uint32_t N, uint32_t K, uint32_t ldx, uint32_t ldy) {                         \
        gemm_skinny<X_BF16, RT, BITS, C, LOADS>(X, W, S, B, Y, M, N, K, ldx, ldy);                \
    }
#define TFQ_SKINNY(TAG, BITS, DT, X_BF16, RT, C)                                                 \
    TFQ_SKINNY_FORM(tfq_gemm_skinny_##TAG##_##DT##_r##RT##_c##C, BITS, X_BF16, RT, C, kLoadsMemory) \
    TFQ_SKINNY_FORM(tfq_gemm_skinny_##TAG##_##DT##_r##RT##_c##C##_few, BITS, X_BF16, RT, C,       \
                    skinny_loads(C))
#define TFQ_SKINNY_C(TAG, BITS, DT, X_BF16, RT)                                                  \
    TFQ_SKINNY(TAG, BITS, DT, X_BF16, RT, 1) TFQ_SKINNY(TAG, BITS, DT, X_BF16, RT, 2)              \
    TFQ_SKINNY(TAG, BITS, DT, X_BF16, RT, 3) TFQ_SKINNY(TAG, BITS, DT, X_BF16, RT, 4)              \
    TFQ_SKINNY(TAG, BITS, DT, X_BF16, RT, 5) TFQ_SKINNY(TAG, BITS, DT, X_BF16, RT, 6)              \
    TFQ_SKINNY(TAG, BITS, DT, X_BF16, RT, 7) TFQ_SKINNY(TAG, BITS, DT, X_BF16, RT, 8)
TFQ_SKINNY_C(q4, 4, f16, false, 1)
TFQ_SKINNY_C(q4, 4, f16, false, 2)
TFQ_SKINNY_C(q4, 4, bf16, true, 1)
TFQ_SKINNY_C(q4, 4, bf16, true, 2)
TFQ_SKINNY_C(q3, 3, f16, false, 1)
TFQ_SKINNY_C(q3, 3, f16, false, 2)
TFQ_SKINNY_C(q3, 3, bf16, true, 1)
TFQ_SKINNY_C(q3, 3, bf16, true, 2)

// int8 rows over a block of tokens (gemm_q8.hpp): RT row tiles, NTT token tiles per block.
#define TFQ_Q8_BLOCK(RT, NTT)                                                                    \
    extern "C" __global__ __launch_bounds__(kQ8BlockThreads, 2) void tfq_q8_block_r##RT##_t##NTT(  \
        Q8Mat m, const uint16_t* X, uint16_t* Y, uint32_t M, uint32_t N, uint32_t K,             \
        uint32_t ldx, uint32_t ldy) {                                                            \
        gemm_q8_block<RT, NTT, false>(m, m, X, Y, M, N, K, ldx, ldy);                            \
    }
#define TFQ_Q8_BLOCK_GATED(RT, NTT)                                                              \
    extern "C" __global__ __launch_bounds__(kQ8BlockThreads, 2) void                             \
        tfq_q8_block_gated_r##RT##_t##NTT(Q8Mat gate, Q8Mat up, const uint16_t* X, uint16_t* Y,  \
                                          uint32_t M, uint32_t N, uint32_t K, uint32_t ldx,      \
                                          uint32_t ldy) {                                        \
        gemm_q8_block<RT, NTT, true>(gate, up, X, Y, M, N, K, ldx, ldy);                         \
    }
TFQ_Q8_BLOCK(1, 1) TFQ_Q8_BLOCK(1, 2) TFQ_Q8_BLOCK(1, 4)
TFQ_Q8_BLOCK_GATED(2, 1) TFQ_Q8_BLOCK_GATED(2, 2) TFQ_Q8_BLOCK_GATED(2, 4)
// many tokens: 64 tokens x 64 rows per block. Two wavefronts per SIMD asked
// for, so that 256 registers are the bound and the accumulators, which the
// scaling reads, stay in vector registers.
extern "C" __global__ __launch_bounds__(kQ8TileThreads, 2) void tfq_q8_tile(Q8Mat m, const uint16_t* X, uint16_t* Y,
                                                                         uint32_t M, uint32_t N, uint32_t K,
                                                                         uint32_t ldx, uint32_t ldy) {
    gemm_q8_tile<false>(m, m, X, Y, M, N, K, ldx, ldy);
}
extern "C" __global__ __launch_bounds__(kQ8TileThreads, 2) void tfq_q8_tile_gated(Q8Mat gate, Q8Mat up,
                                                                               const uint16_t* X, uint16_t* Y,
                                                                               uint32_t M, uint32_t N, uint32_t K,
                                                                               uint32_t ldx, uint32_t ldy) {
    gemm_q8_tile<true>(gate, up, X, Y, M, N, K, ldx, ldy);
}

// router logits of a block of tokens: C = ceil(d / 512) groups per wavefront
#define TFQ_ROUTER_BLOCK(C)                                                                      \
    extern "C" __global__ __launch_bounds__(kQ8BlockThreads, 2) void tfq_router_block_c##C(      \
        Q8Mat m, const uint16_t* h, uint32_t stride, const uint16_t* eff, float* logits,         \
        uint32_t T, uint32_t E, uint32_t K) {                                                    \
        router_block<C>(m, h, stride, eff, logits, T, E, K);                                     \
    }
TFQ_ROUTER_BLOCK(1) TFQ_ROUTER_BLOCK(2) TFQ_ROUTER_BLOCK(3) TFQ_ROUTER_BLOCK(4)
TFQ_ROUTER_BLOCK(5) TFQ_ROUTER_BLOCK(6) TFQ_ROUTER_BLOCK(7) TFQ_ROUTER_BLOCK(8)
