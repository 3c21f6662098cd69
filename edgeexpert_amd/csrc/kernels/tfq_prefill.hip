// tfq_prefill.hip — grouped MoE prefill: device grouping of the routed pairs and the
// grouped gate/up and down launches (MFMA tile for large grouping tiles, weight
// stream for small ones, one launch each), at 4, 3 and 2 bits.
#include "entry_points.hpp"

extern "C" __global__ __launch_bounds__(kGroupThreads) void tfq_moe_group(
    const uint32_t* idx, const uint16_t* w, uint32_t T, uint32_t k, uint32_t E, Pair* sorted,
    uint32_t* offsets, uint32_t* counts, Tile* tiles, uint32_t* n_tiles, uint32_t* status) {
    moe_group(idx, w, T, k, E, sorted, offsets, counts, tiles, n_tiles, status);
}

#define TFQ_GROUPED_DOWN(NAME, BITS, RS, TAB)                                                    \
    extern "C" __global__ __launch_bounds__(kProjThreads, 2) void NAME(                           \
        ExpertPool pool, const Pair* sorted, const Tile* tiles, uint32_t* n_tiles,               \
        const uint16_t* act, uint16_t* partials, uint32_t D, uint32_t F, uint32_t k,             \
        GroupedLaunch gl) {                                                                      \
        moe_grouped_down_launch<BITS, RS, TAB>(pool, sorted, tiles, n_tiles, act, partials, D, F, k, gl); \
    }
// _t: the units' scale/bias tables staged through registers (aligned tables
// that fit), _w: small tiles in units of 256 outputs (both chosen by the host)
#define TFQ_GROUPED(SUFFIX, BITS, TAB)                                                           \
    extern "C" __global__ __launch_bounds__(kProjThreads, 2) void tfq_moe_grouped_gate_up##SUFFIX( \
        ExpertPool pool, const Pair* sorted, const Tile* tiles, uint32_t* n_tiles,               \
        const uint16_t* hidden, uint32_t stride, uint16_t* act, uint32_t D, uint32_t F,          \
        GroupedLaunch gl) {                                                                      \
        moe_grouped_gate_up_launch<BITS, TAB>(pool, sorted, tiles, n_tiles, hidden, stride, act, D, F, gl); \
    }                                                                                            \
    TFQ_GROUPED_DOWN(tfq_moe_grouped_down##SUFFIX, BITS, 2, TAB)                                  \
    TFQ_GROUPED_DOWN(tfq_moe_grouped_down##SUFFIX##_w, BITS, 4, TAB)
TFQ_GROUPED(, 4, false)
TFQ_GROUPED(_b2, 2, false)
TFQ_GROUPED(_b3, 3, false)
TFQ_GROUPED(_t, 4, true)
TFQ_GROUPED(_b2_t, 2, true)
TFQ_GROUPED(_b3_t, 3, true)

// gate/up of a few pairs per expert: CNT = ceil(d/1024)
#define TFQ_STREAM_GATE_UP(BITS, CNT)                                                            \
    extern "C" __global__ __launch_bounds__(kSkinnyThreads) void tfq_moe_stream_gate_up_b##BITS##_c##CNT( \
        ExpertPool pool, const Pair* sorted, const Tile* tiles, const uint32_t* n_tiles,         \
        const uint16_t* hidden, uint32_t stride, uint16_t* act, uint32_t D, uint32_t F) {        \
        moe_stream_gate_up<BITS, CNT>(pool, sorted, tiles, n_tiles, hidden, stride, act, D, F);  \
    }
#define TFQ_STREAM_GATE_UP_BITS(BITS) \
    TFQ_STREAM_GATE_UP(BITS, 1) TFQ_STREAM_GATE_UP(BITS, 2) TFQ_STREAM_GATE_UP(BITS, 3) TFQ_STREAM_GATE_UP(BITS, 4)
TFQ_STREAM_GATE_UP_BITS(2)
TFQ_STREAM_GATE_UP_BITS(3)
TFQ_STREAM_GATE_UP_BITS(4)
