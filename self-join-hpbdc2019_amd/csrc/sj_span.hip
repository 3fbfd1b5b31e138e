// Kernels of the span walk (d = k = 4..8); the device side is sj_span.hpp.
#include "sj_span.hpp"

namespace sj {

// Three waves per SIMD (at most 168 registers): the FP64 filter at K = 8 just
// fits.  K = 4 in FP32 fits four, which makes no difference (2M points, full
// stencil: count 1.95 ms, 1.93 with three).
template <int K, int PASS, bool F32, int MODE>
__global__ __launch_bounds__(JB) __attribute__((amdgpu_waves_per_eu(F32 && K == 4 ? 4 : 3))) void k_span(JoinArgs a) {
    __shared__ SpanLds lds[WPB];
    if (PASS == PASS_FILL && !fill_gate(a)) return;
    LaneStats st;
    TileRec R;
    tile_loop<PASS>(a, st, R, [&](uint32_t tile) __attribute__((always_inline)) {
        process_span<K, PASS, F32, MODE>(a, tile, lds[threadIdx.x >> 6], st, R);
    });
}

// The fill from the record: no coordinates, one kernel for every k and
// precision
__global__ __launch_bounds__(JB) void k_span_rp(JoinArgs a) {
    __shared__ SpanRows lds[WPB];
    if (!fill_gate(a)) return;
    LaneStats st;
    TileRec R;
    tile_loop<PASS_FILL>(a, st, R, [&](uint32_t tile) __attribute__((always_inline)) {
        replay_span(a, tile, lds[threadIdx.x >> 6], st);
    });
}

template <int K, int MODE>
static JoinKernel pick_k(int pass, int prec) {
    if constexpr (MODE == SPAN_DIRECT)  // no filter, so no precision of one
        return pass == PASS_COUNT ? k_span<K, PASS_COUNT, false, MODE> : k_span<K, PASS_FILL, false, MODE>;
    else if (pass == PASS_COUNT)
        return prec ? k_span<K, PASS_COUNT, true, MODE> : k_span<K, PASS_COUNT, false, MODE>;
    else
        return prec ? k_span<K, PASS_FILL, true, MODE> : k_span<K, PASS_FILL, false, MODE>;
}

template <int MODE>
static JoinKernel pick(int k, int pass, int prec) {
    switch (k) {
    case 4: return pick_k<4, MODE>(pass, prec);
    case 5: return pick_k<5, MODE>(pass, prec);
    case 6: return pick_k<6, MODE>(pass, prec);
    case 7: return pick_k<7, MODE>(pass, prec);
    case 8: return pick_k<8, MODE>(pass, prec);
    }
    return nullptr;
}

JoinKernel pick_span(const JoinArgs &a, int pass, int prec, bool replay) {
    if (replay) return k_span_rp;
    if (a.spanDirect) return pick<SPAN_DIRECT>(a.k, pass, prec);
    return a.spanDense ? pick<SPAN_BLOCKS>(a.k, pass, prec) : pick<SPAN_FILTER>(a.k, pass, prec);
}

}  // namespace sj
