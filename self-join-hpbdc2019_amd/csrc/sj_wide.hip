// Plain FP64 wide traversal kernel and its launch; the tile walk itself
// is in sj_wide.hpp.
#include "sj_wide.hpp"

namespace sj {

template <int PASS>
__global__ __launch_bounds__(JB) void k_join_wide(JoinArgs a) {
    __shared__ WideLds lds[WPB];
    if (PASS == PASS_FILL && !fill_gate(a)) return;
    const unsigned wave = threadIdx.x >> 6;
    const unsigned lane = __lane_id();
    WideLds &L = lds[wave];
    const uint32_t nTiles = *a.nTilesDev;
    LaneStats st;
    TileRec R;
    if (a.tileOrder) {
        const uint32_t ns = min(gridDim.x, (uint32_t)QSLICES);
        const uint32_t sl = blockIdx.x % ns;
        const uint32_t nbl = (gridDim.x - sl + ns - 1) / ns;
        uint64_t i = (uint64_t)(blockIdx.x / ns) * WPB + wave;
        for (;;) {
            const uint64_t q = queue_entry(i, sl, ns);
            if (q >= nTiles) break;
            uint32_t nx = 0;
            if (lane == 0) nx = atomicAdd(a.qctr + sl * QSTRIDE, 1u);
            process_tile_wide<PASS, true>(a, a.tileOrder[q], L, st, R);
            i = (uint64_t)nbl * WPB + readlane_u32(nx, 0);
        }
    } else {
        for (uint32_t tile = blockIdx.x * WPB + wave; tile < nTiles; tile += gridDim.x * WPB)
            process_tile_wide<PASS, true>(a, tile, L, st, R);
    }
    flush_stats(a, st);
    // record words this wave's chunks needed, plus its last partial block
    if (PASS == PASS_COUNT && a.recCtr && lane == 0) {
        const uint32_t sl = (blockIdx.x * WPB + wave) % REC_NSLICE;
        atomicAdd(&a.recCtr[REC_SLICE0 + sl * REC_STRIDE + 1], (unsigned long long)(R.want + REC_BLK));
    }
}

// Every grid the K == D tile walk does not cover, up to WIDE_MAXD dims.
bool wide_supported(int d, int k) { return d <= WIDE_MAXD && (d > DEV_MAXK || d != k); }

sj_status launch_join_wide(const JoinArgs &a, int pass, int cu_count, hipStream_t s) {
    const uint64_t len = (uint64_t)a.qEnd - a.qBegin;
    uint64_t blocks = std::min<uint64_t>((uint64_t)cu_count * 8, (len + 63) / 64 / WPB + 1);
    if (blocks == 0) blocks = 1;
    if (pass == PASS_COUNT)
        hipLaunchKernelGGL(k_join_wide<PASS_COUNT>, dim3((unsigned)blocks), dim3(JB), 0, s, a);
    else
        hipLaunchKernelGGL(k_join_wide<PASS_FILL>, dim3((unsigned)blocks), dim3(JB), 0, s, a);
    SJ_LAUNCH_CHECK();
    return SJ_OK;
}

}  // namespace sj
