// Canonical row order (sort_rows): every neighbour row ascending by point
// ID, in place.
//
// Bound: the pass reads and writes every neighbour ID once (129M IDs: 0.21 ms
// at the rate of a large copy); beyond that it is instruction issue.  A row of at most 1024 IDs is sorted in
// the registers of one wave, K IDs per lane (K = 1, 2, 4, 8, 16), by a
// bitonic network whose merges start with a mirrored step, so that every
// compare-exchange is ascending and the padding (INT32_MAX past the row's
// end) never moves below an ID.  Cross-lane partners come from DPP moves
// (distances within 16 lanes) and permlane16/32 swaps, each
// compare-exchange is one v_med3 against a per-lane limit (INT32_MIN keeps
// the smaller, INT32_MAX the larger value), and steps inside a lane's K
// registers need no data movement: no LDS and no synchronisation.  Short
// rows share a wave: four rows of at most 16 IDs or two of at most 32 go
// through one smaller network.  Longer rows are sorted in runs of 1024,
// merged in place through global memory by the wave.
// Measured per join (an LDS bitonic sort of one row per wave -> this): 129M
// IDs in rows of 64 on average 2.34 -> 0.374 ms, 54M in rows of 27 1.20 ->
// 0.195 ms, 24M in rows of 46 0.477 -> 0.094 ms.  The registers matter: at
// eight waves per SIMD with the row sizes' address arithmetic hoisted out of
// the row loop, 57 to 68 registers spilled and the first took 0.93 to 1.18 ms.
// A wave takes 16 rows in turn, which loses a little where there are too few
// rows for the chip (200 rows of 200 22 -> 27 us, 1,000 of 250 23 -> 27 us) and
// nothing from 1,000 rows of 1,000 on (99 -> 85 us; 64,000 of 1,000 1.02 ->
// 0.20 ms); rows above 1,024: 64,000 of 4,000 163 -> 3.3 ms.
#include "sj_common.hpp"

namespace sj {

namespace {

constexpr int SRB = 256;  // threads per block
constexpr int SRW = 16;   // consecutive rows per wave

__device__ __forceinline__ uint64_t readlane64(uint64_t v, int l) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l);
    return ((uint64_t)hi << 32) | lo;
}

// The lane ID, opaque to the compiler: what is derived from it is computed
// where it is used.  Hoisted out of the row loop, the addresses and masks of
// all row sizes together spill.
__device__ __forceinline__ uint32_t local_lane() {
    uint32_t l = __lane_id();
    asm volatile("" : "+v"(l));
    return l;
}

// median of three: the smaller of a and b for lim = INT32_MIN, the larger
// for lim = INT32_MAX
__device__ __forceinline__ int32_t med3(int32_t a, int32_t b, int32_t lim) {
    return max(min(a, b), min(max(a, b), lim));  // one v_med3_i32
}

template <int CTRL>
__device__ __forceinline__ int32_t dpp(int32_t x) {
    return __builtin_amdgcn_mov_dpp(x, CTRL, 0xF, 0xF, true);
}

// the value that lane ^ 2^J (J = 4, 5) holds in y; lim as below for bit J.
// The swap of a register with itself leaves {lower half's, upper half's}.
template <int J>
__device__ __forceinline__ int32_t far_partner(int32_t y, int32_t lim) {
    if constexpr (J == 4) {
        const auto p = __builtin_amdgcn_permlane16_swap((unsigned)y, (unsigned)y, false, false);
        return lim < 0 ? (int32_t)p[1] : (int32_t)p[0];
    } else {
        const auto p = __builtin_amdgcn_permlane32_swap((unsigned)y, (unsigned)y, false, false);
        return lim < 0 ? (int32_t)p[1] : (int32_t)p[0];
    }
}

constexpr int QUAD_X1 = 0xB1, QUAD_X2 = 0x4E, QUAD_X3 = 0x1B;  // lane ^ 1, ^ 2, ^ 3
constexpr int ROW_ROR8 = 0x128, ROW_MIRROR = 0x140, ROW_HALF_MIRROR = 0x141;

// butterfly compare-exchange with lane ^ 2^J
template <int J>
__device__ __forceinline__ int32_t butterfly(int32_t x, const int32_t (&lim)[6]) {
    if constexpr (J == 0) return med3(x, dpp<QUAD_X1>(x), lim[0]);
    else if constexpr (J == 1) return med3(x, dpp<QUAD_X2>(x), lim[1]);
    else if constexpr (J == 2) return med3(x, dpp<QUAD_X3>(dpp<ROW_HALF_MIRROR>(x)), lim[2]);
    else if constexpr (J == 3) return med3(x, dpp<ROW_ROR8>(x), lim[3]);
    else if constexpr (J == 4) {
        const auto p = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)x, false, false);
        return med3((int32_t)p[0], (int32_t)p[1], lim[4]);
    } else {
        const auto p = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)x, false, false);
        return med3((int32_t)p[0], (int32_t)p[1], lim[5]);
    }
}

// mirrored compare-exchange of x with y of lane ^ (2^M - 1)
template <int M>
__device__ __forceinline__ int32_t mirrored(int32_t x, int32_t y, const int32_t (&lim)[6]) {
    if constexpr (M == 1) return med3(x, dpp<QUAD_X1>(y), lim[0]);
    else if constexpr (M == 2) return med3(x, dpp<QUAD_X3>(y), lim[1]);
    else if constexpr (M == 3) return med3(x, dpp<ROW_HALF_MIRROR>(y), lim[2]);
    else if constexpr (M == 4) return med3(x, dpp<ROW_MIRROR>(y), lim[3]);
    else if constexpr (M == 5) return med3(x, far_partner<4>(dpp<ROW_MIRROR>(y), lim[4]), lim[4]);
    else return med3(x, far_partner<5>(far_partner<4>(dpp<ROW_MIRROR>(y), lim[4]), lim[5]), lim[5]);
}

__device__ __forceinline__ void order(int32_t &a, int32_t &b) {
    const int32_t lo = min(a, b), hi = max(a, b);
    a = lo;
    b = hi;
}

// butterfly steps at register distances K/2 .. 1
template <int K>
__device__ __forceinline__ void merge_regs(int32_t (&x)[K]) {
#pragma unroll
    for (int d = K / 2; d > 0; d >>= 1) {
#pragma unroll
        for (int r = 0; r < K; r++)
            if (!(r & d)) order(x[r], x[r | d]);
    }
}

// the K registers of a lane ascending
template <int K>
__device__ __forceinline__ void sort_regs(int32_t (&x)[K]) {
#pragma unroll
    for (int s = 2; s <= K; s <<= 1) {
#pragma unroll
        for (int r = 0; r < K; r++)
            if (!(r & (s / 2))) order(x[r], x[(r | (s - 1)) - (r & (s - 1))]);  // mirrored in the block of s
#pragma unroll
        for (int d = s / 4; d > 0; d >>= 1) {
#pragma unroll
            for (int r = 0; r < K; r++)
                if (!(r & d)) order(x[r], x[r | d]);
        }
    }
}

// butterfly steps at lane distances 2^J .. 1, then the registers
template <int K, int J>
__device__ __forceinline__ void merge_lanes(int32_t (&x)[K], const int32_t (&lim)[6]) {
    if constexpr (J >= 0) {
#pragma unroll
        for (int r = 0; r < K; r++) x[r] = butterfly<J>(x[r], lim);
        merge_lanes<K, J - 1>(x, lim);
    } else {
        merge_regs<K>(x);
    }
}

// merges of 2^M lanes, M from M to ML
template <int K, int M, int ML>
__device__ __forceinline__ void merge_up(int32_t (&x)[K], const int32_t (&lim)[6]) {
    if constexpr (M <= ML) {
#pragma unroll
        for (int r = 0; r < (K + 1) / 2; r++) {
            const int32_t a = mirrored<M>(x[r], x[K - 1 - r], lim);
            if (r != K - 1 - r) x[K - 1 - r] = mirrored<M>(x[K - 1 - r], x[r], lim);
            x[r] = a;
        }
        merge_lanes<K, M - 2>(x, lim);
        merge_up<K, M + 1, ML>(x, lim);
    }
}

// element lane * K + r of each group of 2^ML lanes ascending
template <int K, int ML>
__device__ __forceinline__ void sort_net(int32_t (&x)[K], const int32_t (&lim)[6]) {
    sort_regs<K>(x);
    merge_up<K, 1, ML>(x, lim);
}

// one row of at most 64 K IDs
template <int K>
__device__ __forceinline__ void sort_row(int32_t *v, uint32_t len, const int32_t (&lim)[6]) {
    const uint32_t lane = local_lane();
    int32_t x[K];
    // any order will do on the way in: coalesced
#pragma unroll
    for (int r = 0; r < K; r++) x[r] = lane + 64u * r < len ? v[lane + 64u * r] : INT32_MAX;
    sort_net<K, 6>(x, lim);
    const uint32_t e = lane * K;
    if (K > 1 && e + K <= len) {
        __builtin_memcpy(v + e, x, sizeof x);
    } else {
#pragma unroll
        for (int r = 0; r < K; r++)
            if (e + r < len) v[e + r] = x[r];
    }
}

// the steps at distances 512 .. 1 of a longer merge, on one run of 1024
__device__ __forceinline__ void merge_run(int32_t *v, uint64_t len, const int32_t (&lim)[6]) {
    constexpr int K = 16;
    const uint64_t e = (uint64_t)local_lane() * K;
    int32_t x[K];
#pragma unroll
    for (int r = 0; r < K; r++) x[r] = e + r < len ? v[e + r] : INT32_MAX;
    merge_lanes<K, 5>(x, lim);
#pragma unroll
    for (int r = 0; r < K; r++)
        if (e + r < len) v[e + r] = x[r];
}

__device__ __forceinline__ void wave_mem_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

// rows above 1024 IDs, by one wave in place.  Partners past the row's end
// stand for padding: never smaller, so nothing moves.
__device__ __forceinline__ void sort_long_row(int32_t *v, uint64_t len, const int32_t (&lim)[6]) {
    const uint32_t lane = local_lane();
    for (uint64_t b = 0; b < len; b += 1024) sort_row<16>(v + b, (uint32_t)min<uint64_t>(1024, len - b), lim);
    wave_mem_sync();
    for (uint64_t s = 2048; s / 2 < len; s <<= 1) {
        // mirrored step over blocks of s, then distances s / 4 .. 1024
        for (uint64_t d = s / 2; d >= 1024; d >>= 1) {
            const bool mirrored = d == s / 2;
            for (uint64_t i = lane; i < len / 2 + d; i += 64) {
                // i-th element of the lower halves of the blocks of 2 d
                const uint64_t a = 2 * (i & ~(d - 1)) + (i & (d - 1));
                const uint64_t c = mirrored ? a ^ (s - 1) : a + d;
                if (c < len) {
                    const int32_t x = v[a], y = v[c];
                    if (x > y) {
                        v[a] = y;
                        v[c] = x;
                    }
                }
            }
            wave_mem_sync();
        }
        for (uint64_t b = 0; b < len; b += 1024) merge_run(v + b, len - b, lim);
        wave_mem_sync();
    }
}

// R units of the wave's rows from row i on, all loaded before any is sorted:
// a unit is one row of at most 64 K IDs (ML = 6), or the next 2^(6 - ML)
// rows of at most 2^ML IDs each (K = 1).  off, next: lane l holds the ends
// of the wave's row l (empty past the last).
template <int R, int K, int ML>
__device__ __forceinline__ void sort_units(int32_t *ids, uint64_t off, uint64_t next, int i,
                                           const int32_t (&lim)[6]) {
    static_assert(K == 1 || ML == 6, "short rows take one register");
    const uint32_t lane = local_lane(), e = lane & ((1u << ML) - 1u);
    int32_t x[R][K];
    int32_t *v[R];
    uint32_t len[R];
#pragma unroll
    for (int u = 0; u < R; u++) {
        if constexpr (ML == 6) {
            const uint64_t b = readlane64(off, i + u);
            v[u] = ids + b;
            len[u] = (uint32_t)(readlane64(next, i + u) - b);
        } else {
            const int src = i + (u << (6 - ML)) + (int)(lane >> ML);
            const uint64_t b = __shfl(off, src, 64);
            v[u] = ids + b;
            len[u] = (uint32_t)(__shfl(next, src, 64) - b);
        }
        // any order will do on the way in: coalesced
#pragma unroll
        for (int r = 0; r < K; r++) x[u][r] = e + 64u * r < len[u] ? v[u][e + 64u * r] : INT32_MAX;
    }
#pragma unroll
    for (int u = 0; u < R; u++) sort_net<K, ML>(x[u], lim);
#pragma unroll
    for (int u = 0; u < R; u++) {
        if (K > 1 && (e + 1) * K <= len[u]) {
            __builtin_memcpy(v[u] + e * K, x[u], sizeof x[u]);
        } else {
#pragma unroll
            for (int r = 0; r < K; r++)
                if (e * K + r < len[u]) v[u][e * K + r] = x[u][r];
        }
    }
}

__global__ __launch_bounds__(SRB) __attribute__((amdgpu_waves_per_eu(8))) void k_sort_rows(const uint64_t *offsets, int32_t *ids, uint64_t n,
                                                   uint64_t base, uint64_t idsCap) {
    const unsigned lane = __lane_id();
    const uint64_t row0 = ((uint64_t)blockIdx.x * (SRB / 64) + (threadIdx.x >> 6)) * SRW;
    if (row0 >= n) return;
    if (idsCap && offsets[n] - base > idsCap) return;  // the fill wrote nothing
    const int rows = (int)min<uint64_t>(SRW, n - row0);
    // lane l: row row0 + l (rows past the end are empty)
    const uint64_t off = offsets[row0 + (uint64_t)min((int)lane, rows)] - base;
    const uint64_t next = offsets[row0 + (uint64_t)min((int)lane + 1, rows)] - base;
    const uint64_t len = next - off;
    int32_t lim[6];
#pragma unroll
    for (int b = 0; b < 6; b++) {
        lim[b] = (lane >> b) & 1u ? INT32_MAX : INT32_MIN;
        // opaque: a visible choice of two constants would split every med3
        asm volatile("" : "+v"(lim[b]));
    }
    const uint64_t le16 = __ballot(len <= 16), le32 = __ballot(len <= 32), le64 = __ballot(len <= 64);
    const uint64_t le128 = __ballot(len <= 128);
    for (int i = 0; i < rows;) {
        if (((le16 >> i) & 0xFFFFu) == 0xFFFFu) {
            sort_units<4, 1, 4>(ids, off, next, i, lim);
            i += 16;
        } else if (((le32 >> i) & 0xFFu) == 0xFFu) {
            sort_units<4, 1, 5>(ids, off, next, i, lim);
            i += 8;
        } else if (((le64 >> i) & 0xFu) == 0xFu) {
            sort_units<4, 1, 6>(ids, off, next, i, lim);
            i += 4;
        } else if (((le128 >> i) & 0x3u) == 0x3u) {
            sort_units<2, 2, 6>(ids, off, next, i, lim);
            i += 2;
        } else {
            const uint64_t m = readlane64(len, i);
            int32_t *v = ids + readlane64(off, i);
            if (m <= 256) sort_units<1, 4, 6>(ids, off, next, i, lim);
            else if (m <= 512) sort_row<8>(v, (uint32_t)m, lim);
            else if (m <= 1024) sort_row<16>(v, (uint32_t)m, lim);
            else sort_long_row(v, m, lim);
            i++;
        }
    }
}

}  // namespace

sj_status sort_rows_device(sj_context ctx, const uint64_t *offsets, int32_t *ids, uint64_t n, uint64_t base,
                           uint64_t idsCap) {
    if (!n) return SJ_OK;
    constexpr uint64_t RB = (uint64_t)SRW * (SRB / 64);
    hipLaunchKernelGGL(k_sort_rows, dim3((unsigned)((n + RB - 1) / RB)), dim3(SRB), 0, ctx->stream, offsets, ids, n,
                       base, idsCap);
    SJ_LAUNCH_CHECK();
    return SJ_OK;
}

}  // namespace sj
