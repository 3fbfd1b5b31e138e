// Device side of the span walk: the tile walk for points with d = k >= 4.
//
// In four and more dimensions a cell row (same coordinates in dims 1..k-1)
// holds few points and a tile has 3^(k-1) neighbour rows, so a walk over
// rows spends its time between rows, on half-empty waves.  Here a tile is a
// run of at most 64 points of one cell group: the cells that share the
// coordinates of dims g..k-1 (g >= 1, choose_span).  Cells are sorted
// with dim 0 fastest, so the cells adjacent to a tile's cells inside one of
// the 3^(k-g) neighbour groups lie in one span of sorted positions: from the
// first cell's linear ID minus M = sum of the multipliers of dims < g to the
// last cell's plus M, moved by the group's offset and cut to the group.
//
// All pairs of the tile and 16 candidates of the span at a time go through a
// filter on the matrix cores (v_mfma_*_16x16x4, FP64, or FP32 for
// the FP32+recheck form): with y = x - (the tile's first point), rounded
// once, |q|^2 + |c|^2 - 2 q.c <= T, where the products are the matrix
// instructions, |q|^2 is their accumulator input and |c|^2 sits in the
// threshold each lane compares with.  A candidate's coordinates enter the
// operand from one lane each, so nothing is staged; its norm is two
// cross-lane sums.  The norms are scaled by 1 - alpha and the threshold is
// T1 >= T, which covers every rounding (span_band), so the filter has no
// false misses; each candidate that passes is decided by the canonical FP64
// predicate.  Outside the filter's range (spanDirect: coordinates or eps
// near overflow or underflow) the predicate itself is evaluated for every
// candidate.
//
// Few pairs pass, so they are gathered across blocks and ranges in an LDS
// buffer and decided 64 at a time, one per lane (span_flush): the canonical
// predicate; the candidate in a cell adjacent to the query's (the span holds
// cells further away, and the grid join leaves such pairs out even when
// rounding puts their distance at eps); the form's claim.  Cells are compared
// by their coordinates modulo 4 (posPk, 4 bits per dim): a pair that passes
// the filter lies at most two cells apart, since a grid has fewer than 2^32
// cells per dim and eps is far above underflow.  Under spanDirect neither
// holds for the predicate (the squares of several eps may underflow to 0),
// so there the coordinates themselves are compared.
//
// Hit record: one word per hit, candidate | query << 32 | mirrored slot << 38 |
// (no mirrored hit) << 63, in the order of the walk, so a row's own hits keep
// ascending positions; blocks of candidates decided whole (span_dense) as masks
// of queries.  A tile's words start at recStart and fill the wave's blocks of
// REC_BLK words, whose last word links to the next block; recN counts them.
// The replaying fill reads up to 256 words at a time and looks nothing up.
// Bound: latency.  2M points uniform in 6-D, FP32+recheck: 9.4e9 pairs in
// 3.8 ms, of which the matrix instructions are busy 1.05 ms and the vector
// instructions 1.2 ms; 147 registers allow
// three waves per SIMD, and 46% of their cycles they wait (candidates' loads,
// the gathered pairs' loads and atomics).  Measured against the row walk with
// LDS-staged windows it replaced (count, replayed fill): that case 6.94, 4.11
// -> 3.84, 0.55 ms; 100,000 points in 8-D, FP64 6.23, 1.73 -> 1.25, 0.02 ms; 12
// joins in 2 to 8 dims in one graph 39.0, 33.1 ms -> 2.8 ms for both.  Tried and left: the candidates
// as scalar operands of vector FMAs (8.3 ms in 6-D, waiting for the scalar
// cache), hit masks per lane and 64-candidate piece instead of gathered pairs
// (5.9 ms, fill 1.2 ms), loads four steps ahead (4.1 ms: more registers).
#pragma once

#include "sj_traverse.hpp"

namespace sj {

constexpr int SPAN_MINK = 4;

constexpr uint32_t SPAN_BUF = 63 + 64 * 16;        // gathered pairs: 64 x 16 come in on top of at most 63
constexpr uint32_t SPAN_LINK = REC_BLK - 1u;       // a block's link to the next
constexpr uint64_t SPAN_SLOT_MAX = (1ull << 25) - 1;  // mirrored slots a record word holds
// Other record words, told by two of the bits that a word without a mirrored
// hit leaves 0: the head of a block of candidates (first | number << 32, then
// three words each: queries with hits, with mirrored hits, first slot), and
// the rest of the record block unused.
constexpr uint64_t SPAN_BLOCK = 3ull << 62, SPAN_SKIP = 5ull << 61;

// the tile's query rows (all the replaying fill needs)
struct SpanRows {
    uint64_t pos[64];       // fills: first entry of the query's row, NO_SLOT outside the window
    uint32_t room[64];      // fills: own hits the row holds
    int32_t id[64];         // its point ID
    uint32_t own[64];       // its own hits so far
};
struct SpanLds : SpanRows {
    double nq[64];          // scaled squared norms of the queries
    uint32_t cs0[64], cs1[64];  // the query's own cell as sorted positions
    uint32_t pk[64];        // its cell coordinates
    uint32_t hc[SPAN_BUF];  // gathered pairs: candidate position
    uint8_t hq[SPAN_BUF];   // and query
};

// The matrix instruction of a precision: v_mfma_f64_16x16x4 or
// v_mfma_f32_16x16x4.  Operand A element (i, kk) sits in lane i + 16 kk,
// operand B element (kk, j) in lane j + 16 kk, register r of the result holds
// column lane % 16 and row(lane, r).
template <bool F32>
struct SpanMma;
template <>
struct SpanMma<false> {
    typedef double T;
    typedef double V __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V mma(T a, T b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ unsigned row(unsigned lane, int r) { return (lane >> 4) + 4u * (unsigned)r; }
    // the sum over the lanes with the same lane % 16 (a register swapped with
    // itself leaves the own and the partner's value in some order)
    static __device__ __forceinline__ T sum16(T v) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const uint64_t b = (uint64_t)__double_as_longlong(v);
            const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
            const auto l = s == 0 ? __builtin_amdgcn_permlane16_swap(lo, lo, false, false)
                                  : __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
            const auto h = s == 0 ? __builtin_amdgcn_permlane16_swap(hi, hi, false, false)
                                  : __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
            v = __longlong_as_double((long long)(((uint64_t)h[0] << 32) | l[0])) +
                __longlong_as_double((long long)(((uint64_t)h[1] << 32) | l[1]));
        }
        return v;
    }
};
template <>
struct SpanMma<true> {
    typedef float T;
    typedef float V __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V mma(T a, T b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ unsigned row(unsigned lane, int r) { return 4u * (lane >> 4) + (unsigned)r; }
    static __device__ __forceinline__ T sum16(T v) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const unsigned b = __float_as_uint(v);
            const auto l = s == 0 ? __builtin_amdgcn_permlane16_swap(b, b, false, false)
                                  : __builtin_amdgcn_permlane32_swap(b, b, false, false);
            v = __uint_as_float(l[0]) + __uint_as_float(l[1]);
        }
        return v;
    }
};

// Fields of b - a modulo 4, 4 bits per dim.
__device__ __forceinline__ uint32_t pk_diff(uint32_t b, uint32_t a) { return ((b + 0x44444444u) - a) & 0x33333333u; }
// Any field equal to 2: the cells are not adjacent.
__device__ __forceinline__ bool pk_far(uint32_t z) { return (z & ~(z << 1) & 0x22222222u) != 0u; }

// The span of a tile inside its own group: linear IDs [lo, hi).
struct TileSpan {
    uint64_t lo, hi;
};
template <int K>
__device__ __forceinline__ TileSpan tile_span(const JoinArgs &a, int g, const uint32_t *cF, uint64_t linF,
                                              uint64_t linL) {
    uint64_t M = 0, base = linF;
#pragma unroll
    for (int j = 0; j < K; j++)
        if (j < g) {
            M += (uint64_t)a.mult[j];
            base -= (uint64_t)cF[j] * (uint64_t)a.mult[j];
        }
    const uint64_t size = (uint64_t)a.mult[g - 1] * a.nCells[g - 1];
    TileSpan s;
    s.lo = linF - base > M ? linF - M : base;
    s.hi = min(linL + M + 1, base + size);
    return s;
}

// Neighbour group `my` of 3^(K-g): its offsets in dims >= g (ternary digits,
// dim g fastest, so groups come in ascending linear ID), the linear offset,
// and whether it lies in the grid.
template <int K>
__device__ __forceinline__ bool span_group(const JoinArgs &a, int g, const uint32_t *cF, int my, int (&od)[K],
                                           int64_t &dl) {
    bool inb = true;
    dl = 0;
#pragma unroll
    for (int j = 0; j < K; j++) {
        od[j] = 0;
        if (j >= g) {
            od[j] = my % 3 - 1;
            my /= 3;
            const int64_t v = (int64_t)cF[j] + od[j];
            inb = inb && v >= 0 && v < (int64_t)a.nCells[j];
            dl += (int64_t)od[j] * a.mult[j];
        }
    }
    return inb;
}

__device__ __forceinline__ uint32_t uniform_u32(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) {
    return ((uint64_t)uniform_u32((uint32_t)(v >> 32)) << 32) | uniform_u32((uint32_t)v);
}

// A tile's side of the filter: the centre, operand A (-2 y of the queries,
// 16 per block) and the queries' scaled norms as accumulator inputs.
template <int K, bool F32>
struct SpanQuery {
    using M = SpanMma<F32>;
    using T = typename M::T;
    static constexpr int H = (K + 3) / 4;  // matrix instructions per 16 x 16 pairs
    double ctr[H];  // the centre's dims 4 h + lane / 16
    T A[4][H];
    typename M::V C[4];

    // FP64 coordinates of point t, dims 4 h + lane / 16 (the last dim beyond it)
    static __device__ __forceinline__ void fetch(const JoinArgs &a, uint32_t t, double (&x)[H]) {
        const double *p = a.pts + (uint64_t)t * K;
#pragma unroll
        for (int h = 0; h < H; h++) x[h] = p[min(4u * (unsigned)h + (__lane_id() >> 4), (unsigned)K - 1u)];
    }
    // relative to the centre, 0 beyond the last dim
    __device__ __forceinline__ T y(double x, int h) const {
        const T v = (T)(x - ctr[h]);
        return 4 * h + 3 < K || 4u * (unsigned)h + (__lane_id() >> 4) < (unsigned)K ? v : (T)0;
    }

    __device__ __forceinline__ void load(const JoinArgs &a, SpanLds &L, uint32_t ts0, uint32_t ts1) {
        const unsigned lane = __lane_id(), i = lane & 15u;
        const T scale = (T)a.spanScale;
        fetch(a, ts0, ctr);
        T *nq = reinterpret_cast<T *>(L.nq);
#pragma unroll
        for (int rb = 0; rb < 4; rb++) {
            double x[H];
            fetch(a, min(ts0 + 16u * rb + i, ts1 - 1u), x);
            T nn = (T)0;
#pragma unroll
            for (int h = 0; h < H; h++) {
                const T v = y(x[h], h);
                A[rb][h] = (T)-2 * v;
                nn = F32 ? fmaf(v, v, nn) : fma(v, v, nn);
            }
            nn = M::sum16(nn);
            // past the tile's end: never a hit
            if (lane < 16u) nq[16 * rb + i] = ts0 + 16u * rb + i < ts1 ? nn * scale : (T)INFINITY;
        }
        wave_lds_sync();
#pragma unroll
        for (int rb = 0; rb < 4; rb++)
#pragma unroll
            for (int r = 0; r < 4; r++) C[rb][r] = nq[16u * rb + M::row(lane, r)];
    }

    // Pairs of the 16 candidates [t0, ..) below t1, with coordinates x, that
    // pass the filter, handed to gather(pass, query, candidate) in ascending
    // candidates for each query.
    template <class Gather>
    __device__ __forceinline__ void filter(uint32_t t0, uint32_t t1, const double (&x)[H], T scale, T T1,
                                           Gather &gather) const {
        const unsigned lane = __lane_id(), j = lane & 15u;
        T B[H], nn = (T)0;
#pragma unroll
        for (int h = 0; h < H; h++) {
            B[h] = y(x[h], h);
            nn = F32 ? fmaf(B[h], B[h], nn) : fma(B[h], B[h], nn);
        }
        nn = M::sum16(nn);
        // past the end: never a hit
        const T thr = t0 + j < t1 ? T1 - nn * scale : (T)-INFINITY;
        typename M::V acc[4];
#pragma unroll
        for (int rb = 0; rb < 4; rb++) acc[rb] = M::mma(A[rb][0], B[0], C[rb]);
#pragma unroll
        for (int h = 1; h < H; h++)
#pragma unroll
            for (int rb = 0; rb < 4; rb++) acc[rb] = M::mma(A[rb][h], B[h], acc[rb]);
#pragma unroll
        for (int rb = 0; rb < 4; rb++)
#pragma unroll
            for (int r = 0; r < 4; r++) gather(acc[rb][r] <= thr, 16u * rb + M::row(lane, r), t0 + j);
    }
};

// Room for n <= 64 more record words of the tile in progress (started: it
// has words already): the first goes to the returned word, those from room
// on to the next block.  False when the record space is exhausted: the
// wave's block then may lie past the space (rec_room of an earlier tile of
// another instance), so not even a word that would fit in it is placed.
__device__ __forceinline__ bool span_rec_room(const JoinArgs &a, TileRec &R, uint32_t n, bool started, uint64_t &at,
                                              uint32_t &room, uint64_t &next) {
    room = R.used < SPAN_LINK ? SPAN_LINK - R.used : 0u;
    at = R.blk + R.used;
    next = 0;
    if (!R.ok) return false;
    if (n <= room) {
        R.used += n;
        return true;
    }
    const uint32_t sl = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) % REC_NSLICE;
    uint64_t b = 0;
    if (__lane_id() == 0) b = atomicAdd(&a.recCtr[REC_SLICE0 + sl * REC_STRIDE], 1ull);
    next = (readlane_u64(b, 0) * REC_NSLICE + sl) * REC_BLK;
    R.ok = next + REC_BLK <= a.maskCap;
    if (!R.ok) {
        if (__lane_id() == 0) atomicAdd(&a.recCtr[REC_BAD], 1ull);
        return false;
    }
    if ((started || room) && __lane_id() == 0) a.recMask[R.blk + SPAN_LINK] = next;
    if (!started && !room) at = next;
    R.blk = next;
    R.used = n - room;
    return true;
}

// Per-tile record state of the count.
struct SpanRec {
    bool on = false;
    uint32_t n = 0;
    uint64_t start = 0;
};

// Lanes of `active` with the same low 6 bits of v.
__device__ __forceinline__ uint64_t match6(uint64_t active, uint32_t v) {
    uint64_t peers = active;
#pragma unroll
    for (int b = 0; b < 6; b++) {
        const bool bit = (v >> b) & 1u;
        const uint64_t m = __ballot(bit);
        peers &= bit ? m : ~m;
    }
    return peers;
}

// One slot per lane of `mirror` in its candidate's row: the lanes of one
// candidate take theirs with one atomic (lanes whose candidate differs from
// their group's first in the higher bits only take their own).
template <class Ctr>
__device__ __forceinline__ uint64_t span_slots(Ctr *ctr, bool mirror, uint32_t c) {
    const uint64_t mm = __ballot(mirror);
    if (!mm) return 0;
    const uint64_t peers = match6(mm, c);
    const int lead = mirror ? __builtin_ctzll(peers) : 0;
    const uint32_t lc = __shfl(c, lead, 64);
    const uint64_t group = peers & __ballot(mirror && c == lc);  // the lanes of the leader's candidate
    uint64_t base = 0;
    const bool own = mirror && c != lc;
    if (mirror && (own || __lane_id() == (unsigned)lead)) base = atomicAdd(&ctr[c], (Ctr)(own ? 1 : __popcll(group)));
    const uint32_t lo = __shfl((uint32_t)base, lead, 64), hi = __shfl((uint32_t)(base >> 32), lead, 64);
    return own ? base : ((((uint64_t)hi << 32) | lo) + popc_below64(group));
}

// Variants of the walk: the filter; the filter and blocks decided whole
// (span_dense); the predicate for every pair (spanDirect); the first or the
// third by spanDirect (many joins).  Each has kernels of its own: together
// they spill registers.
enum { SPAN_FILTER = 0, SPAN_BLOCKS = 1, SPAN_DIRECT = 2, SPAN_ANY = 3 };
template <int MODE>
__device__ __forceinline__ bool span_direct(const JoinArgs &a) {
    return MODE == SPAN_DIRECT || (MODE == SPAN_ANY && a.spanDirect);
}

// Whether a query (cells pkq, own cell from position cs0) claims candidate c
// (same: in its own cell), z = pk_diff of their cells.
template <int K>
__device__ __forceinline__ bool span_claim(const JoinArgs &a, uint32_t z, uint32_t pkq, uint32_t c, uint32_t cs0,
                                           bool same) {
    if (pk_far(z)) return false;
    if (a.form == SJ_FORM_LID) return c >= cs0;
    if (a.form == SJ_FORM_FULL || same) return true;
    uint32_t cp[K];  // claims reads only the parities
    int o[K];
#pragma unroll
    for (int j = 0; j < K; j++) {
        const uint32_t f = (z >> (4 * j)) & 3u;
        o[j] = f == 3u ? -1 : (int)f;
        cp[j] = (pkq >> (4 * j)) & 3u;
    }
    return claims<K>(a.form, cp, o, 0, 0);
}

// Records the hits of the lanes in okm: candidate c, query q, mirrored hits'
// slots.
__device__ __forceinline__ void span_record(const JoinArgs &a, TileRec &R, SpanRec &rec, uint64_t okm, bool ok,
                                            uint32_t c, uint32_t q, bool mirror, uint64_t slot) {
    const uint32_t n = (uint32_t)__popcll(okm);
    R.want += n;  // also past the end of the space: the whole demand
    if (!rec.on) return;
    uint64_t at, next;
    uint32_t room;
    slot = mirror ? slot : 0ull;
    bool fits = !__ballot(slot > SPAN_SLOT_MAX);
    if (!fits && __lane_id() == 0) atomicAdd(&a.recCtr[REC_BAD], 1ull);
    fits = fits && span_rec_room(a, R, n, rec.n > 0, at, room, next);
    rec.on = fits;
    if (!fits) return;
    if (rec.n == 0) rec.start = at;
    if (rec.n == 0 && at == next) room = n;  // all of them in the new block
    const uint32_t i = popc_below64(okm);
    if (ok)
        a.recMask[i < room ? at + i : next + (i - room)] =
            (uint64_t)c | ((uint64_t)q << 32) | (slot << 38) | (mirror ? 0ull : 1ull << 63);
    rec.n += n;
}

// The plain FP32 decision of a pair: coordinates relative to the tile's first
// point, FMA chain in dimension order.
template <int K>
__device__ __forceinline__ bool span_plain32(const JoinArgs &a, uint32_t ts0, const double (&xq)[K],
                                             const double (&xc)[K]) {
    float s32 = 0.0f;
#pragma unroll
    for (int j = 0; j < K; j++) {
        const double ctr = a.pts[(uint64_t)ts0 * K + j];
        const float f = (float)(xc[j] - ctr) - (float)(xq[j] - ctr);
        s32 = j == 0 ? f * f : fmaf(f, f, s32);
    }
    return s32 <= (float)a.T;
}

// Whether the plain FP32 decision of a pair at d2 can differ from the exact one:
// its sum errs by at most (2.03 K + 8.02) u s (span_band), s = |q|^2 + |c|^2 <=
// 3 |q|^2 + 2 d2, and fl32(T) by u T; 1.1 covers nq, |q|^2 scaled, and the rest.
// Few pairs are that near eps: deciding all of them took 5% of the 6-D count.
template <int K>
__device__ __forceinline__ bool span_plain_unsure(const JoinArgs &a, double d2, float nq) {
    constexpr double u = 1.1 * 0x1p-24;
    return fabs(d2 - a.T) <= u * ((2.03 * K + 8.02) * (3.0 * (double)nq + 2.0 * d2) + a.T);
}

// Decides the nh <= 64 gathered pairs from buffer position head, one per
// lane, and counts and records them, or writes them to their rows.
template <int K, int PASS, bool F32, int MODE>
__device__ __forceinline__ void span_flush(const JoinArgs &a, SpanLds &L, uint32_t ts0, uint32_t head, uint32_t nh,
                                           LaneStats &st, TileRec &R, SpanRec &rec) {
    const unsigned lane = __lane_id();
    const uint32_t h = head + min(lane, nh - 1u);
    const uint32_t c = L.hc[h], q = L.hq[h];
    const uint32_t cs0 = L.cs0[q], cs1 = L.cs1[q], pkA = L.pk[q];
    double xq[K], xc[K];
#pragma unroll
    for (int j = 0; j < K; j++) xc[j] = a.pts[(uint64_t)c * K + j];
#pragma unroll
    for (int j = 0; j < K; j++) xq[j] = a.pts[(uint64_t)(ts0 + q) * K + j];
    const uint32_t z = pk_diff(a.posPk[c], pkA);
    const bool same = c >= cs0 && c < cs1;  // the query's own cell
    bool ok = lane < nh && span_claim<K>(a, z, pkA, c, cs0, same);
    if (span_direct<MODE>(a)) {
        const uint32_t *cc = a.cellCoord + (uint64_t)a.cellOf[c] * K;
        const uint32_t *cq = a.cellCoord + (uint64_t)a.cellOf[ts0 + q] * K;
#pragma unroll
        for (int j = 0; j < K; j++) ok = ok && cc[j] - cq[j] + 1u <= 2u;
    }
    if (ok) {
        const double d2 = d2_fp64<K>(xq, xc, K);
        ok = d2 <= a.T;
        if (F32 && PASS == PASS_COUNT && !span_direct<MODE>(a)) {
            st.band++;
            if (MODE == SPAN_ANY || span_plain_unsure<K>(a, d2, reinterpret_cast<const float *>(L.nq)[q]))
                st.mis += ok != span_plain32<K>(a, ts0, xq, xc) ? 1u : 0u;
        }
    }
    const uint64_t okm = __ballot(ok);
    if (!okm) return;
    // rank of the hit in its query's row
    const uint64_t peers = match6(okm, q);
    const uint32_t rank = L.own[q] + popc_below64(peers);
    wave_lds_sync();
    if (ok && popc_below64(peers) == 0) L.own[q] = rank + (uint32_t)__popcll(peers);
    const bool mirror = ok && a.form != SJ_FORM_FULL && !same && c >= a.wBegin && c < a.wEnd;
    if constexpr (PASS == PASS_COUNT) {
        const uint64_t slot = span_slots(a.mirCnt, mirror, c);
        span_record(a, R, rec, okm, ok, c, q, mirror, slot);
    } else {
        const uint64_t p0 = L.pos[q];
        if (ok && p0 != NO_SLOT) {
            // more hits than the row has room for: count and fill disagree
            if (rank < L.room[q]) a.ids[p0 + rank] = (int32_t)a.origId[c];
            else st.err++;
        }
        const uint64_t p = span_slots(a.mirCur, mirror, c);
        if (mirror) {
            if (p < a.offS[c + 1u] - a.outBase) a.ids[p] = L.id[q];
            else st.err++;
        }
    }
}

__device__ __forceinline__ double readlane_f64(double v, uint32_t l) {
    return __longlong_as_double((long long)readlane_u64((uint64_t)__double_as_longlong(v), (int)l));
}

// Bit i: candidate i of a block (x, as SpanQuery::fetch leaves it) is within eps
// of the lane's query by the predicate.  Called by the whole wave.
template <int K>
__device__ __forceinline__ uint32_t span_near(const JoinArgs &a, const double (&xq)[K], const double (&x)[(K + 3) / 4]) {
    uint32_t near = 0u;
#pragma unroll 4
    for (uint32_t i = 0; i < 16u; i++) {
        double xc[K];
#pragma unroll
        for (int j = 0; j < K; j++) xc[j] = readlane_f64(x[j / 4], i + 16u * (j % 4));
        near |= d2_fp64<K>(xq, xc, K) <= a.T ? 1u << i : 0u;
    }
    return near;
}

// Room for a run of n < 64 record words in one block: what is left of a
// block too short for it is skipped (SPAN_SKIP).  False when the record space
// is exhausted.
__device__ __forceinline__ bool span_rec_run(const JoinArgs &a, TileRec &R, SpanRec &rec, uint32_t n, uint64_t &at) {
    uint64_t next;
    uint32_t room;
    const uint32_t left = R.used < SPAN_LINK ? SPAN_LINK - R.used : 0u;
    if (R.ok && left > 0 && left < n) {
        if (rec.n) {
            if (__lane_id() == 0) a.recMask[R.blk + R.used] = SPAN_SKIP;
            rec.n++;
        }
        R.used = SPAN_LINK;
    }
    rec.on = span_rec_room(a, R, n, rec.n > 0, at, room, next);
    if (!rec.on) return false;
    if (room < n) at = next;
    if (rec.n == 0) rec.start = at;
    rec.n += n;
    return true;
}

// Writes the hits of nc <= 16 candidates to their rows, lane q those of query
// q.  Lane i holds candidate i's values: the queries with hits and with
// mirrored hits, its ID, the row position of its first mirrored hit and its
// row's end.
__device__ __forceinline__ void span_emit(const JoinArgs &a, SpanRows &L, uint32_t nc, uint64_t okl, uint64_t mml,
                                          int32_t idl, uint64_t base, uint64_t lim, LaneStats &st) {
    const unsigned lane = __lane_id();
    const uint64_t p0 = L.pos[lane];
    const uint32_t room = L.room[lane];
    const int32_t idq = L.id[lane];
    uint32_t own = L.own[lane];
#pragma unroll 1
    for (uint32_t i = 0; i < nc; i++) {
        const uint64_t okm = readlane_u64(okl, (int)i), mm = readlane_u64(mml, (int)i);
        const int32_t id = (int32_t)readlane_u32((uint32_t)idl, (int)i);
        if ((okm >> lane) & 1ull) {
            if (p0 != NO_SLOT) {
                // more hits than the row has room for: count and fill disagree
                if (own < room) a.ids[p0 + own] = id;
                else st.err++;
            }
            own++;
        }
        if (mm) {
            const uint64_t p = readlane_u64(base, (int)i) + popc_below64(mm), end = readlane_u64(lim, (int)i);
            if ((mm >> lane) & 1ull) {
                if (p < end) a.ids[p] = idq;
                else st.err++;
            }
        }
    }
    L.own[lane] = own;
}

// The 16 candidates [t0, ..) below t1, many of whose pairs are hits: lane q
// decides all of them for query q, the candidates' coordinates broadcast from
// the lanes that hold them (x, as SpanQuery::fetch leaves them).  One round
// of loads and atomics and one run of record words serve up to 1,024 pairs,
// where span_flush has one per 64.  Returns the hits.
constexpr uint32_t SPAN_DENSE = 256;  // pairs of 1,024: four rounds of span_flush or one of span_dense
template <int K, int PASS, bool F32>
__device__ __forceinline__ uint32_t span_dense(const JoinArgs &a, SpanLds &L, uint32_t ts0, uint32_t m, uint32_t t0,
                                               uint32_t t1, const double (&x)[(K + 3) / 4], LaneStats &st, TileRec &R,
                                               SpanRec &rec) {
    const unsigned lane = __lane_id();
    double xq[K];
#pragma unroll
    for (int j = 0; j < K; j++) xq[j] = a.pts[(uint64_t)(ts0 + min(lane, m - 1u)) * K + j];
    const uint32_t cp = min(t0 + (lane & 15u), t1 - 1u), nc = min(16u, t1 - t0);
    // the candidates that the query claims, and those that get a mirrored hit
    uint32_t may = (1u << nc) - 1u, mirrored = 0u;
    {
        const uint32_t pkq = L.pk[lane], cs0 = L.cs0[lane], cs1 = L.cs1[lane];
        // nothing to find out when the block lies in every query's own cell
        if (__ballot(lane < m && (t0 < cs0 || t0 + nc > cs1))) {
            const uint32_t pkl = a.posPk[cp];
            may = 0u;
#pragma unroll 1
            for (uint32_t i = 0; i < nc; i++) {
                const uint32_t c = t0 + i;
                const bool same = c >= cs0 && c < cs1;
                const bool ok = span_claim<K>(a, pk_diff(readlane_u32(pkl, (int)i), pkq), pkq, c, cs0, same);
                may |= ok ? 1u << i : 0u;
                mirrored |= ok && !same ? 1u << i : 0u;
            }
            if (a.form == SJ_FORM_FULL) mirrored = 0u;
            mirrored &= (uint32_t)range_bits(t0, a.wBegin, a.wEnd);
        }
        may = lane < m ? may : 0u;
    }
    const uint32_t near = span_near<K>(a, xq, x);
    if constexpr (F32 && PASS == PASS_COUNT) {
        uint32_t plain = 0u;
#pragma unroll 1
        for (uint32_t i = 0; i < nc; i++) {
            double xc[K];
#pragma unroll
            for (int j = 0; j < K; j++) xc[j] = readlane_f64(x[j / 4], i + 16u * (j % 4));
            plain |= span_plain32<K>(a, ts0, xq, xc) ? 1u << i : 0u;
        }
        st.band += (uint32_t)__popc(may);
        st.mis += (uint32_t)__popc((near ^ plain) & may);
    }
    const uint32_t hit = near & may, mir = hit & mirrored;
    uint32_t total = 0;
    uint64_t okl = 0, mml = 0;  // lane i: the queries with a (mirrored) hit on candidate t0 + i
    for (uint32_t i = 0; i < nc; i++) {
        const uint64_t okm = __ballot((hit >> i) & 1u), mm = __ballot((mir >> i) & 1u);
        okl = lane == i ? okm : okl;
        mml = lane == i ? mm : mml;
        total += (uint32_t)__popcll(okm);
    }
    // a slot per mirrored hit
    uint64_t base = 0;
    const uint32_t cnt = (uint32_t)__popcll(mml);
    if (cnt) {
        if constexpr (PASS == PASS_COUNT) base = atomicAdd(&a.mirCnt[cp], cnt);
        else base = atomicAdd(&a.mirCur[cp], (unsigned long long)cnt);
    }
    if constexpr (PASS == PASS_COUNT) {
        L.own[lane] += (uint32_t)__popc(hit);
        R.want += 1u + 3u * nc;
        uint64_t at;
        if (rec.on && span_rec_run(a, R, rec, 1u + 3u * nc, at)) {
            if (lane == 0) a.recMask[at] = SPAN_BLOCK | ((uint64_t)nc << 32) | t0;
            if (lane < nc) {
                uint64_t *e = a.recMask + at + 1u + 3u * lane;
                e[0] = okl;
                e[1] = mml;
                e[2] = base;
            }
        }
    } else {
        const bool inW = lane < nc && cp >= a.wBegin && cp < a.wEnd;
        span_emit(a, L, nc, okl, mml, (int32_t)a.origId[cp], base, inW ? a.offS[cp + 1u] - a.outBase : 0ull, st);
    }
    wave_lds_sync();
    return total;
}

// The tile's queries into LDS (lane q holds query q).
template <int PASS>
__device__ __forceinline__ bool span_queries(const JoinArgs &a, SpanRows &L, uint32_t ts0, uint32_t ts1) {
    const unsigned lane = __lane_id();
    const uint32_t s = min(ts0 + lane, ts1 - 1u);
    const bool ownW = ts0 + lane < ts1 && s >= a.wBegin && s < a.wEnd;
    L.own[lane] = 0u;
    if (PASS == PASS_FILL) {
        L.pos[lane] = ownW ? a.offS[s] - a.outBase : NO_SLOT;
        L.room[lane] = ownW ? a.ownCnt[s] : 0u;
        L.id[lane] = (int32_t)a.origId[s];
    }
    return ownW;
}

// One tile of the span walk.
template <int K, int PASS, bool F32, int MODE>
__device__ __forceinline__ void process_span(const JoinArgs &a, uint32_t tile, SpanLds &L, LaneStats &st,
                                             TileRec &R) {
    const unsigned lane = __lane_id();
    const uint32_t ts0 = uniform_u32(a.tileStart[tile]), ts1 = uniform_u32(a.tileStart[tile + 1]);
    if (ts0 >= ts1) return;
    const uint32_t m = ts1 - ts0;  // queries
    const uint32_t s = min(ts0 + lane, ts1 - 1u);
    const uint32_t cellA = a.cellOf[s];
    L.cs0[lane] = a.cellStart[cellA];
    L.cs1[lane] = a.cellStart[cellA + 1];
    L.pk[lane] = a.posPk[s];
    const bool ownW = span_queries<PASS>(a, L, ts0, ts1);
    const bool anyOwnW = __ballot(ownW) != 0ull;
    const int g = a.spanG;
    // the group's coordinates and the tile's span are wave-uniform
    const uint32_t cellF = uniform_u32(a.cellOf[ts0]), cellL = uniform_u32(a.cellOf[ts1 - 1u]);
    uint32_t cF[K];
#pragma unroll
    for (int j = 0; j < K; j++) cF[j] = uniform_u32(a.cellCoord[(uint64_t)cellF * K + j]);
    const uint64_t linF = uniform_u64(a.cellLinear[cellF]), linL = uniform_u64(a.cellLinear[cellL]);
    const TileSpan sp = tile_span<K>(a, g, cF, linF, linL);
    const uint32_t startF = uniform_u32(a.cellStart[cellF]);
    SpanQuery<K, F32> Q;
    const bool direct = span_direct<MODE>(a);
    if (!direct) Q.load(a, L, ts0, ts1);
    SpanRec rec;
    rec.on = PASS == PASS_COUNT && a.recCtr != nullptr;

    uint32_t nh = 0;  // gathered pairs
    auto gather = [&](bool pass, uint32_t q, uint32_t c) __attribute__((always_inline)) {
        const uint64_t b = __builtin_amdgcn_ballot_w64(pass);
        if (!b) return;
        if (pass) {
            const uint32_t at = nh + popc_below64(b);
            L.hc[at] = c;
            L.hq[at] = (uint8_t)q;
        }
        nh += (uint32_t)__popcll(b);
    };
    // decide 64 at a time until fewer than 64 are left (all: none), which
    // move to the front
    auto drain = [&](bool all) __attribute__((always_inline)) {
        wave_lds_sync();
        uint32_t head = 0;
        while (nh - head >= 64u || (all && nh > head)) {
            const uint32_t n = min(nh - head, 64u);
            span_flush<K, PASS, F32, MODE>(a, L, ts0, head, n, st, R, rec);
            head += n;
        }
        nh -= head;
        if (nh) {
            const uint32_t h = head + min(lane, nh - 1u);
            const uint32_t c = L.hc[h];
            const uint8_t q = L.hq[h];
            wave_lds_sync();
            if (lane < nh) {
                L.hc[lane] = c;
                L.hq[lane] = q;
            }
        }
        wave_lds_sync();
    };
    using T = typename SpanMma<F32>::T;
    const T scale = (T)a.spanScale, T1 = (T)a.spanT1;
    bool rich = false;  // the last block was dense

    int ng = 1;
#pragma unroll
    for (int j = 0; j < K; j++)
        if (j >= g) ng *= 3;
    for (int b0 = 0; b0 < ng; b0 += 64) {
        // neighbour groups 64 at a time: lane l looks up group b0 + l
        const int my = b0 + (int)lane;
        int od[K];
        int64_t dl;
        const bool inb = span_group<K>(a, g, cF, my, od, dl) && my < ng;
        uint32_t r0 = 0u, r1 = 0u;
        if (inb) {
            // LID claims no group of smaller linear IDs and, in its own
            // group, nothing before its first cell; Unicomp claims a whole
            // group by the parity of its highest differing dim
            bool may = true;
            if (a.form == SJ_FORM_LID) may = dl >= 0;
            else if (a.form == SJ_FORM_UNICOMP && dl != 0) may = claims<K>(a.form, cF, od, 0, 0);
            if (may) {
                r0 = pos_lb(a, (uint64_t)((int64_t)sp.lo + dl));
                r1 = pos_lb(a, (uint64_t)((int64_t)sp.hi + dl));
                if (a.form == SJ_FORM_LID && dl == 0) r0 = max(r0, startF);
            }
        }
        uint64_t am = __ballot(r1 > r0);
        while (am) {
            const int bl = __builtin_ctzll(am);
            am &= am - 1ull;
            const uint32_t u0 = readlane_u32(r0, bl), u1 = readlane_u32(r1, bl);
            // nothing of this range lands in the rows written
            if (PASS == PASS_FILL && !anyOwnW && (u1 <= a.wBegin || u0 >= a.wEnd)) continue;
            if (PASS == PASS_COUNT && lane < m) st.cand += u1 - u0;
            if (MODE == SPAN_ANY && direct) {
                // every pair goes on to the predicate
                for (uint32_t t0 = u0; t0 < u1; t0++) {
                    gather(lane < m, lane, t0);
                    if (nh >= 64u) drain(false);
                }
                continue;
            }
            if (MODE == SPAN_DIRECT) {
                // every pair goes to the predicate, those within eps on to
                // the claims.  One candidate and 64 queries at a time through
                // the gathered pairs, 20,000 points in 4-D took 0.97 ms a join
                // instead of 0.31 ms.
                double xq[K], x[Q.H];
#pragma unroll
                for (int j = 0; j < K; j++) xq[j] = a.pts[(uint64_t)s * K + j];
#pragma unroll 1
                for (uint32_t t0 = u0; t0 < u1; t0 += 16u) {
                    Q.fetch(a, min(t0 + (lane & 15u), u1 - 1u), x);
                    // by all lanes: they hold the candidates
                    uint32_t near = span_near<K>(a, xq, x);
                    near &= lane < m ? (1u << min(16u, u1 - t0)) - 1u : 0u;
#pragma unroll 1
                    for (uint32_t i = 0; i < 16u; i++) gather((near >> i) & 1u, lane, t0 + i);
                    if (nh >= 64u) drain(false);
                }
                continue;
            }
            double x[Q.H], nx[Q.H];
            Q.fetch(a, min(u0 + (lane & 15u), u1 - 1u), x);
#pragma unroll 1
            for (uint32_t t0 = u0; t0 < u1; t0 += 16u) {
                // the next candidates' coordinates are on their way meanwhile
                Q.fetch(a, min(t0 + 16u + (lane & 15u), u1 - 1u), nx);
                bool dense = MODE == SPAN_BLOCKS && rich;
                if (!dense) {
                    const uint32_t before = nh;
                    Q.filter(t0, u1, x, scale, T1, gather);
                    if (MODE == SPAN_BLOCKS && nh - before >= SPAN_DENSE) {
                        // decided whole, after the pairs gathered before
                        nh = before;
                        dense = true;
                    }
                    if (dense ? nh > 0u : nh >= 64u) drain(dense);
                }
                if constexpr (MODE == SPAN_BLOCKS) {
                    if (dense)
                        rich = span_dense<K, PASS, F32>(a, L, ts0, m, t0, u1, x, st, R, rec) >= SPAN_DENSE;
                }
#pragma unroll
                for (int h = 0; h < Q.H; h++) x[h] = nx[h];
            }
        }
    }
    if (nh) drain(true);
    if (PASS == PASS_COUNT) {
        wave_lds_sync();
        if (ownW) a.ownCnt[s] = L.own[lane];
        if (rec.on && lane == 0) {
            a.recN[tile] = rec.n;
            a.recStart[tile] = rec.start;
        }
    } else {
        wave_lds_sync();
        if (ownW && L.own[lane] != L.room[lane]) st.err++;
    }
    wave_lds_sync();
}

// The same tile from the count pass's record, up to 64 * REPLAY_U words at a
// time: the loads that depend on them are all in flight together, as are the
// next words.  64 words at a time waited for two loads each: 2M points in
// 4-D with 48 neighbours 832 -> 657 us, 20,000 with 1,000 670 -> 473 us.
constexpr int REPLAY_U = 4;
__device__ __forceinline__ void replay_span(const JoinArgs &a, uint32_t tile, SpanRows &L, LaneStats &st) {
    const unsigned lane = __lane_id();
    const uint32_t ts0 = uniform_u32(a.tileStart[tile]), ts1 = uniform_u32(a.tileStart[tile + 1]);
    if (ts0 >= ts1) return;
    const bool ownW = span_queries<PASS_FILL>(a, L, ts0, ts1);
    uint32_t left = uniform_u32(a.recN[tile]);
    uint64_t at = uniform_u64(a.recStart[tile]);
    // the words from `at` on, within the tile's and the record block's
    uint64_t next[REPLAY_U];
    uint32_t nNext;
    auto load = [&]() __attribute__((always_inline)) {
        nNext = min(min(left, 64u * REPLAY_U), SPAN_LINK - (uint32_t)(at % REC_BLK));
#pragma unroll
        for (int u = 0; u < REPLAY_U; u++)
            next[u] = lane + 64u * u < nNext ? a.recMask[at + lane + 64u * u] : 0ull;
    };
    if (left) load();
    wave_lds_sync();
    while (left) {
        uint64_t w[REPLAY_U];
#pragma unroll
        for (int u = 0; u < REPLAY_U; u++) w[u] = next[u];
        uint32_t n = nNext;
        // up to the first word that is not a hit
        uint64_t special = 0;
#pragma unroll
        for (int u = REPLAY_U - 1; u >= 0; u--) {
            const uint64_t b = __ballot((w[u] >> 61) > 4ull);
            if (b) {
                n = 64u * u + (uint32_t)__builtin_ctzll(b);
                special = readlane_u64(w[u], __builtin_ctzll(b));
            }
        }
        const bool block = special >= SPAN_BLOCK;
        const uint32_t nc = block ? (uint32_t)(special >> 32) & 31u : 0u;
        left -= n;
        at += n;
        // a block's words: lane i those of its candidate i
        uint64_t okl = 0, mml = 0, base = 0, end = 0;
        int32_t idl = 0;
        if (lane < nc) {
            const uint32_t c = (uint32_t)special + lane;
            const uint64_t *e = a.recMask + at + 1u + 3u * lane;
            okl = e[0];
            idl = (int32_t)a.origId[c];
            if (c >= a.wBegin && c < a.wEnd) {
                mml = e[1];
                base = a.offS[c] - a.outBase + a.ownCnt[c] + e[2];
                end = a.offS[c + 1u] - a.outBase;
            }
        }
        if (block) {
            left -= 1u + 3u * nc;
            at += 1u + 3u * nc;
        } else if (special) {
            left--;
            at = at / REC_BLK * REC_BLK + SPAN_LINK;
        }
        if (left) {
            if (at % REC_BLK == SPAN_LINK) at = uniform_u64(a.recMask[at]);
            load();
        }
        int32_t id[REPLAY_U];
        uint64_t p[REPLAY_U], lim[REPLAY_U];
        bool mirror[REPLAY_U];
#pragma unroll
        for (int u = 0; u < REPLAY_U; u++) {
            const bool live = lane + 64u * u < n;
            const uint32_t c = (uint32_t)w[u];
            id[u] = live ? (int32_t)a.origId[c] : 0;
            mirror[u] = live && !(w[u] >> 63) && c >= a.wBegin && c < a.wEnd;
            p[u] = lim[u] = 0;
            if (mirror[u]) {
                p[u] = a.offS[c] - a.outBase + a.ownCnt[c] + (w[u] >> 38);
                lim[u] = a.offS[c + 1u] - a.outBase;
            }
        }
#pragma unroll
        for (int u = 0; u < REPLAY_U; u++) {
            if (64u * u >= n) break;
            const bool live = lane + 64u * u < n;
            const uint32_t q = (uint32_t)(w[u] >> 32) & 63u;
            const uint64_t peers = match6(__ballot(live), q);
            const uint32_t rank = L.own[q] + popc_below64(peers);
            wave_lds_sync();
            if (live && popc_below64(peers) == 0) L.own[q] = rank + (uint32_t)__popcll(peers);
            const uint64_t p0 = L.pos[q];
            if (live && p0 != NO_SLOT) {
                if (rank < L.room[q]) a.ids[p0 + rank] = id[u];
                else st.err++;
            }
            if (mirror[u]) {
                if (p[u] < lim[u]) a.ids[p[u]] = L.id[q];
                else st.err++;
            }
            wave_lds_sync();
        }
        if (nc) {
            span_emit(a, L, nc, okl, mml, idl, base, end, st);
            wave_lds_sync();
        }
    }
    if (ownW && L.own[lane] != L.room[lane]) st.err++;
    wave_lds_sync();
}

// The same for many joins, whose record has no blocks: 64 words at a time.
__device__ __forceinline__ void replay_span_many(const JoinArgs &a, uint32_t tile, SpanRows &L, LaneStats &st) {
    const unsigned lane = __lane_id();
    const uint32_t ts0 = uniform_u32(a.tileStart[tile]), ts1 = uniform_u32(a.tileStart[tile + 1]);
    if (ts0 >= ts1) return;
    const bool ownW = span_queries<PASS_FILL>(a, L, ts0, ts1);
    uint32_t left = uniform_u32(a.recN[tile]);
    uint64_t at = uniform_u64(a.recStart[tile]);
    wave_lds_sync();
    while (left) {
        const uint32_t used = (uint32_t)(at % REC_BLK);
        const uint32_t n = min(min(left, 64u), SPAN_LINK - used);
        const bool live = lane < n;
        const uint64_t w = live ? a.recMask[at + lane] : 0ull;
        left -= n;
        at += n;
        if (left && at % REC_BLK == SPAN_LINK) at = uniform_u64(a.recMask[at]);
        const uint32_t c = (uint32_t)w, q = (uint32_t)(w >> 32) & 63u;
        const uint64_t peers = match6(__ballot(live), q);
        const uint32_t rank = L.own[q] + popc_below64(peers);
        wave_lds_sync();
        if (live && popc_below64(peers) == 0) L.own[q] = rank + (uint32_t)__popcll(peers);
        const uint64_t p0 = L.pos[q];
        if (live && p0 != NO_SLOT) {
            if (rank < a.ownCnt[ts0 + q]) a.ids[p0 + rank] = (int32_t)a.origId[c];
            else st.err++;
        }
        if (live && !(w >> 63) && c >= a.wBegin && c < a.wEnd) {
            const uint64_t p = a.offS[c] - a.outBase + a.ownCnt[c] + (w >> 38);
            if (p < a.offS[c + 1u] - a.outBase) a.ids[p] = L.id[q];
            else st.err++;
        }
        wave_lds_sync();
    }
    if (ownW && L.own[lane] != a.ownCnt[ts0 + lane]) st.err++;
    wave_lds_sync();
}

}  // namespace sj
