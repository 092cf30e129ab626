// Device-wide radix sort, scan and stream compaction for gfx950 (wave64),
// written for this library: the VENOM row sort (reordering.py:219, Python's
// stable `sorted` over per-row keys), the packer's (row, column) and
// (block, row) orders and the proposer's adjacency builds.
//
// Radix sort: LSD over the key's sorted bits (KeyBits: one or two ranges of the
// 64, so that the unused bits between a key's fields cost no pass), digits of at
// most 8 bits, one pass per digit.  A tile is 4,096 keys, 256 per wave of a
// 1,024-thread workgroup.  Every pass ranks a tile's keys the same way: a wave
// takes its keys 64 at a time; the lanes holding one digit find each other
// with a ballot per digit bit, the lowest of them adds the group's size to the
// wave's running count of the digit (LDS), so a key's rank is its wave's count
// so far plus the lanes below it in the group.  Waves' counts are then prefixed in
// wave order, the tile's keys placed in LDS in digit order, and written out with
// consecutive lanes on consecutive output positions.  A pass is bound by this
// chain, not by its bytes, so a tile has 16 waves of 4 rounds (4 waves of 16:
// 12.5 us a pass at 16,384 keys).
//   up to 4,096 keys  all passes in one launch of one workgroup, the keys in
//                     registers and LDS (k_sort_one)
//   up to 65,536      one launch per pass: each tile derives its offsets from
//                     the pass's count table and counts the next pass's digits
//                     for its destination tiles (k_radix_fused); up to 16,384
//                     keys in tiles of 1,024, which spread the ranking's vector
//                     work over 16 CUs (16,384 keys of 33 bits: 65 us on one CU
//                     in one launch, 85 in 6 launches of 4-wave tiles of 4,096)
//   more              three: digit counts per tile (k_radix_hist, digit-major),
//                     a workgroup per digit scanning its tiles' counts
//                     (k_digit_scan), k_radix_scatter (1 M pairs: 39 us a pass
//                     with 4-wave tiles and a three-launch scan, 21 now)
// Every step keeps input order among equal digits, so each pass -- and the
// sort -- is stable.  Passes ping-pong between the output and a scratch
// buffer so the last one lands in the output; the input is never written.
//
// Scan: tiles of 4,096 elements; per-tile totals (k_scan_reduce), then each
// tile scanned in LDS from the sum of the totals before it (k_scan_tile; over
// SCAN_DIRECT tiles one workgroup scans the totals first, k_scan_totals).  Sum and
// max, int32 or uint8 input; at most one tile in one launch (k_scan_small).
// Compaction: exclusive sum of the flags, then a scatter of flagged items.
#include "graph.h"
#include "sortlib.h"

#include <algorithm>

namespace vnm {

namespace {

constexpr int WG = 256;                 // threads per workgroup of the scans
constexpr int NWAVE = WG / 64;
constexpr int ROUNDS = 16;              // elements per thread of a scan tile
constexpr int TILE = WG * ROUNDS;       // 4,096 elements per tile
constexpr int RADIX = 256;
constexpr int SWG = 1024;               // threads per workgroup of the sort
constexpr int SWAVE = SWG / 64;
constexpr int SROUNDS = TILE / SWG;     // 64-key rounds per wave and tile
constexpr int FWG = 256;                // ... of the fused sort's small tiles
constexpr int SCAN_DIRECT = 2048;       // scan tiles whose totals each tile sums itself

// Scratch of the calling host thread, grown on demand (one per thread, so
// concurrent contexts on worker threads do not share it).
struct TempBuf {
    void *p = nullptr;
    size_t bytes = 0;
    int ensure(size_t need) {
        if (need <= bytes && p) return VNM_OK;
        if (p) (void)hipFree(p);  // waits for the device, so no kernel still reads it
        p = nullptr;
        bytes = 0;
        if (device_alloc(&p, need ? need : 1) != hipSuccess) {
            p = nullptr;
            return set_error(VNM_E_OOM, "scratch allocation of %zu bytes failed", need);
        }
        bytes = need;
        return VNM_OK;
    }
    ~TempBuf() {
        if (p) (void)hipFree(p);
    }
};
// Scratch slots per host thread; the current one serves every sort and scan
// (separate slots let launch chains that may run concurrently, such as the
// branches of one captured graph, sort at the same time).
constexpr int SCRATCH_SLOTS = 16;
thread_local TempBuf g_slots[SCRATCH_SLOTS];
thread_local int g_slot = 0;
#define g_tmp (g_slots[g_slot])

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

__device__ __forceinline__ uint64_t lanemask_lt() {
    const int lane = threadIdx.x & 63;
    return lane ? (~0ull >> (64 - lane)) : 0ull;
}

// Inclusive sum over the 64 lanes of a wave.
template <typename T, typename Op>
__device__ __forceinline__ T wave_scan_incl(T v, Op op) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const T o = __shfl_up(v, d, 64);
        if (lane >= d) v = op(v, o);
    }
    return v;
}

// Exclusive scan of one value per thread over the workgroup (wave order),
// identity `id`; *total = the workgroup's reduction.  Uses `sh` (NWAVE Ts).
template <typename T, typename Op>
__device__ __forceinline__ T wg_scan_excl(T v, Op op, T id, T *sh, T *total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const T inc = wave_scan_incl(v, op);
    if (lane == 63) sh[w] = inc;
    __syncthreads();
    T base = id, all = id;
#pragma unroll
    for (int i = 0; i < NWAVE; ++i) {
        if (i < w) base = op(base, sh[i]);
        all = op(all, sh[i]);
    }
    __syncthreads();
    *total = all;
    T ex = __shfl_up(inc, 1, 64);
    if (lane == 0) ex = id;
    return op(base, ex);
}

struct OpSum {
    __device__ __forceinline__ int32_t operator()(int32_t a, int32_t b) const { return a + b; }
    static constexpr int32_t id = 0;
};
struct OpMax {
    __device__ __forceinline__ int32_t operator()(int32_t a, int32_t b) const { return a > b ? a : b; }
    static constexpr int32_t id = INT32_MIN;
};

// ------------------------------------------------------------ radix sort

// LDS of a tile's ranking.
template <int T>
struct RankShared {
    int32_t run[T / 64][RADIX];  // per wave: keys of each digit so far, then in the waves before
    int32_t start[RADIX];       // tile position of each digit's first key
    int32_t sh[RADIX / 64];
};

// Exclusive prefix of one value per thread over threads 0 .. RADIX - 1; every
// thread of the workgroup calls it (the others get nothing of use).
__device__ __forceinline__ int32_t prefix256(int32_t v, int32_t *sh) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int32_t inc = wave_scan_incl(v, [](int32_t a, int32_t b) { return a + b; });
    if (w < RADIX / 64 && lane == 63) sh[w] = inc;
    __syncthreads();
    int32_t base = 0;
#pragma unroll
    for (int i = 0; i < RADIX / 64; ++i) base += i < w ? sh[i] : 0;
    return base + inc - v;
}

// Tile positions of the R * 64 keys a wave holds (key r of lane l is the wave's
// key r * 64 + l; those with !ok(r) take none) in digit order, and the digits.
// Every thread calls it; positions are valid, and S may be read, after it.
template <int T, int R, typename Ok>
__device__ __forceinline__ void rank_tile(RankShared<T> &S, const uint64_t (&key)[R], Ok ok, const Digit &dg,
                                          int (&pos)[R], int (&dig)[R]) {
    constexpr int NW = T / 64;
    const int w = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < NW * RADIX; i += T) (&S.run[0][0])[i] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool in = ok(r);
        const int d = in ? dg.of(key[r]) : 0;
        uint64_t peers = __ballot(in);
        for (int b = 0; b < dg.bits; ++b) {
            const uint64_t bal = __ballot((d >> b) & 1);
            peers &= ((d >> b) & 1) ? bal : ~bal;
        }
        const int below = __popcll(peers & lanemask_lt());
        int r0 = 0;
        if (in) r0 = S.run[w][d];
        // the group's lowest lane advances the digit's count after every
        // lane of the group has read it (same wave: LDS order is program order)
        if (in && below == 0) S.run[w][d] = r0 + __popcll(peers);
        dig[r] = in ? d : -1;
        pos[r] = r0 + below;
    }
    __syncthreads();
    // per digit (thread d): prefix over waves in wave order, tile count
    int32_t c = 0;
    if (threadIdx.x < RADIX) {
        const int d = threadIdx.x;
        int32_t x[NW];
#pragma unroll
        for (int i = 0; i < NW; ++i) x[i] = S.run[i][d];
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            S.run[i][d] = c;
            c += x[i];
        }
    }
    const int32_t st = prefix256(c, S.sh);
    if (threadIdx.x < RADIX) S.start[threadIdx.x] = st;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (dig[r] >= 0) pos[r] += S.start[dig[r]] + S.run[w][dig[r]];
}

// Digit counts of every tile, digit-major; `zero` (nz ints) is cleared for the
// fused passes' tables.
template <int T>
__global__ __launch_bounds__(T) void k_radix_hist(const uint64_t *__restrict__ keys, int64_t n, Digit dg, int tiles,
                                                    int32_t *__restrict__ hist, int32_t *__restrict__ zero, int nz,
                                                    const int *__restrict__ skip) {
    if (skip && *skip) return;  // the caller's flag: this sort is not wanted
    __shared__ int32_t cnt[RADIX];
    if (threadIdx.x < RADIX) cnt[threadIdx.x] = 0;
    for (int i = blockIdx.x * T + threadIdx.x; i < nz; i += gridDim.x * T) zero[i] = 0;
    __syncthreads();
    const int64_t t0 = (int64_t)blockIdx.x * (T * SROUNDS);
#pragma unroll
    for (int j = 0; j < SROUNDS; ++j) {
        const int64_t i = t0 + j * T + threadIdx.x;
        if (i < n) atomicAdd(&cnt[dg.of(keys[i])], 1);
    }
    __syncthreads();
    if (threadIdx.x < RADIX) hist[(int64_t)threadIdx.x * tiles + blockIdx.x] = cnt[threadIdx.x];
}

// Digit blockIdx.x's counts become the keys of that digit in the tiles before;
// its total goes to total[digit].
__global__ __launch_bounds__(SWG) void k_digit_scan(int32_t *__restrict__ hist, int tiles, int32_t *__restrict__ total,
                                                    const int *__restrict__ skip) {
    if (skip && *skip) return;  // the caller's flag: this sort is not wanted
    __shared__ int32_t sh[SWAVE];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int32_t *h = hist + (int64_t)blockIdx.x * tiles;
    int32_t carry = 0;
    for (int b = 0; b < tiles; b += SWG) {
        const int i = b + threadIdx.x;
        const int32_t v = i < tiles ? h[i] : 0;
        const int32_t inc = wave_scan_incl(v, [](int32_t x, int32_t y) { return x + y; });
        if (lane == 63) sh[w] = inc;
        __syncthreads();
        int32_t base = carry, all = 0;
#pragma unroll
        for (int q = 0; q < SWAVE; ++q) {
            base += q < w ? sh[q] : 0;
            all += sh[q];
        }
        if (i < tiles) h[i] = base + inc - v;
        carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

template <bool VALS>
__global__ __launch_bounds__(SWG) void k_radix_scatter(const uint64_t *__restrict__ kin,
                                                       const int32_t *__restrict__ vin,
                                                       uint64_t *__restrict__ kout, int32_t *__restrict__ vout,
                                                       int64_t n, Digit dg, int tiles,
                                                       const int32_t *__restrict__ before,
                                                       const int32_t *__restrict__ total,
                                                       const int *__restrict__ skip) {
    if (skip && *skip) return;  // the caller's flag: this sort is not wanted
    __shared__ RankShared<SWG> S;
    __shared__ int32_t offs[RADIX], psh[RADIX / 64];
    __shared__ uint64_t sk[TILE];
    __shared__ int32_t sv[VALS ? TILE : 1];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t t0 = (int64_t)blockIdx.x * TILE;
    const int64_t base = t0 + w * (64 * SROUNDS) + lane;
    uint64_t key[SROUNDS];
    int32_t val[SROUNDS];
#pragma unroll
    for (int r = 0; r < SROUNDS; ++r) {
        const int64_t i = base + r * 64;
        key[r] = i < n ? kin[i] : 0ull;
        if constexpr (VALS) val[r] = i < n ? vin[i] : 0;
    }
    int32_t tot = 0, bef = 0;
    if (threadIdx.x < RADIX) {
        tot = total[threadIdx.x];
        bef = before[(int64_t)threadIdx.x * tiles + blockIdx.x];
    }
    const int32_t off = prefix256(tot, psh) + bef;
    if (threadIdx.x < RADIX) offs[threadIdx.x] = off;
    int pos[SROUNDS], dig[SROUNDS];
    rank_tile(S, key, [&](int r) { return base + r * 64 < n; }, dg, pos, dig);
#pragma unroll
    for (int r = 0; r < SROUNDS; ++r) {
        if (dig[r] >= 0) {
            sk[pos[r]] = key[r];
            if constexpr (VALS) sv[pos[r]] = val[r];
        }
    }
    __syncthreads();
    // write out: tile position p holds the key of digit dd at offset
    // p - start[dd] of that digit's run
    const int cnt = (int)std::min<int64_t>(TILE, n - t0);
#pragma unroll
    for (int r = 0; r < SROUNDS; ++r) {
        const int p = r * SWG + threadIdx.x;
        if (p >= cnt) break;
        const uint64_t k = sk[p];
        const int dd = dg.of(k);
        const int64_t o = (int64_t)offs[dd] + (p - S.start[dd]);
        kout[o] = k;
        if constexpr (VALS) vout[o] = sv[p];
    }
}

// A whole sort of at most one tile in one workgroup: every pass ranks the
// keys as k_radix_scatter does, places them in LDS in
// digit order and reads them back in the rank layout for the next pass.
template <bool VALS>
__global__ __launch_bounds__(SWG) void k_sort_one(const uint64_t *__restrict__ kin, const int32_t *__restrict__ vin,
                                                  uint64_t *__restrict__ kout, int32_t *__restrict__ vout, int n,
                                                  KeyBits b, const int *__restrict__ skip) {
    if (skip && *skip) return;  // the caller's flag: this sort is not wanted
    __shared__ RankShared<SWG> S;
    constexpr int R = SROUNDS;
    __shared__ uint64_t sk[TILE];  // a pass's keys, then its values
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int base = w * (64 * R) + lane;
    uint64_t key[R];
    int32_t val[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = base + r * 64;
        key[r] = i < n ? kin[i] : 0ull;
        if constexpr (VALS) val[r] = i < n ? vin[i] : 0;
    }
    const int total = b.w0 + b.w1;
    for (int shift = 0; shift < total;) {
        const int bits = digit_bits(total, shift);
        int pos[R], dig[R];
        rank_tile(S, key, [&](int r) { return base + r * 64 < n; }, Digit{b, shift, bits}, pos, dig);
        shift += bits;
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (dig[r] >= 0) sk[pos[r]] = key[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (base + r * 64 < n) key[r] = sk[base + r * 64];
        __syncthreads();
        if constexpr (VALS) {
            int32_t *sv = (int32_t *)sk;
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (dig[r] >= 0) sv[pos[r]] = val[r];
            __syncthreads();
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (base + r * 64 < n) val[r] = sv[base + r * 64];
            __syncthreads();
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = base + r * 64;
        if (i < n) {
            kout[i] = key[r];
            if constexpr (VALS) vout[i] = val[r];
        }
    }
}

// Sorts of up to FUSED_TILES tiles: one launch per pass.  Each workgroup
// derives its tile's offsets itself from the pass's (digit, tile) count
// table, ranks and scatters its tile as k_radix_scatter does, and counts
// the next pass's digits of the keys it writes by destination tile (an LDS
// table, then one atomic add per nonzero count), so no separate histogram
// or scan launch is needed between passes.
constexpr int FUSED_TILES = 16;

template <bool VALS, int T>
__global__ __launch_bounds__(T) void k_radix_fused(const uint64_t *__restrict__ kin, const int32_t *__restrict__ vin,
                                                     uint64_t *__restrict__ kout, int32_t *__restrict__ vout,
                                                     int n, Digit dg, int tiles, const int32_t *__restrict__ hist,
                                                     Digit ndg, int32_t *__restrict__ next_hist,
                                                     const int *__restrict__ skip) {
    if (skip && *skip) return;  // the caller's flag: this sort is not wanted
    constexpr int TL = T * SROUNDS;  // keys of a tile
    __shared__ RankShared<T> S;
    __shared__ int32_t offs[RADIX], psh[RADIX / 64];
    __shared__ uint64_t sk[TL];
    __shared__ int32_t sv[VALS ? TL : 1];
    __shared__ int32_t nh[FUSED_TILES * RADIX];  // next pass: counts per (destination tile, digit)
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int tile = blockIdx.x;
    const int base = tile * TL + w * (64 * SROUNDS) + lane;
    uint64_t key[SROUNDS];
    int32_t val[SROUNDS];
#pragma unroll
    for (int r = 0; r < SROUNDS; ++r) {
        const int i = base + r * 64;
        key[r] = i < n ? kin[i] : 0ull;
        if constexpr (VALS) val[r] = i < n ? vin[i] : 0;
    }
    if (next_hist)
        for (int i = threadIdx.x; i < tiles * RADIX; i += T) nh[i] = 0;
    // this tile's offsets: digits before d over all tiles, then digit d in
    // the tiles before this one (hist is digit-major: hist[d * tiles + t])
    int32_t row = 0, before = 0;
    if (threadIdx.x < RADIX) {
        int32_t x[FUSED_TILES];
#pragma unroll
        for (int t = 0; t < FUSED_TILES; ++t) x[t] = t < tiles ? hist[threadIdx.x * tiles + t] : 0;
#pragma unroll
        for (int t = 0; t < FUSED_TILES; ++t) {
            before += t < tile ? x[t] : 0;
            row += x[t];
        }
    }
    const int32_t off = prefix256(row, psh) + before;
    if (threadIdx.x < RADIX) offs[threadIdx.x] = off;
    int pos[SROUNDS], dig[SROUNDS];
    rank_tile(S, key, [&](int r) { return base + r * 64 < n; }, dg, pos, dig);
#pragma unroll
    for (int r = 0; r < SROUNDS; ++r) {
        if (dig[r] >= 0) {
            sk[pos[r]] = key[r];
            if constexpr (VALS) sv[pos[r]] = val[r];
        }
    }
    __syncthreads();
    const int cnt = min(TL, n - tile * TL);
#pragma unroll
    for (int r = 0; r < SROUNDS; ++r) {
        const int p = r * T + threadIdx.x;
        if (p >= cnt) break;
        const uint64_t k = sk[p];
        const int dd = dg.of(k);
        const int o = offs[dd] + (p - S.start[dd]);
        kout[o] = k;
        if constexpr (VALS) vout[o] = sv[p];
        if (next_hist) atomicAdd(&nh[(o / TL) * RADIX + ndg.of(k)], 1);
    }
    if (next_hist) {
        __syncthreads();
        for (int i = threadIdx.x; i < tiles * RADIX; i += T) {
            const int32_t c = nh[i];
            if (c) atomicAdd(&next_hist[(i % RADIX) * tiles + i / RADIX], c);
        }
    }
}

// ------------------------------------------------------------ scan

// Scan input as int32: flags count as 0 or 1.
__device__ __forceinline__ int32_t load_as(const int32_t *p, int64_t i) { return p[i]; }
__device__ __forceinline__ int32_t load_as(const uint8_t *p, int64_t i) { return p[i] != 0; }

template <typename In, typename Op>
__global__ __launch_bounds__(WG) void k_scan_reduce(const In *__restrict__ in, int64_t n,
                                                    int32_t *__restrict__ totals, const int *__restrict__ skip) {
    if (skip && *skip) return;  // the caller's flag: this sort is not wanted
    __shared__ int32_t sh[NWAVE];
    const Op op;
    const int64_t t0 = (int64_t)blockIdx.x * TILE;
    int32_t acc = Op::id;
    for (int j = 0; j < ROUNDS; ++j) {
        const int64_t i = t0 + j * WG + threadIdx.x;
        if (i < n) acc = op(acc, load_as(in, i));
    }
    int32_t total;
    (void)wg_scan_excl<int32_t>(acc, op, Op::id, sh, &total);
    if (threadIdx.x == 0) totals[blockIdx.x] = total;
}

// One workgroup: exclusive scan of the tile totals in place.
template <typename Op>
__global__ __launch_bounds__(WG) void k_scan_totals(int32_t *__restrict__ totals, int tiles, const int *__restrict__ skip) {
    if (skip && *skip) return;  // the caller's flag: this sort is not wanted
    __shared__ int32_t sh[NWAVE];
    const Op op;
    int32_t carry = Op::id;
    for (int b = 0; b < tiles; b += WG) {
        const int i = b + threadIdx.x;
        const int32_t v = i < tiles ? totals[i] : Op::id;
        int32_t total;
        const int32_t ex = wg_scan_excl<int32_t>(v, op, Op::id, sh, &total);
        if (i < tiles) totals[i] = op(carry, ex);
        carry = op(carry, total);
    }
}

// Tile scan: elements staged in LDS, each thread scans 16 consecutive ones.
// totals: of every tile (direct), or the tiles' offsets.
template <typename In, typename Op, bool EXCL>
__global__ __launch_bounds__(WG) void k_scan_tile(const In *__restrict__ in, int32_t *__restrict__ out, int64_t n,
                                                  const int32_t *__restrict__ totals, bool direct,
                                                  const int *__restrict__ skip) {
    if (skip && *skip) return;  // the caller's flag: this sort is not wanted
    __shared__ int32_t s[TILE + TILE / 32];  // one pad word per 32 to spread the banks
    __shared__ int32_t sh[NWAVE];
    const Op op;
    const int64_t t0 = (int64_t)blockIdx.x * TILE;
    auto at = [](int i) { return i + (i >> 5); };
    for (int j = 0; j < ROUNDS; ++j) {
        const int i = j * WG + threadIdx.x;
        s[at(i)] = t0 + i < n ? load_as(in, t0 + i) : Op::id;
    }
    __syncthreads();
    int32_t v[ROUNDS];
    int32_t acc = Op::id;
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
        v[j] = s[at(threadIdx.x * ROUNDS + j)];
        acc = op(acc, v[j]);
    }
    int32_t total, offset;
    if (direct) {
        int32_t t = Op::id;
        for (int i = threadIdx.x; i < (int)blockIdx.x; i += WG) t = op(t, totals[i]);
        (void)wg_scan_excl<int32_t>(t, op, Op::id, sh, &offset);
        __syncthreads();
    } else {
        offset = totals[blockIdx.x];
    }
    int32_t run = op(offset, wg_scan_excl<int32_t>(acc, op, Op::id, sh, &total));
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
        const int32_t next = op(run, v[j]);
        s[at(threadIdx.x * ROUNDS + j)] = EXCL ? run : next;
        run = next;
    }
    __syncthreads();
    for (int j = 0; j < ROUNDS; ++j) {
        const int i = j * WG + threadIdx.x;
        if (t0 + i < n) out[t0 + i] = s[at(i)];
    }
}

template <typename In, typename Op, bool EXCL>
// A whole scan of at most TILE elements in one workgroup (one launch).
__global__ __launch_bounds__(WG) void k_scan_small(const In *__restrict__ in, int32_t *__restrict__ out, int n, const int *__restrict__ skip) {
    if (skip && *skip) return;  // the caller's flag: this sort is not wanted
    __shared__ int32_t s[TILE + TILE / 32];
    __shared__ int32_t sh[NWAVE];
    const Op op;
    auto at = [](int i) { return i + (i >> 5); };
    for (int j = 0; j < ROUNDS; ++j) {
        const int i = j * WG + threadIdx.x;
        s[at(i)] = i < n ? load_as(in, i) : Op::id;
    }
    __syncthreads();
    int32_t v[ROUNDS];
    int32_t acc = Op::id;
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
        v[j] = s[at(threadIdx.x * ROUNDS + j)];
        acc = op(acc, v[j]);
    }
    int32_t total;
    int32_t run = wg_scan_excl<int32_t>(acc, op, Op::id, sh, &total);
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
        const int32_t next = op(run, v[j]);
        s[at(threadIdx.x * ROUNDS + j)] = EXCL ? run : next;
        run = next;
    }
    __syncthreads();
    for (int j = 0; j < ROUNDS; ++j) {
        const int i = j * WG + threadIdx.x;
        if (i < n) out[i] = s[at(i)];
    }
}

__global__ void k_select_scatter(const int32_t *__restrict__ in, const uint8_t *__restrict__ flags,
                                 const int32_t *__restrict__ pos, int64_t n, int32_t *__restrict__ out,
                                 int32_t *__restrict__ count) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const bool f = flags[i] != 0;
    if (f) out[pos[i]] = in[i];
    if (i == n - 1) *count = pos[i] + (f ? 1 : 0);
}

int tiles_of(int64_t n) { return (int)((n + TILE - 1) / TILE); }

// Scan of n elements with `totals` (>= tiles_of(n) ints) as scratch.
template <typename In, typename Op, bool EXCL>
int scan_with(const In *in, int32_t *out, int64_t n, int32_t *totals, hipStream_t st,
              const int *skip = nullptr) {
    if (n <= TILE) {
        hipLaunchKernelGGL((k_scan_small<In, Op, EXCL>), dim3(1), dim3(WG), 0, st, in, out, (int)n, skip);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return set_error(VNM_E_HIP, "scan launch failed: %s", hipGetErrorString(e));
        return VNM_OK;
    }
    const int tiles = tiles_of(n);
    hipLaunchKernelGGL((k_scan_reduce<In, Op>), dim3(tiles), dim3(WG), 0, st, in, n, totals, skip);
    const bool direct = tiles <= SCAN_DIRECT;
    if (!direct) hipLaunchKernelGGL((k_scan_totals<Op>), dim3(1), dim3(WG), 0, st, totals, tiles, skip);
    hipLaunchKernelGGL((k_scan_tile<In, Op, EXCL>), dim3(tiles), dim3(WG), 0, st, in, out, n, totals, direct, skip);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(VNM_E_HIP, "scan launch failed: %s", hipGetErrorString(e));
    return VNM_OK;
}

template <bool VALS>
int radix_sort(const uint64_t *kin, uint64_t *kout, const int32_t *vin, int32_t *vout, int64_t n, KeyBits b,
               hipStream_t st, const int *skip = nullptr) {
    if (n <= 0) return VNM_OK;
    if (n > (int64_t)INT32_MAX) return set_error(VNM_E_ARG, "radix sort of %lld keys", (long long)n);
    const int total = b.w0 + b.w1, passes = passes_of(b);
    const bool small = n <= FUSED_TILES * FWG * SROUNDS;  // 1,024-key tiles
    const int tiles = small ? (int)((n + FWG * SROUNDS - 1) / (FWG * SROUNDS)) : tiles_of(n);
    if (n <= TILE) {
        hipLaunchKernelGGL((k_sort_one<VALS>), dim3(1), dim3(SWG), 0, st, kin, vin, kout, vout, (int)n, b, skip);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return set_error(VNM_E_HIP, "radix sort launch failed: %s", hipGetErrorString(e));
        return VNM_OK;
    }
    // scratch: keys and values of the other buffer, then one count table per
    // pass (fused) or one and its digits' totals
    const bool fused = tiles <= FUSED_TILES;
    const size_t kb = align256((size_t)n * 8), vb = VALS ? align256((size_t)n * 4) : 0;
    const int64_t tab = (int64_t)RADIX * tiles;
    int rc = g_tmp.ensure(kb + vb + align256((size_t)(fused ? tab * passes : tab + RADIX) * 4));
    if (rc) return rc;
    uint64_t *ktmp = (uint64_t *)g_tmp.p;
    int32_t *vtmp = (int32_t *)((char *)g_tmp.p + kb);
    int32_t *hist = (int32_t *)((char *)g_tmp.p + kb + vb);
    const uint64_t *ks = kin;
    const int32_t *vs = vin;
    int shift = 0;
    for (int p = 0; p < passes; ++p) {
        // the last pass writes the output
        uint64_t *kd = ((passes - 1 - p) % 2 == 0) ? kout : ktmp;
        int32_t *vd = ((passes - 1 - p) % 2 == 0) ? vout : vtmp;
        const Digit dg{b, shift, digit_bits(total, shift)};
        shift += dg.bits;
        if (fused) {
            const bool last = p + 1 == passes;
            int32_t *h = hist + tab * p;
            const Digit ndg{b, shift, last ? 1 : digit_bits(total, shift)};
            int32_t *nh = last ? nullptr : h + tab;
            const int nz = (int)(tab * (passes - 1));
            if (small) {
                if (p == 0)  // the first table counted, the others cleared
                    hipLaunchKernelGGL(k_radix_hist<FWG>, dim3(tiles), dim3(FWG), 0, st, ks, n, dg, tiles, h, h + tab, nz, skip);
                hipLaunchKernelGGL((k_radix_fused<VALS, FWG>), dim3(tiles), dim3(FWG), 0, st, ks, vs, kd, vd, (int)n, dg,
                                   tiles, h, ndg, nh, skip);
            } else {
                if (p == 0)
                    hipLaunchKernelGGL(k_radix_hist<SWG>, dim3(tiles), dim3(SWG), 0, st, ks, n, dg, tiles, h, h + tab, nz, skip);
                hipLaunchKernelGGL((k_radix_fused<VALS, SWG>), dim3(tiles), dim3(SWG), 0, st, ks, vs, kd, vd, (int)n, dg,
                                   tiles, h, ndg, nh, skip);
            }
        } else {
            hipLaunchKernelGGL(k_radix_hist<SWG>, dim3(tiles), dim3(SWG), 0, st, ks, n, dg, tiles, hist, nullptr, 0, skip);
            hipLaunchKernelGGL(k_digit_scan, dim3(RADIX), dim3(SWG), 0, st, hist, tiles, hist + tab, skip);
            hipLaunchKernelGGL((k_radix_scatter<VALS>), dim3(tiles), dim3(SWG), 0, st, ks, vs, kd, vd, n, dg, tiles, hist,
                               hist + tab, skip);
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return set_error(VNM_E_HIP, "radix sort launch failed: %s", hipGetErrorString(e));
        ks = kd;
        vs = vd;
    }
    return VNM_OK;
}

}  // namespace

int sort_keys_u64(const uint64_t *in, uint64_t *out, int64_t n, KeyBits bits, hipStream_t st) {
    return radix_sort<false>(in, out, nullptr, nullptr, n, bits, st);
}

int sort_keys_u64_if(const uint64_t *in, uint64_t *out, int64_t n, KeyBits bits, hipStream_t st, const int *skip) {
    return radix_sort<false>(in, out, nullptr, nullptr, n, bits, st, skip);
}

int sort_scratch_slot(int slot) {
    const int prev = g_slot;
    if (slot >= 0 && slot < SCRATCH_SLOTS) g_slot = slot;
    return prev;
}

int sort_scratch_reserve(int64_t n) {
    if (n <= TILE) return VNM_OK;
    // keys and values, count tables of 8 passes (fused) or one with its totals
    const int64_t tab = (int64_t)RADIX * std::max<int64_t>(tiles_of(n), FUSED_TILES);
    return g_tmp.ensure(align256((size_t)n * 8) + align256((size_t)n * 4) + align256((size_t)(tab * 8 + RADIX) * 4));
}

int sort_pairs_u64_i32(const uint64_t *kin, uint64_t *kout, const int32_t *vin, int32_t *vout, int64_t n,
                       KeyBits bits, hipStream_t st) {
    return radix_sort<true>(kin, kout, vin, vout, n, bits, st);
}

int scan_excl_i32(const int32_t *in, int32_t *out, int64_t n, hipStream_t st) {
    if (n <= 0) return VNM_OK;
    int rc = g_tmp.ensure(align256((size_t)tiles_of(n) * 4));
    if (rc) return rc;
    return scan_with<int32_t, OpSum, true>(in, out, n, (int32_t *)g_tmp.p, st);
}

int scan_incl_max_i32(const int32_t *in, int32_t *out, int64_t n, hipStream_t st) {
    if (n <= 0) return VNM_OK;
    int rc = g_tmp.ensure(align256((size_t)tiles_of(n) * 4));
    if (rc) return rc;
    return scan_with<int32_t, OpMax, false>(in, out, n, (int32_t *)g_tmp.p, st);
}

int select_flagged_i32(const int32_t *in, const uint8_t *flags, int32_t *out, int32_t *d_count, int64_t n,
                       hipStream_t st) {
    if (n <= 0) {
        hipError_t e = hipMemsetAsync(d_count, 0, sizeof(int32_t), st);
        return e == hipSuccess ? VNM_OK : set_error(VNM_E_HIP, "select: %s", hipGetErrorString(e));
    }
    const size_t pb = align256((size_t)n * 4);
    int rc = g_tmp.ensure(pb + align256((size_t)tiles_of(n) * 4));
    if (rc) return rc;
    int32_t *pos = (int32_t *)g_tmp.p;
    if ((rc = scan_with<uint8_t, OpSum, true>(flags, pos, n, (int32_t *)((char *)g_tmp.p + pb), st))) return rc;
    hipLaunchKernelGGL(k_select_scatter, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, in, flags, pos, n, out,
                       d_count);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? VNM_OK : set_error(VNM_E_HIP, "select launch failed: %s", hipGetErrorString(e));
}

}  // namespace vnm


extern "C" int vnm_sort_pairs(vnm_ctx *ctx, const uint64_t *keys_in, uint64_t *keys_out, const int32_t *vals_in,
                              int32_t *vals_out, int64_t n, int end_bit) {
    if (!ctx || (n > 0 && (!keys_in || !keys_out))) return vnm::set_error(VNM_E_ARG, "sort: null argument");
    if (n < 0 || end_bit < 1 || end_bit > 64) return vnm::set_error(VNM_E_ARG, "sort: n >= 0, end_bit in [1, 64]");
    if ((vals_in == nullptr) != (vals_out == nullptr))
        return vnm::set_error(VNM_E_ARG, "sort: values in and out must both be given or both be NULL");
    if (keys_in == keys_out || (vals_in && vals_in == vals_out))
        return vnm::set_error(VNM_E_ARG, "sort: output must not alias the input");
    const vnm::KeyBits bits = vnm::key_range(0, end_bit);
    int rc = vals_in ? vnm::sort_pairs_u64_i32(keys_in, keys_out, vals_in, vals_out, n, bits, ctx->stream)
                     : vnm::sort_keys_u64(keys_in, keys_out, n, bits, ctx->stream);
    if (rc) return rc;
    ctx->launches += 5 * ((end_bit + 7) / 8);
    return VNM_OK;
}
