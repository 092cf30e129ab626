// V:N:M (N = 2) packer and SpMM for gfx950.
//
// Replaces the reference's SpMM paths (kernel/spmm.cu: the 16x16 WMMA BSR
// kernel :44-161 and the cuSPARSELt 2:4 prune/compress/matmul :324-500,
// which densify A first, kernel/eval.h:12-18).
//
// Format (VENOM with row compression).  A is cut into V x M blocks (V rows,
// one segment of M columns).  Each stored block keeps 4 of its M columns --
// the subset maximising sum over rows of min(2, |row & S|), ties to the
// lexicographically smallest subset -- and each row keeps at most 2 values
// inside them (2:4): the two largest |v|, ties to the lower column.  Blocks
// store their segment, the 4 column offsets (4 bits each) and, for FP8, one
// FP32 scale (absmax / 448).  Rows of a block that keep anything store one
// "row entry": two values and two 2-bit selector indices.  Row entries are
// laid out row-major (CSR over rows), so the SpMM accumulates each output row
// in registers and writes it once.
//
//   bytes(A) = 4 (R + 1) + E (4 + 4 + 1 + 2 s_v) + nb (4 + 2 + 4)
// (rowptr; per row entry its row, block, selector byte and two values; per
// block its segment, selectors and scale).
//
// SpMM: C[R x n] = A_vnm B, FP32 accumulation.  Packing also writes the
// SpMM's value stream: every kept value of the row entries as (B row, FP32
// weight = value x block scale), 8 bytes per value, so the SpMM reads no block
// data and branches on no selector.  A work item is a whole row of at most 64
// values or a 64-value chunk of a longer row; items and stream are sorted by
// item length.  A wave takes 64 / LPR items for one column tile, LPR lanes per
// item: one load instruction gathers the tiles of 64 / LPR B rows, 16 bytes per
// lane, with the values' B rows and weights spread over the lanes by DPP, and the
// row is stored once, after its last value (rows that keep nothing are written in
// the gaps).  The chunks of a long row store partial sums into slots, and a
// fix-up pass adds each cut row's slots in chunk order, so C is bit-identical
// for every launch shape and run: no atomics.  When the tile count T divides 8,
// tile t runs on its own 8/T XCDs, so each XCD's L2 serves one 1/T slice of B.
// FP8 B is decoded by the gfx950 e4m3 conversion instruction.
//
// Measured (us per product, fix-up pass included; before: one item of mixed row
// lengths per wave, the B row's offset a scalar, 2 to 8 bytes per lane, the width
// timed on first use): R-MAT 65,536, 128:2:8, n = 256: FP32 88 -> 76, BF16 82 ->
// 49; R-MAT 131,072 degree 24, 64:2:4, BF16 n = 128: 107 -> 68; Chung-Lu 20,011
// FP8 n = 384: 45 -> 26.  The FP32 gather moves 1.07 GB through L1s that take
// 33 us for it when every request hits, 37 when every one hits L2; the rest is L2
// misses (a copy of the loop without row ends or weights' FMAs: 60).
#include "graph.h"
#include "hip_common.h"
#include "packed.h"
#include "sortlib.h"

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <memory>
#include <vector>

namespace vnm {

static int grid_of(int64_t n, int block) {
    int64_t g = (n + block - 1) / block;
    return (int)std::max<int64_t>(1, std::min<int64_t>(g, 1 << 20));
}

// ------------------------------------------------------------ value codecs

// ------------------------------------------------------------ packer kernels

__global__ void k_nz_keys(const int32_t *__restrict__ row, const int32_t *__restrict__ col,
                          const float *__restrict__ val, int64_t nnz, int32_t ncolseg,
                          uint64_t *__restrict__ keys, int32_t *__restrict__ idx) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < nnz; i += (int64_t)gridDim.x * blockDim.x) {
        const bool ok = val[i] != 0.0f && col[i] < ncolseg;
        keys[i] = ok ? (((uint64_t)(uint32_t)row[i] << 32) | (uint32_t)col[i]) : ~0ull;
        idx[i] = (int32_t)i;
    }
}

// Run heads of the sorted keys; dropped entries' all-ones keys, sorted last, head
// none, and the last key before them gives the number of the others.
__global__ void k_pk_heads(const uint64_t *__restrict__ k, int64_t n, int M, int32_t *__restrict__ head,
                           int32_t *__restrict__ nz) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t a = k[i];
        const bool kept = a != ~0ull;
        bool h = kept;
        if (i > 0) {
            const uint64_t b = k[i - 1];
            h = kept && ((a >> 32) != (b >> 32) || (uint32_t)a / M != (uint32_t)b / M);
        }
        head[i] = h;
        if (kept && (i + 1 == n || k[i + 1] == ~0ull)) *nz = (int32_t)(i + 1);
    }
}

// The total of n flags whose exclusive sums are `excl`.
__global__ void k_pk_total(const int32_t *__restrict__ excl, const int32_t *__restrict__ flag, int64_t n,
                           int32_t *__restrict__ total) {
    *total = excl[n - 1] + flag[n - 1];
}

__global__ void k_pk_runs(const uint64_t *__restrict__ k, const int32_t *__restrict__ head,
                          const int32_t *__restrict__ excl, int64_t n, int M, uint32_t *__restrict__ bits,
                          int32_t *__restrict__ rstart, int32_t *__restrict__ rlen, uint64_t *__restrict__ bkey,
                          int32_t *__restrict__ rid) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t key = k[i];
        const uint32_t c = (uint32_t)key, r = (uint32_t)(key >> 32);
        const int u = excl[i] + head[i] - 1;
        atomicOr(&bits[u], 1u << (M - 1 - (c % M)));
        atomicAdd(&rlen[u], 1);
        if (head[i]) {
            rstart[u] = (int32_t)i;
            // (segment, row): a block's runs, rows r / V of one segment, lie together
            bkey[u] = ((uint64_t)(c / M) << 32) | r;
            rid[u] = u;
        }
    }
}

__global__ void k_blk_heads(const uint64_t *__restrict__ bk, int U, int V, int32_t *__restrict__ head) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < U)
        head[i] = (i == 0) || ((bk[i] >> 32) != (bk[i - 1] >> 32)) ||
                  (uint32_t)bk[i] / (uint32_t)V != (uint32_t)bk[i - 1] / (uint32_t)V;
}

// The selected subset's 4 column offsets (ascending), 4 bits each.
__device__ __forceinline__ uint16_t subset_sel(uint32_t S, int M) {
    uint16_t sel = 0;
    int k = 0;
    for (int c = 0; c < M && k < 4; ++c)
        if (S & (1u << (M - 1 - c))) sel |= (uint16_t)(c << (4 * k++));
    return sel;
}

constexpr int LANE_RUNS = 8;  // runs of a block that one lane scores

// Block selection, one lane per block of at most LANE_RUNS runs (nearly all
// blocks of sparse graphs): the run bitmaps stay in registers and the
// subsets are scored in ascending index order with strict > (ties to the
// smallest), the order k_blk_select's argmax yields.  Longer blocks are
// listed for k_blk_select.
__global__ __launch_bounds__(256) void k_blk_select_lane(
    const uint64_t *__restrict__ bk, const int32_t *__restrict__ rid_sorted, int U, int nb, int M,
    const uint32_t *__restrict__ bits, const uint32_t *__restrict__ subs, int nsub,
    const int32_t *__restrict__ blk_first, int32_t *__restrict__ blk_seg, uint16_t *__restrict__ blk_sel,
    uint32_t *__restrict__ blk_mask, int32_t *__restrict__ run_blk, unsigned long long *__restrict__ retained,
    int32_t *__restrict__ longb, int32_t *__restrict__ nlong) {
    int kept = 0;
    for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < nb; b += gridDim.x * blockDim.x) {
        const int first = blk_first[b];
        const int last = b + 1 < nb ? blk_first[b + 1] : U;
        const int n = last - first;
        if (n > LANE_RUNS) {
            longb[atomicAdd(nlong, 1)] = b;
        } else {
            uint32_t r[LANE_RUNS];
#pragma unroll
            for (int j = 0; j < LANE_RUNS; ++j) r[j] = j < n ? bits[rid_sorted[first + j]] : 0u;
            int best_score = -1, best_idx = 0;
            for (int s = 0; s < nsub; ++s) {
                const uint32_t S = subs[s];
                int sc = 0;
#pragma unroll
                for (int j = 0; j < LANE_RUNS; ++j) sc += min(2, popc32(r[j] & S));
                if (sc > best_score) {
                    best_score = sc;
                    best_idx = s;
                }
            }
            const uint32_t S = subs[best_idx];
            blk_seg[b] = (int32_t)(bk[first] >> 32);
            blk_sel[b] = subset_sel(S, M);
            blk_mask[b] = S;
            kept += best_score;
            for (int j = 0; j < n; ++j) run_blk[rid_sorted[first + j]] = b;
        }
    }
    // one atomic per workgroup: atomics on a single address serialise at the
    // L2, so the grid is capped and the workgroup sums first
    __shared__ int wsum[4];
    for (int d = 32; d >= 1; d >>= 1) kept += __shfl_xor(kept, d, 64);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = kept;
    __syncthreads();
    if (threadIdx.x == 0) {
        const int t = wsum[0] + wsum[1] + wsum[2] + wsum[3];
        if (t) atomicAdd(retained, (unsigned long long)t);
    }
}

// One wave per listed block: best 4-column subset (lexicographic order of
// ascending column tuples; ties to the smallest).  nsub = C(M, 4) <= 70.
__global__ __launch_bounds__(256) void k_blk_select(const uint64_t *__restrict__ bk, const int32_t *__restrict__ rid_sorted,
                             int U, int nb, int M, const uint32_t *__restrict__ bits,
                             const uint32_t *__restrict__ subs, int nsub,
                             const int32_t *__restrict__ blk_first, int32_t *__restrict__ blk_seg,
                             uint16_t *__restrict__ blk_sel, uint32_t *__restrict__ blk_mask,
                             int32_t *__restrict__ run_blk, unsigned long long *__restrict__ retained,
                             const int32_t *__restrict__ list, const int32_t *__restrict__ nlist) {
    const int lane = threadIdx.x & 63;
    const int wpb = blockDim.x / 64;
    const int count = *nlist;
    // listed blocks in a grid-stride loop per wave; the retained count is
    // summed per wave and added once (one atomic per block on a single
    // address serialises at the L2)
    unsigned long long kept = 0;
    for (int i = blockIdx.x * wpb + (threadIdx.x >> 6); i < count; i += gridDim.x * wpb) {
        const int b = list[i];
        const int first = blk_first[b];
        int last = U;
        if (b + 1 < nb) last = blk_first[b + 1];
        // scores of 128 subsets at a time (lane and lane + 64; one round for
        // M <= 8): the block's run bitmaps are loaded 64 at a time, one per
        // lane, and broadcast
        int best_score = -1, best_idx = 0x7FFFFFFF;
        for (int s0 = 0; s0 < nsub; s0 += 128) {
            const int i0 = s0 + lane, i1 = s0 + 64 + lane;
            const uint32_t S0 = i0 < nsub ? subs[i0] : 0u;
            const uint32_t S1 = i1 < nsub ? subs[i1] : 0u;
            int sc0 = 0, sc1 = 0;
            for (int base = first; base < last; base += 64) {
                const int q = base + lane;
                const int mine = q < last ? (int)bits[rid_sorted[q]] : 0;
                const int n = min(64, last - base);
                for (int j = 0; j < n; ++j) {
                    const uint32_t bj = (uint32_t)__builtin_amdgcn_readlane(mine, j);
                    sc0 += min(2, popc32(bj & S0));
                    sc1 += min(2, popc32(bj & S1));
                }
            }
            // ascending subset index per lane: strict > keeps the smaller on ties
            if (i0 < nsub && sc0 > best_score) { best_score = sc0; best_idx = i0; }
            if (i1 < nsub && sc1 > best_score) { best_score = sc1; best_idx = i1; }
        }
        // wave argmax (score desc, index asc)
        for (int d = 32; d >= 1; d >>= 1) {
            int os = __shfl_xor(best_score, d, 64), oi = __shfl_xor(best_idx, d, 64);
            if (os > best_score || (os == best_score && oi < best_idx)) { best_score = os; best_idx = oi; }
        }
        const uint32_t S = subs[best_idx];
        if (lane == 0) {
            blk_seg[b] = (int32_t)(bk[first] >> 32);
            blk_sel[b] = subset_sel(S, M);
            blk_mask[b] = S;
            kept += (unsigned long long)best_score;
        }
        for (int q = first + lane; q < last; q += 64) run_blk[rid_sorted[q]] = b;
    }
    // one atomic per workgroup (lane 0 of each wave holds the wave's sum)
    __shared__ unsigned long long wsum[4];
    if (lane == 0) wsum[threadIdx.x >> 6] = kept;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long t = wsum[0] + wsum[1] + wsum[2] + wsum[3];
        if (t) atomicAdd(retained, t);
    }
}

__global__ void k_blk_first(const int32_t *__restrict__ head, const int32_t *__restrict__ excl, int U,
                            int32_t *__restrict__ blk_first) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < U && head[i]) blk_first[excl[i]] = i;
}

// Per run: the kept values (<= 2) among the block's selected columns.
__global__ void k_run_keep(const uint64_t *__restrict__ keys, const int32_t *__restrict__ eidx,
                           const float *__restrict__ val, int U, int M,
                           const int32_t *__restrict__ rstart, const int32_t *__restrict__ rlen,
                           const int32_t *__restrict__ run_blk, const uint32_t *__restrict__ blk_mask,
                           float *__restrict__ kv, uint8_t *__restrict__ kidx,
                           int32_t *__restrict__ nkeep, uint32_t *__restrict__ blk_absmax) {
    int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= U) return;
    const int b = run_blk[u];
    const uint32_t S = blk_mask[b];
    // selector index of column offset c within S (ascending order)
    float v0 = 0.f, v1 = 0.f;
    int c0 = -1, c1 = -1;
    const int beg = rstart[u], len = rlen[u];
    for (int q = beg; q < beg + len; ++q) {
        const int c = (int)((uint32_t)keys[q] % (uint32_t)M);
        if (!(S & (1u << (M - 1 - c)))) continue;
        const float v = val[eidx[q]];
        const float a = fabsf(v);
        // entries come in ascending column order: strict > keeps the lower
        // column on ties
        if (c0 < 0 || a > fabsf(v0)) { v1 = v0; c1 = c0; v0 = v; c0 = c; }
        else if (c1 < 0 || a > fabsf(v1)) { v1 = v; c1 = c; }
    }
    int n = (c0 >= 0) + (c1 >= 0);
    uint8_t code = 0;
    if (n > 0) {
        int i0 = popc32(S >> (M - c0)), i1 = c1 >= 0 ? popc32(S >> (M - c1)) : 0;
        code = (uint8_t)(i0 | (i1 << 2) | (c1 >= 0 ? 0x10 : 0));
        float m = fmaxf(fabsf(v0), c1 >= 0 ? fabsf(v1) : 0.f);
        atomicMax(&blk_absmax[b], __float_as_uint(m));
    }
    kv[2 * u] = v0;
    kv[2 * u + 1] = c1 >= 0 ? v1 : 0.f;
    kidx[u] = code;
    nkeep[u] = n;
}

// Kept runs per row.  Runs are sorted by row, so a wave's lanes of one row
// are contiguous: the last lane of each such segment adds the segment's
// kept count (one atomic per row and wave; a hub row's thousands of runs
// would otherwise serialise on one address).
__global__ void k_row_counts(const uint64_t *__restrict__ keys, const int32_t *__restrict__ rstart,
                             const int32_t *__restrict__ nkeep, const int32_t *__restrict__ run_blk,
                             const int32_t *__restrict__ dmap, int U, int32_t *__restrict__ rcnt,
                             uint8_t *__restrict__ flag) {
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const bool valid = u < U;
    // runs of dense blocks (dmap >= 0) go to the sparse-MFMA part instead
    const bool keep = valid && nkeep[u] > 0 && (dmap == nullptr || dmap[run_blk[u]] < 0);
    const int row = valid ? (int)(keys[rstart[u]] >> 32) : -1;
    if (valid) flag[u] = keep;
    const uint64_t kmask = __ballot(keep);
    const int prev = __shfl_up(row, 1, 64), next = __shfl_down(row, 1, 64);
    const uint64_t heads = __ballot(lane == 0 || row != prev);
    const bool tail = lane == 63 || row != next;
    if (valid && tail) {
        const uint64_t upto = lane == 63 ? ~0ull : ((2ull << lane) - 1);
        const int start = 63 - __builtin_clzll(heads & upto);
        const int c = __popcll(kmask & upto & ~((1ull << start) - 1));
        if (c) atomicAdd(&rcnt[row], c);
    }
}

__global__ void k_iota_i(int32_t *p, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}

__global__ void k_scales(const uint32_t *__restrict__ absmax, int nb, int fp8, float *__restrict__ sc) {
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    float m = __uint_as_float(absmax[b]);
    sc[b] = (fp8 && m > 0.f) ? m / 448.0f : 1.0f;
}

__global__ void k_emit(const int32_t *__restrict__ sel_runs, int E, const int32_t *__restrict__ run_blk,
                       const uint64_t *__restrict__ keys, const int32_t *__restrict__ rstart,
                       const float *__restrict__ kv, const uint8_t *__restrict__ kidx,
                       const float *__restrict__ sc, const int32_t *__restrict__ blk_seg,
                       const uint16_t *__restrict__ blk_sel, int M, int dtype,
                       int32_t *__restrict__ ent_row, int32_t *__restrict__ ent_col,
                       int32_t *__restrict__ ent_blk, uint8_t *__restrict__ ent_idx,
                       uint8_t *__restrict__ ent_val) {
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const int u = sel_runs[e];
    const int b = run_blk[u];
    ent_row[e] = (int32_t)(keys[rstart[u]] >> 32);
    // selector indices -> columns: first value absolute, second as offset
    const uint32_t code = kidx[u], sel = blk_sel[b];
    ent_col[e] = blk_seg[b] * M + (int)((sel >> (4 * (code & 3u))) & 15u);
    ent_idx[e] = (code & 0x10u) ? (uint8_t)(0x10u | ((sel >> (4 * ((code >> 2) & 3u))) & 15u)) : (uint8_t)0;
    if (dtype == VNM_DT_FP8) ent_blk[e] = b;
    const float v0 = kv[2 * u], v1 = kv[2 * u + 1];
    if (dtype == VNM_DT_F32) {
        float *p = (float *)ent_val;
        p[2 * e] = v0;
        p[2 * e + 1] = v1;
    } else if (dtype == VNM_DT_BF16) {
        uint16_t *p = (uint16_t *)ent_val;
        p[2 * e] = f32_to_bf16(v0);
        p[2 * e + 1] = f32_to_bf16(v1);
    } else if (dtype == VNM_DT_F16) {
        __half *p = (__half *)ent_val;
        p[2 * e] = __float2half(v0);
        p[2 * e + 1] = __float2half(v1);
    } else {
        const float s = sc[b];
        ent_val[2 * e] = f32_to_e4m3(v0 / s);
        ent_val[2 * e + 1] = f32_to_e4m3(v1 / s);
    }
}

// ------------------------------------------------------------ SpMM

// ------------------------------------------------------------ value stream

// Values per row entry (1 or 2), and entry E's count 0 (the scan's total).
__global__ void k_val_counts(const uint8_t *__restrict__ ent_idx, int E, int32_t *__restrict__ nv) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e < E) nv[e] = (ent_idx[e] & 0x10u) ? 2 : 1;
    else if (e == E) nv[e] = 0;
}

// Where the values of a row go: piece c of row r (the row, or its c-th chunk of
// ITEM values) starts at pdst[pbase[r] + c] of the value stream.
struct Pieces {
    const int32_t *vrp, *pbase, *pdst;
};

// Value i (in row-major order) of row r: B row c, weight w.
__device__ __forceinline__ void put_value(const Pieces &P, int i, int r, int c, float w, uint2 *__restrict__ vrec) {
    const int k = i - P.vrp[r];
    vrec[P.pdst[P.pbase[r] + k / ITEM] + k % ITEM] = make_uint2((uint32_t)c, __float_as_uint(w));
}

template <int DT>
__device__ __forceinline__ void emit_values(int e, int M, const int32_t *__restrict__ voff, const Pieces &P,
                                            const int32_t *__restrict__ ent_row, const int32_t *__restrict__ ent_col,
                                            const uint8_t *__restrict__ ent_idx, const uint8_t *__restrict__ ent_val,
                                            const int32_t *__restrict__ ent_blk, const float *__restrict__ blk_scale,
                                            uint2 *__restrict__ vrec) {
    const int o = voff[e];
    const int r = ent_row[e], c0 = ent_col[e];
    const uint32_t code = ent_idx[e];
    const float sc = DT == VNM_DT_FP8 ? blk_scale[ent_blk[e]] : 1.f;
    put_value(P, o, r, c0, load_aval<DT>(ent_val, 2 * e) * sc, vrec);
    if (code & 0x10u)
        put_value(P, o + 1, r, (c0 & ~(M - 1)) | (int)(code & 15u), load_aval<DT>(ent_val, 2 * e + 1) * sc, vrec);
}

// The SpMM's value stream: row entry e's values (its first, then its second),
// each weight being the stored value times the block scale (FP8; 1 otherwise)
// rounded to FP32 once.
__global__ void k_values(int E, int M, int dtype, const int32_t *__restrict__ voff, Pieces P,
                         const int32_t *__restrict__ ent_row, const int32_t *__restrict__ ent_col,
                         const uint8_t *__restrict__ ent_idx, const uint8_t *__restrict__ ent_val,
                         const int32_t *__restrict__ ent_blk, const float *__restrict__ blk_scale,
                         uint2 *__restrict__ vrec) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    switch (dtype) {
        case VNM_DT_F32:
            emit_values<VNM_DT_F32>(e, M, voff, P, ent_row, ent_col, ent_idx, ent_val, ent_blk, blk_scale, vrec);
            break;
        case VNM_DT_BF16:
            emit_values<VNM_DT_BF16>(e, M, voff, P, ent_row, ent_col, ent_idx, ent_val, ent_blk, blk_scale, vrec);
            break;
        case VNM_DT_F16:
            emit_values<VNM_DT_F16>(e, M, voff, P, ent_row, ent_col, ent_idx, ent_val, ent_blk, blk_scale, vrec);
            break;
        default:
            emit_values<VNM_DT_FP8>(e, M, voff, P, ent_row, ent_col, ent_idx, ent_val, ent_blk, blk_scale, vrec);
            break;
    }
}

// Row pointers over values: vrp[r] = voff[rowptr[r]], r <= R.
__global__ void k_vrowptr(const int32_t *__restrict__ rowptr, const int32_t *__restrict__ voff, int R,
                          int32_t *__restrict__ vrp) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r <= R) vrp[r] = voff[rowptr[r]];
}

// ------------------------------------------------------------ work items

// Rows without values from row r on, counted up to GAP_MAX + 1.
__device__ __forceinline__ int empty_run(const int32_t *__restrict__ vrp, int R, int r) {
    int n = 0;
    while (n <= GAP_MAX && r + n < R && vrp[r + n + 1] == vrp[r + n]) ++n;
    return n;
}

// Per row: its pieces (np), a cut row's first slot (slot0), the rows without
// values written after an uncut row (gap), and the rows of the fix-up pass --
// cut rows, and rows without values that no uncut row writes: those before the
// first row with values, after a cut row, or in a run of more than GAP_MAX.
// cnt: slots, hub rows, other listed rows.  Slots and list positions come from
// counters, so they differ from one packing to the next; nothing computed does.
__global__ __launch_bounds__(256) void k_row_pieces(const int32_t *__restrict__ vrp, int R, int32_t *__restrict__ np,
                                                    int32_t *__restrict__ slot0, uint8_t *__restrict__ gap,
                                                    int32_t *__restrict__ cnt, int4 *__restrict__ fix) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r > R) return;
    const int len = r < R ? vrp[r + 1] - vrp[r] : 0;
    const int pieces = (len + ITEM - 1) / ITEM;
    np[r] = pieces;
    if (r == R) return;
    bool list = false;
    int s0 = 0, ns = 0;
    if (len > ITEM) {
        list = true;
        ns = pieces;
        s0 = atomicAdd(&cnt[0], ns);
        slot0[r] = s0;
        gap[r] = 0;
    } else if (len > 0) {
        const int e = empty_run(vrp, R, r + 1);
        gap[r] = (uint8_t)(e <= GAP_MAX ? e : 0);
    } else {
        int b = 1;  // the row with values before this one is r - b
        while (b <= GAP_MAX && r - b >= 0 && vrp[r - b + 1] == vrp[r - b]) ++b;
        list = b > GAP_MAX || r - b < 0 || vrp[r - b + 1] - vrp[r - b] > ITEM ||
               empty_run(vrp, R, r - b + 1) > GAP_MAX;
    }
    const bool hub = list && ns > HUB_SLOTS;
    const bool rest = list && !hub;
    if (hub) fix[atomicAdd(&cnt[1], 1)] = make_int4(r, s0, ns, 0);
    const uint64_t m = __ballot(rest);  // one atomic per wave
    if (rest) {
        const int lane = threadIdx.x & 63;
        int base = 0;
        const int lead = __builtin_ctzll(m);
        if (lane == lead) base = atomicAdd(&cnt[2], (int)__popcll(m));
        base = __shfl(base, lead, 64);
        fix[R - 1 - (base + (int)__popcll(m & ((1ull << lane) - 1)))] = make_int4(r, s0, ns, 0);
    }
}

// The pieces in row order: sort key (long pieces first; slots of the arrays past
// the last piece sort behind them), and what the work item will hold.
__global__ __launch_bounds__(256) void k_pieces(const int32_t *__restrict__ vrp, int R, const int32_t *__restrict__ pbase,
                                                const int32_t *__restrict__ slot0, const uint8_t *__restrict__ gap,
                                                int cap, uint64_t *__restrict__ key, int32_t *__restrict__ id,
                                                int2 *__restrict__ info) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < R) {
        const int len = vrp[t + 1] - vrp[t], p0 = pbase[t];
        const bool cut = len > ITEM;
        for (int c = 0; c * ITEM < len; ++c) {
            const int l = min(ITEM, len - c * ITEM);
            key[p0 + c] = (uint64_t)(ITEM - l);
            id[p0 + c] = p0 + c;
            info[p0 + c] = make_int2(cut ? slot0[t] + c : t, l | (cut ? 1 << 16 : (int)gap[t] << 8));
        }
    }
    for (int i = pbase[R] + t; i < cap; i += gridDim.x * blockDim.x) {
        key[i] = ITEM;
        id[i] = i;
        info[i] = make_int2(0, 0);
    }
}

__global__ void k_piece_lens(const int32_t *__restrict__ order, const int2 *__restrict__ info, int cap,
                             int32_t *__restrict__ len) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cap) len[i] = info[order[i]].y & 0xFF;
}

// The work items: the sorted pieces (beg: their starts in the value stream), in
// groups of GROUP neighbours -- the most a wave walks side by side, so those
// have one length -- whose order steps through the sorted list by about 0.62 of
// it.  In sorted order the launch gathers only at first and mostly stores at
// the end: R-MAT 65,536, FP32, n = 256: 110 us sorted, 80 mixed.
constexpr int GROUP = 8;
__global__ __launch_bounds__(256) void k_items(const int32_t *__restrict__ npieces, const int32_t *__restrict__ order,
                                               const int2 *__restrict__ info, const int32_t *__restrict__ beg,
                                               int32_t *__restrict__ pdst, int4 *__restrict__ items) {
    __shared__ int step;
    const int n = *npieces, ng = n / GROUP;
    if (threadIdx.x == 0) {
        // a step coprime to the group count visits every group once
        int s = max(1, (int)(ng * 0.618f));
        for (;; ++s) {
            int x = s, y = ng;
            while (y) {
                const int r = x % y;
                x = y;
                y = r;
            }
            if (x <= 1 || ng <= 1) break;
        }
        step = s;
    }
    __syncthreads();
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const int g = j / GROUP;
    const int i = g < ng ? (int)((int64_t)g * step % ng) * GROUP + j % GROUP : j;
    const int id = order[i];
    const int2 f = info[id];
    pdst[id] = beg[i];
    const Piece p{beg[i], f.y & 0xFF, f.x, (int16_t)((f.y >> 8) & 0xFF), (int16_t)(f.y >> 16)};
    items[j] = *(const int4 *)&p;
}

// ------------------------------------------------------------ SpMM kernel

template <int BT, int LPR, int LB, bool EXTRA>
__global__ __launch_bounds__(256) void k_spmm(SpmmArgs a, int T, int per_g) {
    constexpr int NV = LB / bsize<BT>();
    __shared__ __align__(16) float turn[NV > 4 ? 4 : 1][NV > 4 ? 64 * NV : 4];
    const int wv = threadIdx.x >> 6;
    // workgroups are dealt round-robin over the 8 XCDs
    const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
    int tile, iwg;
    if (8 % T == 0) {  // tile t on XCDs [t*8/T, (t+1)*8/T)
        const int gs = 8 / T;
        tile = xcd / gs;
        iwg = (xcd % gs) * per_g + slot;
    } else {
        const int lwg = xcd * per_g + slot;
        tile = lwg % T;
        iwg = lwg / T;
    }
    const int item0 = __builtin_amdgcn_readfirstlane((iwg * 4 + wv) * (64 / LPR));
    if (item0 >= a.items) return;
    spmm_items<BT, LPR, LB, EXTRA>(a, item0, __builtin_amdgcn_readfirstlane(tile), turn[NV > 4 ? wv : 0]);
}

// Fix-up pass: rows cut into chunks get the sum of their partial-sum slots
// in item order; a matrix without work items, the bias or zero in every row.
__global__ __launch_bounds__(256) void k_spmm_fix(const int4 *__restrict__ hubs, int nhub,
                                                  const int4 *__restrict__ rest, int nrest,
                                                  const float *__restrict__ part, int pn, int n,
                                                  float *__restrict__ C, int ldc, const float *__restrict__ bias,
                                                  const uint8_t *__restrict__ dvb, int V) {
    // wave-uniform, so the list entry is a scalar load
    int w = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    const int hp = n / 64, cp = (n + 255) / 256;
    const bool hub = w < nhub * hp;
    if (!hub) w -= nhub * hp;
    const int i = hub ? w / hp : w / cp;
    if (!hub && i >= nrest) return;
    const int4 f = hub ? hubs[i] : rest[i];
    float *crow = C + (size_t)f.x * ldc;
    const bool dense = dvb != nullptr && dvb[f.x / V] != 0;
    if (hub) fix_row<1, 32>(crow, part, pn, f.y, f.z, w % hp * 64, n, bias, dense);
    else fix_row<4, 8>(crow, part, pn, f.y, f.z, w % cp * 256, n, bias, dense);
}

// ------------------------------------------------------------ host

static std::vector<uint32_t> subsets4(int M) {
    std::vector<uint32_t> out;
    if (M <= 4) {
        out.push_back((1u << M) - 1);
        return out;
    }
    for (int a = 0; a < M; ++a)
        for (int b = a + 1; b < M; ++b)
            for (int c = b + 1; c < M; ++c)
                for (int d = c + 1; d < M; ++d)
                    out.push_back((1u << (M - 1 - a)) | (1u << (M - 1 - b)) | (1u << (M - 1 - c)) |
                                  (1u << (M - 1 - d)));
    return out;
}

// SpMM work items from the value row pointers, on the device: the pieces of
// every row, sorted by length, and where each starts in the value stream
// (pbase, pdst).  At most cap pieces.
struct PieceBufs {
    DBuf<int32_t> np, slot0, pbase, id, order, len, beg, pdst, cnt;
    DBuf<uint8_t> gap;
    DBuf<uint64_t> key, key2;
    DBuf<int2> info;
};

static int build_items(vnm_packed *p, const int32_t *vrp, int64_t values, PieceBufs &P) {
    hipStream_t st = p->ctx->stream;
    const int R = p->nrows;
    // a row of at most ITEM values is one piece, and the others' chunks hold
    // ITEM values but for one per row
    const int cap = (int)(R + values / ITEM + 1);
    int rc;
    if ((rc = p->item.alloc(cap)) || (rc = p->fix.alloc(R)) || (rc = P.np.alloc(R + 1)) || (rc = P.pbase.alloc(R + 1)) ||
        (rc = P.slot0.alloc(R)) || (rc = P.gap.alloc(R)) || (rc = P.cnt.alloc(4)) || (rc = P.key.alloc(cap)) ||
        (rc = P.key2.alloc(cap)) || (rc = P.id.alloc(cap)) || (rc = P.order.alloc(cap)) || (rc = P.info.alloc(cap)) ||
        (rc = P.len.alloc(cap)) || (rc = P.beg.alloc(cap)) || (rc = P.pdst.alloc(cap)))
        return rc;
    VNM_HIP_TRY(hipMemsetAsync(P.cnt.p, 0, 16, st));
    hipLaunchKernelGGL(k_row_pieces, dim3(grid_of((int64_t)R + 1, 256)), dim3(256), 0, st, vrp, R, P.np.p, P.slot0.p,
                       P.gap.p, P.cnt.p, p->fix.p);
    if ((rc = scan_excl_i32(P.np.p, P.pbase.p, R + 1, st))) return rc;
    hipLaunchKernelGGL(k_pieces, dim3(grid_of(R, 256)), dim3(256), 0, st, vrp, R, P.pbase.p, P.slot0.p, P.gap.p, cap,
                       P.key.p, P.id.p, P.info.p);
    if ((rc = sort_pairs_u64_i32(P.key.p, P.key2.p, P.id.p, P.order.p, cap, key_range(0, 7), st))) return rc;
    hipLaunchKernelGGL(k_piece_lens, dim3(grid_of(cap, 256)), dim3(256), 0, st, P.order.p, P.info.p, cap, P.len.p);
    if ((rc = scan_excl_i32(P.len.p, P.beg.p, cap, st))) return rc;
    hipLaunchKernelGGL(k_items, dim3(grid_of(cap, 256)), dim3(256), 0, st, P.pbase.p + R, P.order.p, P.info.p, P.beg.p,
                       P.pdst.p, p->item.p);
    p->ctx->launches += 4;
    VNM_LAUNCH_CHECK("pack items");
    return VNM_OK;
}

int pack(vnm_graph *g, int V, int dtype, int dense_min, vnm_packed **out, int64_t *retained_only) {
    const int M = g->M;
    if (dense_min < 0 || (dense_min > 0 && (dtype != VNM_DT_BF16 || V % 16 != 0)))
        return set_error(VNM_E_ARG, "the sparse-MFMA part needs BF16 values and V a multiple of 16 "
                                    "(dense_min %d, dtype %d, V %d)", dense_min, dtype, V);
    if (V <= 0 || V > 256) return set_error(VNM_E_ARG, "V must be in [1, 256] (got %d)", V);
    if (M != 4 && M != 8 && M != 16) return set_error(VNM_E_ARG, "M must be 4, 8 or 16");
    if (dtype < VNM_DT_F32 || dtype > VNM_DT_FP8) return set_error(VNM_E_ARG, "bad dtype %d", dtype);
    if (g->col_overflow)
        return set_error(VNM_E_ARG, "entries lie past the padded column count after a relabel of a matrix "
                                    "with fewer columns than rows");
    hipStream_t st = g->ctx->stream;
    const int R = g->nrows;
    const int nseg = (g->ncols + M - 1) / M;
    const int nblk = (R + V - 1) / V;
    const int64_t nnz = g->nnz;
    const size_t e1 = std::max<int64_t>(nnz, 1);
    int rc;
    DBuf<uint64_t> keys, keys2, bkey, bkey2;
    DBuf<int32_t> idx, idx2, head, excl, rstart, rlen, rid, rid2, bhead, bexcl, blk_first, run_blk,
        nkeep, rcnt, sel_runs, cnt;
    DBuf<uint32_t> bits, blk_mask, absmax, dsubs;
    DBuf<float> kv;
    DBuf<uint8_t> kidx, flag;
    DBuf<unsigned long long> dret;
    DBuf<int32_t> longb, nlong;
    if ((rc = keys.alloc(e1)) || (rc = keys2.alloc(e1)) || (rc = idx.alloc(e1)) ||
        (rc = idx2.alloc(e1)) || (rc = head.alloc(e1)) || (rc = excl.alloc(e1)) ||
        (rc = dret.alloc(1)) || (rc = cnt.alloc(4)))
        return rc;
    const int gb = grid_of(nnz, 256);
    hipLaunchKernelGGL(k_nz_keys, dim3(gb), dim3(256), 0, st, g->row.p, g->col.p, g->val.p, nnz,
                       nseg * M, keys.p, idx.p);
    // rows are below R and columns below nseg * M; dropped entries' all-ones
    // keys sort last
    if ((rc = sort_pairs_u64_i32(keys.p, keys2.p, idx.p, idx2.p, nnz,
                                 key_halves(bits_for((int64_t)nseg * M - 1), bits_for(R)), st)))
        return rc;
    // the kept entries and their runs, counted on the device: one host read (a
    // binary search for the first all-ones key read the host 20 times, 0.3 ms)
    int64_t nz = 0;
    int U = 0;
    if (nnz > 0) {
        VNM_HIP_TRY(hipMemsetAsync(cnt.p, 0, 16, st));
        hipLaunchKernelGGL(k_pk_heads, dim3(gb), dim3(256), 0, st, keys2.p, nnz, M, head.p, cnt.p);
        if ((rc = scan_excl_i32(head.p, excl.p, nnz, st))) return rc;
        hipLaunchKernelGGL(k_pk_total, dim3(1), dim3(1), 0, st, excl.p, head.p, nnz, cnt.p + 1);
        int32_t h[2];
        VNM_HIP_TRY(hipMemcpyAsync(h, cnt.p, 8, hipMemcpyDeviceToHost, st));
        VNM_HIP_TRY(hipStreamSynchronize(st));
        nz = h[0];
        U = h[1];
    }
    const size_t u1 = std::max(U, 1);
    if ((rc = bits.alloc(u1)) || (rc = rstart.alloc(u1)) || (rc = rlen.alloc(u1)) ||
        (rc = bkey.alloc(u1)) || (rc = bkey2.alloc(u1)) || (rc = rid.alloc(u1)) ||
        (rc = rid2.alloc(u1)) || (rc = bhead.alloc(u1)) || (rc = bexcl.alloc(u1)) ||
        (rc = run_blk.alloc(u1)) || (rc = nkeep.alloc(u1)) || (rc = kv.alloc(2 * u1)) ||
        (rc = kidx.alloc(u1)) || (rc = flag.alloc(u1)) || (rc = sel_runs.alloc(u1)) ||
        (rc = rcnt.alloc(R + 1)))
        return rc;
    int nb = 0;
    std::vector<uint32_t> subs = subsets4(M);
    if ((rc = dsubs.alloc(subs.size()))) return rc;
    VNM_HIP_TRY(hipMemcpyAsync(dsubs.p, subs.data(), subs.size() * 4, hipMemcpyHostToDevice, st));
    VNM_HIP_TRY(hipMemsetAsync(dret.p, 0, 8, st));
    if (U > 0) {
        VNM_HIP_TRY(hipMemsetAsync(bits.p, 0, (size_t)U * 4, st));
        VNM_HIP_TRY(hipMemsetAsync(rlen.p, 0, (size_t)U * 4, st));
        hipLaunchKernelGGL(k_pk_runs, dim3(grid_of(nz, 256)), dim3(256), 0, st, keys2.p, head.p,
                           excl.p, nz, M, bits.p, rstart.p, rlen.p, bkey.p, rid.p);
        if ((rc = sort_pairs_u64_i32(bkey.p, bkey2.p, rid.p, rid2.p, U,
                                     key_halves(bits_for(R - 1), bits_for(nseg - 1)), st)))
            return rc;
        hipLaunchKernelGGL(k_blk_heads, dim3(grid_of(U, 256)), dim3(256), 0, st, bkey2.p, U, V, bhead.p);
        if ((rc = scan_excl_i32(bhead.p, bexcl.p, U, st))) return rc;
        hipLaunchKernelGGL(k_pk_total, dim3(1), dim3(1), 0, st, bexcl.p, bhead.p, (int64_t)U, cnt.p + 2);
        VNM_HIP_TRY(hipMemcpyAsync(&nb, cnt.p + 2, 4, hipMemcpyDeviceToHost, st));
        VNM_HIP_TRY(hipStreamSynchronize(st));
    }
    vnm_packed *p = new vnm_packed();
    p->ctx = g->ctx;
    p->V = V; p->M = M; p->nrows = R; p->ncols = g->ncols; p->dtype = dtype; p->nblocks = nb;
    const size_t b1 = std::max(nb, 1);
    if ((rc = blk_first.alloc(b1)) || (rc = blk_mask.alloc(b1)) || (rc = absmax.alloc(b1)) ||
        (rc = p->blk_seg.alloc(b1)) || (rc = p->blk_sel.alloc(b1)) || (rc = p->blk_scale.alloc(b1))) {
        delete p;
        return rc;
    }
    if (nb > 0) {
        hipLaunchKernelGGL(k_blk_first, dim3(grid_of(U, 256)), dim3(256), 0, st, bhead.p, bexcl.p, U,
                           blk_first.p);
        // short blocks one per lane; the rest one per wave, from a list the
        // lane kernel fills (its length read on the device: no host wait)
        if ((rc = longb.alloc(b1)) || (rc = nlong.alloc(1))) {
            delete p;
            return rc;
        }
        VNM_HIP_TRY(hipMemsetAsync(nlong.p, 0, 4, st));
        hipLaunchKernelGGL(k_blk_select_lane, dim3(std::min(grid_of(nb, 256), 2048)), dim3(256), 0, st, bkey2.p, rid2.p, U, nb,
                           M, bits.p, dsubs.p, (int)subs.size(), blk_first.p, p->blk_seg.p, p->blk_sel.p,
                           blk_mask.p, run_blk.p, dret.p, longb.p, nlong.p);
        hipLaunchKernelGGL(k_blk_select, dim3(std::min((nb + 3) / 4, 4096)), dim3(256), 0, st, bkey2.p, rid2.p,
                           U, nb, M, bits.p, dsubs.p, (int)subs.size(), blk_first.p, p->blk_seg.p,
                           p->blk_sel.p, blk_mask.p, run_blk.p, dret.p, longb.p, nlong.p);
        VNM_HIP_TRY(hipMemsetAsync(absmax.p, 0, (size_t)nb * 4, st));
        hipLaunchKernelGGL(k_run_keep, dim3(grid_of(U, 256)), dim3(256), 0, st, keys2.p, idx2.p,
                           g->val.p, U, M, rstart.p, rlen.p, run_blk.p, blk_mask.p, kv.p, kidx.p,
                           nkeep.p, absmax.p);
        hipLaunchKernelGGL(k_scales, dim3(grid_of(nb, 256)), dim3(256), 0, st, absmax.p, nb,
                           dtype == VNM_DT_FP8, p->blk_scale.p);
    }
    unsigned long long ret = 0;
    VNM_HIP_TRY(hipMemcpyAsync(&ret, dret.p, 8, hipMemcpyDeviceToHost, st));
    VNM_HIP_TRY(hipStreamSynchronize(st));
    p->retained = (int64_t)ret;
    VNM_LAUNCH_CHECK("pack select");
    if (retained_only) {
        *retained_only = p->retained;
        delete p;
        return VNM_OK;
    }
    // dense blocks to the sparse-MFMA part
    DBuf<int32_t> dmap;
    if (dense_min > 0 && nb > 0 &&
        (rc = build_dense(p, dense_min, U, nb, nblk, run_blk.p, nkeep.p, blk_first.p, bkey2.p, keys2.p, rstart.p,
                          kv.p, kidx.p, dmap))) {
        delete p;
        return rc;
    }
    // row entries (runs of the other blocks that keep something), row-major
    VNM_HIP_TRY(hipMemsetAsync(rcnt.p, 0, (size_t)(R + 1) * 4, st));
    int E = 0;
    if (U > 0) {
        hipLaunchKernelGGL(k_row_counts, dim3(grid_of(U, 256)), dim3(256), 0, st, keys2.p, rstart.p,
                           nkeep.p, run_blk.p, p->ngroups > 0 ? dmap.p : nullptr, U, rcnt.p, flag.p);
        hipLaunchKernelGGL(k_iota_i, dim3(grid_of(U, 256)), dim3(256), 0, st, rid.p, U);
        if ((rc = select_flagged_i32(rid.p, flag.p, sel_runs.p, cnt.p, U, st))) { delete p; return rc; }
        VNM_HIP_TRY(hipMemcpyAsync(&E, cnt.p, 4, hipMemcpyDeviceToHost, st));
        VNM_HIP_TRY(hipStreamSynchronize(st));
    }
    p->nent = E;
    const int vs = dtype == VNM_DT_F32 ? 4 : dtype == VNM_DT_FP8 ? 1 : 2;
    if ((rc = p->rowptr.alloc(R + 1)) || (rc = p->ent_col.alloc(std::max(E, 1))) ||
        (rc = p->ent_blk.alloc(dtype == VNM_DT_FP8 ? std::max(E, 1) : 1)) ||
        (rc = p->ent_row.alloc(std::max(E, 1))) ||
        (rc = p->ent_idx.alloc(std::max(E, 1))) ||
        (rc = p->ent_val.alloc((size_t)std::max(E, 1) * 2 * vs))) {
        delete p;
        return rc;
    }
    if ((rc = scan_excl_i32(rcnt.p, p->rowptr.p, R + 1, st))) { delete p; return rc; }
    if (E > 0)
        hipLaunchKernelGGL(k_emit, dim3(grid_of(E, 256)), dim3(256), 0, st, sel_runs.p, E, run_blk.p,
                           keys2.p, rstart.p, kv.p, kidx.p, p->blk_scale.p, p->blk_seg.p, p->blk_sel.p,
                           M, dtype, p->ent_row.p, p->ent_col.p, p->ent_blk.p, p->ent_idx.p, p->ent_val.p);
    g->ctx->launches += 17;
    VNM_LAUNCH_CHECK("pack emit");
    // the value stream and its row pointers
    DBuf<int32_t> nv, voff, vrp;
    if ((rc = nv.alloc((size_t)E + 1)) || (rc = voff.alloc((size_t)E + 1)) || (rc = vrp.alloc((size_t)R + 1))) {
        delete p;
        return rc;
    }
    hipLaunchKernelGGL(k_val_counts, dim3(grid_of((int64_t)E + 1, 256)), dim3(256), 0, st, p->ent_idx.p, E, nv.p);
    if ((rc = scan_excl_i32(nv.p, voff.p, (int64_t)E + 1, st))) { delete p; return rc; }
    hipLaunchKernelGGL(k_vrowptr, dim3(grid_of((int64_t)R + 1, 256)), dim3(256), 0, st, p->rowptr.p, voff.p, R,
                       vrp.p);
    // the most values the row entries hold: two each, and every kept value is an
    // entry of its own.  (The retained count is no bound: it counts positions, and a
    // relabel that is not one-to-one leaves a position's entries side by side, of
    // which a row entry keeps two.)
    const int64_t values = std::min<int64_t>(nz, 2 * (int64_t)E);
    PieceBufs P;
    if ((rc = p->vrec.alloc(std::max<int64_t>(values, 1))) || (rc = build_items(p, vrp.p, values, P))) {
        delete p;
        return rc;
    }
    if (E > 0)
        hipLaunchKernelGGL(k_values, dim3(grid_of(E, 256)), dim3(256), 0, st, E, M, dtype, voff.p,
                           Pieces{vrp.p, P.pbase.p, P.pdst.p}, p->ent_row.p, p->ent_col.p, p->ent_idx.p,
                           p->ent_val.p, p->ent_blk.p, p->blk_scale.p, p->vrec.p);
    g->ctx->launches += 4;
    VNM_LAUNCH_CHECK("pack values");
    int32_t cn[3], np = 0, nval = 0;
    VNM_HIP_TRY(hipMemcpyAsync(cn, P.cnt.p, 12, hipMemcpyDeviceToHost, st));
    VNM_HIP_TRY(hipMemcpyAsync(&np, P.pbase.p + R, 4, hipMemcpyDeviceToHost, st));
    VNM_HIP_TRY(hipMemcpyAsync(&nval, voff.p + E, 4, hipMemcpyDeviceToHost, st));
    VNM_HIP_TRY(hipStreamSynchronize(st));  // the scratch is freed on return
    p->nval = nval;
    p->nitems = np;
    p->nslots = cn[0];
    p->nhub = cn[1];
    p->nfix = cn[1] + cn[2];
    *out = p;
    return VNM_OK;
}

// Rows of n floats of SpMM scratch: the partial-sum slots of rows cut into
// chunks, then the dense units' slots (V rows each).
size_t scratch_rows(const vnm_packed *p) { return (size_t)p->nslots + (size_t)p->ndslots * p->V; }

// Partial-sum slots for n output columns, grown on demand.
int ensure_part(vnm_packed *p, int n) {
    const size_t need = std::max<size_t>(scratch_rows(p) * n, 1);
    if (p->part.n >= need) return VNM_OK;
    VNM_HIP_TRY(hipStreamSynchronize(p->ctx->stream));  // the old buffer may be in use
    return p->part.alloc(need);
}

int bsize_of(int bt) { return bt == VNM_DT_F32 ? 4 : bt == VNM_DT_BF16 ? 2 : 1; }

// Column tiles of 64 * vec values usable for (bt, n): a tile is 128 to 1,024
// bytes of a B row (8 to 64 lanes of 16 bytes) and divides n; FP8 rows of an odd
// number of 64-column groups, which have no such tile, take 64-byte ones (vec 1).
bool vec_ok(int bt, int n, int vec) {
    if (vec != 1 && vec != 2 && vec != 4 && vec != 8 && vec != 16) return false;
    const int bytes = vec * bsize_of(bt);
    return (bytes >= 2 || n % 128 != 0) && bytes <= 16 && n % (64 * vec) == 0;
}

// The tile taken unless the caller fixes one: 256 bytes where they divide the
// row, else 128; wider where that leaves more than 8 tiles, which no longer have
// XCDs of their own.  With 8 tiles or fewer, 256 and 512 bytes are within 3 % of
// each other, 128 up to 15 % slower (twice the item and value reads per byte),
// 1,024 20-30 % (no slice of B stays with an XCD): us at 128 / 256 / 512 / 1,024
// bytes, R-MAT 65,536 n = 256 FP32 - / 76.3 / 76.4 / 98.7, BF16 54.4 / 49.0 / 52.5 /
// -; R-MAT 131,072 n = 128 BF16 68.2 / 69.9.  Past 8 tiles of 256 bytes, at 256 /
// 512 / 1,024 bytes: FP32 n = 1,024 (16 / 8 / 4 tiles) R-MAT 65,536 562 / 340 / 389,
// ER 100,000 degree 10 582 / 598 / 607, 4,096 rows of 200 values 356 / 139 / 143; n =
// 2,048 R-MAT 1,037 / 1,031 / 667.  Where the tile count does not divide 8 (n = 384:
// 6 / 3 tiles, n = 768: 12 / 6 / 3), every XCD reads all of B and the widths are within
// 10 % of each other: R-MAT 137 / 137 and 320 / 317 / 324, ER 227 / 233 and 435 / 461 /
// 471, rows of 200 84 / 79 and 247 / 238 / 237.  (The width was timed per matrix before,
// with one item a wave: such rows, all of them cut and B in L2, took 77 us at n = 384, 75
// at 512, now 82, and 142 at 1,024; every other matrix here took longer than now.)
int default_vec(int bt, int n) {
    int v = 4 / bsize_of(bt);
    while (v > 1 && !vec_ok(bt, n, v)) v /= 2;
    while (n / (64 * v) > 8 && vec_ok(bt, n, 2 * v)) v *= 2;
    return v;
}

// default_vec for a matrix: the widest tile where B is far larger than the caches and
// few values lie in cut rows.  Without hubs nothing of B is read again soon, so slices of
// their own leave the XCDs nothing to keep, and a row of B in one piece is the better
// access to memory: ER 2^20 at 256 / 512 / 1,024 bytes, FP32 n = 256 (1 GiB of B) 1,707 /
// 1,636 / 1,583 us, n = 512 3,744 / 3,630 / 3,555; 2^18 (256 MiB) n = 256 331 / 340 / 337;
// but R-MAT 2^20 n = 256 2,353 / 2,748 / 3,124.
int shape_of(const vnm_packed *p, int bt, int n) {
    constexpr uint64_t FAR_B = 512ull << 20;
    int v = default_vec(bt, n);
    if ((uint64_t)p->ncols * n * bsize_of(bt) >= FAR_B && (int64_t)p->nslots * ITEM * 16 <= p->nval)
        while (vec_ok(bt, n, 2 * v)) v *= 2;
    return v;
}

// Items one wave walks: 64 lanes over the lanes of a tile.
int tile_items(int bt, int vec) {
    const int bytes = 64 * vec * bsize_of(bt);
    return bytes >= 128 ? 1024 / bytes : 8;
}

SpmmArgs packed_args(const vnm_packed *p, const void *B, int ldb, const float *bs, float *C, int ldc,
                     const float *bias, float *part, int pn) {
    SpmmArgs a;
    a.pieces = p->item.p;
    a.vrec = p->vrec.p;
    a.B = (const uint8_t *)B;
    a.b_scales = bs;
    a.C = C;
    a.part = part;
    a.bias = bias;
    a.items = p->nitems;
    a.ldb = ldb;
    a.ldc = ldc;
    a.pn = pn;
    a.b_rows = p->ncols;
    a.c_rows = p->nrows;
    a.dvb = p->ngroups > 0 ? p->dvb.p : nullptr;
    a.V = p->V;
    return a;
}

template <int BT, int LPR, int LB = 16>
static void launch_v(const SpmmArgs &args, int n, hipStream_t st) {
    const int T = n * bsize<BT>() / (LPR * LB);
    const int per_wg = 4 * (64 / LPR);  // items of a workgroup
    const int iwg = (args.items + per_wg - 1) / per_wg;
    int per_g;
    if (8 % T == 0) {
        const int gs = 8 / T;
        per_g = (iwg + gs - 1) / gs;
    } else {
        per_g = (iwg * T + 7) / 8;
    }
    if (args.bias || args.dvb)
        hipLaunchKernelGGL((k_spmm<BT, LPR, LB, true>), dim3(8 * per_g), dim3(256), 0, st, args, T, per_g);
    else
        hipLaunchKernelGGL((k_spmm<BT, LPR, LB, false>), dim3(8 * per_g), dim3(256), 0, st, args, T, per_g);
}

// The value stream carries FP32 weights, so the kernel depends on B's dtype
// and the tile width only.
static void launch_b(const SpmmArgs &args, int vec, int n, int bt, hipStream_t st) {
    if (bt == VNM_DT_F32) {
        if (vec == 4) launch_v<VNM_DT_F32, 64>(args, n, st);
        else if (vec == 2) launch_v<VNM_DT_F32, 32>(args, n, st);
        else launch_v<VNM_DT_F32, 16>(args, n, st);
    } else if (bt == VNM_DT_BF16) {
        if (vec == 8) launch_v<VNM_DT_BF16, 64>(args, n, st);
        else if (vec == 4) launch_v<VNM_DT_BF16, 32>(args, n, st);
        else if (vec == 2) launch_v<VNM_DT_BF16, 16>(args, n, st);
        else launch_v<VNM_DT_BF16, 8>(args, n, st);
    } else {
        if (vec == 16) launch_v<VNM_DT_FP8, 64>(args, n, st);
        else if (vec == 8) launch_v<VNM_DT_FP8, 32>(args, n, st);
        else if (vec == 4) launch_v<VNM_DT_FP8, 16>(args, n, st);
        else if (vec == 2) launch_v<VNM_DT_FP8, 8>(args, n, st);
        else launch_v<VNM_DT_FP8, 8, 8>(args, n, st);
    }
}

// One SpMM with `vec` values per lane and the partial-sum slots at `part`
// (nslots x n floats): the gather kernel, then the fix-up pass.
int spmm_run(vnm_packed *p, int vec, const void *B, int ldb, int n, int bt, const float *bs, float *C,
                    int ldc, const float *bias, float *part, bool timed) {
    hipStream_t st = p->ctx->stream;
    const SpmmArgs args = packed_args(p, B, ldb, bs, C, ldc, bias, part, n);
    // the dense blocks' 2:4 products first: the row-entry pass adds to them
    int rc = spmm_dense(p, (const uint16_t *)B, ldb, n, C, ldc, part + (size_t)p->nslots * n, st, timed);
    if (rc) return rc;
    if (p->nitems > 0) {
        KernelTimer kt(timed ? p->ctx : nullptr, "k_spmm");
        launch_b(args, vec, n, bt, st);
        kt.stop();
        p->ctx->launches++;
    }
    if (p->nfix > 0) {
        hipLaunchKernelGGL(k_spmm_fix, dim3((unsigned)((fix_waves(p->nfix, p->nhub, n) + 3) / 4)), dim3(256), 0, st,
                           p->fix.p, p->nhub, p->fix_rest(), p->nfix - p->nhub, part, n, n, C,
                           ldc, bias, args.dvb, p->V);
        p->ctx->launches++;
    }
    VNM_LAUNCH_CHECK("k_spmm");
    return VNM_OK;
}

// spmm_run with the packed matrix's own slots.
static int spmm_v(vnm_packed *p, int vec, const void *B, int ldb, int n, int bt, const float *bs, float *C,
                  int ldc, const float *bias, bool timed) {
    int rc = ensure_part(p, n);
    if (rc) return rc;
    return spmm_run(p, vec, B, ldb, n, bt, bs, C, ldc, bias, p->part.p, timed);
}

int shape_key(int bt, int n) { return (bt << 24) | n; }

int spmm_check(const vnm_packed *p, const void *B, int ldb, int n, int bt, const float *bs,
                      const float *C, int ldc) {
    if (!p || !B || !C || n <= 0 || n % 64 != 0 || ldb < n || ldc < n)
        return set_error(VNM_E_ARG, "spmm: n must be a positive multiple of 64 with ldb, ldc >= n");
    if (bt != VNM_DT_F32 && bt != VNM_DT_BF16 && bt != VNM_DT_FP8)
        return set_error(VNM_E_ARG, "spmm: B dtype must be F32, BF16 or FP8");
    if (bt == VNM_DT_FP8 && !bs) return set_error(VNM_E_ARG, "spmm: FP8 B needs per-128-row scales");
    // vector loads of up to 16 bytes of B, stores of up to 16 bytes of C
    if ((ldb * bsize_of(bt)) % 16 != 0 || (ldc % 4) != 0 || ((uintptr_t)B & 15) || ((uintptr_t)C & 15))
        return set_error(VNM_E_ARG, "spmm: B and C must be 16-byte aligned with rows of whole 16-byte "
                                    "units (ldb * sizeof(B value) and 4 * ldc multiples of 16)");
    if ((uint64_t)p->ncols * (uint64_t)ldb * (uint64_t)bsize_of(bt) > 0xFFFFFFFFull)
        return set_error(VNM_E_ARG, "spmm: B (ncols x ldb) must be smaller than 4 GiB");
    if (p->ngroups > 0 && bt != VNM_DT_BF16)
        return set_error(VNM_E_ARG, "spmm: a matrix packed with a sparse-MFMA part takes BF16 B");
    return VNM_OK;
}

int spmm(vnm_packed *p, const void *B, int ldb, int n, int bt, const float *bs, float *C, int ldc,
         const float *bias) {
    int rc = spmm_check(p, B, ldb, n, bt, bs, C, ldc);
    if (rc) return rc;
    // the shape stays with the packed matrix: vnm_spmm_get_shape reports it
    const int v = p->shapes.emplace(shape_key(bt, n), shape_of(p, bt, n)).first->second;
    return spmm_v(p, v, B, ldb, n, bt, bs, C, ldc, bias, true);
}

}  // namespace vnm

using namespace vnm;

extern "C" {

int vnm_retained_nnz(vnm_graph *g, int V, int N, int64_t *out) {
    if (!g || !out) return set_error(VNM_E_ARG, "null argument");
    PoolScope pool(g->ctx->pool);
    if (N != 2) return set_error(VNM_E_ARG, "the V:N:M format keeps N = 2 per row (got %d)", N);
    return pack(g, V, VNM_DT_F32, 0, nullptr, out);
}

int vnm_pack(vnm_graph *g, int V, int dtype, vnm_packed **out) {
    if (!g || !out) return set_error(VNM_E_ARG, "null argument");
    PoolScope pool(g->ctx->pool);
    return pack(g, V, dtype, 0, out, nullptr);
}

int vnm_pack_ex(vnm_graph *g, int V, int dtype, int dense_min, vnm_packed **out) {
    if (!g || !out) return set_error(VNM_E_ARG, "null argument");
    PoolScope pool(g->ctx->pool);
    return pack(g, V, dtype, dense_min, out, nullptr);
}

int vnm_packed_info_get(const vnm_packed *p, vnm_packed_info *info) {
    if (!p || !info) return set_error(VNM_E_ARG, "null argument");
    info->V = p->V;
    info->M = p->M;
    info->nrows = p->nrows;
    info->ncols = p->ncols;
    info->nblocks = p->nblocks;
    info->dtype = p->dtype;
    info->retained_nnz = p->retained;
    const int vs = p->dtype == VNM_DT_F32 ? 4 : p->dtype == VNM_DT_FP8 ? 1 : 2;
    const int blk = p->dtype == VNM_DT_FP8 ? 4 : 0;  // per-entry block index for the FP8 scale
    info->bytes = 4ll * (p->nrows + 1) + (int64_t)p->nent * (4 + 4 + 1 + 2 * vs + blk) +
                  (int64_t)p->nblocks * (4 + 2 + 4);
    // the SpMM's value stream: (B row, FP32 weight) per value
    info->bytes += (int64_t)p->nval * 8;
    // what k_spmm reads: the value stream and the item table
    info->spmm_bytes = (int64_t)p->nval * 8 + (int64_t)p->nitems * (int64_t)sizeof(Piece);
    info->items = p->nitems;
    info->slots = (int32_t)scratch_rows(p);
    info->dense_blocks = p->ndense;
    info->dense_chunks = p->nchunks;
    // the sparse-MFMA part reads per chunk its 64 column indices and per
    // 16-row slice 64 lanes x (16 value bytes + 4 position bytes)
    info->spmm_bytes += (int64_t)p->nchunks * (64 * 4 + (int64_t)(p->V / 16) * 64 * 20) + (int64_t)p->ngroups * 16;
    info->bytes += (int64_t)p->nchunks * (64 * 4 + (int64_t)(p->V / 16) * 64 * 20) + (int64_t)p->ngroups * 16 +
                   (p->ngroups ? (int64_t)((p->nrows + p->V - 1) / p->V) : 0);
    return VNM_OK;
}

void vnm_packed_destroy(vnm_packed *p) {
    if (!p) return;
    if (p->ctx && p->ctx->stream) (void)hipStreamSynchronize(p->ctx->stream);
    delete p;
}

int vnm_spmm(vnm_packed *p, const void *B, int ldb, int n, int b_dtype, const float *b_scales,
             float *C, int ldc) {
    PoolScope pool(p ? p->ctx->pool : nullptr);
    return spmm(p, B, ldb, n, b_dtype, b_scales, C, ldc, nullptr);
}

int vnm_spmm_set_shape(vnm_packed *p, int b_dtype, int n, int cols_per_lane) {
    if (!p) return set_error(VNM_E_ARG, "null argument");
    if (cols_per_lane == 0) {
        p->shapes.erase(shape_key(b_dtype, n));
        return VNM_OK;
    }
    if (!vec_ok(b_dtype, n, cols_per_lane))
        return set_error(VNM_E_ARG, "spmm: %d columns per lane do not fit n = %d for B dtype %d",
                         cols_per_lane, n, b_dtype);
    p->shapes[shape_key(b_dtype, n)] = cols_per_lane;
    return VNM_OK;
}

int vnm_spmm_get_shape(const vnm_packed *p, int b_dtype, int n, int32_t *cols_per_lane) {
    if (!p || !cols_per_lane) return set_error(VNM_E_ARG, "null argument");
    auto it = p->shapes.find(shape_key(b_dtype, n));
    *cols_per_lane = it == p->shapes.end() ? 0 : it->second;
    return VNM_OK;
}

}  // extern "C"
