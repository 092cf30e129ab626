// The packed V:N:M format and the SpMM device code shared by the single and
// batched SpMM kernels (pack.hip, batch.hip).  Format and kernel design are
// described in pack.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <cstring>
#include <type_traits>
#include <map>
#include <memory>

#include "graph.h"
#include "hip_common.h"

struct vnm_packed {
    vnm_ctx *ctx = nullptr;
    int32_t V = 0, M = 0, nrows = 0, ncols = 0, dtype = 0;
    int32_t nblocks = 0, nent = 0;
    int64_t retained = 0;
    vnm::DBuf<int32_t> rowptr, ent_row, ent_col, ent_blk, blk_seg;
    vnm::DBuf<uint8_t> ent_idx, ent_val;                   // values: 2 per entry, dtype-sized
    vnm::DBuf<uint16_t> blk_sel;
    vnm::DBuf<float> blk_scale;
    // the SpMM's value stream: every value of the row entries as (B row, FP32
    // weight), in the order of the work items -- pieces: whole rows of at most
    // ITEM values, and the ITEM-value chunks of longer rows, whose partial sums go
    // to slots -- which are sorted by length
    int32_t nval = 0;
    vnm::DBuf<uint2> vrec;
    int32_t nitems = 0, nslots = 0, nfix = 0, nhub = 0;
    vnm::DBuf<int4> item;                                  // vnm::Piece
    // rows the fix-up pass writes (empty or cut), {row, first slot, slots, 0}:
    // the nhub hub rows from the front, the other nfix - nhub at the end
    vnm::DBuf<int4> fix;
    const int4 *fix_rest() const { return fix.p + (fix.n - (size_t)(nfix - nhub)); }
    vnm::DBuf<float> part;                                 // nslots x n partial sums
    // 2:4 sparse-MFMA part (dense.hip): blocks keeping >= dense_min values
    int32_t dense_min = 0, ndense = 0, nchunks = 0, ngroups = 0, nmulti = 0, ndslots = 0;
    vnm::DBuf<int4> dgrp;                                  // units {V-row block, first chunk, chunks, slot or -1}
    vnm::DBuf<int4> dmulti;                                // {V-row block, first slot, slots, 0}
    vnm::DBuf<int32_t> dcol;                               // chunks x 64 B rows (-1: none)
    vnm::DBuf<uint32_t> dfrag;                             // chunks x V/16 x 64 lanes x 8 BF16
    vnm::DBuf<uint32_t> didx;                              // chunks x V/16 x 64 lanes: positions
    vnm::DBuf<uint8_t> dvb;                                // per V-row block: 1 = C holds a dense sum
    std::map<int, int> shapes;                             // (b dtype << 24 | n) -> values per lane
    vnm::DBuf<uint16_t> gcn_h;                             // X W of the last GCN layer (BF16)
};

namespace vnm {

constexpr int ITEM = 64;      // most values of a work item, and values of a long row's chunk
constexpr int SBLK = 8;       // gathers in flight per lane group of the SpMM
constexpr int GAP_MAX = 8;    // runs of rows without entries up to this long, after an uncut row,
                              // are written with that row; other such rows by the fix-up pass

// A work item of the SpMM: `len` values from `beg` on in the value stream,
// whose sum goes to row `row` of C (and `gap` rows without values after it get
// the bias or zero) or, with `slot` set, to partial-sum slot `row`.
struct Piece {
    int32_t beg, len, row;
    int16_t gap, slot;
};
static_assert(sizeof(Piece) == 16, "read as one int4");

// ------------------------------------------------------------ value codecs

// OCP FP8 E4M3 (bias 7, no infinities, 0x7F = NaN, max 448): round to
// nearest even, saturating to +-448.
__host__ __device__ inline uint8_t f32_to_e4m3(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    const uint8_t sign = (uint8_t)((u >> 24) & 0x80u);
    const uint32_t a = u & 0x7FFFFFFFu;
    if (a > 0x7F800000u) return (uint8_t)(sign | 0x7F);  // NaN
    float af;
    memcpy(&af, &a, 4);
    if (af >= 448.0f) return (uint8_t)(sign | 0x7E);      // saturate
    const int e = (int)(a >> 23) - 127;                    // unbiased exponent
    if (e < -6) {
        // subnormal range: value = m * 2^-9, m in [0, 7]
        float q = af * 512.0f;                             // exact scaling
        // round half to even
        float r = q - floorf(q);
        uint32_t m = (uint32_t)floorf(q);
        if (r > 0.5f || (r == 0.5f && (m & 1u))) m += 1;
        return (uint8_t)(sign | m);                        // m == 8 -> smallest normal 0x08
    }
    // normal: keep 3 mantissa bits, round half to even on the 20 dropped bits
    uint32_t mant = a & 0x7FFFFFu;
    uint32_t keep = mant >> 20, rest = mant & 0xFFFFFu;
    uint32_t exp8 = (uint32_t)(e + 7);
    if (rest > 0x80000u || (rest == 0x80000u && (keep & 1u))) {
        keep += 1;
        if (keep == 8) { keep = 0; exp8 += 1; }
    }
    uint32_t code = (exp8 << 3) | keep;
    if (code > 0x7E) code = 0x7E;
    return (uint8_t)(sign | code);
}

__host__ __device__ inline float e4m3_to_f32(uint8_t c) {
    const uint32_t s = c & 0x80u, e = (c >> 3) & 0xFu, m = c & 7u;
    float v;
    if (e == 0) v = (float)m * (1.0f / 512.0f);
    else if (e == 15 && m == 7) v = __builtin_nanf("");
    else {
        uint32_t u = ((e + 120u) << 23) | (m << 20);
        memcpy(&v, &u, 4);
    }
    return s ? -v : v;
}

// ------------------------------------------------------------ SpMM device code

template <int BT>
constexpr int bsize() { return BT == VNM_DT_F32 ? 4 : BT == VNM_DT_BF16 ? 2 : 1; }

typedef float f32x2_t __attribute__((ext_vector_type(2)));

// LB bytes of one B row, as one lane gathers them: NV = LB / sizeof(value)
// values.
template <int LB>
struct BRaw {
    uint32_t w[LB / 4];
};

// acc += w * (decoded raw)
template <int BT, int LB>
__device__ __forceinline__ void fma_raw(float (&acc)[LB / bsize<BT>()], float w, const BRaw<LB> &raw) {
    constexpr int NV = LB / bsize<BT>();
    if constexpr (BT == VNM_DT_F32) {
#pragma unroll
        for (int i = 0; i < NV; ++i) acc[i] = fmaf(w, __uint_as_float(raw.w[i]), acc[i]);
    } else if constexpr (BT == VNM_DT_BF16) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const uint32_t x = raw.w[i / 2];
            acc[i] = fmaf(w, __uint_as_float((i & 1) ? (x & 0xFFFF0000u) : (x << 16)), acc[i]);
        }
    } else {
        // OCP e4m3 through the gfx950 conversion, two values per call
#pragma unroll
        for (int i = 0; i < NV; i += 4) {
            const uint32_t x = raw.w[i / 4];
            const f32x2_t lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)x, false);
            const f32x2_t hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)x, true);
            acc[i] = fmaf(w, lo.x, acc[i]);
            acc[i + 1] = fmaf(w, lo.y, acc[i + 1]);
            acc[i + 2] = fmaf(w, hi.x, acc[i + 2]);
            acc[i + 3] = fmaf(w, hi.y, acc[i + 3]);
        }
    }
}

// A lane's NB runs of 4 columns, RUN columns apart: partial sums, rows of C
// (nontemporal, so that the output stream does not push the gathered B rows out
// of L2), and values added to them.
template <int NB, int RUN>
__device__ __forceinline__ void store_runs(float *__restrict__ p, const float (&v)[4 * NB]) {
#pragma unroll
    for (int i = 0; i < NB; ++i)
        *(float4 *)(p + i * RUN) = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
}

template <int NB, int RUN>
__device__ __forceinline__ void store_runs_nt(float *__restrict__ p, const float (&v)[4 * NB]) {
    typedef float f4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int i = 0; i < NB; ++i)
        __builtin_nontemporal_store(f4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]}, (f4 *)(p + i * RUN));
}

template <int NB, int RUN>
__device__ __forceinline__ void add_runs(float (&v)[4 * NB], const float *__restrict__ p) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const float4 x = *(const float4 *)(p + i * RUN);
        v[4 * i] += x.x; v[4 * i + 1] += x.y; v[4 * i + 2] += x.z; v[4 * i + 3] += x.w;
    }
}

// One packed matrix as the SpMM kernels see it.
struct SpmmArgs {
    const int4 *pieces;  // the work items (Piece)
    const uint2 *vrec;   // the value stream: {B row, weight}
    const uint8_t *B;
    const float *b_scales;
    float *C;
    float *part;        // nslots x pn partial sums of cut rows
    const float *bias;  // nullptr or n floats added to every output row
    const uint8_t *dvb; // nullptr, or per V-row block 1 when C already holds the block's dense sums
    int items, ldb, ldc, pn;  // pn = n, the columns of the product
    int b_rows;         // rows of B (columns of A); b_rows * ldb * sizeof(value) < 2^32
    int c_rows;         // rows of C (of A)
    int V;
};

// LB bytes of one B row for this lane.
template <int LB>
__device__ __forceinline__ BRaw<LB> load_row(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
    BRaw<LB> r;
    if constexpr (LB == 16) {
        const auto t = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, 0);
        r.w[0] = t[0]; r.w[1] = t[1]; r.w[2] = t[2]; r.w[3] = t[3];
    } else {
        const auto t = __builtin_amdgcn_raw_buffer_load_b64(rs, (int)off, 0, 0);
        r.w[0] = t[0]; r.w[1] = t[1];
    }
    return r;
}

// Value i of the value array as a float (per lane).
template <int DT>
__device__ __forceinline__ float load_aval(const uint8_t *__restrict__ p, int i) {
    if constexpr (DT == VNM_DT_F32) return ((const float *)p)[i];
    else if constexpr (DT == VNM_DT_BF16) return bf16_to_f32(((const uint16_t *)p)[i]);
    else if constexpr (DT == VNM_DT_F16) return __half2float(((const __half *)p)[i]);
    else return e4m3_to_f32(p[i]);
}

// Value J (< SBLK) of this lane's group, from the lane that holds it: lanes
// J and 8 + J of every row of 16 hold value J of their group.
template <int LPR, int J>
__device__ __forceinline__ uint32_t group_bcast(uint32_t v) {
    constexpr int NEWBCAST = 0x150;  // DPP row_newbcast: one lane of a row of 16 to the whole row
    if constexpr (LPR >= 16) {
        return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, NEWBCAST + J, 0xF, 0xF, true);
    } else {
        // the two groups of a row of 16 one after the other (bank masks)
        const int lo = __builtin_amdgcn_update_dpp((int)v, (int)v, NEWBCAST + J, 0xF, 0x3, false);
        return (uint32_t)__builtin_amdgcn_update_dpp(lo, (int)v, NEWBCAST + 8 + J, 0xF, 0xC, false);
    }
}

// f(integral_constant<int, J>) for J = 0 .. SBLK - 1.
template <int J = 0, typename F>
__device__ __forceinline__ void each_step(F &&f) {
    if constexpr (J < SBLK) {
        f(std::integral_constant<int, J>());
        each_step<J + 1>(f);
    }
}

// C = A_vnm B for 64 / LPR consecutive work items from item0 on and column
// tile `tile` (LPR * LB bytes of every B row), one wave: LPR lanes per item, LB
// bytes of a B row per lane.
//
// What bounds it is the gather: every kept value reads one B row's tile
// through the vector L1, and a CU's L1 takes one 64-byte request a cycle, so
// loads of 16 bytes per lane are the cheapest per byte.  Groups of lanes that
// walk items of their own keep 16-byte loads whatever the tile width: one load
// instruction fetches 64 / LPR tiles, one per item, and a tile can be as
// narrow as 128 bytes of BF16 or FP8.  (One item per wave, with the B row's
// offset a scalar, read 2 to 8 bytes per lane there.)
//
// Items are sorted by length, so the groups of a wave walk items of one length
// (but where it changes) and end together.  Lane J of a group reads value J of a
// block of SBLK: its B row's offset and weight reach the group's lanes by DPP.  The
// gathers of a block are all in flight before its FMAs; the next block's values
// are loaded before them.  Every output value is one fixed sequence of FP32
// operations (the row's values in order; the fix-up pass adds a cut row's
// chunks in order), whatever the launch shape.
//
// EXTRA: there is a bias, or rows that hold a dense part's sum.  turn: 64 NV
// floats of LDS of the wave's own (NV = values of a lane) when NV > 4.
template <int BT, int LPR, int LB, bool EXTRA>
__device__ __forceinline__ void spmm_items(const SpmmArgs &a, int item0, int tile, float *turn) {
    constexpr int SB = bsize<BT>(), NV = LB / SB;
    const int lane = threadIdx.x & 63;
    const int item = item0 + lane / LPR;
    int4 pc = make_int4(0, 0, 0, 0);
    if (item < a.items) pc = a.pieces[item];
    const int len = pc.y;
    const uint32_t rowb = (uint32_t)a.ldb * SB;
    const uint32_t bytes = (uint32_t)(a.b_rows - 1) * rowb + (uint32_t)a.pn * SB;  // B up to its last value
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)a.B, 0, (int)bytes, 0x00020000);
    const uint32_t voff = (uint32_t)(tile * LPR + lane % LPR) * LB;
    // a lane without a value gathers from past B's end, where a buffer load
    // reads nothing (or, when B ends within a row of 4 GiB, from some row of
    // B), and only its own group's sum, which is complete, is kept below
    const uint32_t none = 0xFFFFFF00u - rowb;
    const uint2 *__restrict__ vals = a.vrec + pc.x;
    const int mine = lane % SBLK;
    float acc[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) acc[i] = 0.f;
    uint2 v = mine < len ? vals[mine] : make_uint2(0u, 0u);
    // one block of values from k0 on: all SBLK of them, or (LAST) the first
    // `m` only, m uniform over the wave
    auto block = [&](auto LAST, int k0, int m) {
        constexpr bool last = decltype(LAST)::value;
        const bool live = k0 + mine < len;
        uint32_t off = live ? v.x * rowb : none, w = v.y;
        if constexpr (BT == VNM_DT_FP8) w = __float_as_uint(__uint_as_float(w) * a.b_scales[v.x >> 7]);
        if (!last && k0 + SBLK + mine < len) v = vals[k0 + SBLK + mine];
        BRaw<LB> raw[SBLK];
        each_step([&](auto J) {
            constexpr int j = decltype(J)::value;
            if (!last || j < m) raw[j] = load_row<LB>(rs, voff + group_bcast<LPR, j>(off));
        });
        if (!last && k0 + SBLK <= len) {
            each_step([&](auto J) {
                constexpr int j = decltype(J)::value;
                fma_raw<BT, LB>(acc, __uint_as_float(group_bcast<LPR, j>(w)), raw[j]);
            });
        } else {
            each_step([&](auto J) {
                constexpr int j = decltype(J)::value;
                if (last && j >= m) return;
                const float wj = __uint_as_float(group_bcast<LPR, j>(w));
                if (k0 + j < len) fma_raw<BT, LB>(acc, wj, raw[j]);
            });
        }
    };
    // items come in descending length, so the wave's longest is its first
    const int mlen = __builtin_amdgcn_readfirstlane(len);
    int k0 = 0;
    for (; k0 + SBLK <= mlen; k0 += SBLK) block(std::false_type(), k0, SBLK);
    if (k0 < mlen) block(std::true_type(), k0, mlen - k0);
    // lane l of a group of BF16 or FP8 lanes holds columns NV l .. NV l + NV - 1
    // of the tile: through LDS to 4 l .. 4 l + 3 of each run of 4 LPR columns, so
    // that a store writes whole lines (partial ones cost FP8 4 times the requests)
    constexpr int NB = NV / 4;
    const int l = lane % LPR;
    if constexpr (NB > 1) {
        float *t = turn + (lane - l) * NV;
#pragma unroll
        for (int i = 0; i < NV; i += 4) *(float4 *)(t + l * NV + i) = make_float4(acc[i], acc[i + 1], acc[i + 2], acc[i + 3]);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const float4 x = *(const float4 *)(t + i * 4 * LPR + 4 * l);
            acc[4 * i] = x.x; acc[4 * i + 1] = x.y; acc[4 * i + 2] = x.z; acc[4 * i + 3] = x.w;
        }
    }
    if (len == 0) return;
    const int c0 = tile * LPR * NV + 4 * l;  // first column of run 0
    constexpr int RUN = 4 * LPR;
    if (pc.w >> 16) {
        store_runs<NB, RUN>(a.part + (size_t)pc.z * a.pn + c0, acc);
        return;
    }
    float *cp = a.C + (size_t)pc.z * a.ldc + c0;
    const int gap = pc.w & 0xFFFF;
    for (int i = 0; i <= gap; ++i) {
        if constexpr (EXTRA) {
            // rows whose V-row block has a dense part hold its sum already
            // (written by the dense kernel): row sums add to it
            if (a.dvb != nullptr && a.dvb[(pc.z + i) / a.V] != 0) add_runs<NB, RUN>(acc, cp);
            if (a.bias) add_runs<NB, RUN>(acc, a.bias + c0);
        }
        store_runs_nt<NB, RUN>(cp, acc);
#pragma unroll
        for (int q = 0; q < NV; ++q) acc[q] = 0.f;
        cp += a.ldc;
    }
}

// Fix-up of some columns of one listed row (a wave, W columns per lane from
// c0 + W lane on): the sum of its `ns` partial-sum slots from `s0` on, in slot
// order, plus the row's dense sum when it has one, plus the bias.  What bounds it
// is the chain of round trips: FB slots' loads go out before they are added, in
// order.  Most cut rows have a few slots: those and the rows without values
// (ns = 0) take 4 columns per lane and 8 slots at a time; the hub rows, listed
// first, 1 column per lane and 32 slots.
constexpr int HUB_SLOTS = 16;  // a row of more slots is a hub row
template <int W, int FB>
__device__ __forceinline__ void fix_row(float *__restrict__ crow, const float *__restrict__ part, int pn, int s0,
                                        int ns, int c0, int n, const float *__restrict__ bias, bool dense) {
    typedef float vec __attribute__((ext_vector_type(W)));
    const int c = c0 + W * (threadIdx.x & 63);
    if (c >= n) return;
    vec acc = (vec)0.f;
    const float *pc = part + (size_t)s0 * pn + c;
    for (int j0 = 0; j0 < ns; j0 += FB) {
        vec v[FB];
#pragma unroll
        for (int j = 0; j < FB; ++j) v[j] = j0 + j < ns ? *(const vec *)(pc + (size_t)(j0 + j) * pn) : (vec)0.f;
#pragma unroll
        for (int j = 0; j < FB; ++j)
            if (j0 + j < ns) acc += v[j];
    }
    if (dense) acc += *(const vec *)(crow + c);  // written by the dense kernel
    if (bias) acc += *(const vec *)(bias + c);
    *(vec *)(crow + c) = acc;
}

// Waves of a fix-up pass over nfix rows, the first nhub of them hub rows, and
// wave w's row and first column.
__host__ __device__ inline int64_t fix_waves(int nfix, int nhub, int n) {
    return (int64_t)nhub * (n / 64) + (int64_t)(nfix - nhub) * ((n + 255) / 256);
}

// ------------------------------------------------------------ host helpers (pack.hip)

int ensure_part(vnm_packed *p, int n);
size_t scratch_rows(const vnm_packed *p);
int bsize_of(int bt);
bool vec_ok(int bt, int n, int vec);
int default_vec(int bt, int n);
int shape_of(const vnm_packed *p, int bt, int n);
int tile_items(int bt, int vec);
SpmmArgs packed_args(const vnm_packed *p, const void *B, int ldb, const float *bs, float *C, int ldc,
                     const float *bias, float *part, int pn);
int spmm(vnm_packed *p, const void *B, int ldb, int n, int bt, const float *bs, float *C, int ldc,
         const float *bias);
int spmm_check(const vnm_packed *p, const void *B, int ldb, int n, int bt, const float *bs, const float *C, int ldc);
int spmm_run(vnm_packed *p, int vec, const void *B, int ldb, int n, int bt, const float *bs, float *C, int ldc,
             const float *bias, float *part, bool timed);
int shape_key(int bt, int n);
int build_dense(vnm_packed *p, int dense_min, int U, int nb, int nblk, const int32_t *run_blk,
                const int32_t *nkeep, const int32_t *blk_first, const uint64_t *bkey, const uint64_t *keys,
                const int32_t *rstart, const float *kv, const uint8_t *kidx, DBuf<int32_t> &dmap);
int spmm_dense(vnm_packed *p, const uint16_t *B, int ldb, int n, float *C, int ldc, float *dslot, hipStream_t st,
               bool timed);

}  // namespace vnm
