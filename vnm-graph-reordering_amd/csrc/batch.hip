// Batched V:N:M SpMM and the GCN aggregation layer (gfx950).
//
// Batch: many packed matrices of uneven size multiplied in one persistent
// launch.  The work units (the items of one wave x one column tile) of all
// matrices form one list (prefix offsets per matrix); a fixed grid of 8
// workgroups per CU walks it, each XCD taking a contiguous range so neighbouring
// units of one matrix share that XCD's L2.  A device table holds every matrix's
// pointers (SpmmArgs).  The batch is captured once as a HIP graph of two kernels
// -- the SpMM and the fix-up pass (rows cut into chunks, whose partial sums are
// added in chunk order) -- replayed by vnm_batch_run.  24 Chung-Lu graphs of 1,000
// to 40,000 nodes, BF16, n = 256: 338 us with the single SpMM's earlier kernel
// and a width timed per batch, 275 now.
//
// GCN layer (the consumer of gnn/single/pyg_gcn.py:41-74, aggr='add'):
// Y = A_vnm (X W) + bias.  X W runs on MFMA (BF16 inputs, FP32 accumulation,
// BF16 result into a workspace kept with the packed matrix), then the SpMM
// with the bias folded into its row stores and fix-up pass.
#include "graph.h"
#include "hip_common.h"
#include "packed.h"

#include <algorithm>
#include <chrono>
#include <vector>

struct vnm_batch {
    vnm_ctx *ctx = nullptr;
    int count = 0, n = 0, bt = 0, at = 0, vec = 0, T = 1;
    int total_units = 0, nfix = 0, nhub = 0, grid = 0, per_xcd = 0, waves_per_xcd = 0;
    bool has_bias = false;  // some matrix has a bias
    vnm::DBuf<vnm::SpmmArgs> descs;
    vnm::DBuf<int32_t> unit_off;
    vnm::DBuf<int4> fix;          // {matrix, row, first slot, slots}
    vnm::DBuf<float> part;        // partial-sum slots of every matrix
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    ~vnm_batch() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
    }
};

namespace vnm {

template <int BT, int LPR, int LB, bool EXTRA>
__global__ __launch_bounds__(256) void k_spmm_batch(const SpmmArgs *__restrict__ descs,
                                                    const int32_t *__restrict__ unit_off, int count, int T,
                                                    int total, int per_xcd, int waves_per_xcd) {
    constexpr int NV = LB / bsize<BT>();
    __shared__ __align__(16) float turn[NV > 4 ? 4 : 1][NV > 4 ? 64 * NV : 4];
    // wave-uniform; readfirstlane lets the unit's reads be scalar loads
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
    for (int u = slot * 4 + wv; u < per_xcd; u += waves_per_xcd) {
        const int unit = xcd * per_xcd + u;
        if (unit >= total) break;  // wave-uniform: every wave reaches the end
        // matrix of this unit: the last g with unit_off[g] <= unit
        int lo = 0, hi = count - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (unit_off[mid] <= unit) lo = mid;
            else hi = mid - 1;
        }
        const int local = unit - unit_off[lo];
        spmm_items<BT, LPR, LB, EXTRA>(descs[lo], local / T * (64 / LPR), local % T, turn[NV > 4 ? wv : 0]);
    }
}

// Fix-up of the listed (matrix, row) pairs, hub rows first: cut rows get the
// sum of their slots in item order (rows of a matrix without work items, the
// bias or zero).
__global__ __launch_bounds__(256) void k_fix_batch(const int4 *__restrict__ list, int nf, int nhub, int n,
                                                   const SpmmArgs *__restrict__ descs) {
    int w = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    const int hp = n / 64, cp = (n + 255) / 256;
    const bool hub = w < nhub * hp;
    if (!hub) w -= nhub * hp;
    const int i = hub ? w / hp : nhub + w / cp;
    if (i >= nf) return;
    const int4 e = list[i];
    const SpmmArgs &a = descs[e.x];
    float *crow = a.C + (size_t)e.y * a.ldc;
    if (hub) fix_row<1, 32>(crow, a.part, a.pn, e.z, e.w, w % hp * 64, n, a.bias, false);
    else fix_row<4, 8>(crow, a.part, a.pn, e.z, e.w, w % cp * 256, n, a.bias, false);
}

// Rows of a matrix's fix-up list into the batch's.
__global__ void k_tag_fix(const int4 *__restrict__ fix, int nf, int g, int4 *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nf) out[i] = make_int4(g, fix[i].x, fix[i].y, fix[i].z);
}

template <int BT, int LPR, int LB = 16>
static void launch_batch_v(vnm_batch *b, hipStream_t st) {
    if (b->has_bias)
        hipLaunchKernelGGL((k_spmm_batch<BT, LPR, LB, true>), dim3(b->grid), dim3(256), 0, st, b->descs.p,
                           b->unit_off.p, b->count, b->T, b->total_units, b->per_xcd, b->waves_per_xcd);
    else
        hipLaunchKernelGGL((k_spmm_batch<BT, LPR, LB, false>), dim3(b->grid), dim3(256), 0, st, b->descs.p,
                           b->unit_off.p, b->count, b->T, b->total_units, b->per_xcd, b->waves_per_xcd);
}

static void launch_batch_b(vnm_batch *b, hipStream_t st) {
    const int v = b->vec;
    if (b->bt == VNM_DT_F32) {
        if (v == 4) launch_batch_v<VNM_DT_F32, 64>(b, st);
        else if (v == 2) launch_batch_v<VNM_DT_F32, 32>(b, st);
        else launch_batch_v<VNM_DT_F32, 16>(b, st);
    } else if (b->bt == VNM_DT_BF16) {
        if (v == 8) launch_batch_v<VNM_DT_BF16, 64>(b, st);
        else if (v == 4) launch_batch_v<VNM_DT_BF16, 32>(b, st);
        else if (v == 2) launch_batch_v<VNM_DT_BF16, 16>(b, st);
        else launch_batch_v<VNM_DT_BF16, 8>(b, st);
    } else {
        if (v == 16) launch_batch_v<VNM_DT_FP8, 64>(b, st);
        else if (v == 8) launch_batch_v<VNM_DT_FP8, 32>(b, st);
        else if (v == 4) launch_batch_v<VNM_DT_FP8, 16>(b, st);
        else if (v == 2) launch_batch_v<VNM_DT_FP8, 8>(b, st);
        else launch_batch_v<VNM_DT_FP8, 8, 8>(b, st);
    }
}

// Set the launch shape for tiles of 64 * vec columns: tile count, units, grid.
static void batch_shape(vnm_batch *b, const std::vector<int> &items, int vec, std::vector<int32_t> &off) {
    b->vec = vec;
    b->T = b->n / (64 * vec);
    off.assign(b->count + 1, 0);
    const int per = tile_items(b->bt, vec);  // items of a unit
    for (int g = 0; g < b->count; ++g) off[g + 1] = off[g] + (items[g] + per - 1) / per * b->T;
    b->total_units = off[b->count];
    int ncu = 256;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, b->ctx->device) != hipSuccess || ncu < 8)
        ncu = 256;
    b->grid = std::max(8, (ncu * 8) / 8 * 8);  // 8 workgroups of 4 waves per CU
    b->per_xcd = (b->total_units + 7) / 8;
    b->waves_per_xcd = (b->grid / 8) * 4;
}

static int batch_enqueue(vnm_batch *b, hipStream_t st) {
    if (b->total_units > 0) {
        launch_batch_b(b, st);
    }
    if (b->nfix > 0)
        hipLaunchKernelGGL(k_fix_batch, dim3((unsigned)((fix_waves(b->nfix, b->nhub, b->n) + 3) / 4)), dim3(256), 0, st,
                           b->fix.p, b->nfix, b->nhub, b->n,
                           b->descs.p);
    VNM_LAUNCH_CHECK("k_spmm_batch");
    return VNM_OK;
}

static int batch_create(vnm_ctx *ctx, vnm_packed *const *ps, int count, const void *const *B, const int32_t *ldb,
                        int n, int bt, const float *const *bs, float *const *C, const int32_t *ldc,
                        const float *const *bias, int vec, vnm_batch **out) {
    if (!ctx || !ps || count < 1 || !B || !ldb || !C || !ldc || !out) return set_error(VNM_E_ARG, "bad arguments");
    if (n <= 0 || n % 64) return set_error(VNM_E_ARG, "batch: n must be a positive multiple of 64");
    if (bt != VNM_DT_F32 && bt != VNM_DT_BF16 && bt != VNM_DT_FP8)
        return set_error(VNM_E_ARG, "batch: B dtype must be F32, BF16 or FP8");
    const int at = ps[0] ? ps[0]->dtype : 0;
    for (int g = 0; g < count; ++g) {
        const vnm_packed *p = ps[g];
        if (!p || p->ctx != ctx) return set_error(VNM_E_ARG, "batch: matrix %d missing or on another context", g);
        if (p->dtype != at) return set_error(VNM_E_ARG, "batch: every matrix needs the same value dtype");
        if (p->ngroups > 0)
            return set_error(VNM_E_ARG, "batch: matrix %d has a sparse-MFMA part (pack it with vnm_pack)", g);
        if (!B[g] || !C[g] || ldb[g] < n || ldc[g] < n || (bt == VNM_DT_FP8 && (!bs || !bs[g])))
            return set_error(VNM_E_ARG, "batch: operands of matrix %d", g);
        if ((ldb[g] * bsize_of(bt)) % 16 || ldc[g] % 4 || ((uintptr_t)B[g] & 15) || ((uintptr_t)C[g] & 15) ||
            (bias && bias[g] && ((uintptr_t)bias[g] & 15)))
            return set_error(VNM_E_ARG, "batch: matrix %d operands must be 16-byte aligned", g);
        if ((uint64_t)p->ncols * (uint64_t)ldb[g] * (uint64_t)bsize_of(bt) > 0xFFFFFFFFull)
            return set_error(VNM_E_ARG, "batch: B of matrix %d must be smaller than 4 GiB", g);
    }
    if (vec && !vec_ok(bt, n, vec)) return set_error(VNM_E_ARG, "batch: %d values per lane do not fit n", vec);
    hipStream_t st = ctx->stream;
    auto b = std::make_unique<vnm_batch>();
    b->ctx = ctx;
    b->count = count;
    b->n = n;
    b->bt = bt;
    b->at = at;
    for (int g = 0; g < count; ++g) b->has_bias |= bias && bias[g];
    std::vector<SpmmArgs> d(count);
    std::vector<int> items(count);
    std::vector<size_t> part_off(count + 1, 0);
    std::vector<int> hub_off(count + 1, 0), fix_off(count + 1, 0);  // hub rows, and the other listed rows
    int rc;
    for (int g = 0; g < count; ++g) {
        items[g] = ps[g]->nitems;
        part_off[g + 1] = part_off[g] + (size_t)ps[g]->nslots * n;
        hub_off[g + 1] = hub_off[g] + ps[g]->nhub;
        fix_off[g + 1] = fix_off[g] + ps[g]->nfix - ps[g]->nhub;
    }
    b->nhub = hub_off[count];
    b->nfix = b->nhub + fix_off[count];
    if ((rc = b->descs.alloc(count)) || (rc = b->unit_off.alloc(count + 1)) ||
        (rc = b->fix.alloc(std::max(b->nfix, 1))) || (rc = b->part.alloc(std::max<size_t>(part_off[count], 1))))
        return rc;
    for (int g = 0; g < count; ++g)
        d[g] = packed_args(ps[g], B[g], ldb[g], bs ? bs[g] : nullptr, C[g], ldc[g], bias ? bias[g] : nullptr,
                           b->part.p + part_off[g], n);
    VNM_HIP_TRY(hipMemcpyAsync(b->descs.p, d.data(), count * sizeof(SpmmArgs), hipMemcpyHostToDevice, st));
    for (int g = 0; g < count; ++g) {
        const int hubs = ps[g]->nhub, rest = ps[g]->nfix - hubs;
        if (hubs)
            hipLaunchKernelGGL(k_tag_fix, dim3((hubs + 255) / 256), dim3(256), 0, st, ps[g]->fix.p, hubs, g,
                               b->fix.p + hub_off[g]);
        if (rest)
            hipLaunchKernelGGL(k_tag_fix, dim3((rest + 255) / 256), dim3(256), 0, st, ps[g]->fix_rest(), rest, g,
                               b->fix.p + b->nhub + fix_off[g]);
    }
    VNM_LAUNCH_CHECK("k_tag_fix");
    std::vector<int32_t> off;
    if (vec == 0) vec = default_vec(bt, n);
    batch_shape(b.get(), items, vec, off);
    VNM_HIP_TRY(hipMemcpyAsync(b->unit_off.p, off.data(), (count + 1) * 4, hipMemcpyHostToDevice, st));
    VNM_HIP_TRY(hipStreamSynchronize(st));
    // capture the two kernels once; vnm_batch_run replays them
    VNM_HIP_TRY(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    rc = batch_enqueue(b.get(), st);
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamEndCapture(st, &graph);
    if (rc) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc;
    }
    if (e != hipSuccess) return set_error(VNM_E_HIP, "batch capture failed: %s", hipGetErrorString(e));
    b->graph = graph;
    e = hipGraphInstantiate(&b->exec, graph, nullptr, nullptr, 0);
    if (e != hipSuccess) return set_error(VNM_E_HIP, "batch graph instantiation failed: %s", hipGetErrorString(e));
    ctx->launches += 2;
    *out = b.release();
    return VNM_OK;
}

// ------------------------------------------------------------ GCN layer

// A barrier for LDS data only: pending global loads stay in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// f32_to_bf16 without branches (round to nearest even, NaN kept quiet).
__device__ __forceinline__ uint32_t bf16_bits(float f) {
    const uint32_t u = __float_as_uint(f);
    const uint32_t r = (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
    return (u & 0x7FFFFFFFu) > 0x7F800000u ? ((u >> 16) | 0x40u) : r;
}

// H[R x N] (BF16) = X[R x K] (BF16, leading dimension ldx) W[K x N]; K a multiple
// of 16, N of 64.  A workgroup of four waves takes a tile of 64 HF rows, 16 HF a
// wave, and 64-column panels of W: blockIdx.y, + gridDim.y, ...  With K <= GKT
// (every row of X fits the wave's registers) X is read once for all of them.
// Bound by X and H in memory (R 65,536, K = N = 256: 67 MB in 22.3 us, 3.0 TB/s of
// a copy's 4.9: reading, then multiplying and writing, in step over the chip; 30 us
// with X read once a panel and W transposed by a launch of its own, 7.5 us).
//
// The panel lies transposed in LDS, K-contiguous per column, for 16-byte reads of
// 8 k: a thread loads two columns' 8 k as eight words, straight from W, and packs
// them into two 16-byte writes; the next panel's words are in flight while the
// current one is multiplied, and go to the other half of the LDS buffer.
// gfx950's v_mfma_f32_16x16x32_bf16 takes the W fragment as its first operand
// (lane l: row l%16 of the fragment, k 8(l/16)..+7) and the X fragment as its
// second (row l%16, the same k), so it produces H transposed: lane l holds rows
// 4(l/16)..+3 of the W fragment for one row of X.  Row 4g + i of fragment nt is
// column 16g + 4nt + i of the panel, so that a lane's four fragments are 16
// consecutive columns, stored as two 16-byte pieces.  LDS rows are padded by 16
// bytes and the 16-byte chunks of fragment nt's rows exchanged by 4nt, which keeps
// both the fragment reads and the transposing writes off each other's banks.
// In step s lane group g = l/16 takes k 32s + 8g .. +7; where K is an odd
// multiple of 16, the last step's upper groups hold zeros in both operands.
constexpr int GEMM_WG = 256;
constexpr int GEMM_K = 256;  // k of a stage

template <int GKT>
struct GemmStage {  // two columns x 8 k each, of up to GKT k
    static constexpr int PT = (GKT / 8) * 32 / GEMM_WG;
    uint32_t r[PT][8];
    __device__ __forceinline__ void load(const uint16_t *__restrict__ W, int N, int n0, int kn) {
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const int i = threadIdx.x + GEMM_WG * j, c = i % 32, k = min(i / 32 * 8, kn - 8);
#pragma unroll
            for (int q = 0; q < 8; ++q)  // W may be 2-byte aligned
                __builtin_memcpy(&r[j][q], W + (size_t)(k + q) * N + n0 + 2 * c, 4);
        }
    }
    __device__ __forceinline__ void store(uint16_t *w, int kn) const {
        const int kr = (kn + 31) / 32 * 32;  // zeros up to the last step's end
#pragma unroll
        for (int j = 0; j < PT; ++j) {
            const int i = threadIdx.x + GEMM_WG * j, c = i % 32 * 2, kb = i / 32;
            if (kb * 8 >= kr) continue;
            const bool live = kb * 8 < kn;
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                lo[q] = live ? __builtin_amdgcn_perm(r[j][2 * q + 1], r[j][2 * q], 0x05040100u) : 0u;
                hi[q] = live ? __builtin_amdgcn_perm(r[j][2 * q + 1], r[j][2 * q], 0x07060302u) : 0u;
            }
            const int nt = (c >> 2) & 3, row = nt * 16 + (c >> 4) * 4 + (c & 3);
            uint16_t *d = w + row * (GKT + 8) + ((kb ^ (4 * nt)) * 8);
            *(uint4 *)d = make_uint4(lo[0], lo[1], lo[2], lo[3]);
            *(uint4 *)(d + GKT + 8) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        }
    }
};

template <int HF, int GKT>
__global__ __launch_bounds__(GEMM_WG) void k_gemm_xw(int R, int K, int N, const uint16_t *__restrict__ X, int ldx,
                                                     const uint16_t *__restrict__ W, uint16_t *__restrict__ H) {
    typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
    typedef float f32x4_t __attribute__((ext_vector_type(4)));
    constexpr int GS = GKT / 32, BUF = 64 * (GKT + 8);
    __shared__ __align__(16) uint16_t w[2 * BUF];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int m = lane & 15, g = lane >> 4;
    const int r0 = (blockIdx.x * 4 + wv) * 16 * HF;
    const int P = N / 64;
    const bool once = K <= GKT;
    bf16x8_t a[HF][GS];
    auto load_x = [&](int kc, int kn) {
#pragma unroll
        for (int h = 0; h < HF; ++h) {
            const uint16_t *xp = X + (size_t)min(r0 + h * 16 + m, R - 1) * ldx + kc;
#pragma unroll
            for (int st = 0; st < GS; ++st) {
                if (32 * st >= kn) break;
                const int k0 = 32 * st + 8 * g;
                uint4 v;
                __builtin_memcpy(&v, __builtin_assume_aligned(xp + min(k0, kn - 8), 8), 16);
                if (k0 >= kn) v = make_uint4(0u, 0u, 0u, 0u);
                a[h][st] = __builtin_bit_cast(bf16x8_t, v);
            }
        }
    };
    f32x4_t acc[HF][4];
    auto clear = [&] {
#pragma unroll
        for (int h = 0; h < HF; ++h)
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) acc[h][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    };
    auto multiply = [&](const uint16_t *wb, int kn) {
#pragma unroll
        for (int st = 0; st < GS; ++st) {
            if (32 * st >= kn) break;
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                const bf16x8_t b = *(const bf16x8_t *)&wb[(nt * 16 + m) * (GKT + 8) + ((4 * st + g) ^ (4 * nt)) * 8];
#pragma unroll
                for (int h = 0; h < HF; ++h)
                    acc[h][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a[h][st], acc[h][nt], 0, 0, 0);
            }
        }
    };
    // lane (m, g): row r0 + 16h + m, columns n0 + 16g .. +15
    auto store_h = [&](int n0) {
#pragma unroll
        for (int h = 0; h < HF; ++h) {
            const int rr = r0 + h * 16 + m;
            if (rr >= R) continue;
            uint32_t v[8];
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                v[2 * nt] = bf16_bits(acc[h][nt][0]) | (bf16_bits(acc[h][nt][1]) << 16);
                v[2 * nt + 1] = bf16_bits(acc[h][nt][2]) | (bf16_bits(acc[h][nt][3]) << 16);
            }
            uint4 *d = (uint4 *)(H + (size_t)rr * N + n0 + 16 * g);
            d[0] = make_uint4(v[0], v[1], v[2], v[3]);
            d[1] = make_uint4(v[4], v[5], v[6], v[7]);
        }
    };
    GemmStage<GKT> sg;
    if (once) {
        int p = blockIdx.y, cur = 0;
        sg.load(W, N, p * 64, K);
        load_x(0, K);
        sg.store(w, K);
        lds_barrier();
        for (; p < P; p += gridDim.y) {
            const int np = p + gridDim.y;
            if (np < P) sg.load(W, N, np * 64, K);
            clear();
            multiply(w + cur * BUF, K);
            store_h(p * 64);
            if (np < P) {
                cur ^= 1;
                sg.store(w + cur * BUF, K);
                lds_barrier();
            }
        }
    } else {
        for (int p = blockIdx.y; p < P; p += gridDim.y) {
            clear();
            for (int kc = 0; kc < K; kc += GKT) {
                const int kn = min(GKT, K - kc);  // a multiple of 16
                sg.load(W + (size_t)kc * N, N, p * 64, kn);
                load_x(kc, kn);
                lds_barrier();  // the chunk before has been read
                sg.store(w, kn);
                lds_barrier();
                multiply(w, kn);
            }
            store_h(p * 64);
        }
    }
}

static int gcn_layer(vnm_packed *p, const uint16_t *X, int ldx, int K, const uint16_t *W, int N,
                     const float *bias, float *Y, int ldy) {
    if (!p || !X || !W || !Y) return set_error(VNM_E_ARG, "gcn: null argument");
    if (K <= 0 || K % 16 || N <= 0 || N % 64 || ldx < K || ldx % 4 || ldy < N || ldy % 4)
        return set_error(VNM_E_ARG, "gcn: K must be a multiple of 16, N of 64, ldx >= K and ldy >= N (multiples of 4)");
    if (((uintptr_t)X & 7) || ((uintptr_t)Y & 15) || (bias && ((uintptr_t)bias & 15)))
        return set_error(VNM_E_ARG, "gcn: X must be 8-byte and Y, bias 16-byte aligned");
    const int R = p->ncols;  // X W has one row per column of A
    hipStream_t st = p->ctx->stream;
    int rc;
    if (p->gcn_h.n < (size_t)R * N) {
        p->gcn_h.release();
        if ((rc = p->gcn_h.alloc((size_t)R * N))) return rc;
    }
    KernelTimer kt(p->ctx, "k_gemm_xw");
    // Tiles of 128 rows share every W fragment between two X fragments; 64-row ones
    // where 128-row tiles and panels are fewer workgroups than CUs (R 3,008, N 256:
    // 6.0 us against 7.2; equal at 8,192).  A workgroup takes every panel, X read
    // once, where the row tiles alone give each CU one (R 65,536: 22.3 us against
    // 33.2 with a panel each; 32,768: 18.6 against 23.1; 16,384: 18.0 against 14.2).
    int ncu = 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, p->ctx->device) != hipSuccess || ncu < 8)
        ncu = 8;
    const int P = N / 64, tiles = (R + 127) / 128;
    if ((int64_t)tiles * P < ncu)
        hipLaunchKernelGGL((k_gemm_xw<1, GEMM_K>), dim3((R + 63) / 64, P), dim3(GEMM_WG), 0, st, R, K, N, X, ldx, W,
                           p->gcn_h.p);
    else
        hipLaunchKernelGGL((k_gemm_xw<2, GEMM_K>), dim3(tiles, K <= GEMM_K && tiles >= ncu ? 1 : P), dim3(GEMM_WG), 0,
                           st, R, K, N, X, ldx, W, p->gcn_h.p);
    kt.stop();
    p->ctx->launches++;
    VNM_LAUNCH_CHECK("k_gemm_xw");
    return spmm(p, p->gcn_h.p, N, N, VNM_DT_BF16, nullptr, Y, ldy, bias);
}

}  // namespace vnm

using namespace vnm;

extern "C" {

int vnm_batch_create(vnm_ctx *ctx, vnm_packed *const *ps, int count, const void *const *B, const int32_t *ldb,
                     int n, int b_dtype, const float *const *b_scales, float *const *C, const int32_t *ldc,
                     const float *const *bias, int cols_per_lane, vnm_batch **out) {
    PoolScope pool(ctx ? ctx->pool : nullptr);
    return batch_create(ctx, ps, count, B, ldb, n, b_dtype, b_scales, C, ldc, bias, cols_per_lane, out);
}

int vnm_batch_run(vnm_batch *b) {
    if (!b) return set_error(VNM_E_ARG, "null batch");
    KernelTimer kt(b->ctx, "k_spmm_batch");
    hipError_t e = hipGraphLaunch(b->exec, b->ctx->stream);
    kt.stop();
    if (e != hipSuccess) return set_error(VNM_E_HIP, "batch graph launch failed: %s", hipGetErrorString(e));
    b->ctx->launches += 2;
    return VNM_OK;
}

int vnm_batch_info(const vnm_batch *b, int32_t *cols_per_lane, int32_t *units, int32_t *zero_rows) {
    if (!b) return set_error(VNM_E_ARG, "null batch");
    if (cols_per_lane) *cols_per_lane = b->vec;
    if (units) *units = b->total_units;
    if (zero_rows) *zero_rows = b->nfix;
    return VNM_OK;
}

void vnm_batch_destroy(vnm_batch *b) {
    if (!b) return;
    if (b->ctx && b->ctx->stream) (void)hipStreamSynchronize(b->ctx->stream);
    delete b;
}

int vnm_gcn_layer(vnm_packed *p, const uint16_t *X, int ldx, int K, const uint16_t *W, int N, const float *bias,
                  float *Y, int ldy) {
    PoolScope pool(p ? p->ctx->pool : nullptr);
    return gcn_layer(p, X, ldx, K, W, N, bias, Y, ldy);
}

}  // extern "C"
