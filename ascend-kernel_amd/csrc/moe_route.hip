// Routing for the grouped ops on gfx950: router logits -> top-k experts per token -> rows sorted
// by expert + the cumulative group_list that grouped_gemm / grouped_soft_gemv read
// (grouped_gemm/op_kernel/grouped_matmul_utils.h:304-320 defines that tensor; the reference leaves
// building it to its caller).  Everything stays on the device: no host round trip between the
// router and the expert GEMMs.
//
// Order of the sorted rows: by expert id, then by flat choice index t * topk + j (a stable sort), so
// the result is deterministic and independent of the launch geometry.
//
//   route_topk_kernel     one wavefront per token: softmax statistics and top-k by repeated arg-max
//   route_count_kernel    per 1024-choice block, a histogram over experts (LDS atomics)
//   route_scan_kernel     (many blocks only) the counts' prefix over the blocks, per expert
//   route_rank_kernel     per block: prefix of the counts over experts and earlier blocks (group_list), then every
//                         choice's rank among the earlier choices of its expert -> its sorted row
//   route_scatter_kernel  a token's x row read once and written to the sorted row of each of its choices
//   route_small_kernel    all of it in one launch for a decode step's few tokens
#include <atomic>

#include "moe_device.h"
#include "moe_internal.h"

namespace moe {

constexpr int RT_BLOCK = 1024;     // choices per block of the count / rank kernels
constexpr int RT_MAX_E = 1024;     // experts (one thread each in the scan kernel)
constexpr int RT_MAX_PER_LANE = RT_MAX_E / 64;

// Maximum over the wavefront by DPP moves (a few cycles each; the same reduction by ds_bpermute shuffles waits for six LDS
// round trips, topk + 1 times per token).  The last lane has it; every lane gets it.
template <int CTRL>
__device__ __forceinline__ float max_from_lane(float v) {
    const int b = __builtin_bit_cast(int, v);
    return fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(b, b, CTRL, 0xf, 0xf, false)));
}
__device__ __forceinline__ float wave_max(float v) {
    v = max_from_lane<0x111>(v);   // row_shr 1, 2, 4, 8: lane 15 of each row of 16 holds the row's maximum
    v = max_from_lane<0x112>(v);
    v = max_from_lane<0x114>(v);
    v = max_from_lane<0x118>(v);
    v = max_from_lane<0x142>(v);   // row_bcast 15, row_bcast 31
    v = max_from_lane<0x143>(v);
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// Softmax statistics and top-k of one token by one wavefront; found(j, expert, weight) is called by the lane that holds the
// j-th choice, all choices of a token (64 at a time) at once.  PL = logits per lane (E <= 64 PL).
// The order is lexicographic in (value descending, expert ascending); NaN logits are no candidates.  Every lane sorts its
// logits first, so that a round of the arg-max looks at the heads of the lanes only: a max-reduction, then the expert of the
// one lane that holds it; only when several lanes hold the maximum a second reduction picks the lowest expert among them.
// (Rounds over all PL logits, each with its own outputs: 64 tokens of 256 experts routed in 18.4 instead of 11.6 us.)
template <int PL, typename FOUND>
__device__ __forceinline__ void token_topk(const float* __restrict__ row, int E, int topk, int lane, FOUND found) {
    constexpr int NONE = 0x7fffffff;   // no candidate: behind every expert, whatever its logit
    float v[PL];
    int id[PL];
    float mx = -INFINITY;
#pragma unroll
    for (int c = 0; c < PL; ++c) {
        const int e = c * 64 + lane;
        v[c] = e < E ? row[e] : -INFINITY;
        mx = fmaxf(mx, v[c]);
    }
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < PL; ++c)
        if (c * 64 + lane < E) sum += __expf(v[c] - mx);
    sum = wave_reduce_sum(sum);
    const float inv = 1.f / sum;
#pragma unroll
    for (int c = 0; c < PL; ++c) {
        const bool candidate = c * 64 + lane < E && v[c] == v[c];
        id[c] = candidate ? c * 64 + lane : NONE;
        v[c] = candidate ? v[c] : -INFINITY;
    }
    // odd-even merge sort network, best first
    auto order = [&](int a, int b) {
        const bool swap = v[b] > v[a] || (v[b] == v[a] && id[b] < id[a]);
        const float va = v[a];
        const int ia = id[a];
        v[a] = swap ? v[b] : va;
        v[b] = swap ? va : v[b];
        id[a] = swap ? id[b] : ia;
        id[b] = swap ? ia : id[b];
    };
#pragma unroll
    for (int p = 1; p < PL; p *= 2)
#pragma unroll
        for (int k = p; k >= 1; k /= 2)
#pragma unroll
            for (int j = k % p; j + k < PL; j += 2 * k)
#pragma unroll
                for (int i = 0; i < k; ++i)
                    if (i + j + k < PL && (i + j) / (2 * p) == (i + j + k) / (2 * p)) order(i + j, i + j + k);
    for (int j0 = 0; j0 < topk; j0 += 64) {
        const int n = min(64, topk - j0);
        float best_v = 0.f;   // lane j: choice j0 + j
        int best_e = 0;
        for (int j = 0; j < n; ++j) {
            const float gv = wave_max(v[0]);
            const unsigned long long holders = __ballot(v[0] == gv);
            int ge;
            if (__popcll(holders) == 1) {
                ge = __builtin_amdgcn_readlane(id[0], __ffsll(holders) - 1);
            } else {
                ge = v[0] == gv ? id[0] : NONE;
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) ge = min(ge, __shfl_xor(ge, off, 64));
            }
            best_v = lane == j ? gv : best_v;
            best_e = lane == j ? ge : best_e;
            const bool mine = id[0] == ge;
#pragma unroll
            for (int c = 0; c < PL; ++c) {
                v[c] = mine ? (c + 1 < PL ? v[c + 1 < PL ? c + 1 : c] : -INFINITY) : v[c];
                id[c] = mine ? (c + 1 < PL ? id[c + 1 < PL ? c + 1 : c] : NONE) : id[c];
            }
        }
        if (lane < n) found(j0 + lane, best_e, __expf(best_v - mx) * inv);
    }
}

template <int PL>
__global__ __launch_bounds__(256) void route_topk_kernel(const float* __restrict__ logits, float* __restrict__ weight,
                                                         int32_t* __restrict__ ids, int T, int E, int topk) {
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= T) return;
    token_topk<PL>(logits + (int64_t)t * E, E, topk, lane, [&](int j, int e, float w) {
        ids[(int64_t)t * topk + j] = e;
        weight[(int64_t)t * topk + j] = w;
    });
}

// Lanes of the wavefront that hold the same id as this one (bits: number of bits an id has; lanes with `in` false match
// nobody's id that matters: they are left out)
__device__ __forceinline__ unsigned long long same_id_lanes(int id, bool in, int bits) {
    unsigned long long same = __ballot(in);
    for (int b = 0; b < bits; ++b) {
        const unsigned long long ones = __ballot((id >> b) & 1);
        same &= ((id >> b) & 1) ? ones : ~ones;
    }
    return same;
}

// Exclusive prefix over the threads of a 1024-thread workgroup; part: 16 integers of LDS.  One barrier.
__device__ __forceinline__ int block_exclusive_prefix(int v, int* part) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int up = __shfl_up(incl, off, 64);
        if (lane >= off) incl += up;
    }
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    int before = 0;
#pragma unroll
    for (int w = 0; w < RT_BLOCK / 64; ++w) before += w < wave ? part[w] : 0;
    return before + incl - v;
}

// Routing of a decode step in one launch: at most RT_SMALL_T tokens and RT_BLOCK choices.  Such a call is bound by launches
// and by chains of dependent latencies, not by work: so every workgroup routes all tokens by itself (16 wavefronts, a token
// each), ranks the choices in LDS and then copies one token's row of x to its choices' sorted rows; the first workgroup
// writes everything else.  1 / 16 tokens, top 8 of 256 experts, K = 7168: 16.6 / 17.8 us with four kernels and the arg-max over
// all logits, 9.3 / 10.7 with three kernels and the one below, 6.4 / 8.3 in one launch; with 32 tokens, two per wavefront,
// 12.0 against 11.1.  Dynamic LDS: (16 + 1) * E + RT_BLOCK integers.
constexpr int RT_SMALL_T = 16;
template <int PL>
__global__ __launch_bounds__(RT_BLOCK) void route_small_kernel(const float* __restrict__ logits, float* __restrict__ weight, int32_t* __restrict__ ids,
                                                               int64_t* __restrict__ group_list, int32_t* __restrict__ row_token,
                                                               int32_t* __restrict__ row_of_choice, const u32x4_t* __restrict__ x,
                                                               u32x4_t* __restrict__ x_sorted, int T, int E, int topk, int units, int bits) {
    extern __shared__ int small_lds[];
    int* wh = small_lds;                 // [16][E] choices of expert e in wavefront w -> in the wavefronts before w
    int* base = wh + 16 * E;             // [E] first sorted row of expert e
    int* choice = base + E;              // [RT_BLOCK] expert, then sorted row, of every choice
    __shared__ int part[RT_BLOCK / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = T * topk;
    const bool writer = blockIdx.x == 0;
    const int waves_n = (n + 63) >> 6;   // wavefronts that hold choices
    for (int j = tid; j < waves_n * E; j += RT_BLOCK) wh[j] = 0;
    if (logits) {
        for (int t = wave; t < T; t += RT_BLOCK / 64)
            token_topk<PL>(logits + (int64_t)t * E, E, topk, lane, [&](int j, int e, float w) {
                choice[t * topk + j] = e;
                if (writer) {
                    ids[t * topk + j] = e;
                    weight[t * topk + j] = w;
                }
            });
    } else if (tid < n) {
        choice[tid] = ids[tid];
    }
    __syncthreads();
    const int my = tid < n ? choice[tid] : -1;
    const bool valid = (unsigned)my < (unsigned)E;   // ids outside [0, E) are dropped
    const unsigned long long same = same_id_lanes(my, valid, bits);
    const unsigned long long below = same & ((1ull << lane) - 1);
    if (valid && below == 0) wh[wave * E + my] = __popcll(same);
    __syncthreads();
    int total = 0;
    if (tid < E)
        for (int w = 0; w < waves_n; ++w) {
            const int c = wh[w * E + tid];
            wh[w * E + tid] = total;
            total += c;
        }
    const int first = block_exclusive_prefix(total, part);
    if (tid < E) {
        base[tid] = first;
        if (writer) group_list[tid] = first + total;
    }
    __syncthreads();
    if (tid < n) {
        const int dst = valid ? base[my] + wh[wave * E + my] + __popcll(below) : -1;
        choice[tid] = dst;
        if (writer) {
            row_of_choice[tid] = dst;
            if (valid) row_token[dst] = tid / topk;
        }
    }
    if (!x) return;
    __syncthreads();
    const int t = blockIdx.x;
    for (int u = tid; u < units; u += RT_BLOCK) {
        const u32x4_t v = x[(int64_t)t * units + u];
        for (int c = 0; c < topk; ++c) {
            const int r = choice[t * topk + c];
            if (r >= 0) x_sorted[(int64_t)r * units + u] = v;
        }
    }
}

__global__ __launch_bounds__(RT_BLOCK) void route_count_kernel(const int32_t* __restrict__ ids, int32_t* __restrict__ block_counts,
                                                               int64_t n, int E) {
    __shared__ int hist[RT_MAX_E];
    for (int e = threadIdx.x; e < E; e += RT_BLOCK) hist[e] = 0;
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * RT_BLOCK + threadIdx.x;
    if (i < n) {
        const int e = ids[i];
        if ((unsigned)e < (unsigned)E) atomicAdd(&hist[e], 1);   // ids outside [0, E) are dropped
    }
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += RT_BLOCK) block_counts[(int64_t)blockIdx.x * E + e] = hist[e];
}

// Many blocks: the per-block counts [nblocks][E] become, in place, each expert's exclusive prefix over the
// blocks, and row nblocks receives the experts' totals.  One wavefront per expert, 64 blocks per round
// (wavefront scan by shuffles, the running total carried from round to round).
constexpr int RT_FUSED_SCAN_MAX_BLOCKS = 64;   // up to here every rank block sums the counts itself
__global__ __launch_bounds__(256) void route_scan_kernel(int32_t* __restrict__ block_counts, int E, int nblocks) {
    const int lane = threadIdx.x & 63;
    const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (e >= E) return;
    int carry = 0;
    for (int b0 = 0; b0 < nblocks; b0 += 64) {
        const int b = b0 + lane;
        const int c = b < nblocks ? block_counts[(int64_t)b * E + e] : 0;
        int incl = c;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int up = __shfl_up(incl, off, 64);
            if (lane >= off) incl += up;
        }
        if (b < nblocks) block_counts[(int64_t)b * E + e] = carry + incl - c;
        carry += __shfl(incl, 63, 64);
    }
    if (lane == 0) block_counts[(int64_t)nblocks * E + e] = carry;
}

// Rank of every choice of block b among the choices of its expert, and with it the sorted row:
//   row = (choices of lower experts) + (choices of this expert in earlier blocks) + (in earlier wavefronts of
//         this block) + (in lower lanes of this wavefront)
// With few blocks every block derives the first two terms from the per-block counts itself (nblocks x E integers
// per block: cheaper than a kernel of its own for the scan, but quadratic in the number of blocks); with more than
// RT_FUSED_SCAN_MAX_BLOCKS of them route_scan_kernel has turned the counts into prefixes and totals (prefixed != 0).
// Block 0 also writes group_list.  The third term comes from per-wavefront histograms in LDS, the fourth from the lanes
// with the same expert.  A single block (nblocks 1) needs no counts from before: the histograms are all there is.  Dynamic
// LDS: (16 + 1) * E integers.
__global__ __launch_bounds__(RT_BLOCK) void route_rank_kernel(const int32_t* __restrict__ ids, const int32_t* __restrict__ block_counts,
                                                              int64_t* __restrict__ group_list,
                                                              int32_t* __restrict__ row_token, int32_t* __restrict__ row_of_choice,
                                                              int64_t n, int E, int topk, int nblocks, int prefixed, int bits) {
    extern __shared__ int rank_lds[];
    int* base = rank_lds;            // [E] first sorted row of this block's choices of expert e
    int* wh = base + E;              // [16][E] choices of expert e in wavefront w -> in the wavefronts before w
    __shared__ int part[RT_BLOCK / 64];
    const int e = threadIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int blk = blockIdx.x;
    const int64_t i = (int64_t)blk * RT_BLOCK + threadIdx.x;
    const int my = i < n ? ids[i] : -1;
    int total = 0, before = 0;
    if (e < E && prefixed) {
        before = block_counts[(int64_t)blk * E + e];
        total = block_counts[(int64_t)nblocks * E + e];
    } else if (e < E && nblocks > 1) {
        // independent loads, 4 blocks at a time
        int b = 0;
        for (; b + 4 <= nblocks; b += 4) {
            const int c0 = block_counts[(int64_t)b * E + e], c1 = block_counts[(int64_t)(b + 1) * E + e];
            const int c2 = block_counts[(int64_t)(b + 2) * E + e], c3 = block_counts[(int64_t)(b + 3) * E + e];
            total += c0 + c1 + c2 + c3;
            before += (b < blk ? c0 : 0) + (b + 1 < blk ? c1 : 0) + (b + 2 < blk ? c2 : 0) + (b + 3 < blk ? c3 : 0);
        }
        for (; b < nblocks; ++b) {
            const int c = block_counts[(int64_t)b * E + e];
            total += c;
            before += b < blk ? c : 0;
        }
    }
    for (int j = threadIdx.x; j < 16 * E; j += RT_BLOCK) wh[j] = 0;
    const bool valid = (unsigned)my < (unsigned)E;   // ids outside [0, E) are dropped
    const unsigned long long same = same_id_lanes(my, valid, bits);
    const unsigned long long below = same & ((1ull << lane) - 1);
    __syncthreads();
    if (valid && below == 0) wh[wave * E + my] = __popcll(same);
    __syncthreads();
    if (e < E) {
        int run = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            const int t = wh[w * E + e];
            wh[w * E + e] = run;
            run += t;
        }
        if (nblocks <= 1) total = run;
    }
    const int first = block_exclusive_prefix(total, part);
    if (e < E) {
        base[e] = first + before;
        if (blk == 0) group_list[e] = first + total;
    }
    __syncthreads();
    if (i >= n) return;
    if (!valid) {
        row_of_choice[i] = -1;
        return;
    }
    const int dst = base[my] + wh[wave * E + my] + __popcll(below);
    row_token[dst] = (int32_t)(i / topk);
    row_of_choice[i] = dst;
}

// x rows copied into sorted order, token by token: a workgroup reads one token's row once (16 bytes per
// thread and load, 4 loads in flight) and writes it to the sorted row of each of its choices.  Dropped
// choices (row_of_choice < 0) write nothing, so the rows past group_list[E - 1] stay untouched.
__global__ __launch_bounds__(256) void route_scatter_kernel(const u32x4_t* __restrict__ x, const int32_t* __restrict__ row_of_choice,
                                                            u32x4_t* __restrict__ x_sorted, int topk, int units) {
    const int t = blockIdx.x;
    const u32x4_t* src = x + (int64_t)t * units;
    const int32_t* roc = row_of_choice + (int64_t)t * topk;
    for (int u0 = threadIdx.x; u0 < units; u0 += 4 * 256) {
        u32x4_t v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (u0 + 256 * j < units) v[j] = src[u0 + 256 * j];
        for (int c = 0; c < topk; ++c) {
            const int r = __builtin_amdgcn_readfirstlane(roc[c]);
            if (r < 0) continue;
            u32x4_t* dst = x_sorted + (int64_t)r * units;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (u0 + 256 * j < units) __builtin_nontemporal_store(v[j], dst + u0 + 256 * j);
        }
    }
}

size_t route_workspace_bytes(const moe_route_args* a) {
    const int64_t n = a->T * a->topk;
    const int64_t nblocks = (n + RT_BLOCK - 1) / RT_BLOCK;
    return (size_t)((nblocks + 1) * a->E) * sizeof(int32_t);   // per-block counts, and a row of totals
}

// Scratch of moe_route_static: the per-block counts (and the row of totals) live in this array instead of a
// caller-provided workspace.  One copy per GPU, held until the process ends; every call on a GPU uses
// that GPU's copy (the count kernel rewrites all of the part a call reads, so nothing needs clearing,
// but two calls that overlap in time on one GPU race on it).
static __device__ __align__(256) unsigned char scratch[MOE_ROUTE_STATIC_SCRATCH_BYTES];

// Device address of `scratch` on each GPU (the array's name is only a host-side handle).  Filled on the
// first call on a device, with that device current.
constexpr int RT_MAX_DEVICES = 64;
static std::atomic<void*> scratch_addr[RT_MAX_DEVICES];

int launch_route_static(const moe_route_args* a, hipStream_t stream) {
    if (route_workspace_bytes(a) > (size_t)MOE_ROUTE_STATIC_SCRATCH_BYTES) return MOE_ERR_TOO_LARGE;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= RT_MAX_DEVICES) return MOE_ERR_NO_DEVICE;
    void* ptr = scratch_addr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return MOE_ERR_NO_DEVICE;
        scratch_addr[dev].store(ptr, std::memory_order_release);   // a race stores the same address twice
    }
    moe_route_args b = *a;
    b.workspace = ptr;
    return launch_route(&b, stream);
}

template <int PL>
static int launch_route_small(const moe_route_args* a, int bits, hipStream_t stream) {
    static std::atomic<uint64_t> lds_set{0};
    if (const int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&route_small_kernel<PL>), (17 * RT_MAX_E + RT_BLOCK) * (int)sizeof(int), lds_set))
        return rc;
    const size_t lds = (size_t)(17 * a->E + RT_BLOCK) * sizeof(int);
    hipLaunchKernelGGL(route_small_kernel<PL>, dim3(a->x ? (unsigned)a->T : 1u), dim3(RT_BLOCK), lds, stream, static_cast<const float*>(a->logits),
                       static_cast<float*>(a->topk_weight), static_cast<int32_t*>(a->topk_ids), static_cast<int64_t*>(a->group_list),
                       static_cast<int32_t*>(a->row_token), static_cast<int32_t*>(a->row_of_choice), static_cast<const u32x4_t*>(a->x),
                       static_cast<u32x4_t*>(a->x_sorted), (int)a->T, (int)a->E, (int)a->topk, (int)(a->K / 8), bits);
    return hipGetLastError() == hipSuccess ? MOE_OK : MOE_ERR_LAUNCH;
}

int launch_route(const moe_route_args* a, hipStream_t stream) {
    const int64_t n = a->T * a->topk;
    const int nblocks = (int)((n + RT_BLOCK - 1) / RT_BLOCK);
    int32_t* ids = static_cast<int32_t*>(a->topk_ids);
    int32_t* counts = static_cast<int32_t*>(a->workspace);
    const int bits = a->E > 1 ? 32 - __builtin_clz((unsigned)(a->E - 1)) : 0;   // of a valid expert id
    if (a->T > 0 && a->T <= RT_SMALL_T && n <= RT_BLOCK) {   // a token per wavefront, see route_small_kernel
        if (a->E <= 64) return launch_route_small<1>(a, bits, stream);
        if (a->E <= 128) return launch_route_small<2>(a, bits, stream);
        if (a->E <= 256) return launch_route_small<4>(a, bits, stream);
        if (a->E <= 512) return launch_route_small<8>(a, bits, stream);
        return launch_route_small<RT_MAX_PER_LANE>(a, bits, stream);
    }
    if (a->logits && a->T > 0) {
        const dim3 grid((unsigned)((a->T + 3) / 4));
        const float* lg = static_cast<const float*>(a->logits);
        float* tw = static_cast<float*>(a->topk_weight);
        const int T = (int)a->T, E = (int)a->E, topk = (int)a->topk;
        if (E <= 64) hipLaunchKernelGGL(route_topk_kernel<1>, grid, dim3(256), 0, stream, lg, tw, ids, T, E, topk);
        else if (E <= 128) hipLaunchKernelGGL(route_topk_kernel<2>, grid, dim3(256), 0, stream, lg, tw, ids, T, E, topk);
        else if (E <= 256) hipLaunchKernelGGL(route_topk_kernel<4>, grid, dim3(256), 0, stream, lg, tw, ids, T, E, topk);
        else if (E <= 512) hipLaunchKernelGGL(route_topk_kernel<8>, grid, dim3(256), 0, stream, lg, tw, ids, T, E, topk);
        else hipLaunchKernelGGL(route_topk_kernel<RT_MAX_PER_LANE>, grid, dim3(256), 0, stream, lg, tw, ids, T, E, topk);
        if (hipGetLastError() != hipSuccess) return MOE_ERR_LAUNCH;
    }
    if (nblocks > 1)
        hipLaunchKernelGGL(route_count_kernel, dim3((unsigned)nblocks), dim3(RT_BLOCK), 0, stream, ids, counts, n, (int)a->E);
    const int prefixed = nblocks > RT_FUSED_SCAN_MAX_BLOCKS ? 1 : 0;
    if (prefixed)
        hipLaunchKernelGGL(route_scan_kernel, dim3((unsigned)((a->E + 3) / 4)), dim3(256), 0, stream, counts, (int)a->E, nblocks);
    // one block even without choices: it writes group_list (all zeros then)
    const size_t lds = (size_t)17 * a->E * sizeof(int);
    static std::atomic<uint64_t> lds_set{0};
    if (const int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&route_rank_kernel), 17 * RT_MAX_E * (int)sizeof(int), lds_set))
        return rc;
    hipLaunchKernelGGL(route_rank_kernel, dim3((unsigned)(nblocks > 0 ? nblocks : 1)), dim3(RT_BLOCK), lds, stream, ids, counts,
                       static_cast<int64_t*>(a->group_list), static_cast<int32_t*>(a->row_token),
                       static_cast<int32_t*>(a->row_of_choice), n, (int)a->E, (int)a->topk, nblocks, prefixed, bits);
    if (hipGetLastError() != hipSuccess) return MOE_ERR_LAUNCH;
    if (a->x && n > 0) {
        hipLaunchKernelGGL(route_scatter_kernel, dim3((unsigned)a->T), dim3(256), 0, stream,
                           static_cast<const u32x4_t*>(a->x), static_cast<const int32_t*>(a->row_of_choice),
                           static_cast<u32x4_t*>(a->x_sorted), (int)a->topk, (int)(a->K / 8));
        if (hipGetLastError() != hipSuccess) return MOE_ERR_LAUNCH;
    }
    return MOE_OK;
}

}  // namespace moe
