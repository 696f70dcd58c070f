// Grouped GEMM with weight antiquant for MoE prefill on gfx950.
//
//   y[rows of expert g, :] = x[rows of expert g, :] . dequant(W[g])     bf16 x bf16 -> fp32 -> bf16
//
// Replaces grouped_matmul_antiquant (grouped_gemm/op_kernel/grouped_matmul_antiquant.h:225-364,
// grouped_matmul.h:147-463).  The reference decodes each weight slab to a bf16 copy in
// global memory and then runs a bf16 matmul on it; here the packed weights are decoded
// in registers straight into bf16 MFMA fragments and never go back to HBM.
//
// Work decomposition.  A tile is (expert, chunk of rows, 256 columns).  The tile list is derived
// inside the kernel from the device-resident cumulative group_list (no host sync); a persistent
// grid walks it with an XCD-aware order so that the workgroups of one XCD share the x rows and
// weight slices of the same experts in that XCD's L2, and takes the last two or three tiles of every
// workgroup from a work counter (see tile_queue).  Every wavefront owns its columns for ALL
// rows of the tile, so each weight element is dequantized exactly once per tile.  Three tile routines:
//   gemm_tile_pair  every quantized container (int4, int8, the K-contiguous fp4 containers, the
//                   reference's fp4 and fp8); x, packed weights and scales arrive by LDS-direct loads into a
//                   ring of stages walked by an unrolled k loop.  Either 8 wavefronts, the two of a SIMD
//                   splitting the k range (int8, fp8, K-contiguous fp4 in launches of few tiles), or 4 wavefronts
//                   that each take their 64 columns through all of k, two such workgroups per CU (int4 and fp4 prefill);
//                   tiles of up to 160 rows, or of up to 32 / 16 rows with small stages (decode batches,
//                   and the GEMV op's arithmetic on the N-contiguous containers)
//   gemm_tile_fp4_k the K-contiguous fp4 containers: 4 wavefronts, two workgroups per CU, tiles of up to 144 rows; x in a
//                   ring of 32-k stages, every wavefront's own weights and scales 256 k at a time
//   gemm_tile_bf16  the bf16 container: 8 wavefronts, tiles of up to 224 rows, x and weights by LDS-direct loads into
//                   two rings
//
// MFMA: v_mfma_f32_16x16x32_bf16.  Lane l = 16*q + i holds, for A, row i and
// k = 8q..8q+7 of the 16x32 block; for B, column i and the same k; for the result,
// column i and rows 4q..4q+3.  The contraction index may be permuted freely as long
// as A and B agree, and so may the column <-> (MFMA, lane) assignment; each weight
// container picks the assignment that makes its global loads wide and contiguous.
#include <algorithm>
#include <type_traits>

#include "moe_device.h"
#include "moe_internal.h"
#include "scale_group.h"

namespace moe {

constexpr int GM_BN = 256;     // columns per workgroup

struct GemmParams {
    const uint16_t* x;
    const uint8_t* w;
    const void* scale;
    const uint16_t* offset;
    const int64_t* gl;
    uint16_t* y;
    int64_t M;
    int K, N, G, scale_rows;
    int epilogue;   // moe_epilogue
    int slot;       // this launch's counter in tile_queue; -1: none, every tile in the fixed order
    unsigned long long stamp;   // what this launch raises its counter to before it draws from it
    // what the scheduler keeps in LDS: 3 the first tile of every expert, the experts' clamped row bounds and the order
    // in which the experts are taken (see order_experts); 2 the first two; 1 the
    // first tiles only (the row bounds are read from group_list per tile); 0 neither fits: the first tile of every
    // thread's run of experts only, and a tile is found by walking its run (any number of experts)
    int table_mode;
    // N-contiguous 4-bit containers: turns a 32-k sub-step index into its scale row
    ScaleRowDivider scale_div;
    int nt_rows;   // experts of up to so many rows: nontemporal weight loads, see nontemporal_rows
};

// Work queue of the persistent grid.  Workgroups do not run at one speed (of two that share a CU the one
// placed first runs about 1.5 times as fast as the other while both are resident, and the XCDs differ by a few
// per cent), so an even split of the tiles leaves most of the chip waiting for the slowest workgroup.  All but
// the last two or three tiles of a workgroup's share are handed out in a fixed, XCD-aware order; the rest
// (the tail) are taken one at a time, front to back, from a counter in the library's device memory.  (One
// counter per XCD, each for a run of its own or for every eighth chunk of the tail, and stealing between them
// at the end, kept more of the tail's reads in the XCDs' L2s but was 1.5 - 2 % slower on the prefill shapes and
// 5 % on the weight-streaming decode shapes.)
//
// A launch owns one slot = one 64-bit counter.  The host numbers the launches (64 bits, never reused); launch L
// uses slot L % GM_QUEUE_SLOTS and the stamp (L / GM_QUEUE_SLOTS + 1) << GM_QUEUE_COUNT_BITS, which grows with
// every use of the slot.  The first workgroups raise the counter to the stamp when they start (atomic max, fire and
// forget, one tile's time before anybody's first draw); a draw is a fetch-and-add, and the value it returns minus
// the stamp is the ticket.  Whatever an earlier launch left in the slot is smaller than the stamp and simply disappears, so
// nothing has to be cleared at the end of a kernel and no state a kernel leaves behind can mislead a later one.
// A launch that only starts after a later launch has taken its slot (its stream was held back for
// GM_QUEUE_SLOTS launches) sees that from the counter, which every workgroup reads once when it starts, and never draws:
// it walks all of its tiles in the fixed order and disturbs nobody.  A draw that returns a value outside
// [stamp, stamp + 2^GM_QUEUE_COUNT_BITS) means that the slot was taken over while this launch was running: the
// workgroup then walks its share of the tail in the fixed order -- tiles that were already handed out get
// computed twice, which only rewrites the same values -- but its stray draws have cost the later launch
// tickets, i.e. tiles: a launch that is still running when the GM_QUEUE_SLOTS-th launch after it starts is
// the one thing callers must not arrange.  A launch that is being captured into a HIP graph gets no slot at
// all (slot -1): its kernel node would keep slot and stamp for every replay while the ring moves on, so it
// walks all of its tiles in the fixed order.
constexpr int GM_QUEUE_SLOTS = 4096;
constexpr int GM_QUEUE_STRIDE = 8;        // 64-bit words per slot: a cache line of its own
constexpr int GM_QUEUE_TAIL_SWEEPS = 2;   // tiles per workgroup that are left to the counter (plus the remainder)
constexpr unsigned GM_QUEUE_COUNT_BITS = 24;
typedef unsigned long long queue_word_t;
__device__ queue_word_t tile_queue[GM_QUEUE_SLOTS * GM_QUEUE_STRIDE];
static std::atomic<uint64_t> queue_launches{0};   // launches of every kind of kernel in this file, for slot and stamp

// What a workgroup does with the launch's counter when it starts: it reads it (an ordinary load, issued ahead of the
// group_list loads and back with them) to see whether the slot is still this launch's, and the first 8 workgroups,
// one per XCD, raise it to the launch's stamp.  Not every workgroup: 512 atomics on one address at the start of a
// kernel held everybody's first loads up (tile table ready after 8 us instead of 2), and an atomic's own return
// value came back 2.5 us behind the loads.  A workgroup that draws before any of those stamps has arrived (it
// cannot be the usual case: draws start one tile into the kernel) gets a value below the stamp, takes it for a lost
// slot and does its share in the fixed order.
__device__ __forceinline__ bool queue_open(queue_word_t* q, queue_word_t stamp, bool stamps) {
    const queue_word_t now = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (stamps) (void)__hip_atomic_fetch_max(q, stamp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return now < stamp + (1ull << GM_QUEUE_COUNT_BITS);   // else: a later launch holds the slot
}
// A draw adds 1 to the counter's low word only (the count never carries out of it) and gets that word back: one
// register in flight instead of two in the tile routines, which have none to spare.  The word still shows the
// low 32 - GM_QUEUE_COUNT_BITS bits of the launch's use of the slot, enough to tell a slot that was taken over.
__device__ __forceinline__ unsigned queue_draw_raw(queue_word_t* q) {
    return __hip_atomic_fetch_add(reinterpret_cast<unsigned*>(q), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The ticket in a counter's low word raw, for a launch with the given stamp; -1: the slot is not this launch's
__device__ __forceinline__ int queue_ticket_of_draw(unsigned raw, queue_word_t stamp) {
    const unsigned d = raw - (unsigned)stamp;
    return d < (1u << GM_QUEUE_COUNT_BITS) ? (int)d : -1;
}
__device__ __forceinline__ int queue_draw(queue_word_t* q, queue_word_t stamp) { return queue_ticket_of_draw(queue_draw_raw(q), stamp); }
// A tile routine that is handed a counter draws the workgroup's next ticket from it while it finishes its own
// tile (the counter's round trip, about 3 us under load, overlaps the tile's reduction and stores) and leaves
// the ticket in *out behind its last barrier.
struct Ticket {
    queue_word_t* counter;   // null: the caller draws the ticket itself
    int* out;
    int* arrivals;           // a word of LDS for the tile routine's arrival counter (see gemm_tile_pair)
    int* wide;               // 5 words of LDS: not 0 if the tile is to be looked at again (see wide_scales), and its g, row0, rows, n0
};

// Buffer resources keep the addressing compact: one 128-bit descriptor in SGPRs per
// tensor slab, one 32-bit per-lane offset that is constant for the whole tile, and a
// wave-uniform (scalar) offset per load.  Reads beyond the slab return 0.
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t make_rsrc(const void* p, int64_t bytes) {
    const uint32_t n = bytes > 0xffffffffLL ? 0xffffffffu : (uint32_t)bytes;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, n, 0x00020000);
}
// D = A * B + D with the accumulator tied in place.  Written as inline asm because the
// compiler, given many live accumulators, stops accumulating in place and shuttles them
// through copies, which halves the MFMA rate.  Hazards: A/B come from VALU or waited
// loads (interlocked); accumulators are only read by other MFMAs until the epilogue,
// which waits out the MFMA latency first.  (The accumulators are ordinary VGPRs: a kernel that uses no AGPRs at all may
// use the whole unified register file as VGPRs, otherwise the compiler splits it in two halves.)
__device__ __forceinline__ void mfma_16x16x32_v(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
}

// ---------------------------------------------------------------------------------
// x tile: rows x BK bf16 in LDS, 16-byte chunks, chunk c of row r stored at
// position c ^ (r & 7) so that the 8 lanes a ds_read_b128 serves together hit
// distinct banks both when writing (consecutive chunks of one row) and when
// reading fragments (same chunk of 8 consecutive rows).
// ---------------------------------------------------------------------------------
template <int BK>
__device__ __forceinline__ int a_lds_unit(int row, int c) {
    return row * (BK / 8) + (c ^ (row & 7));
}

// The same for tile rows of 32 k (four 16-byte chunks, 64 bytes): chunk c of row r at position c ^ ((r >> 1) & 3).
// A 16-byte LDS read is served 8 lanes (128 bytes of banks) at a time: the 8 consecutive rows such a group reads the
// same chunk of then lie in 8 different 16-byte slots modulo 128 bytes (two rows share a 128-byte line; the pairs
// take the four positions in turn).  (With (r >> 2) & 3 in its place the counters showed two lanes per slot:
// SQ_LDS_BANK_CONFLICT at 39 % of the cycles the LDS was active.)
__device__ __forceinline__ int a_lds_unit32(int row, int c) {
    return row * 4 + (c ^ ((row >> 1) & 3));
}

// ---------------------------------------------------------------------------------
// LDS-direct loads (buffer_load_dwordx4 ... lds): lane l of the wavefront writes bytes
// [16 l, 16 l + 16) after the instruction's LDS base.  No staging registers and no LDS store
// instructions, so a tile routine can keep a ring of stages filled several k steps (a few
// microseconds of HBM latency) ahead of their use.
// ---------------------------------------------------------------------------------
#define MOE_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))
__device__ __forceinline__ void lds_load16(rsrc_t r, const u32x4_t* dst, int voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, MOE_LDS_PTR(const_cast<u32x4_t*>(dst)), 16, voff, soff, 0, 0);
}
// The same with the destination as a byte address in LDS (wave-uniform).
__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)MOE_LDS_PTR(p));
}
// AUX: LOAD_NT, or 0.
constexpr int LOAD_NT = 2;   // nontemporal
template <int AUX = 0>
__device__ __forceinline__ void lds_load16_at(rsrc_t r, uint32_t dst, int voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(uintptr_t)dst, 16, voff, soff, 0, AUX);
}
// A wave-uniform value the compiler must take as it finds it: whatever is derived from the result is computed
// where it is used instead of once per variant ahead of an unrolled loop (where it would occupy an SGPR each).
__device__ __forceinline__ uint32_t here(uint32_t v) {
    asm volatile("" : "+s"(v));
    return v;
}

// ---------------------------------------------------------------------------------
// Tile routine for the quantized containers (int4, int8, reference fp4 / fp8, K-contiguous fp4) with two
// wavefronts per SIMD that split the k range.  Described for int4; what differs for the others follows.
//
// A single wavefront issues at most one instruction every ~5 cycles whatever its kind, and an
// MFMA holds the SIMD's vector issue port for about 8 of its 16 cycles: with one wavefront
// per SIMD the decode instructions and the MFMAs of a k step add up instead of overlapping.
// Here the workgroup has 8 wavefronts.  Wavefront wv owns the 64 columns of group wv & 3 for
// all rows of the tile (4 MFMAs per x fragment), but only one of the two 32-k sub-steps of
// every 64-k step: the pair (wv, wv + 4) shares a SIMD and accumulates two partial sums that
// are added once per tile through LDS.  Every weight element is still decoded exactly once
// per tile, a lane decodes 4 nibbles of a dword at a time (2.25 VALU instructions per
// element), and each wavefront reads half of the x fragments.
//
// Each wavefront alternates a decode phase (its sub-step of the packed stage -> 4 bf16 B
// fragments in registers) and an MFMA phase; one wavefront of a SIMD multiplies while the other
// decodes.  The steps of the 8 wavefronts are tied together by a split barrier, an arrival counter
// in LDS (see ring_arrive / ring_wait in gemm_tile_pair): a wavefront that is done with a step says
// so and goes on decoding the next one; it waits for the others only in front of its next MFMA phase.
//
// Everything the k loop consumes -- x tile, packed weight tile, scales -- is brought in by
// LDS-direct loads into a ring of S = 5 stages.  The loads of stage kt+4 (it replaces stage kt-1,
// which every wavefront has left when all have arrived kt times) and the LDS reads of the packed
// dwords of stage kt+1 are spread between the MFMAs of step kt; before it arrives at the end of step
// kt each wavefront waits until its own loads of stage kt+2 have landed.  vmcnt counts a wavefront's loads in order and every
// wavefront issues the same number NI of them per step (waves without a row block of their
// own repeat one: measured, the repeated loads cost nothing, a branch around them does), so "at most
// (S - 3) NI outstanding" means exactly that.
//
// Decode of a k-row pair (a, b) of one dword column: v_perm gathers the two bytes of each row this lane owns, row a's
// into the low, row b's into the high half of a dword.  Masked with 0x000f and put under 0x6400 a half is the fp16
// 1024 + q (0x00f0: 1024 + 16 q), so v_fma_mix_f32 converts a weight and takes its scale and the zero point in one
// instruction: (1024 + q) s - 1032 s, or (1024 + 16 q) s / 16 - 72 s, is (q - 8) s exactly (12 bits).
// From scales of 2^117.98 on 1032 s is beyond fp32 and the weight no number: see wide_scales.
// 2.25 instructions per weight; masks, conversions from e4m3 and fmas took 2.5.  us, before / now: a prefill layer of 4096
// tokens x 8 on 256 experts of 7168 x 2048 2883 / 2842, decode layers of 64 x 8 and 16 x 8 1059 / 998 and 413 / 391, 512 rows
// on 64 experts of 2048 x 4096 122 / 117.
//
// The same routine serves the reference's pre-shuffled fp4 container: its 64 x 128-byte tile is
// brought in by the same loads, a lane's 8 k rows of its 2 bytes are two 16-byte LDS reads, each
// byte pair decodes to 4 floats with v_cvt_scalef32_pk_f32_fp4 and takes one multiply by the
// column's scale of that 16-k block (4 scale rows per step instead of 2).
//
// int8 and the reference fp8 container: a step's tile is 64 rows of 256 bytes (two load instructions
// per wavefront), which leaves room for S = 4 stages; a lane's 4 columns are one dword of each of its 8 k
// rows.  int8 keeps its per-channel scale and offset in registers (and folds them into one fma where that gives
// the bits of the two rounded operations, see i8_one_rounding); fp8 decodes two codes at a time by the hardware's
// conversions, or where a code is NaN to those through fp16 (see decode_f8_plain), and gets the fp32 scale of its
// 128 x 128 block through the ring, 4 bytes per wavefront and step.
//
// K-contiguous fp4 (weight [N, K/2]): a step's tile is 256 weight rows x 32 bytes; MFMA t of a lane takes
// weight row 64 cw + 16 t + i, whose 8 codes of the sub-step are one dword; the scales [N, K/block] are
// fetched 16 bytes per row at a time into buffers of their own (see kc_issue_scale).
// ---------------------------------------------------------------------------------
// Kernel variants.
//   GK_PAIR     quantized containers: 8 wavefronts, k range split between the two wavefronts of a SIMD, tiles of
//               up to 160 rows
//   GK_PAIR_SMALL  GK_PAIR with tiles of at most 32 rows: x stages of 4 KB leave LDS for a second workgroup per
//               CU (decode-sized batches on the 4-bit containers)
//   GK_PAIR_EXACT  GK_PAIR_SMALL with the GEMV op's arithmetic (weights not rounded to bf16)
//   GK_PAIR_EXACT16  GK_PAIR_EXACT with tiles of at most 16 rows (the fp4 container: its 32-row tile routine
//               needs 153 registers, the 16-row one 97, which lets two workgroups share a CU)
//   GK_QUAD     the large tiles of GK_PAIR without the k split: workgroups of 4 wavefronts, each wavefront takes its
//               64 columns through the whole k range in steps of 32 k, two workgroups per CU.  The two wavefronts
//               of a SIMD belong to different workgroups and work on different tiles: no partial sums to
//               exchange, a barrier spans 4 wavefronts instead of 8, and while one workgroup is between two tiles
//               (stores, tile search, first loads) the other has the SIMDs to itself.  (The N-contiguous containers.)
//   GK_FP4_K    gemm_tile_fp4_k
//   GK_BF16     gemm_tile_bf16
//   GK_BF16_128 the same with tiles of at most 128 rows (a limit read at run time instead costs the small calls of either 1.5 %)
enum { GK_PAIR = 2, GK_PAIR_EXACT = 3, GK_PAIR_SMALL = 4, GK_PAIR_EXACT16 = 5, GK_QUAD = 6, GK_BF16 = 7, GK_BF16_128 = 8, GK_FP4_K = 9 };
constexpr bool pair_exact(int kind) { return kind == GK_PAIR_EXACT || kind == GK_PAIR_EXACT16; }
constexpr int pair_waves(int kind) { return kind == GK_QUAD ? 4 : 8; }
constexpr int pair_bk(int kind) { return kind == GK_QUAD ? 32 : 64; }   // k per step

constexpr int PAIR_CAPB = PAIR_ROWS / 16;             // x stages hold 160 rows
constexpr int PAIR_MT_MAX = 10;
constexpr int PAIR_SMALL_MT_MAX = 2;                  // row blocks per tile of the small-stage kinds
constexpr bool pair_small(int kind) { return kind != GK_PAIR && kind != GK_QUAD; }
// 16-byte units of one x stage: 160 rows, or the 32 rows of the small-stage kinds
constexpr int pair_mt_max(int kind) { return !pair_small(kind) ? PAIR_MT_MAX : kind == GK_PAIR_EXACT16 ? 1 : PAIR_SMALL_MT_MAX; }
constexpr int pair_a_units(int kind) { return 16 * (pair_small(kind) ? pair_mt_max(kind) : PAIR_CAPB) * (pair_bk(kind) / 8); }
// packed tile of one k step: rows of 128 bytes (4-bit codes) or of 256 bytes (int8, fp8)
template <int FMT>
constexpr int pair_b_units(int kind) { return pair_bk(kind) * ((FMT == MOE_FMT_INT8 || FMT == MOE_FMT_FP8_REF) ? 16 : 8); }
// Small-stage kinds on the 4-bit N-contiguous containers: two workgroups per CU, one computes while the other
// waits at its barrier or between two tiles (512 rows over 256 experts of 7168 x 2048: int4 425 -> 387 us, fp4
// 440 -> 425 us; the fp4 tile routine with the GEMV op's arithmetic fits four wavefronts per SIMD only in its
// 16-row form).  A deeper ring in the LDS the small x stages free does not pay instead (fp4 10 stages
// 515 us against 510 us with 5; fp8 7 stages 572 us against 552 us with 4: a tile's first stages take longer
// to fill), and the one-byte containers at two workgroups per CU are left with 3 stages (fp8 641 us).
template <int FMT>
constexpr int pair_wg_per_cu(int kind) {
    if (kind == GK_QUAD) return 2;
    if (!pair_small(kind)) return 1;
    return (FMT == MOE_FMT_INT4 || (FMT == MOE_FMT_FP4_REF && kind != GK_PAIR_EXACT)) ? 2 : 1;
}
// ring depth: what fits into LDS next to the 160-row x stages; the 4-wavefront kind runs best with 4 stages (a tile's
// first stages are filled sooner: int4 1790 against 1818 us at K = 7168, 949 against 952 us at K = 2048)
template <int FMT>
constexpr int pair_stages(int kind) { return (FMT == MOE_FMT_INT8 || FMT == MOE_FMT_FP8_REF || kind == GK_QUAD) ? 4 : 5; }
// 16-byte units of scales per k step: rows of 256 bf16, int4 one per 32-k sub-step (groups are multiples
// of 32), the reference fp4 container one per 16 k; fp8 one unit per wavefront holding the fp32 scale of
// its 128 x 128 block; int8 none (per-channel scales stay in registers)
template <int FMT>
constexpr int pair_sc_units(int kind) {
    return (FMT == MOE_FMT_FP4_REF ? 128 : FMT == MOE_FMT_INT4 ? 64 : FMT == MOE_FMT_FP8_REF ? 8 : 0) * pair_bk(kind) / 64;
}
// The K-contiguous fp4 containers keep their scales [N, K/block] outside the stages: 16 bytes (2 or 4 steps'
// worth) per weight row at a time, three buffers of 256 rows
template <int FMT>
constexpr int pair_kc_scale_units() { return (FMT == MOE_FMT_FP4_B32 || FMT == MOE_FMT_FP4_B16) ? 3 * 256 : 0; }
// GK_QUAD, tiles of up to 3 row blocks: they wait for their weights, of which 3 stages ahead of two workgroups are 30 KB on their way
// per CU, enough for about 4 TB/s; their x needs little of the LDS, so they get 6 stages.  us, 4 / 6 stages: 16 rows each on 256
// experts of 7168 x 2048, fp4 514 / 459, int4 519 / 476; 1511 tokens x 8 unevenly routed over the same, fp4 SwiGLU 568 / 540, int4
// (skew 1) 584 / 551; 5600 rows on 64 of 2048 x 4096, fp4 131 / 124.  8 stages are no faster, and with 4 or 5 row blocks fp4 loses (64 rows
// each on 128 experts 327 / 331).  A launch with a tile per workgroup at most keeps 4: it gains nothing from more and pays for fetching
// the code of the longer ring (416 rows on 16 of 3328 x 2048: 42.0 / 43.2).  The one-byte containers are here for experts of many rows.
constexpr int QUAD_DEEP_MT = 3, QUAD_DEEP_STAGES = 6;
// Row blocks of the largest tiles that have a form with nontemporal weight loads (see nontemporal_rows)
constexpr int nt_mt_max(int kind) { return kind == GK_PAIR ? 4 : kind == GK_QUAD ? 0 : 1; }
// Rounded weights of int4 and fp8: the usual decodes take scales below 2^117.98 (int4) and 2^120 (fp8, columns with a 0x7F or 0xFF among
// the wavefront's codes).  A tile with a larger one has columns that are no number; a wavefront that finds one in its sums says so in LDS
// (Ticket::wide), and the workgroup then looks whether such a scale is the reason and if so computes the tile once more, 16 rows at a
// time, with a decode that takes all scales (redo_wide).  A check of the scales in every step instead, with a branch: int4 1.3 to 2.5 % slower in
// decode-like launches, 0.6 to 1.2 % in others; fp8 with random codes 2 to 3 %.
template <int FMT>
constexpr bool wide_scales(int kind) { return (FMT == MOE_FMT_INT4 || FMT == MOE_FMT_FP8_REF) && !pair_exact(kind); }
template <int FMT>
constexpr int pair_lds_units(int kind) {
    return pair_stages<FMT>(kind) * (pair_a_units(kind) + pair_b_units<FMT>(kind) + pair_sc_units<FMT>(kind)) + pair_kc_scale_units<FMT>();
}

// End of a k-split tile.  The two wavefronts of a pair (same columns, the two k halves) hold partial sums of the
// whole tile; each hands the row blocks the other will finish to it through LDS, adds what it receives to the
// row blocks it keeps and stores those: the first half of the tile's 16-row blocks is finished by the h == 0
// wavefront, the second by h == 1, so both reduce and store at the same time.  Rounds of at most 4 row
// blocks (8 wavefronts x 4 blocks x 4 KB fit the x stage area, free now).
// WHOLE: the wavefront holds the whole sums (no k split): it stores all of its row blocks, nothing is exchanged.
template <int MT, bool KC, bool WHOLE = false>
__device__ __forceinline__ void pair_finish(const GemmParams& P, u32x4_t* smem, f32x4_t (&acc)[MT][4], int h, int cw, int lane,
                                            int col0, int64_t row0, int rows, int n0, const Ticket& tk) {
    const int i = lane & 15, q = lane >> 4;
    const bool takes = tk.counter != nullptr && threadIdx.x == 0;
    unsigned next_tile = 0;
    if (takes) next_tile = queue_draw_raw(tk.counter);
    constexpr int MH = (MT + 1) / 2, RR = MH < 4 ? MH : 4, ROUNDS = (MH + RR - 1) / RR;
    // the last tile of an N that is not a multiple of 256 (the reference's fp8 container: multiples of 128)
    // computes columns past N from whatever follows in the slab: they are not stored
    const bool live = KC || n0 + col0 < P.N;
    const bool swi = P.epilogue == MOE_EPILOGUE_SWIGLU;
    // stores go through a buffer resource that ends after the tile's last valid row: those to padded rows
    // fall outside it and are dropped
    const int NO = swi ? P.N >> 1 : P.N;
    const rsrc_t ry = make_rsrc(P.y + row0 * (int64_t)NO, (int64_t)rows * NO * 2);
    auto store_block = [&](int mt) {
        if (!live) return;
        if (swi && KC) {
            // K-contiguous containers: the weight rows come in blocks of 32 = (16 gate rows, 16 up rows), which are
            // the MFMAs t = (0, 1) and (2, 3) of this lane; y has N / 2 columns
            const int vo = (4 * q * NO + ((n0 + 64 * cw) >> 1) + i) * 2;
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    __builtin_amdgcn_raw_buffer_store_b16(
                        (uint16_t)(pack_bf16_rne(swiglu(acc[mt][2 * u][r], acc[mt][2 * u + 1][r]), 0.f) & 0xffffu), ry,
                        vo + 32 * u, (16 * mt + r) * NO * 2, 0);
        } else if (swi) {
            // this lane's 4 columns are (gate, gate, up, up) of 2 output columns; y has N / 2 columns
            const int vo = (4 * q * NO + ((n0 + col0) >> 1)) * 2;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                __builtin_amdgcn_raw_buffer_store_b32(
                    pack_bf16_rne(swiglu(acc[mt][0][r], acc[mt][2][r]), swiglu(acc[mt][1][r], acc[mt][3][r])), ry, vo,
                    (16 * mt + r) * NO * 2, 0);
        } else if (KC) {
            // K-contiguous containers: MFMA t holds column 64 cw + 16 t + i, one 2-byte store each
            const int vy = (4 * q * P.N + n0 + 64 * cw + i) * 2;
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(pack_bf16_rne(acc[mt][t][r], 0.f) & 0xffffu), ry,
                                                          vy + 32 * t, (16 * mt + r) * P.N * 2, 0);
        } else {
            const int vy = (4 * q * P.N + n0 + col0) * 2;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                u32x2_t v;
                v[0] = pack_bf16_rne(acc[mt][0][r], acc[mt][1][r]);
                v[1] = pack_bf16_rne(acc[mt][2][r], acc[mt][3][r]);
                __builtin_amdgcn_raw_buffer_store_b64(v, ry, vy, (16 * mt + r) * P.N * 2, 0);
            }
        }
    };
    // Barrier between the LDS writes and reads of the exchange: it orders LDS traffic only.  (__syncthreads
    // would also wait for this wavefront's global stores of the previous round to complete, 2-3 us each time.)
    auto lds_barrier = []() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    // H: which half this wavefront finishes (a compile-time constant in each branch, so that every register
    // index is one); both kinds of wavefront take the same barriers
    auto finish = [&](auto HC) __attribute__((always_inline)) {
        constexpr int H = decltype(HC)::value;
        constexpr int KEEP0 = H == 0 ? 0 : MH, KEEPN = H == 0 ? MH : MT - MH;
        constexpr int SEND0 = H == 0 ? MH : 0, SENDN = MT - KEEPN;
        u32x4_t* out_slot = smem + (cw * 2 + (1 - H)) * (RR * 4 * 64) + lane;
        const u32x4_t* in_slot = smem + (cw * 2 + H) * (RR * 4 * 64) + lane;
#pragma unroll
        for (int rd = 0; rd < ROUNDS; ++rd) {
            if (rd > 0) lds_barrier();   // the previous round's slots are read
#pragma unroll
            for (int b = rd * RR; b < (rd + 1) * RR && b < SENDN; ++b)
#pragma unroll
                for (int t = 0; t < 4; ++t) out_slot[((b - rd * RR) * 4 + t) * 64] = __builtin_bit_cast(u32x4_t, acc[SEND0 + b][t]);
            lds_barrier();
#pragma unroll
            for (int b = rd * RR; b < (rd + 1) * RR && b < KEEPN; ++b) {
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[KEEP0 + b][t] += __builtin_bit_cast(f32x4_t, in_slot[((b - rd * RR) * 4 + t) * 64]);
                store_block(KEEP0 + b);
            }
        }
    };
    if constexpr (WHOLE) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) store_block(mt);
    } else if (h == 0) {
        finish(std::integral_constant<int, 0>{});
    } else {
        finish(std::integral_constant<int, 1>{});
    }
    if (takes) *tk.out = queue_ticket_of_draw(next_tile, P.stamp);
    lds_barrier();   // the slots are read: the next tile may load into the ring (the stores are still in flight)
}

// EXACT selects the arithmetic of the GEMV op (grouped_soft_gemv/op_kernel/gemv_impl.h:147-199: the
// dequantized weights stay fp32): the B fragments then hold the codes themselves, which are exact in
// bf16, every MFMA covers k of one scale group only and its result is multiplied by that group's fp32
// scale on the way into the accumulators.  The fp4 container has a scale per 16 k, half an MFMA: the x
// fragment is split into its lanes q < 2 and q >= 2 (the other half zeroed) and each half takes its
// own MFMA.  These MFMAs are compiler-visible builtins (their results feed ordinary VALU code).
//
// STACK2 (that arithmetic on the fp4 container, tiles of at most 8 rows): the two scale groups of an MFMA's 32 k
// are told apart by the row of the 16 x 16 product instead of by two MFMAs.  Row r < 8 of the x fragment holds
// x row r in its first 16 k and zeros in the others, row 8 + r holds x row r in the last 16 k only (the zeros are
// read from the rows 8..15 of the x stage, which are padding for such a tile).  One MFMA per 16 columns then
// leaves the first group's sums in the lanes q < 2 and the second group's in q >= 2, each lane applies the
// scale of its own group, and the two halves are added once at the end of the tile: half the MFMAs and half
// the multiplies of the general case, and no masking.
//
// DEEP (GK_QUAD, small tiles): the longer ring, see QUAD_DEEP_STAGES.  NT: nontemporal loads of the weights, see nontemporal_rows.
// WIDE: int4 and fp8 with any scale, see wide_scales.
template <int FMT, int MT, int KIND, bool STACK2 = false, bool DEEP = false, bool NT = false, bool WIDE = false>
__device__ __forceinline__ void gemm_tile_pair(const GemmParams& P, u32x4_t* smem, int g, int64_t row0, int rows, int n0, const Ticket& tk) {
    static_assert(FMT != MOE_FMT_BF16, "the k-split tile routine decodes quantized containers");
    constexpr bool EXACT = pair_exact(KIND);
    static_assert(!STACK2 || (EXACT && FMT == MOE_FMT_FP4_REF && MT == 1), "two scale groups stacked in one MFMA: fp4, at most 8 rows");
    static_assert(!EXACT || FMT == MOE_FMT_INT4 || FMT == MOE_FMT_FP4_REF || FMT == MOE_FMT_FP8_REF,
                  "un-rounded weights: the N-contiguous containers of the GEMV op");
    constexpr bool FP4 = FMT == MOE_FMT_FP4_REF, I8 = FMT == MOE_FMT_INT8, F8 = FMT == MOE_FMT_FP8_REF;
    // K-contiguous fp4 (weight [N, K/2], scales [N, K/KBLK]): the step's tile is 256 weight rows x 32 bytes
    constexpr bool KC = FMT == MOE_FMT_FP4_B32 || FMT == MOE_FMT_FP4_B16;
    constexpr int KBLK = FMT == MOE_FMT_FP4_B32 ? 32 : 16;
    constexpr bool B8 = I8 || F8;   // one byte per weight: tiles of 64 rows x 256 bytes
    // Q4: the kind without the k split (GK_QUAD): 4 wavefronts, steps of 32 k, every wavefront in every step
    constexpr bool Q4 = KIND == GK_QUAD;
    static_assert(!Q4 || FMT == MOE_FMT_INT4 || FMT == MOE_FMT_INT8 || FMT == MOE_FMT_FP4_REF || FMT == MOE_FMT_FP8_REF,
                  "the 4-wavefront kind serves the N-contiguous containers");
    constexpr int NW = pair_waves(KIND);
    constexpr int BK = pair_bk(KIND), S = DEEP ? QUAD_DEEP_STAGES : pair_stages<FMT>(KIND), PAIR_SC_UNITS = pair_sc_units<FMT>(KIND);
    constexpr int PAIR_B_UNITS = pair_b_units<FMT>(KIND);
    constexpr int AHEAD = S - 1;   // a step's loads fill the stage of step kt + AHEAD
    // Kinds of which two workgroups share a CU (decode batches, HBM bound) keep one s_barrier per step, placed so
    // that the two wavefronts of a SIMD alternate (those of sub-step 0 take it after their MFMA phase, those of
    // sub-step 1 half way through their decode); with one workgroup per CU the split barrier described below is
    // faster (measured on 512 rows over 256 experts of 7168 x 2048: two per CU 335 against 340 us (int4), 390 against
    // 395 us (fp4) with the plain barrier; one per CU, fp8, 555 against 580 us with the split one).
    constexpr bool SPLIT_BARRIER = pair_wg_per_cu<FMT>(KIND) == 1;
    constexpr int PAIR_A_UNITS = DEEP ? 64 * MT : pair_a_units(KIND);
    // The next step's packed dwords are read ahead of the MFMAs instead of behind the first ones: with 4 or 8 MFMAs a step their
    // latency otherwise ends in the next decode (int4, a tile per CU, 2 rows: 64 experts of 2048 x 1024 22.6 / 21.3 us).
    // fp4 gains nothing from it, the GEMV op's kinds lose 0.5 to 4 %: they still need the scales of the step being multiplied.
    constexpr bool EARLY_RAW = FMT == MOE_FMT_INT4 && KIND == GK_PAIR_SMALL;
    constexpr int W_AUX = NT ? LOAD_NT : 0;   // (fp4: of the scales too, whose rows are read once; those of int4 serve four steps)
    static_assert(S * (PAIR_A_UNITS + PAIR_B_UNITS + PAIR_SC_UNITS) <= pair_lds_units<FMT>(KIND), "stages beyond the LDS of the kernel");
    static_assert(16 * MT * (BK / 8) <= PAIR_A_UNITS, "tile rows beyond the x stage");
    u32x4_t* lds_a = smem;
    u32x4_t* lds_b = lds_a + S * PAIR_A_UNITS;
    u32x4_t* lds_s = lds_b + S * PAIR_B_UNITS;

    // (the thread id is taken as found: what is derived from it is worked out per tile and does not hold
    // registers from tile to tile, where the routine has none to spare)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int i = lane & 15, q = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cw = wv & 3;                                    // column group: 64 columns
    // the sub-step of every step this wavefront owns (Q4: a step is one sub-step)
    const int h = Q4 ? 0 : 1 - (wv >> 2);
    // this lane's 4 columns (MFMA t = column col0 + t): half of a dword of 8 4-bit codes, or a dword of 4 bytes
    const int col0 = B8 ? 64 * cw + 4 * i : 128 * (cw >> 1) + 8 * i + 4 * (cw & 1);
    const int nk = P.K / BK;

    const int64_t KN = (int64_t)P.K * P.N;
    const rsrc_t rw = B8 ? make_rsrc(P.w + g * KN, KN) : make_rsrc(P.w + g * (KN >> 1), KN >> 1);
    const rsrc_t rs = KC ? make_rsrc(static_cast<const uint16_t*>(P.scale) + g * (KN / KBLK), (KN / KBLK) * 2)
                         : make_rsrc(static_cast<const uint16_t*>(P.scale) + (int64_t)g * P.scale_rows * P.N,
                                     (int64_t)P.scale_rows * P.N * 2);
    // fp8: the expert's fp32 block scales [K/128, N/128]; this wavefront's 128-column block
    const rsrc_t rs8 = make_rsrc(static_cast<const float*>(P.scale) + (int64_t)g * (P.K >> 7) * (P.N >> 7),
                                 (int64_t)(P.K >> 7) * (P.N >> 7) * 4);
    const int cs8 = ((n0 + 64 * cw) >> 7) * 4;
    auto scale_row = [&](uint32_t sub) { return (int)moe::scale_row(P.scale_div, sub); };
    // x rows through a buffer resource that ends after the last valid row (padded rows read as
    // zeros).  Load instruction j covers rows 8j + (lane >> 3); position lane & 7 of a row
    // holds chunk (lane & 7) ^ (row & 7), the swizzle a_lds_unit expects.
    // (Q4, rows of 64 bytes: instruction j covers rows 16j + (lane >> 2); position lane & 3 of a row holds
    // chunk (lane & 3) ^ ((row >> 1) & 3), see a_lds_unit32)
    const rsrc_t rx = make_rsrc(P.x + row0 * (int64_t)P.K, (int64_t)rows * P.K * 2);
    const int va = Q4 ? ((lane >> 2) * P.K + (((lane & 3) ^ ((lane >> 3) & 3)) * 8)) * 2
                      : ((lane >> 3) * P.K + (((lane & 7) ^ (lane >> 3)) * 8)) * 2;
    // packed tile: instruction wv brings rows 8 wv + (lane >> 3) into the 1 KB block wv of the stage;
    // the two 64-byte halves of the rows with odd (row >> 3) are swapped, so that the four q groups
    // of a wavefront read from both halves of the banks
    // int8 / fp8 (rows of 256 bytes): instruction e of wavefront wv brings rows 8 wv + 4 e + (lane >> 4); the
    // 64-byte quarters of a row are permuted by (row >> 3) & 3 = wv & 3, so that the four q groups read
    // from different quarters of the banks
    // K-contiguous fp4: LDS unit 64 wv + lane of the stage holds one 16-byte half of weight row
    // n = 32 wv + (lane >> 1); the halves of the rows with odd (n >> 3) are swapped (bank spread)
    const int kc_n = 32 * wv + (lane >> 1);
    const int vb = KC   ? kc_n * (P.K >> 1) + 16 * ((lane & 1) ^ ((kc_n >> 3) & 1))
                   : B8 ? (lane >> 4) * P.N + (((lane & 15) ^ (4 * (wv & 3))) * 16)
                        : (lane >> 3) * (P.N >> 1) + (((lane & 7) ^ (4 * (wv & 1))) * 16);
    constexpr int XI = Q4 ? MT : 2 * MT;          // x load instructions per step (1 KB each: 16 or 8 rows)
    constexpr int XROWS = Q4 ? 16 : 8;
    constexpr int NA = (XI + NW - 1) / NW;        // ... per wavefront
    constexpr int NB = B8 ? 2 : 1;                // packed-tile instructions
    constexpr int NI = NA + NB + ((PAIR_SC_UNITS || KC) ? 1 : 0);   // + this wavefront's share of the step's scales
    int ja[NA], ca[NA];
#pragma unroll
    for (int m = 0; m < NA; ++m) {
        int j = wv + NW * m;
        if (NW * NA > XI) j = j % XI;   // repeat a block rather than issue fewer loads
        ja[m] = j * 64;
        ca[m] = XROWS * j * P.K * 2;
    }
    // (Q4 on the reference's fp4 container: the 32 k of a step are the rows [16 hp, +16) and [32 + 16 hp, +16) of the
    // container's 64-row tile, hp = step & 1: wavefront wv brings the 8 rows from 32 (wv >> 1) + 16 hp + 8 (wv & 1) on)
    const int cb = KC            ? n0 * (P.K >> 1)
                   : B8          ? 8 * wv * P.N + n0
                   : (Q4 && FP4) ? (32 * (wv >> 1) + 8 * (wv & 1)) * (P.N >> 1) + (n0 >> 1)
                                 : 8 * wv * (P.N >> 1) + (n0 >> 1);
    const int kb_step = KC ? BK / 2 : B8 ? BK * P.N : BK * (P.N >> 1);
    // byte offset of step kp's packed rows in the expert's slab
    auto b_step_offset = [&](int kp) {
        if constexpr (Q4 && FP4)
            return ((kp >> 1) * 64 + (kp & 1) * 16) * (P.N >> 1);
        else
            return kp * kb_step;
    };
    // K-contiguous fp4 scales.  Fetching the 4 or 8 bytes a weight row needs per step costs a request per
    // row and step (measured: 20 % of the kernel); instead 16 bytes of a row -- the scales of SUP steps --
    // are fetched at a time: the load slot of step kt brings, for step index kp = kt + KC_D, the rows
    // [RPS (kp % SUP), + RPS) of super-block kp / SUP (one lane per row, RPW rows per wavefront) into buffer
    // (kp / SUP) % 3 of 256 rows x 16 bytes behind the stages.  KC_D = SUP + 3: a load issued in step t is
    // visible after barrier t + 2, and the scales of step s are read during step s - 1.  Three buffers: the
    // first load into a buffer comes after the last read of its previous occupant.
    constexpr int SUP = KBLK == 32 ? 4 : 2, KC_D = SUP + 3, RPS = 256 / SUP, RPW = RPS / 8;
    const int kc_vs = lane * (P.K / KBLK) * 2;
    auto kc_issue_scale = [&](int kp) {
        const int sb = kp / SUP, j = kp % SUP, row = RPS * j + RPW * wv;
        if (lane < RPW)
            lds_load16(rs, lds_s + (sb % 3) * 256 + row, kc_vs, (n0 + row) * (P.K / KBLK) * 2 + sb * 16);
    };
    // scales of a step: int4 2 rows of 512 bytes, 128 bytes (8 lanes) per wavefront: bytes [128 (wv & 3), +128) of
    // row wv >> 2; fp4 4 rows (one per 16 k), 256 bytes (16 lanes) per wavefront: bytes [256 (wv & 1), +256) of row wv >> 1
    const int cs = FP4 ? n0 * 2 + (wv & 1) * 256 : n0 * 2 + (wv & 3) * 128;
    const int lane16 = lane * 16;
    const bool s_lane = lane < (FP4 ? 16 : 8);
    // where this wavefront's loads land in stage 0 (byte addresses in LDS)
    uint32_t a_at[NA];
#pragma unroll
    for (int m = 0; m < NA; ++m) a_at[m] = lds_address(lds_a + ja[m]);
    const uint32_t b_at = lds_address(lds_b + wv * (PAIR_B_UNITS / NW));
    const uint32_t s_at = lds_address(lds_s + wv * (F8 ? 1 : PAIR_SC_UNITS / NW));
    // m-th load of group kt (stage kt+AHEAD of x, packed tile and scales), into LDS stage ST
    auto issue = [&](int m, int kt, int ST) {
        if (m < NA) {
            lds_load16_at(rx, here(a_at[m]) + ST * (PAIR_A_UNITS * 16), va, ca[m] + (kt + AHEAD) * (BK * 2));
        } else if (m < NA + NB) {
            const int e = m - NA;
            lds_load16_at<W_AUX>(rw, here(b_at) + ST * (PAIR_B_UNITS * 16) + e * 1024, vb,
                          cb + (B8 ? 4 * e * P.N : 0) + b_step_offset(kt + AHEAD));
        } else if constexpr (KC) {
            kc_issue_scale(kt + KC_D);
        } else if constexpr (F8) {
            // the block scale of the stage's 128-k block, 4 bytes by lane 0 (past K: reads as 0, unused)
            if (lane == 0)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rs8, (__attribute__((address_space(3))) void*)(uintptr_t)(here(s_at) + ST * (PAIR_SC_UNITS * 16)), 4, 0,
                    ((kt + AHEAD) >> (Q4 ? 2 : 1)) * (P.N >> 7) * 4 + cs8, 0, 0);
        } else {
            const int grow = FP4  ? (kt + AHEAD) * (Q4 ? 2 : 4) + (wv >> 1)
                             : Q4 ? scale_row((uint32_t)(kt + AHEAD))
                                  : scale_row((uint32_t)((kt + AHEAD) * 2 + (wv >> 2)));
            if (s_lane) lds_load16_at<FP4 ? W_AUX : 0>(rs, here(s_at) + ST * (PAIR_SC_UNITS * 16), lane16, grow * (P.N * 2) + cs);
        }
    };
    auto issue_group = [&](int kt, int ST) {
#pragma unroll
        for (int m = 0; m < NI; ++m) issue(m, kt, ST);
    };

    // perm selector: bytes 2hh, 2hh+1 of row a, then of row b (hh = half of the dword this lane owns)
    const uint32_t h2 = 2u * (uint32_t)(cw & 1);
    // (int4 with the GEMV op's arithmetic: row a and row b interleaved, so that a 16-bit word holds a k pair)
    constexpr bool I4X = EXACT && FMT == MOE_FMT_INT4;
    uint32_t sel = I4X ? h2 | ((4u + h2) << 8) | ((h2 + 1u) << 16) | ((5u + h2) << 24)
                       : h2 | ((h2 + 1u) << 8) | ((4u + h2) << 16) | ((5u + h2) << 24);
    uint32_t mask = FMT == MOE_FMT_INT4 && !EXACT ? 0x000f000fu : 0x0f0f0f0fu, mask_hi = 0x00f000f0u, magic = 0x64006400u;
    asm volatile("" : "+s"(mask), "+s"(sel));   // kept opaque so that each stays one SGPR operand
    if constexpr (FMT == MOE_FMT_INT4 && !EXACT) asm volatile("" : "+s"(mask_hi), "+v"(magic));
    const int d = 16 * (cw >> 1) + i;            // dword column of this lane
    const int unit = (d >> 2) ^ (4 * (q & 1));
    // row of the x stage this lane's fragment row i comes from (STACK2: see above)
    const int xrow = STACK2 ? (((i >> 3) == (q >> 1)) ? (i & 7) : 8 + (i & 7)) : i;
    // LDS unit (within a stage) of this lane's 8 k of tile row `row`
    auto x_unit = [&](int row) {
        if constexpr (Q4)
            return a_lds_unit32(row, q);
        else
            return a_lds_unit<64>(row, 4 * h + q);
    };

    // The accumulators are zeroed by asm so that the compiler cannot re-materialize the zeros
    // right in front of the first MFMA that accumulates into them: a VALU write of an MFMA's
    // accumulator input needs wait states the compiler only inserts for MFMAs it can see.
    // (Done behind the prologue's loads, below: up to 160 moves that would otherwise delay the first request.)
    f32x4_t acc[MT][4];
    u32x4_t bf[4], afr[4];
    constexpr int RING = 3;
    constexpr int R = RING < MT ? RING : MT;   // x fragments read ahead of their MFMAs

    // int8: per-channel scale and offset of this lane's 4 columns, fixed for the tile (ordinary loads,
    // older than every ring load: the counted waits below cover them)
    float ch_s[4] = {0.f, 0.f, 0.f, 0.f}, ch_o[4] = {0.f, 0.f, 0.f, 0.f};
    u32x2_t ch_sb = {0u, 0u}, ch_ob = {0u, 0u};
    if constexpr (I8) {
        ch_sb = *reinterpret_cast<const u32x2_t*>(static_cast<const uint16_t*>(P.scale) + (int64_t)g * P.N + n0 + col0);
        ch_ob = *reinterpret_cast<const u32x2_t*>(P.offset + (int64_t)g * P.N + n0 + col0);
    }
    // groups -AHEAD .. -1: stages 0 .. AHEAD-1; stages 0 and 1 must have landed before the first barrier
    // (WAITN: the loads of the S - 3 youngest groups may still be in flight at a barrier)
    constexpr int WAITN = (S - 3) * NI;
    // wait until this wavefront's loads of all but the S - 3 youngest groups have landed, then a barrier (prologue)
    auto ring_barrier = [&]() { asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(WAITN) : "memory"); };
    // Inside the k loop the step's barrier is split in two.  A wavefront "arrives" at the end of step kt: it is
    // done with stage kt, and its loads of stage kt + 2 have landed; it adds 1 to a counter in LDS.  It only
    // "waits" -- polls the counter until all 8 wavefronts have arrived kt times -- at the start of the MFMA phase
    // of step kt + 1, in front of the first things that need the others: the loads that overwrite stage kt and
    // the packed dwords of stage kt + 2.  A whole decode phase lies between the two, so a wavefront that is late
    // by less than that stalls nobody (measured against one s_barrier per step: 7 % at K = 7168, 4 % at K = 2048).
    // Everything is inline asm so that the compiler can move nothing across it; every wavefront arrives once in
    // every step of a tile, so every wait ends.  The counter is zeroed per tile, ahead of the prologue's barrier.
    // (the counter's address stays in an SGPR; the asm makes its vector operands on the spot, so that no vector
    // register is held for them through the decode)
    const uint32_t arrivals_at = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)MOE_LDS_PTR(tk.arrivals));
    const __attribute__((address_space(3))) uint32_t* arrivals_lds =
        reinterpret_cast<const __attribute__((address_space(3))) uint32_t*>(MOE_LDS_PTR(tk.arrivals));
    uint32_t arrivals_seen = 0u;
    if (tid == 0) {
        uint32_t va, vz;
        asm volatile("v_mov_b32 %0, %2\n\tv_mov_b32 %1, 0\n\ts_nop 0\n\tds_write_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(va), "=&v"(vz) : "s"(arrivals_at) : "memory");
    }
    auto ring_arrive = [&]() {
        uint32_t va, v1;
        asm volatile("s_waitcnt vmcnt(%2)\n\tv_mov_b32 %0, %3\n\tv_mov_b32 %1, 1\n\ts_mov_b64 exec, 1\n\tds_add_u32 %0, %1\n\ts_mov_b64 exec, -1"
                     : "=&v"(va), "=&v"(v1) : "n"(WAITN), "s"(arrivals_at) : "memory");
    };
    // early: the counter as read half a decode phase ago (usually enough, and its latency is hidden)
    auto ring_wait = [&](uint32_t steps, uint32_t early) {
        uint32_t seen_v, seen_s;
        asm volatile("v_readfirstlane_b32 %1, %4\n\ts_cmp_ge_u32 %1, %3\n\ts_cbranch_scc1 2f\n"
                     "1:\n\tv_mov_b32 %0, %2\n\ts_nop 0\n\tds_read_b32 %0, %0\n\ts_waitcnt lgkmcnt(0)\n\tv_readfirstlane_b32 %1, %0\n\ts_cmp_ge_u32 %1, %3\n\t"
                     "s_cbranch_scc1 2f\n\ts_sleep 1\n\ts_branch 1b\n2:"
                     : "=&v"(seen_v), "=&s"(seen_s) : "s"(arrivals_at), "s"((uint32_t)NW * steps), "v"(early) : "memory", "scc");
    };
    if constexpr (KC) {
        // the scale loads the groups below do not cover (older than all of them: landed by the first barrier)
#pragma unroll
        for (int kp = 0; kp < KC_D - AHEAD; ++kp) kc_issue_scale(kp);
    }
#pragma unroll
    for (int st0 = 0; st0 < AHEAD; ++st0) issue_group(st0 - AHEAD, st0);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if constexpr (EXACT)
                acc[mt][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            else
                asm volatile("v_mov_b32 %0, 0\n\tv_mov_b32 %1, 0\n\tv_mov_b32 %2, 0\n\tv_mov_b32 %3, 0"
                             : "=v"(acc[mt][t][0]), "=v"(acc[mt][t][1]), "=v"(acc[mt][t][2]), "=v"(acc[mt][t][3]));
        }
    ring_barrier();
    // int8: (q + offset) * scale is defined as two rounded fp32 operations.  Where q + offset cannot round (an
    // offset of 0, or of a magnitude in [2^-8, 2^22]: the sum of an 8-bit integer and an 8-bit significand then fits
    // 24 bits) and offset * scale is exact and normal (scale positive and far from the ends of the range), one fma
    // q * scale + offset * scale rounds the same real number once and gives the same bits: 2.5 instead of 3.5
    // instructions per weight.  Decided per wavefront and tile from its lanes' channels.
    float ch_os[4] = {0.f, 0.f, 0.f, 0.f};
    bool i8_one_rounding = false;
    if constexpr (I8) {
        ch_s[0] = bf16_lo(ch_sb[0]); ch_s[1] = bf16_hi(ch_sb[0]); ch_s[2] = bf16_lo(ch_sb[1]); ch_s[3] = bf16_hi(ch_sb[1]);
        ch_o[0] = bf16_lo(ch_ob[0]); ch_o[1] = bf16_hi(ch_ob[0]); ch_o[2] = bf16_lo(ch_ob[1]); ch_o[3] = bf16_hi(ch_ob[1]);
        bool ok = true;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float ao = fabsf(ch_o[t]);
            ok = ok && ch_s[t] >= 0x1p-60f && ch_s[t] <= 0x1p60f && (ao == 0.f || (ao >= 0x1p-8f && ao <= 0x1p22f));
            ch_os[t] = ch_o[t] * ch_s[t];
        }
        i8_one_rounding = __all(ok);
    }

    // this lane's packed dwords and scales of its sub-step of LDS stage st
    uint32_t r[8];
    u32x2_t sc = {0u, 0u}, sc2 = {0u, 0u};   // sc2: with EXACT, the fp4 scales of the second 16 k of the sub-step
    // (s: the step the stage belongs to)
    auto read_raw = [&](int st, int s) {
        const uint16_t* sc16 = reinterpret_cast<const uint16_t*>(lds_s + st * PAIR_SC_UNITS);
        if constexpr (FP4) {
            // Reference pre-shuffle (grouped_gemm/test/python/test_group_gemm_fp4.py:129-142): the tile row
            // 32 j + 8 i' + p holds, in its 32-byte run q', the 8 k rows 16 i' + 8 j + [0, 8) (one dword each)
            // of byte columns 16 p + 4 q' + [0, 4).  This lane's 8 k are 32 h + 8 q + [0, 8) and its two
            // bytes start at byte column 64 (cw >> 1) + 4 i + 2 (cw & 1): p = 4 (cw >> 1) + (i >> 2), q' = i & 3.
            // (Q4: the stage holds the step's 32 rows of that tile packed together, see cb)
            const int trow = Q4 ? 16 * (q & 1) + 8 * (q >> 1) + 4 * (cw >> 1) + (i >> 2)
                                : 32 * (q & 1) + 8 * (2 * h + (q >> 1)) + 4 * (cw >> 1) + (i >> 2);
            const int swz = 4 * ((trow >> 3) & 1);   // the halves of the rows with odd (row >> 3) are swapped (see vb)
            const u32x4_t* tb = lds_b + st * PAIR_B_UNITS + trow * 8;
            const u32x4_t lo4 = tb[(2 * (i & 3)) ^ swz], hi4 = tb[(2 * (i & 3) + 1) ^ swz];
#pragma unroll
            for (int j = 0; j < 4; ++j) { r[j] = lo4[j]; r[4 + j] = hi4[j]; }
            if constexpr (EXACT && !STACK2) {
                sc = *reinterpret_cast<const u32x2_t*>(sc16 + 256 * (2 * h) + col0);
                sc2 = *reinterpret_cast<const u32x2_t*>(sc16 + 256 * (2 * h + 1) + col0);
            } else {
                sc = *reinterpret_cast<const u32x2_t*>(sc16 + 256 * (2 * h + (q >> 1)) + col0);
            }
        } else if constexpr (KC) {
            // MFMA t takes weight row n = 64 cw + 16 t + i: its 8 codes k = 32 h + 8 q + [0, 8) are dword q of
            // the row's half h; the scale of that block
            const uint32_t* t32 = reinterpret_cast<const uint32_t*>(lds_b + st * PAIR_B_UNITS);
            // the row's 8 scales of super-block s / SUP; this lane's block among them
            const uint16_t* sup = reinterpret_cast<const uint16_t*>(lds_s + ((s / SUP) % 3) * 256) +
                                  (KBLK == 16 ? 4 * (s % SUP) + 2 * h + (q >> 1) : 2 * (s % SUP) + h);
            uint32_t s4[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int n = 64 * cw + 16 * t + i;
                r[t] = t32[(2 * n + (h ^ ((i >> 3) & 1))) * 4 + q];
                s4[t] = sup[8 * n];
            }
            sc[0] = s4[0] | (s4[1] << 16);
            sc[1] = s4[2] | (s4[3] << 16);
        } else if constexpr (B8) {
            // dword 16 cw + i of each of this lane's 8 k rows; the quarter of the row it lies in is
            // permuted by (row >> 3) & 3 = q (see vb)
            const uint32_t* t32 = reinterpret_cast<const uint32_t*>(lds_b + st * PAIR_B_UNITS);
#pragma unroll
            for (int j = 0; j < 8; ++j) r[j] = t32[(32 * h + 8 * q + j) * 64 + 16 * (cw ^ q) + i];
            if constexpr (F8) sc[0] = *reinterpret_cast<const uint32_t*>(lds_s + st * PAIR_SC_UNITS + wv);
        } else {
            const uint32_t* t32 = reinterpret_cast<const uint32_t*>(lds_b + st * PAIR_B_UNITS);
#pragma unroll
            for (int j = 0; j < 8; ++j) r[j] = t32[((32 * h + 8 * q + j) * 8 + unit) * 4 + (d & 3)];
            sc = *reinterpret_cast<const u32x2_t*>(sc16 + 256 * h + col0);
        }
    };
    read_raw(0, 0);

    // int4, WIDE: k rows 2 p0 .. 2 p0 + 3 of the sub-step: q - 8 first (exact), then its product with the scale
    auto decode_i4_wide = [&](int p0) __attribute__((always_inline)) {
        const float s[4] = {bf16_lo(sc[0]), bf16_hi(sc[0]), bf16_lo(sc[1]), bf16_hi(sc[1])};
#pragma unroll
        for (int p = p0; p < p0 + 2; ++p) {
            const uint32_t pr = __builtin_amdgcn_perm(r[2 * p + 1], r[2 * p], sel);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t h4 = ((t < 2 ? pr : pr >> 8) & (t & 1 ? mask_hi : mask)) | magic;
                const float one = t & 1 ? 0.0625f : 1.f, zero_point = t & 1 ? -72.f : -1032.f;
                bf[t][p] = pack_bf16_rne(fp16_lo_fma(h4, one, zero_point) * s[t], fp16_hi_fma(h4, one, zero_point) * s[t]);
            }
        }
    };
    // fp8, k rows 2 p0 .. 2 p0 + 3 of the sub-step.  decode_f8: byte t of the dwords of two k rows as a pair through fp16 (see
    // e4m3_ref_pair_over_256), where 0x7F and 0xFF are the reference's +-480; the 2^8 goes into the block scale (WIDE: into the
    // fp16 pair, half an instruction per weight more).
    auto decode_f8 = [&](int p0) __attribute__((always_inline)) {
        const float scl = __uint_as_float(sc[0]) * (WIDE ? 1.f : 256.f);
        float nz = -0.0f;
        asm volatile("" : "+v"(nz));   // kept in a register: not an inline constant
#pragma unroll
        for (int p = p0; p < p0 + 2; ++p) {
            const uint32_t a = r[2 * p], b = r[2 * p + 1];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t sel8 = (uint32_t)t | 0x0c00u | ((uint32_t)(4 + t) << 16) | 0x0c000000u;   // [a.byte t, 0, b.byte t, 0]
                uint32_t h2 = e4m3_ref_pair_over_256_fp16(__builtin_amdgcn_perm(b, a, sel8));
                if constexpr (WIDE) h2 = fp16_pair_times_256(h2);
                if constexpr (EXACT) {
                    // the e4m3 values themselves (worth 2^-8): exact in bf16
                    typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
                    const half2_t hv = __builtin_bit_cast(half2_t, h2);
                    bf[t][p] = pack_bf16_rne((float)hv[0], (float)hv[1]);
                } else {
                    bf[t][p] = pack_bf16_rne(fp16_lo_times(h2, scl, nz), fp16_hi_times(h2, scl, nz));
                }
            }
        }
    };
    // decode_f8_plain: by the hardware conversions, two codes at a time: 2 instructions per weight (EXACT: 0.75) instead of 3.5.
    // They make NaN of 0x7F and 0xFF.  seen_nan collects the step's fragments (v_pk_maximum3_f16 keeps NaN, and a bf16 NaN is an
    // fp16 NaN; so is a bf16 beyond 2^121, which the other decode serves as well): 0.25 instructions per weight.  us, decode_f8
    // alone / this one: 256 experts of 7168 x 2048, 16 rows each 699 / 642; 8 of 4096 x 14336, 512 rows 508 / 472; GEMV op, 128 rows
    // on 64 of 2048 x 1024 29.6 / 26.5.  With random bytes for weights, where every tile changes over at once: 0 to 2 % slower.
    // (Both decodes in one loop, by a flag: 6 to 8 % slower then.)
    uint32_t seen_nan = 0u;
    auto decode_f8_plain = [&](int p0) __attribute__((always_inline)) {
        const float scl = __uint_as_float(sc[0]);
        if (p0 == 0) seen_nan = 0u;
#pragma unroll
        for (int p = p0; p < p0 + 2; ++p) {
            const uint32_t a = r[2 * p], b = r[2 * p + 1];
            if constexpr (EXACT) {
                const uint32_t lo = __builtin_amdgcn_perm(b, a, 0x05010400u), hi = __builtin_amdgcn_perm(b, a, 0x07030602u);   // a.byte t, b.byte t
                bf[0][p] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 0x1p-8f, false));
                bf[1][p] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 0x1p-8f, true));
                bf[2][p] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 0x1p-8f, false));
                bf[3][p] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 0x1p-8f, true));
            } else {
                const f32x2_t a01 = __builtin_amdgcn_cvt_pk_f32_fp8(a, false), a23 = __builtin_amdgcn_cvt_pk_f32_fp8(a, true);
                const f32x2_t b01 = __builtin_amdgcn_cvt_pk_f32_fp8(b, false), b23 = __builtin_amdgcn_cvt_pk_f32_fp8(b, true);
                bf[0][p] = pack_bf16_rne(a01[0] * scl, b01[0] * scl);
                bf[1][p] = pack_bf16_rne(a01[1] * scl, b01[1] * scl);
                bf[2][p] = pack_bf16_rne(a23[0] * scl, b23[0] * scl);
                bf[3][p] = pack_bf16_rne(a23[1] * scl, b23[1] * scl);
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) asm("v_pk_maximum3_f16 %0, %1, %2, %0" : "+v"(seen_nan) : "v"(bf[t][p0]), "v"(bf[t][p0 + 1]));
    };
    bool f8_plain = true;   // this wavefront has met no 0x7F or 0xFF in this tile

    // One data step; st = step mod S is its LDS stage, sn the next one, sl the stage this step's loads
    // go to (wave-uniform).
    // PLAIN (fp8): decode_f8_plain
    auto step = [&](int kt, int st, int sn, int sl, auto PLAIN) __attribute__((always_inline)) {
        const u32x4_t* la = lds_a + st * PAIR_A_UNITS;
        // ---- decode phase: this wavefront's sub-step of the packed stage -> bf[0..3]
        float m[4], z[4];
        const float s0 = bf16_lo(sc[0]), s1 = bf16_hi(sc[0]), s2 = bf16_lo(sc[1]), s3 = bf16_hi(sc[1]);
        // with EXACT: the scales of the step being multiplied (sc is refilled during the MFMA phase)
        const float f8s = __uint_as_float(sc[0]) * 256.f;   // fp8: the step's block scale (times the 2^8 the decode leaves out)
        const float sa[4] = {F8 ? f8s : s0, F8 ? f8s : s1, F8 ? f8s : s2, F8 ? f8s : s3};
        const float sb[4] = {bf16_lo(sc2[0]), bf16_hi(sc2[0]), bf16_lo(sc2[1]), bf16_hi(sc2[1])};
        if constexpr (EXACT) {
            m[0] = m[1] = m[2] = m[3] = FP4 ? 1.f : 512.f;
            z[0] = z[1] = z[2] = z[3] = FP4 ? 0.f : -8.f;
        } else if constexpr (FP4 || KC) {
            m[0] = s0; m[1] = s1; m[2] = s2; m[3] = s3;
            z[0] = z[1] = z[2] = z[3] = 0.f;
        } else {
            m[0] = s0; m[1] = s1 * 0.0625f; m[2] = s2; m[3] = s3 * 0.0625f;
            z[0] = -1032.f * s0; z[1] = -72.f * s1; z[2] = -1032.f * s2; z[3] = -72.f * s3;
        }
        // Written stage by stage over two row pairs at a time so that consecutive instructions are
        // independent (a VALU result is not available to the very next instruction); the fences
        // keep the scheduler from folding the stages back into per-element chains.
#pragma unroll
        for (int p0 = 0; p0 < 4; p0 += 2) {
            if (p0 == 2) {
                if constexpr (SPLIT_BARRIER) {
                    arrivals_seen = *arrivals_lds;   // a first look at the counter, checked after the decode
                } else if (h == 1) {
                    // barrier kt-1 for the wavefronts that own sub-step 1, half way through their decode
                    // (not in the tile's first step: the barrier of the prologue stands for it)
                    if (kt > 0) ring_barrier();
                }
                // first x fragments of the MFMA phase, read under the rest of the decode
#pragma unroll
                for (int f = 0; f < R; ++f) afr[f & 3] = la[x_unit(16 * f + xrow)];
            }
            if constexpr (KC) {
                // dword r[t] = 8 consecutive k of MFMA t's weight row: byte p = the k pair p
#pragma unroll
                for (int t = p0; t < p0 + 2; ++t) {
                    const f32x2_t f0 = e2m1_pair_to_f32<0>(r[t]), f1 = e2m1_pair_to_f32<1>(r[t]);
                    const f32x2_t f2 = e2m1_pair_to_f32<2>(r[t]), f3 = e2m1_pair_to_f32<3>(r[t]);
                    bf[t][0] = pack_bf16_rne(f0[0] * m[t], f0[1] * m[t]);
                    bf[t][1] = pack_bf16_rne(f1[0] * m[t], f1[1] * m[t]);
                    bf[t][2] = pack_bf16_rne(f2[0] * m[t], f2[1] * m[t]);
                    bf[t][3] = pack_bf16_rne(f3[0] * m[t], f3[1] * m[t]);
                }
                __builtin_amdgcn_sched_barrier(0);
                continue;
            }
            if constexpr (F8) {
                if constexpr (PLAIN)
                    decode_f8_plain(p0);
                else
                    decode_f8(p0);
                __builtin_amdgcn_sched_barrier(0);
                continue;
            }
            if constexpr (I8) {
                // byte t of the dwords of k rows 2p, 2p+1 -> (q + offset) * scale as two rounded fp32
                // operations (or the one fma that equals them, see i8_one_rounding) -> bf16 pair along k
                if (i8_one_rounding) {
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const uint32_t a = r[2 * (p0 + p)], b = r[2 * (p0 + p) + 1];
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            const float qa = (float)(int)(int8_t)(a >> (8 * t)), qb = (float)(int)(int8_t)(b >> (8 * t));
                            bf[t][p0 + p] = pack_bf16_rne(__fmaf_rn(qa, ch_s[t], ch_os[t]), __fmaf_rn(qb, ch_s[t], ch_os[t]));
                        }
                    }
                } else {
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const uint32_t a = r[2 * (p0 + p)], b = r[2 * (p0 + p) + 1];
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            const float qa = (float)(int)(int8_t)(a >> (8 * t)), qb = (float)(int)(int8_t)(b >> (8 * t));
                            bf[t][p0 + p] = pack_bf16_rne(__fmul_rn(__fadd_rn(qa, ch_o[t]), ch_s[t]),
                                                          __fmul_rn(__fadd_rn(qb, ch_o[t]), ch_s[t]));
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                continue;
            }
            if constexpr (FMT == MOE_FMT_INT4 && WIDE) {
                decode_i4_wide(p0);
                __builtin_amdgcn_sched_barrier(0);
                continue;
            }
            uint32_t pr[2];
            float wa[2][4], wb[2][4];
#pragma unroll
            for (int p = 0; p < 2; ++p) pr[p] = __builtin_amdgcn_perm(r[2 * (p0 + p) + 1], r[2 * (p0 + p)], sel);   // a.b0 a.b1 b.b0 b.b1
            if constexpr (FP4) {
                // e2m1: each byte of pr is two columns of one k row; exact decode, one multiply by the
                // column's scale, RNE to bf16 (W = bf16(e2m1 * scale) as the reference's antiquant phase)
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const f32x2_t a01 = e2m1_pair_to_f32<0>(pr[p]), a23 = e2m1_pair_to_f32<1>(pr[p]);
                    const f32x2_t b01 = e2m1_pair_to_f32<2>(pr[p]), b23 = e2m1_pair_to_f32<3>(pr[p]);
                    if constexpr (EXACT) {
                        bf[0][p0 + p] = pack_bf16_rne(a01[0], b01[0]);
                        bf[1][p0 + p] = pack_bf16_rne(a01[1], b01[1]);
                        bf[2][p0 + p] = pack_bf16_rne(a23[0], b23[0]);
                        bf[3][p0 + p] = pack_bf16_rne(a23[1], b23[1]);
                    } else {
                        bf[0][p0 + p] = pack_bf16_rne(a01[0] * m[0], b01[0] * m[0]);
                        bf[1][p0 + p] = pack_bf16_rne(a01[1] * m[1], b01[1] * m[1]);
                        bf[2][p0 + p] = pack_bf16_rne(a23[0] * m[2], b23[0] * m[2]);
                        bf[3][p0 + p] = pack_bf16_rne(a23[1] * m[3], b23[1] * m[3]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                continue;
            }
            if constexpr (I4X) {
                // The codes themselves as bf16, two at a time: a nibble read as e4m3 is q / 512, and the scaled
                // convert (scale 2^9: only the exponent of that operand counts) yields the bf16 pair (q_a, q_b) of
                // one column.  The zero point is taken off in the MFMA phase.
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const uint32_t lo = pr[p] & mask, hi = (pr[p] >> 4) & mask;
                    bf[0][p0 + p] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.f, false));
                    bf[2][p0 + p] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.f, true));
                    bf[1][p0 + p] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.f, false));
                    bf[3][p0 + p] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.f, true));
                }
                __builtin_amdgcn_sched_barrier(0);
                continue;
            }
            // int4: halves (a, b) as fp16, one fma each (see the head of this routine)
            uint32_t h4[2][4];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const uint32_t up = pr[p] >> 8;
                h4[p][0] = (pr[p] & mask) | magic;
                h4[p][1] = (pr[p] & mask_hi) | magic;
                h4[p][2] = (up & mask) | magic;
                h4[p][3] = (up & mask_hi) | magic;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 4; t += 2) {
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int u = t; u < t + 2; ++u) {
                        wa[p][u] = fp16_lo_fma(h4[p][u], m[u], z[u]);
                        wb[p][u] = fp16_hi_fma(h4[p][u], m[u], z[u]);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int t = 0; t < 4; ++t) bf[t][p0 + p] = pack_bf16_rne(wa[p][t], wb[p][t]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (F8 && PLAIN) {
            asm("v_pk_maximum3_f16 %0, %0, %0, %0 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "+v"(seen_nan));   // both halves
            if (__any(__builtin_isnan(__builtin_bit_cast(_Float16, (uint16_t)seen_nan)))) [[unlikely]] {
                f8_plain = false;
                decode_f8(0);
                decode_f8(2);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // ---- MFMA phase, at raised issue priority: the other wavefront of the SIMD is decoding
        // meanwhile and would otherwise win the arbitration whenever both are ready, starving
        // the matrix pipe; its VALU instructions fit into the gaps the MFMAs leave
        // every wavefront has arrived kt times (none in the tile's first step: the prologue's barrier stands for it)
        if constexpr (SPLIT_BARRIER) ring_wait((uint32_t)kt, arrivals_seen);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(3);
        if constexpr (EARLY_RAW) {
            read_raw(sn, kt + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        // Everybody is done with stage kt-1 and has its part of stage kt+1 in LDS: this step's loads (stage kt+4
        // replaces stage kt-1) and the packed dwords of the next step (stage kt+1) are fetched between the MFMAs.
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if (mt + R < MT) afr[(mt + R) & 3] = la[x_unit(16 * (mt + R) + xrow)];
            if constexpr (EXACT) {
                const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
                if constexpr (STACK2) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const f32x4_t dd = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8_t, afr[mt & 3]), __builtin_bit_cast(bf16x8_t, bf[t]), zero, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[mt][t][e] = fmaf(dd[e], sa[t], acc[mt][t][e]);
                    }
                } else if constexpr (FP4) {
                    const uint32_t mlo = q < 2 ? 0xffffffffu : 0u;
                    u32x4_t xlo, xhi;
#pragma unroll
                    for (int j = 0; j < 4; ++j) { xlo[j] = afr[mt & 3][j] & mlo; xhi[j] = afr[mt & 3][j] & ~mlo; }
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const f32x4_t dlo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8_t, xlo), __builtin_bit_cast(bf16x8_t, bf[t]), zero, 0, 0, 0);
                        const f32x4_t dhi = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8_t, xhi), __builtin_bit_cast(bf16x8_t, bf[t]), zero, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[mt][t][e] = fmaf(dhi[e], sb[t], fmaf(dlo[e], sa[t], acc[mt][t][e]));
                    }
                } else {
                    // int4: the fragments hold q, not q - 8: each product starts from -8 sum_k x[m][k] (one more
                    // MFMA per x fragment, against a constant fragment of -8.0), so dd = sum_k x (q - 8)
                    f32x4_t start = zero;
                    if constexpr (I4X) {
                        const u32x4_t m8 = {0xc100c100u, 0xc100c100u, 0xc100c100u, 0xc100c100u};
                        start = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8_t, afr[mt & 3]), __builtin_bit_cast(bf16x8_t, m8), zero, 0, 0, 0);
                    }
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const f32x4_t dd = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            __builtin_bit_cast(bf16x8_t, afr[mt & 3]), __builtin_bit_cast(bf16x8_t, bf[t]), start, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[mt][t][e] = fmaf(dd[e], sa[t], acc[mt][t][e]);
                    }
                }
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t) mfma_16x16x32_v(acc[mt][t], afr[mt & 3], bf[t]);
            }
#pragma unroll
            for (int m = (mt * NI + MT - 1) / MT; m < ((mt + 1) * NI + MT - 1) / MT; ++m) issue(m, kt, sl);
            if (mt == 0 && !EARLY_RAW) read_raw(sn, kt + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        if constexpr (SPLIT_BARRIER) {
            ring_arrive();
        } else if (h == 0) {
            ring_barrier();   // barrier kt
        }
    };
    // unrolled over the ring, so that every stage number is a constant and the LDS addresses of a step are
    // immediate offsets (with run-time stage numbers a step spent 9 vector and about 25 scalar instructions on
    // them: measured 10 % of the kernel's time at K = 7168); a tile starts at stage 0
    // (the K-contiguous containers keep run-time stage numbers: their routine has no registers left for the
    // unrolled form)
    if constexpr (!KC) {
        if constexpr (F8) {
            // fragments with a NaN among them are decoded again, and from the next turn of the ring on the tile goes through decode_f8
            int kt0 = 0;
            for (; kt0 < nk && f8_plain && !WIDE; kt0 += S) {
#pragma unroll
                for (int u = 0; u < S; ++u)
                    if (kt0 + u < nk) step(kt0 + u, u, (u + 1) % S, (u + S - 1) % S, std::true_type{});
            }
            for (; kt0 < nk; kt0 += S) {
#pragma unroll
                for (int u = 0; u < S; ++u)
                    if (kt0 + u < nk) step(kt0 + u, u, (u + 1) % S, (u + S - 1) % S, std::false_type{});
            }
        } else {
            for (int kt0 = 0; kt0 < nk; kt0 += S) {
#pragma unroll
                for (int u = 0; u < S; ++u)
                    if (kt0 + u < nk) step(kt0 + u, u, (u + 1) % S, (u + S - 1) % S, std::false_type{});
            }
        }
    } else {
        for (int kt = 0, st = 0, sl = S - 1; kt < nk; ++kt) {
            const int sn = st == S - 1 ? 0 : st + 1;
            step(kt, st, sn, sl, std::false_type{});
            st = sn;
            sl = sl == S - 1 ? 0 : sl + 1;
        }
    }
    if constexpr (!SPLIT_BARRIER)
        if (h == 1) ring_barrier();   // barrier nk-1
    // drain this wavefront's loads (they target stages past K and are never read); the
    // accumulators were last written by MFMAs the compiler cannot see: wait out their latency
    // (and the last arrivals are counted before anybody zeroes the counter for the next tile)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15\n\ts_barrier" ::: "memory");

    if constexpr (STACK2) {
        // the lanes q and q + 2 hold the two scale groups' sums of the same rows
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[0][t][e] += __shfl_xor(acc[0][t][e], 32);
    }
    if constexpr (wide_scales<FMT>(KIND) && !WIDE) {
        // a weight that is no number leaves none in its column, in any row: row block 0 tells (see redo_wide); fp8: the hardware's
        // conversions take any scale
        if (!F8 || !f8_plain) {
            float bad[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < 4; ++t) asm volatile("" : "+v"(acc[0][t]));   // not read ahead of the wait above
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) bad[e] = fmaf(acc[0][t][e], 0.f, bad[e]);
            if (__any(__builtin_isnan((bad[0] + bad[1]) + (bad[2] + bad[3])))) [[unlikely]] {
                if (lane == 0) {
                    tk.wide[0] = 1; tk.wide[1] = g; tk.wide[2] = (int)row0; tk.wide[3] = rows; tk.wide[4] = n0;
                }
            }
        }
    }
    pair_finish<MT, KC, Q4>(P, smem, acc, h, cw, lane, col0, row0, rows, n0, tk);
}

// ---------------------------------------------------------------------------------
// Tile routine for the K-contiguous fp4 containers (weights [N, K/2], scales [N, K/16 or K/32]): workgroups of 4 wavefronts,
// two per CU, as GK_QUAD: wavefront cw takes columns 64 cw .. + 63 of the tile through all of k for up to 144 rows.
//
// Bound by issue, as the N-contiguous kinds: 2 vector instructions per weight (exact convert, times its scale, rounded to
// bf16) beside the MFMAs, and next to that by requests to L2.  Two workgroups per CU hide each other's barriers and the time
// between tiles, which the 8 wavefronts of GK_PAIR do not; with a single tile per CU GK_PAIR is ahead (see moe_dispatch.cpp).
// us, GK_PAIR / this one: 128 experts of 2048 x 7168, 2047 tokens x 8 rows: fp4_b16 686 / 570 (843 TFLOP/s), fp4_b32
// 635 / 551; 7168 x 2048 the same rows, fp4_b32: 624 / 593; 4608 x 3072, 1245 tokens x 8, unevenly routed, fp4_b16: 490 / 436; 8 of
// 3968 x 13568, 841 rows each, fp4_b32: 699 / 627.  (The reference's fp4 container on GK_QUAD: 522, 534 on the first and third.)
//
// The weight rows of a wavefront's columns are read by that wavefront alone, so its weights and scales are its own business:
// it loads them for 256 k at a time, whole 128-byte lines of 64 rows, into registers during the first steps of the period before, puts
// them into its own LDS when the last of that period is read, and shares no barrier for them.  (Loads are counted in order: the wait for x at
// the end of a step also waits for the weights requested two steps earlier, so they have 2 to 3 steps to land, not the 4 to 8 until
// they are needed.)  (64 bytes of a row at a time, straight to
// LDS: the other half of a line was gone from L2 when its turn came, 64 workgroups of 256 lines each on an XCD; 1.6 GB fetched
// instead of 1.2, by counters, and 635 us instead of 593 at K = 7168.  Both halves back to back but in instructions of 16 rows x
// 64 bytes: 615 us, twice the requests.)  Only x is shared: a ring of four 32-k stages, three steps ahead, one barrier per step.
//
// Step u of a period reads dword q of 16-byte unit u of every weight row: the 8 codes k = 32 u + 8 q + [0, 8).  Unit u of the
// row in slot s lies at position u ^ ((s >> 1) & 7), so that the 64 lanes of a read (16 rows x 4 dwords) hit 64 banks.
// Column t of a lane is 4 i + t (SwiGLU: two gate and two up rows of two adjacent output columns), as in gemm_tile_bf16.
// ---------------------------------------------------------------------------------
constexpr int FK_MT_MAX = 9;                         // row blocks of 16; a tenth leaves no registers for the weights ahead
constexpr int FK_XS = 4;                             // x stages
constexpr int FK_X_UNITS = 16 * FK_MT_MAX * 4;       // 32 k
constexpr int FK_W_UNITS = GM_BN * 8;                // 256 weight rows x 256 k
constexpr int FK_S_UNITS = GM_BN * 2;                // their scales: 32 bytes a row (fp4_b32: 16)
static_assert(16 * FK_MT_MAX == FP4_K_ROWS, "what the dispatch goes by");
constexpr int fk_lds_units() { return FK_XS * FK_X_UNITS + FK_W_UNITS + FK_S_UNITS; }
template <int FMT, int MT>
__device__ __forceinline__ void gemm_tile_fp4_k(const GemmParams& P, u32x4_t* smem, int g, int64_t row0, int rows, int n0, const Ticket& tk) {
    constexpr int BLK = FMT == MOE_FMT_FP4_B32 ? 32 : 16, SL = 32 / BLK;   // SL: load instructions of a period's scales
    constexpr int NW = 4, NA = (MT + NW - 1) / NW, AHEAD = FK_XS - 1;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, i = lane & 15, q = lane >> 4;
    const int cw = __builtin_amdgcn_readfirstlane(tid >> 6);
    u32x4_t* const lds_w = smem + FK_XS * FK_X_UNITS + cw * (FK_W_UNITS / 4);   // this wavefront's own
    u32x4_t* const lds_s = smem + FK_XS * FK_X_UNITS + FK_W_UNITS + cw * (FK_S_UNITS / 4);
    const int nk = P.K >> 5;                                     // a multiple of 4
    const int k2 = P.K * 2, kh = P.K >> 1, ks = P.K / BLK * 2;   // bytes of a row of x, weights, scales
    const int64_t KN = (int64_t)P.K * P.N;
    const bool swi = P.epilogue == MOE_EPILOGUE_SWIGLU;
    // x as in GK_QUAD: load instructions of 16 rows x 64 bytes, see a_lds_unit32
    const rsrc_t rx = make_rsrc(P.x + row0 * (int64_t)P.K, (int64_t)rows * k2);
    const int va = (lane >> 2) * k2 + ((lane & 3) ^ ((lane >> 3) & 3)) * 16;
    int ca[NA];
    uint32_t a_at[NA];
#pragma unroll
    for (int m = 0; m < NA; ++m) {
        int j = cw + NW * m;
        if (NW * NA > MT) j = j % MT;   // repeat a block rather than issue fewer loads
        a_at[m] = lds_address(smem + j * 64);
        ca[m] = 16 * j * k2;
    }
    auto issue_x = [&](int m, int kt, int st) { lds_load16_at(rx, here(a_at[m]) + st * (FK_X_UNITS * 16), va, ca[m] + kt * 64); };
    // Slot 16 t + i of a wavefront's weights and scales is the weight row that lane i multiplies in MFMA t, row lane_row(i) +
    // mfma_row(t) of its 64.  Weights: load e brings slots 8 e + (l >> 3), the whole 128 bytes of each
    const int lane_rows = swi ? 2 : 4;   // lanes i and i + 1 (i + 8: 32 rows, either way)
    auto mfma_row = [&](int t) { return swi ? (t & 1) + 16 * (t >> 1) : t; };
    const rsrc_t rw = make_rsrc(P.w + g * (KN >> 1), KN >> 1);
    const int cb = (n0 + 64 * cw) * kh;
    const int vb0 = (lane >> 3) * lane_rows * kh + ((lane & 7) ^ (lane >> 4)) * 16;
    const int vb1 = (lane >> 3) * lane_rows * kh + ((lane & 7) ^ (lane >> 4) ^ 4) * 16;
    u32x4_t wreg[8], sreg[SL];
    auto load_w = [&](int e, int p) {
        wreg[e] = __builtin_amdgcn_raw_buffer_load_b128(rw, e & 1 ? vb1 : vb0, cb + (mfma_row(e >> 1) + 32 * (e & 1)) * kh + p * 128, 0);
    };
    // scales: fp4_b32 the 16 bytes of slot l; fp4_b16 load e the 32 bytes of slots 32 e + (l >> 1)
    const rsrc_t rs = make_rsrc(static_cast<const uint16_t*>(P.scale) + g * (KN / BLK), (KN / BLK) * 2);
    const int sl = SL == 1 ? lane : lane >> 1;   // slot
    const int vs = (32 * ((sl >> 3) & 1) + lane_rows * (sl & 7) + mfma_row(sl >> 4)) * ks + (SL == 1 ? 0 : (lane & 1) * 16);
    const int cs = (n0 + 64 * cw) * ks;
    auto load_s = [&](int e, int p) { sreg[e] = __builtin_amdgcn_raw_buffer_load_b128(rs, vs, cs + mfma_row(2) * e * ks + p * (16 * SL), 0); };
    auto put = [&]() {
#pragma unroll
        for (int e = 0; e < SL; ++e) lds_s[e * 64 + lane] = sreg[e];
#pragma unroll
        for (int e = 0; e < 8; ++e) lds_w[e * 64 + lane] = wreg[e];
    };

#pragma unroll
    for (int e = 0; e < SL; ++e) load_s(e, 0);
#pragma unroll
    for (int e = 0; e < 8; ++e) load_w(e, 0);
#pragma unroll
    for (int st = 0; st < AHEAD; ++st)
#pragma unroll
        for (int m = 0; m < NA; ++m) issue_x(m, st, st);
    f32x4_t acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < 4; ++t)
            asm volatile("v_mov_b32 %0, 0\n\tv_mov_b32 %1, 0\n\tv_mov_b32 %2, 0\n\tv_mov_b32 %3, 0"
                         : "=v"(acc[mt][t][0]), "=v"(acc[mt][t][1]), "=v"(acc[mt][t][2]), "=v"(acc[mt][t][3]));
    put();
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * NA) : "memory");   // x stage 0 is there

    uint32_t r[4], sk[4];
    // this lane's codes and scales of step u of the period
    const uint32_t* const t32 = reinterpret_cast<const uint32_t*>(lds_w) + i * 32 + q;
    const uint16_t* const s16 = reinterpret_cast<const uint16_t*>(lds_s) + i * (8 * SL) + (BLK == 16 ? q >> 1 : 0);
    auto read_raw = [&](int u) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            r[t] = t32[16 * t * 32 + (u ^ (i >> 1)) * 4];
            sk[t] = s16[16 * t * (8 * SL) + u * SL];
        }
    };
    read_raw(0);

    constexpr int R = MT == 9 ? 2 : MT < 3 ? MT : 3, RB = R + 1;   // x fragments read ahead of their MFMAs (nine blocks: registers)
    // what step u requests of the next period's weights and scales (0 for u < 0 too)
    constexpr auto extra = [](int u) { return u >= 0 && u < 4 ? 2 + (u < SL ? 1 : 0) : 0; };
    // step u of period p; MORE: with requests for the next period (or the counts below would include loads that nothing reads and
    // that the compiler therefore takes out)
    auto step = [&](auto U, auto MORE, int p) __attribute__((always_inline)) {
        constexpr int u = decltype(U)::value, st = u % FK_XS, here_n = MORE ? extra(u) : 0, before_n = MORE ? extra(u - 1) : 0;
        const u32x4_t* la = smem + st * FK_X_UNITS + a_lds_unit32(i, q);
        u32x4_t bf[4], afr[RB];
#pragma unroll
        for (int t0 = 0; t0 < 4; t0 += 2) {
            if (t0 == 2)
#pragma unroll
                for (int f = 0; f < R; ++f) afr[f] = la[f * 64];
#pragma unroll
            for (int t = t0; t < t0 + 2; ++t) {
                const float m = bf16_bits_to_f32(sk[t]);
                const f32x2_t f0 = e2m1_pair_to_f32<0>(r[t]), f1 = e2m1_pair_to_f32<1>(r[t]);
                const f32x2_t f2 = e2m1_pair_to_f32<2>(r[t]), f3 = e2m1_pair_to_f32<3>(r[t]);
                bf[t][0] = pack_bf16_rne(f0[0] * m, f0[1] * m);
                bf[t][1] = pack_bf16_rne(f1[0] * m, f1[1] * m);
                bf[t][2] = pack_bf16_rne(f2[0] * m, f2[1] * m);
                bf[t][3] = pack_bf16_rne(f3[0] * m, f3[1] * m);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(3);
        // the x stage three steps ahead replaces the one everybody has left at the barrier; a quarter of the next weights
        constexpr int NI = NA + extra(u);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if (mt + R < MT) afr[(mt + R) % RB] = la[(mt + R) * 64];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if constexpr (MT == 1)   // (few enough for the compiler, which moves them to other registers behind the loop)
                    acc[0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, afr[0]), __builtin_bit_cast(bf16x8_t, bf[t]), acc[0][t], 0, 0, 0);
                else
                    mfma_16x16x32_v(acc[mt][t], afr[mt % RB], bf[t]);
            }
#pragma unroll
            for (int m = (mt * NI + MT - 1) / MT; m < ((mt + 1) * NI + MT - 1) / MT; ++m) {
                if (m < NA)
                    issue_x(m, 8 * p + u + AHEAD, (u + AHEAD) % FK_XS);
                else if (!MORE)
                    break;
                else if (m < NA + 2)
                    load_w(2 * u + m - NA, p + 1);
                else
                    load_s(u, p + 1);
            }
            if (mt == 0) {
                if constexpr (u == 7) put();
                read_raw((u + 1) & 7);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        // x of the next step (requested two steps ago) has landed: behind it are all requests of the last step and this one
        // (whole steps: within a step the compiler may order the requests as it likes)
        constexpr int WAITN = 2 * NA + before_n + here_n;
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(WAITN) : "memory");
    };
    // (the half period of a K that is no multiple of 256 stands behind the loop: a path from step 3 to step 0, with loads into wreg
    // on their way, would make the compiler wait in every step)
    const int np = nk >> 3;
    const auto half = [&](auto FIRST, auto MORE, int p) __attribute__((always_inline)) {
        constexpr int u = decltype(FIRST)::value;
        step(std::integral_constant<int, u>{}, MORE, p);
        step(std::integral_constant<int, u + 1>{}, MORE, p);
        step(std::integral_constant<int, u + 2>{}, MORE, p);
        step(std::integral_constant<int, u + 3>{}, MORE, p);
    };
    for (int p = 0; p < np; ++p) {
        half(std::integral_constant<int, 0>{}, std::true_type{}, p);
        half(std::integral_constant<int, 4>{}, std::true_type{}, p);
    }
    if (nk & 4) half(std::integral_constant<int, 0>{}, std::false_type{}, np);
    // the last loads are for steps past K and never read; wait out the last MFMAs' latency
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15\n\ts_barrier" ::: "memory");
    pair_finish<MT, false, true>(P, smem, acc, 0, cw, lane, 64 * cw + 4 * i, row0, rows, n0, tk);
}

// ---------------------------------------------------------------------------------
// Tile routine for the bf16 container (weights [N, K], K-contiguous, nothing to decode): 8 wavefronts, one workgroup per
// CU, tiles of up to 224 rows x 256 columns; wavefront (wr, cw) multiplies half wr of the rows by the 64 columns of
// group cw.
//
// What bounds it: with up to about 200 rows per expert the weights (2 bytes each) are read once from HBM, and the rate
// follows from how many of their bytes are on their way, i.e. from how much LDS is left for them; with more rows per
// expert the latency of L2 misses that a step cannot look far enough ahead for.  With all loads taken out the loop runs
// at 1.5 PFLOP/s, with all of them hitting L2 at 1.3.  Hence one workgroup per CU, so that x is held once (two of 4
// wavefronts with 144 rows each, three 25 KB stages: no faster than the routine this replaced), and two rings: x, which
// the neighbouring column tiles read too and L2 usually holds, two or three pairs of steps deep, the weights three or four.
// A load instruction brings 64 bytes (one 32-k step) of 16 rows; the two halves of a 128-byte line are requested back
// to back, in pairs of steps: asked for a step apart the line travels from L2 twice (measured: 535 and 480 us).
// Weights straight into registers, two steps of 64 k ahead, lose: such loads of 16 rows each cost the CU's
// vector memory path twice the cycles of LDS-direct ones (498 us, and 616 instead of 570 us on the large shape below).
//
// 64 experts, K = 7168, N = 2048, 900 / 1021 tokens x 8 rows (the second unevenly routed): 416 / 542 us with the
// 4-wavefront routine this replaced, now 391 / 489 (5.1 / 4.1 TB/s); 100 tokens: 361 -> 320 us (5.9 TB/s);
// 8 experts of 512 rows, K = 4096, N = 14336: 554 -> 491 us (979 TFLOP/s).
//
// Column t of a lane is 4 i + t, so that a lane stores 4 adjacent columns in one instruction (the rows of the weight
// may be assigned to MFMAs and lanes freely); with the SwiGLU epilogue the lane takes the two gate rows and the two up
// rows of two adjacent output columns, which makes its 4 accumulators what the N-contiguous containers have.
// ---------------------------------------------------------------------------------
constexpr int BF_MT_MAX = 7;                                   // row blocks of a wavefront: tiles of 224 rows
static_assert(32 * BF_MT_MAX == BF16_ROWS, "what the dispatch goes by");
constexpr int BF_B_UNITS = GM_BN * 4;                          // 256 weight rows x 32 k
constexpr int bf_a_units(int mt) { return 32 * mt * 4; }       // 32 mt rows x 32 k
// pairs of steps in the two rings: what fits into 156 KB
constexpr int bf_x_pairs(int mt) { return mt == 4 || mt == 5 ? 3 : 2; }
constexpr int bf_w_pairs(int mt) { return mt > 3 ? 3 : 4; }
constexpr int bf_lds_units() {
    int most = 0;
    for (int mt = 1; mt <= BF_MT_MAX; ++mt) {
        const int units = 2 * (bf_x_pairs(mt) * bf_a_units(mt) + bf_w_pairs(mt) * BF_B_UNITS);
        if (units > most) most = units;
    }
    return most;
}
template <int MT>
__device__ __forceinline__ void gemm_tile_bf16(const GemmParams& P, u32x4_t* smem, int g, int64_t row0, int rows, int n0, const Ticket& tk) {
    constexpr int XP = bf_x_pairs(MT), WP = bf_w_pairs(MT), NW = 8;
    constexpr int AU = bf_a_units(MT), BU = BF_B_UNITS;   // units of a half step
    u32x4_t* const lds_w = smem + XP * 2 * AU;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, i = lane & 15, q = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wv >> 2, cw = wv & 3;
    const int np = P.K >> 6;
    // Where in K a column tile starts (it goes round).  L2's 16 channels take 256 bytes in turn: with weight rows a multiple
    // of 4 KB apart all rows of all tiles, which run nearly in step, would ask one channel at a time, so each column tile
    // starts in the next one.  K = 2048, 256 experts of N = 1024, 8 rows each: 239 us without, 201 with (212 with the 4-wavefront
    // routine this replaced); 64 of N = 2048, 48 rows:
    // 139 / 122.  Other K gain nothing and lose the x rows that neighbouring tiles find in L2 (prefill, K = 7168: 481 / 491).
    const int rot = P.K % 2048 ? 0 : (int)((unsigned)(2 * (g * ((P.N + GM_BN - 1) / GM_BN) + n0 / GM_BN)) % (unsigned)np);
    auto pair_at = [&](int p) { return p + rot < np ? p + rot : p + rot - np; };
    const int64_t KN = (int64_t)P.K * P.N;
    const int k2 = P.K * 2;
    const bool swi = P.epilogue == MOE_EPILOGUE_SWIGLU;
    // Load instructions of 16 rows x 64 bytes: lane l brings the 16-byte chunk (l & 3) ^ ((l >> 3) & 3) of row l >> 2 to
    // position l & 3 (see a_lds_unit32); both 64-byte halves of a row's 128-byte line are requested back to back
    const int li = lane >> 2, vc = ((lane & 3) ^ ((lane >> 3) & 3)) * 16;
    const rsrc_t rx = make_rsrc(P.x + row0 * (int64_t)P.K, (int64_t)rows * k2);
    const int va = li * k2 + vc;
    const rsrc_t rw = make_rsrc(P.w + g * (KN * 2), KN * 2);
    const int vb = (swi ? 32 * (li >> 3) + 2 * (li & 7) : 4 * li) * k2 + vc;
    constexpr int XI = 2 * MT, NA = (XI + NW - 1) / NW, NB = 2;
    int ca[NA], cb[NB];
    uint32_t a_at[NA];
#pragma unroll
    for (int m = 0; m < NA; ++m) {
        int j = wv + NW * m;
        if (NW * NA > XI) j = j % XI;   // repeat a block rather than issue fewer loads
        a_at[m] = lds_address(smem + j * 64);
        ca[m] = 16 * j * k2;
    }
#pragma unroll
    for (int e = 0; e < NB; ++e) {
        const int j = NB * wv + e, t = j & 3;   // rows of MFMA t of column group j >> 2
        cb[e] = (n0 + 64 * (j >> 2) + (swi ? (t & 1) + 16 * (t >> 1) : t)) * k2;
    }
    const uint32_t b_at = lds_address(lds_w + NB * wv * 64);
    auto issue_x = [&](int m, int p, int slot) {
        const int h = m & 1, e = m >> 1;
        lds_load16_at(rx, here(a_at[e]) + slot * (2 * AU * 16) + h * (AU * 16), va, ca[e] + p * 128 + h * 64);
    };
    auto issue_w = [&](int m, int p, int slot) {
        const int h = m & 1, e = m >> 1;
        lds_load16_at(rw, here(b_at) + slot * (2 * BU * 16) + h * (BU * 16) + e * 1024, vb, cb[e] + p * 128 + h * 64);
    };
#pragma unroll
    for (int p = 0; p < WP - 1; ++p) {   // (in the order of the loop below: x a ring's depth ahead, then the weights)
        if (p >= WP - XP)
#pragma unroll
            for (int m = 0; m < 2 * NA; ++m) issue_x(m, pair_at(p - (WP - XP)), p - (WP - XP));
#pragma unroll
        for (int m = 0; m < 2 * NB; ++m) issue_w(m, pair_at(p), p);
    }
    f32x4_t acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < 4; ++t)
            asm volatile("v_mov_b32 %0, 0\n\tv_mov_b32 %1, 0\n\tv_mov_b32 %2, 0\n\tv_mov_b32 %3, 0"
                         : "=v"(acc[mt][t][0]), "=v"(acc[mt][t][1]), "=v"(acc[mt][t][2]), "=v"(acc[mt][t][3]));
    // the next pair's x and weights have landed: of what was requested behind them, one pair's weights (and its x, where
    // that ring holds three pairs) may be on their way
    constexpr int WAITN = (XP - 2) * 2 * NA + 2 * NB;
    auto pair_barrier = [&]() { asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(WAITN) : "memory"); };
    pair_barrier();
    const u32x4_t* const xf = smem + a_lds_unit32(16 * MT * wr + i, q);
    const u32x4_t* const wf = lds_w + a_lds_unit32(64 * cw + i, q);
    constexpr int NI = 2 * (NA + NB);
    constexpr int F = 2 * MT, R = 3 < F ? 3 : F;   // x fragments of a pair, read R ahead of their MFMAs
    for (int p = 0, xs = 0, ws = 0; p < np; ++p) {
        const int px = pair_at(p + XP - 1), pw = pair_at(p + WP - 1);
        const int x_to = xs == 0 ? XP - 1 : xs - 1, w_to = ws == 0 ? WP - 1 : ws - 1;
        const u32x4_t* lx = xf + xs * (2 * AU);
        const u32x4_t* lw = wf + ws * (2 * BU);
        u32x4_t bf[2][4], afr[4];
        auto read_x = [&](int f) { afr[f & 3] = lx[(f / MT) * AU + (f % MT) * 64]; };
#pragma unroll
        for (int t = 0; t < 4; ++t) bf[0][t] = lw[t * 64];
#pragma unroll
        for (int f = 0; f < R; ++f) read_x(f);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(3);
#pragma unroll
        for (int f = 0; f < F; ++f) {
            if (f + R < F) read_x(f + R);
            if (f == (MT + 1) / 2 - 1)
#pragma unroll
                for (int t = 0; t < 4; ++t) bf[1][t] = lw[BU + t * 64];
#pragma unroll
            for (int t = 0; t < 4; ++t) mfma_16x16x32_v(acc[f % MT][t], afr[f & 3], bf[f / MT][t]);
#pragma unroll
            for (int m = (f * NI + MT - 1) / MT; f < MT && m < ((f + 1) * NI + MT - 1) / MT; ++m) {
                if (m < 2 * NA)
                    issue_x(m, px, x_to);
                else
                    issue_w(m - 2 * NA, pw, w_to);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_setprio(0);
        pair_barrier();
        xs = xs == XP - 1 ? 0 : xs + 1;
        ws = ws == WP - 1 ? 0 : ws + 1;
    }
    // the last loads are for pairs behind the last one and never read; wait out the last MFMAs' latency
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15\n\ts_barrier" ::: "memory");
    pair_finish<MT, false, true>(P, smem, acc, 0, cw, lane, 64 * cw + 4 * i, row0 + 16 * MT * wr, max(rows - 16 * MT * wr, 0), n0, tk);
}

// ---------------------------------------------------------------------------------
// Tile scheduler (role of GMMAntiquantProcess::Process,
// grouped_gemm/op_kernel/grouped_matmul_antiquant.h:241-288).  Expert g with m_g rows
// has ceil(m_g/BLOCK) row blocks, cut into the fewest chunks of <= MT_MAX blocks, as
// even as possible; each chunk has N/256 tiles.  prefix[] (in LDS) is the exclusive
// scan of the tile counts.
// ---------------------------------------------------------------------------------
template <int MT_MAX, int BLOCK>
__device__ __forceinline__ void expert_chunks(int m, int& chunks, int& bpc) {
    const int nblk = (m + BLOCK - 1) / BLOCK;
    if (nblk <= MT_MAX) {   // the usual case, without the division
        chunks = nblk ? 1 : 0;
        bpc = nblk;
        return;
    }
    chunks = (nblk + MT_MAX - 1) / MT_MAX;
    bpc = (nblk + chunks - 1) / chunks;
}

// Inclusive sums over the lanes of a row of 16: DPP shifts (a shuffle goes through LDS, about 100 cycles)
__device__ __forceinline__ int row_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    return v;
}

// The order in which a launch takes its experts: those with the largest tiles (most row blocks per chunk) first, those
// without rows last, otherwise as they come.  A tile's time goes by its row blocks, and with the largest tiles up to half
// of a launch long, one that starts among the last leaves most of the chip waiting for it.
// us as they come / in this order, rows unevenly routed (skew: see moe_dispatch.cpp): fp4 SwiGLU, 1511 tokens x 8 on 256
// experts of 7168 x 2048, skew 1: 578 / 563, skew 0.25: 628 / 615; int4, 2000 x 4 on 64 of 7168 x 2048, skew 0.25: 307 / 282.
// It takes 0.55 us of every workgroup with 4 wavefronts, 0.8 with 8 (an earlier form with shuffles and a second pass over the experts
// 1.1 and 1.3), which small launches and those that need no order lose: only launches of KernelCfg::ORDER_MIN_WORK do it.  Times as fast as
// unordered, median (worst, best) evenly routed, by balanced top-k routing and at a skew of 1: int4 and fp4 on GK_QUAD, 0.25 to 0.5
// million tiles times k (20 us) 0.966 (0.93), 0.968 (0.94), 1.05; 0.5 to 1 million 0.99 (0.967), 0.995 (0.95), 1.0; 1 to 3 million
// (50 to 100 us) 0.99 (0.95), 0.995 (0.965), 1.06 (0.95, 1.26); more 0.995 (0.973), 1.0 (0.96), 1.07 (0.966, 1.3).  int8 and fp8 on
// GK_PAIR, 0.5 to 3 million (40 to 110 us) 0.987 (0.97), 0.975 (0.9), 1.01 (0.92, 1.22); more 0.997 (0.973), 0.995 (0.966),
// 1.035 (0.955, 1.15).  (The scan that follows stays on shuffles: with DPP it saves 0.25 us more, but the k loops of int8 on GK_QUAD, laid out
// a little differently around it, came out 1 to 4 % slower at K = 7168.)
// Not for bf16, whose tiles wait for memory or for the matrix cores by their size: large and small ones side by side use both, and
// that goes either way.  1021 x 8 on 64 of 7168 x 2048, three routings each of skew 0.25 and 0.5: 508 / 485, 457 / 472, 462 / 476
// and 510 / 470, 496 / 474, 502 / 476; 1500 x 2 on 16 of 4096 x 8192, skew 1: 287 / 302; 700 x 8 on 64 of 7168 x 2048, skew 0:
// 359 / 366.  (Largest and median ones in turn: 0.955 to 1.077 times as fast as unordered over the same calls.)
// Every workgroup works the same order out: a counting sort, ranks from ballots; 64 experts of a wavefront at a
// time leave one count per class in scratch (LDS of the tile routine, [rounds * WAVES][16]).
template <int MTM, int BLOCK, int WAVES, typename Rows>
__device__ __forceinline__ void order_experts(int G, int ntile_n, int tid, int* scratch, uint16_t* order, int* tiles, Rows expert_rows) {
    static_assert(MTM < 15, "classes 0 .. MTM, 15 for no expert");
    const int lane = tid & 63, wave = tid >> 6, col = lane & 15, rounds = (G + 64 * WAVES - 1) / (64 * WAVES);
    int c = 15, n_tiles = 0;   // of this thread's expert in the round
    auto look = [&](int g) {
        c = 15;
        if (g < G) {
            int first, chunks, bpc;
            expert_chunks<MTM, BLOCK>(expert_rows(g, first), chunks, bpc);
            c = MTM - bpc;
            n_tiles = chunks * ntile_n;
        }
    };
    for (int r = 0; r < rounds; ++r) {
        look(r * 64 * WAVES + tid);
        int n = 0;
#pragma unroll
        for (int k = 0; k <= MTM; ++k) {
            const int in = __popcll(__ballot(c == k));
            if (lane == k) n = in;
        }
        if (lane < 16) scratch[(r * WAVES + wave) * 16 + lane] = n;
    }
    __syncthreads();
    // lane k (mod 16): where class k starts for the next 64 experts of this wavefront
    int all = 0, next = 0;
    for (int r = 0; r < rounds; ++r)
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const int n = scratch[(r * WAVES + w) * 16 + col];
            all += n;
            next += r == 0 && w < wave ? n : 0;
        }
    next += row_scan(all) - all;
    for (int r = 0;;) {
        const int g = r * 64 * WAVES + tid;
        if (rounds > 1) look(g);
        unsigned long long same = 0;
#pragma unroll
        for (int k = 0; k <= MTM; ++k) {
            const unsigned long long in = __ballot(c == k);
            if (c == k) same = in;
        }
        const int at = __shfl(next, c, 64) + __popcll(same & ((1ull << lane) - 1));
        if (g < G) {
            order[at] = (uint16_t)g;
            tiles[at] = n_tiles;
        }
        if (++r == rounds) break;
        // before the wavefront's next 64 experts come these, those of the wavefronts behind it and the next of those in front
#pragma unroll
        for (int w = 0; w < WAVES; ++w) next += scratch[((w < wave ? r : r - 1) * WAVES + w) * 16 + col];
    }
    __syncthreads();
}

template <int FMT, int KIND>
struct KernelCfg {
    static constexpr bool PAIR = KIND == GK_PAIR || KIND == GK_PAIR_SMALL || KIND == GK_QUAD || pair_exact(KIND);
    static constexpr bool FP4_K = KIND == GK_FP4_K;
    static_assert(PAIR == (FMT != MOE_FMT_BF16 && !FP4_K) && (!FP4_K || FMT == MOE_FMT_FP4_B32 || FMT == MOE_FMT_FP4_B16), "the routine of the container");
    static constexpr int WAVES = PAIR ? pair_waves(KIND) : FP4_K ? 4 : 8;
    static constexpr int BLOCK = PAIR || FP4_K ? 16 : 32;   // rows per row block of a tile routine's template argument
    static constexpr int BN = GM_BN;                                             // columns per tile
    static constexpr int pair_wgs() {
        if constexpr (PAIR) return pair_wg_per_cu<FMT>(KIND); else return FP4_K ? 2 : 1;
    }
    static constexpr int WG_PER_CU = pair_wgs();
    static constexpr int WAVES_PER_SIMD = WG_PER_CU * WAVES / 4;
    static constexpr int MTM = PAIR ? pair_mt_max(KIND) : FP4_K ? FK_MT_MAX : KIND == GK_BF16_128 ? 4 : BF_MT_MAX;   // row blocks per tile
    // tiles of up to 32 rows take the time of their weights, in any order; bf16: see order_experts; K-contiguous fp4 on GK_PAIR has
    // a tile per CU or evenly filled ones (6 % slower in this order at 256 tiles, evenly routed)
    static constexpr bool ORDERED = KIND == GK_QUAD || KIND == GK_FP4_K || (KIND == GK_PAIR && (FMT == MOE_FMT_INT8 || FMT == MOE_FMT_FP8_REF));
    // ... in launches of at least that many tiles (an upper bound) times k
    static constexpr int64_t ORDER_MIN_WORK = KIND == GK_PAIR ? 3 << 20 : 1 << 19;
    // tiles of mt row blocks have a form with nontemporal weight loads
    static constexpr bool nontemporal(int mt) { return PAIR && FMT != MOE_FMT_FP4_B32 && FMT != MOE_FMT_FP4_B16 && mt <= nt_mt_max(KIND); }
    // 16-byte LDS units of the tile routine (the tile prefix array follows them)
    static constexpr int lds_units() {
        if constexpr (PAIR)
            return pair_lds_units<FMT>(KIND);
        else
            return FP4_K ? fk_lds_units() : bf_lds_units();
    }
};

template <int FMT, int MT, int KIND>
__device__ __forceinline__ void run_tile(const GemmParams& P, u32x4_t* smem, int g, int64_t row0, int rows, int n0, const Ticket& tk, bool deep, bool nt) {
    using C = KernelCfg<FMT, KIND>;
    if constexpr (C::PAIR) {
        if constexpr (C::nontemporal(MT)) {
            if (nt) {
                if constexpr (FMT == MOE_FMT_FP4_REF && pair_exact(KIND)) {
                    if (rows <= 8) return gemm_tile_pair<FMT, MT, KIND, true, false, true>(P, smem, g, row0, rows, n0, tk);
                }
                return gemm_tile_pair<FMT, MT, KIND, false, false, true>(P, smem, g, row0, rows, n0, tk);
            }
        }
        if constexpr (KIND == GK_QUAD && MT <= QUAD_DEEP_MT && (FMT == MOE_FMT_INT4 || FMT == MOE_FMT_FP4_REF)) {
            if (deep) return gemm_tile_pair<FMT, MT, KIND, false, true>(P, smem, g, row0, rows, n0, tk);
        }
        if constexpr (FMT == MOE_FMT_FP4_REF && pair_exact(KIND) && MT == 1) {
            if (rows <= 8) return gemm_tile_pair<FMT, MT, KIND, true>(P, smem, g, row0, rows, n0, tk);
        }
        gemm_tile_pair<FMT, MT, KIND>(P, smem, g, row0, rows, n0, tk);
    } else if constexpr (C::FP4_K) {
        gemm_tile_fp4_k<FMT, MT>(P, smem, g, row0, rows, n0, tk);
    } else {
        gemm_tile_bf16<MT>(P, smem, g, row0, rows, n0, tk);
    }
}

// The tile that a wavefront has found columns in that are no number: if one of its scales is beyond what the usual decode takes, once
// more with the decode that takes all (see wide_scales); else x is the reason.  The whole workgroup comes here together; tk draws no
// ticket (the tile has drawn the next one).
template <int FMT, int KIND>
__device__ __forceinline__ void redo_wide(const GemmParams& P, u32x4_t* smem, const Ticket& tk) {
    const int tid = threadIdx.x;
    auto word = [&](int e) { return __builtin_amdgcn_readfirstlane(tk.wide[e]); };
    const int g = word(1), row0 = word(2), rows = word(3), n0 = word(4);
    // everybody has read them, and the tile's stores have ended: the second time another wavefront may store a row block
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) tk.wide[0] = 0;
    __syncthreads();
    constexpr bool F8 = FMT == MOE_FMT_FP8_REF;
    // the tile's scales: [rows of scales][columns] out of rows of `stride`
    const int per = F8 ? 128 : 1, stride = P.N / per, columns = (min(P.N - n0, KernelCfg<FMT, KIND>::BN) + per - 1) / per;
    const int64_t scale_rows = F8 ? P.K / 128 : P.scale_rows, first = g * scale_rows * stride + n0 / per;
    bool found = false;
    for (int64_t e = tid; e < scale_rows * columns; e += blockDim.x) {
        const int64_t at = first + e / columns * stride + e % columns;
        if constexpr (F8)
            found = found || fabsf(static_cast<const float*>(P.scale)[at]) >= 0x1p120f;
        else
            found = found || (static_cast<const uint16_t*>(P.scale)[at] & 0x7fffu) >= 0x7a00u;   // 2^117
    }
    if (found) tk.wide[0] = 1;
    __syncthreads();
    const int wide = word(0);
    __syncthreads();
    if (tid == 0) tk.wide[0] = 0;
    if (!wide) return;
    for (int r = 0; r < rows; r += 16)
        gemm_tile_pair<FMT, 1, KIND, false, false, false, true>(P, smem, g, row0 + r, min(rows - r, 16), n0, tk);
}

template <int FMT, int KIND>
__global__ __launch_bounds__((64 * KernelCfg<FMT, KIND>::WAVES), (KernelCfg<FMT, KIND>::WAVES_PER_SIMD)) void grouped_gemm_kernel(GemmParams P) {
    using C = KernelCfg<FMT, KIND>;
    constexpr int WAVES = C::WAVES;
    extern __shared__ u32x4_t smem[];
    constexpr int THREADS = 64 * WAVES;
    constexpr int MTM = C::MTM;
    // [G + 1] first tile of every expert; table_mode 0: [THREADS + 1] first tile of every thread's run of experts
    int* prefix = reinterpret_cast<int*>(smem + C::lds_units());
    // [G + 1] row bounds: rowc[g] = group_list[g - 1] clamped to [0, M] (rowc[0] = 0); expert g owns the rows
    // [rowc[g], rowc[g + 1]) if that is not empty (same result as clamping start and end separately).  Kept in
    // LDS so that the scheduler does not wait for a global load per tile (2 to 4 us under a streaming kernel).
    int* rowc = prefix + (P.G + 1);
    // [G] table_mode 3: the expert at each place of prefix[]
    uint16_t* order = reinterpret_cast<uint16_t*>(rowc + (P.G + 1));
    const int tid = threadIdx.x;
    const int ntile_n = (P.N + C::BN - 1) / C::BN;
    // scan partials (one per wavefront); later part[0] carries the ticket drawn from the queue, part[1] the tile
    // resolved from it, part[2] the tile routine's arrival counter
    __shared__ int part[32];
    constexpr int PART_WIDE = 20;    // Ticket::wide
    constexpr int PART_FIXED = 16;   // first whether this workgroup uses the launch's counter, then its number of fixed sweeps
    auto clamp_row = [&](int64_t v) { return (int)min(max(v, (int64_t)0), P.M); };
    auto expert_rows = [&](int g, int& first) {
        int hi;
        if (P.table_mode >= 2) {
            first = rowc[g];
            hi = rowc[g + 1];
        } else {
            first = g ? clamp_row(P.gl[g - 1]) : 0;
            hi = clamp_row(P.gl[g]);
        }
        return max(hi - first, 0);
    };

    // the launch's counter is looked at, and raised to the launch's stamp, now: long before the first draw from it
    if (tid == 0) part[PART_FIXED] = P.slot >= 0 && queue_open(tile_queue + GM_QUEUE_STRIDE * max(P.slot, 0), P.stamp, blockIdx.x < 8);

    if (wide_scales<FMT>(KIND) && tid == 0) part[PART_WIDE] = 0;   // (set by the tile routine, cleared by redo_wide)

    // exclusive scan of tiles per expert: each thread takes a contiguous run of experts
    const int per = (P.G + THREADS - 1) / THREADS;
    const int entries = P.table_mode ? P.G : THREADS;   // the table has entries + 1 elements
    {
        const int g0 = min(P.G, tid * per), g1 = min(P.G, g0 + per);
        if (P.table_mode >= 2) {
            for (int g = g0; g < g1; ++g) rowc[g + 1] = clamp_row(P.gl[g]);
            if (tid == 0) rowc[0] = 0;
            __syncthreads();
        }
        if constexpr (C::ORDERED)
            if (P.table_mode == 3) order_experts<MTM, C::BLOCK, WAVES>(P.G, ntile_n, tid, reinterpret_cast<int*>(smem), order, prefix, expert_rows);
        // tiles of the expert at place e (order_experts has left them in the table)
        auto tiles_at = [&](int e) {
            if (C::ORDERED && P.table_mode == 3) return prefix[e];
            int first, chunks, bpc;
            expert_chunks<MTM, C::BLOCK>(expert_rows(e, first), chunks, bpc);
            return chunks * ntile_n;
        };
        int sum = 0;
        for (int e = g0; e < g1; ++e) sum += tiles_at(e);
        // scan over the threads: within a wavefront by shuffles, across wavefronts through their totals in
        // LDS (a loop of one thread over all partial sums took 8 us at the start of every workgroup)
        const int lane = tid & 63, wave = tid >> 6;
        int incl = sum;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int up = __shfl_up(incl, off, 64);
            if (lane >= off) incl += up;
        }
        if (lane == 63) part[wave] = incl;
        __syncthreads();
        int before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const int v = part[w];
            before += w < wave ? v : 0;
            all += v;
        }
        if (tid == 0) prefix[entries] = all;
        int run = before + incl - sum;
        if (P.table_mode) {
            for (int e = g0; e < g1; ++e) {
                const int n = tiles_at(e);
                prefix[e] = run;
                run += n;
            }
        } else {
            prefix[tid] = run;
        }
        __syncthreads();
    }
    const int total = __builtin_amdgcn_readfirstlane(prefix[entries]);

    // more than one tile per workgroup (see QUAD_DEEP_STAGES)
    const bool deep = total > (int)gridDim.x;

    // XCD-aware order: workgroup b runs on XCD b % 8; give each XCD a contiguous run of
    // tiles in every sweep so that its workgroups share x rows in its own L2.
    const int nwg = gridDim.x;
    const int per_xcd = (nwg + 7) / 8;
    const int vid = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    const int sweep = per_xcd * 8;   // == nwg: the grid is a multiple of 8
    // The number of sweeps in the fixed order lives in LDS, not in a register that would stay live across the tile
    // routines; GM_NO_QUEUE: a launch without counters (captured into a HIP graph, or one whose slot a later launch
    // holds by now) walks every tile in the fixed order, sweep after sweep until the tile number passes the last.
    constexpr int GM_NO_QUEUE = 0x7fffffff;
    // (at least one sweep in the fixed order before the first draw, so that the stamp is there by then; launches of
    // at most one tile per workgroup have nothing to balance)
    if (tid == 0) part[PART_FIXED] = part[PART_FIXED] && total > sweep ? max(1, total / sweep - GM_QUEUE_TAIL_SWEEPS) : GM_NO_QUEUE;
    __syncthreads();

    bool have_ticket = false;   // the previous tile routine left its ticket in part[0]
    queue_word_t* const q_own = tile_queue + GM_QUEUE_STRIDE * max(P.slot, 0);
    auto ticket_from = [&](queue_word_t* counter) { return Ticket{counter, part, part + 2, part + PART_WIDE}; };
    for (int sw = 0;; ++sw) {
        int T;
        const int look_again = wide_scales<FMT>(KIND) ? part[PART_WIDE] : 0;
        int fixed = __builtin_amdgcn_readfirstlane(part[PART_FIXED]);
        if constexpr (wide_scales<FMT>(KIND)) {
            // the previous tile's (set ahead of the barrier that ends the tile routine, and not again before one that every wavefront
            // reaches after this; read here, beside the other word: behind the tile routine it cost 1 % of decode-like launches)
            if (__builtin_amdgcn_readfirstlane(look_again)) [[unlikely]] redo_wide<FMT, KIND>(P, smem, ticket_from(nullptr));
        }
        if (sw >= fixed) {
            if (fixed == GM_NO_QUEUE) break;
            if (!have_ticket) {
                __syncthreads();   // part[] of the previous round is read
                if (tid == 0) part[0] = queue_draw(q_own, P.stamp);
                __syncthreads();
            }
            const int own = __builtin_amdgcn_readfirstlane(part[0]);
            if (own >= 0) {
                T = fixed * sweep + own;
                if (T >= total) break;
            } else {
                // the slot belongs to a later launch: this workgroup's share of the tail in the fixed order
                __syncthreads();   // everyone has read this round's part[PART_FIXED]
                if (tid == 0) part[PART_FIXED] = GM_NO_QUEUE;
                sw = fixed;
                fixed = GM_NO_QUEUE;
            }
        }
        if (sw < fixed) {
            // (the last, partial sweep of a launch without a counter goes to the workgroups in launch order, i.e.
            // round-robin over the XCDs and to different CUs first, not to the first XCDs' workgroups only: where two
            // workgroups share a CU the tiles per CU, which is what its time follows, then differ by at most one)
            T = sw * sweep + ((sw + 1) * sweep > total ? (int)blockIdx.x : vid);
            if (T >= total) break;
        }
        // from the last tile of the fixed order on, the tile routines draw the next ticket themselves
        const bool take = fixed != GM_NO_QUEUE && sw + 1 >= fixed;
        const Ticket tk = ticket_from(take ? q_own : nullptr);
        have_ticket = take;
        // largest e with prefix[e] <= T (empty experts have prefix[e] == prefix[e+1]): every wavefront looks at 64
        // evenly spaced entries at once, then at the entries between two of them -- two LDS round trips
        // instead of the ten of a binary search
        const int lane64 = tid & 63;
        const int stride = (entries + 63) >> 6;                  // entries per lane of the first step
        const int probe = min(lane64 * stride, entries);
        const unsigned long long le1 = __ballot(prefix[probe] <= T && lane64 * stride <= entries);
        const int seg = 63 - __builtin_clzll(le1 | 1ull);        // last lane whose entry is <= T (lane 0: prefix[0] = 0)
        // (the entries <= T of a segment are its first ones: count them, 64 at a time; one pass up to 4096 entries)
        int upto = 0;
        for (int o = 0; o < stride; o += 64) {
            const int idx2 = seg * stride + o + lane64;
            const int n_le = __popcll(__ballot(o + lane64 < stride && idx2 < entries && prefix[idx2] <= T));
            upto += n_le;
            if (n_le < 64) break;
        }
        // everything below is wave-uniform; readfirstlane lets the compiler keep it in SGPRs
        const int found = __builtin_amdgcn_readfirstlane(seg * stride + max(upto, 1) - 1);
        int g = found, local = __builtin_amdgcn_readfirstlane(T - prefix[found]);
        if (C::ORDERED && P.table_mode == 3) {
            g = __builtin_amdgcn_readfirstlane((int)order[found]);
        } else if (P.table_mode == 0) {
            // found is a thread's run of experts: walk it 64 experts at a time (group_list from memory, the tile
            // counts summed across the wavefront) up to the expert that holds tile number `local` of the run
            const int e_end = min(P.G, (found + 1) * per);
            g = -1;
            for (int e0 = found * per, base = 0; e0 < e_end && g < 0; e0 += 64) {
                const int ge = e0 + lane64;
                int tiles = 0;
                if (ge < e_end) {
                    int first, ch, bp;
                    expert_chunks<MTM, C::BLOCK>(expert_rows(ge, first), ch, bp);
                    tiles = ch * ntile_n;
                }
                int incl = tiles;
#pragma unroll
                for (int off = 1; off < 64; off <<= 1) {
                    const int up = __shfl_up(incl, off, 64);
                    if (lane64 >= off) incl += up;
                }
                const unsigned long long hit = __ballot(base + incl > local);
                if (hit) {
                    const int l = __ffsll(hit) - 1;
                    g = e0 + l;
                    local -= base + __shfl(incl - tiles, l, 64);
                } else {
                    base += __shfl(incl, 63, 64);
                }
            }
            g = __builtin_amdgcn_readfirstlane(g);
            local = __builtin_amdgcn_readfirstlane(local);
            if (g < 0) break;   // cannot happen: the run holds the tile
        }
        int gfirst;
        const int m = __builtin_amdgcn_readfirstlane(expert_rows(g, gfirst));
        const int64_t gbeg = gfirst;
        int chunks, bpc;
        expert_chunks<MTM, C::BLOCK>(m, chunks, bpc);
        // row chunks innermost: the tiles that share a weight column tile are neighbours in the order, run at
        // the same time on one XCD and pull that slice of the expert's weights into its L2 once
        const int nt = chunks == 1 ? local : local / chunks, chunk = chunks == 1 ? 0 : local % chunks;
        const int rbeg = chunk * bpc * C::BLOCK;
        const int rows = min(m - rbeg, bpc * C::BLOCK);
        const int mt = (rows + C::BLOCK - 1) / C::BLOCK;
        const int rlo = __builtin_amdgcn_readfirstlane((int)(uint32_t)(gbeg & 0xffffffffLL));
        const int rhi = __builtin_amdgcn_readfirstlane((int)(gbeg >> 32));
        const int64_t row0 = (((int64_t)rhi << 32) | (uint32_t)rlo) + rbeg;
        const int n0 = nt * C::BN;
        const bool nontemporal = m <= P.nt_rows;   // the expert's only tile of these columns
        switch (mt) {
            case 1:
                if constexpr (MTM >= 1) run_tile<FMT, 1, KIND>(P, smem, g, row0, rows, n0, tk, deep, nontemporal);
                break;
            case 2:
                if constexpr (MTM >= 2) run_tile<FMT, 2, KIND>(P, smem, g, row0, rows, n0, tk, deep, nontemporal);
                break;
            case 3:
                if constexpr (MTM >= 3) run_tile<FMT, 3, KIND>(P, smem, g, row0, rows, n0, tk, deep, nontemporal);
                break;
            case 4:
                if constexpr (MTM >= 4) run_tile<FMT, 4, KIND>(P, smem, g, row0, rows, n0, tk, deep, nontemporal);
                break;
            case 5:
                if constexpr (MTM >= 5) run_tile<FMT, 5, KIND>(P, smem, g, row0, rows, n0, tk, deep, nontemporal);
                break;
            case 6:
                if constexpr (MTM >= 6) run_tile<FMT, 6, KIND>(P, smem, g, row0, rows, n0, tk, deep, nontemporal);
                break;
            case 7:
                if constexpr (MTM >= 7) run_tile<FMT, 7, KIND>(P, smem, g, row0, rows, n0, tk, deep, nontemporal);
                break;
            case 8:
                if constexpr (MTM >= 8) run_tile<FMT, 8, KIND>(P, smem, g, row0, rows, n0, tk, deep, nontemporal);
                break;
            case 9:
                if constexpr (MTM >= 9) run_tile<FMT, 9, KIND>(P, smem, g, row0, rows, n0, tk, deep, nontemporal);
                break;
            case 10:
                if constexpr (MTM >= 10) run_tile<FMT, 10, KIND>(P, smem, g, row0, rows, n0, tk, deep, nontemporal);
                break;
            default: have_ticket = false; break;
        }
    }
}

int64_t gemm_shift_launch_number(int64_t delta) {
    return (int64_t)(queue_launches.fetch_add((uint64_t)delta, std::memory_order_relaxed) + (uint64_t)delta);
}

// Compute units of the current device, looked up once per device.
static int device_cu_count() {
    static std::atomic<int> cached[64];
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return -1;
    int cus = cached[dev].load(std::memory_order_relaxed);
    if (cus == 0) {
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) return -1;
        cached[dev].store(cus, std::memory_order_relaxed);
    }
    return cus;
}

template <int FMT, int KIND>
static int launch_gemm_kind(const GemmParams& P, const moe_grouped_args* a, hipStream_t stream) {
    using C = KernelCfg<FMT, KIND>;
    constexpr size_t lds_max = (160 * 1024 - 512) / C::WG_PER_CU;
    const size_t table = ((size_t)a->G + 1) * sizeof(int);
    // tile table, and the row bounds next to it where they fit; else the scheduler reads group_list per tile; else,
    // with more experts than LDS holds a table for, it keeps one entry per thread and walks group_list (see
    // GemmParams::table_mode)
    constexpr size_t units = (size_t)C::lds_units() * 16, thread_table = (size_t)(64 * C::WAVES + 1) * sizeof(int);
    static_assert(units + thread_table <= lds_max, "any number of experts");
    int table_mode = units + 2 * table <= lds_max ? 2 : units + table <= lds_max ? 1 : 0;
    size_t lds = units + (table_mode ? table_mode * table : thread_table);
    static std::atomic<uint64_t> lds_set{0};
    if (const int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&grouped_gemm_kernel<FMT, KIND>), (int)lds_max, lds_set))
        return rc;
    const int cus = device_cu_count();
    if (cus <= 0) return MOE_ERR_NO_DEVICE;
    // persistent grid: as many workgroups as the CUs hold, but no more than an upper bound on the
    // tile count that needs no look at group_list (every expert adds at most one partly filled chunk)
    const int64_t max_chunks = a->M / (C::BLOCK * C::MTM) + a->G;
    const int64_t max_tiles = max_chunks * ((a->N + C::BN - 1) / C::BN);
    const int64_t want = max_tiles < (int64_t)cus * C::WG_PER_CU ? max_tiles : (int64_t)cus * C::WG_PER_CU;
    // where a workgroup may get more than one tile, the experts with the largest ones come first (as far as LDS has room, and in
    // launches long enough for it, see order_experts)
    if (C::ORDERED && table_mode == 2 && max_tiles > want && max_tiles * a->K >= C::ORDER_MIN_WORK && lds + (size_t)a->G * sizeof(uint16_t) <= lds_max) {
        table_mode = 3;
        lds += (size_t)a->G * sizeof(uint16_t);
    }
    // a multiple of 8 so that the XCD-aware order covers every tile index
    const int64_t grid = want > 0 ? (want + 7) / 8 * 8 : 8;
    GemmParams Q = P;
    // A launch that is being captured into a graph gets no counters (see tile_queue); so does one whose
    // stream cannot be queried.  (The null stream cannot be captured and is not asked.)
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (stream != nullptr && hipStreamIsCapturing(stream, &capture) != hipSuccess) {
        (void)hipGetLastError();
        capture = hipStreamCaptureStatusActive;
    }
    if (capture == hipStreamCaptureStatusNone) {
        const uint64_t launch = queue_launches.fetch_add(1, std::memory_order_relaxed);
        Q.slot = (int)(launch % GM_QUEUE_SLOTS);
        Q.stamp = (launch / GM_QUEUE_SLOTS + 1) << GM_QUEUE_COUNT_BITS;
    } else {
        Q.slot = -1;
        Q.stamp = 0;
    }
    Q.table_mode = table_mode;
    hipLaunchKernelGGL((grouped_gemm_kernel<FMT, KIND>), dim3((unsigned)grid), dim3(64 * C::WAVES), lds, stream, Q);
    return hipGetLastError() == hipSuccess ? MOE_OK : MOE_ERR_LAUNCH;
}

// Nontemporal weight loads.  A weight line that is read once in a launch, whole, only pushes others out of L2 and the 256 MB behind
// it.  So: the N-contiguous containers on GK_PAIR and the small-stage kinds, for experts whose rows are one tile (GK_PAIR: of up to 4 row
// blocks, small stages: of one), in launches that may read more weights (min(M, G) experts, if each has rows) than those caches
// can keep for the next launch that reads them.  us, without / with: GEMV op, 512 rows on 128 experts of 7168 x
// 2048, fp8 307 / 270, on 256, int4 311 / 292, fp4 359 / 331; GEMM op, 512 rows on 256, fp4 374 / 355, int4 350 / 336; fp8, 128 rows on
// 64 of 2048 x 1024 28.0 / 25.5, 1024 on 256 of 7168 x 2048 599 / 562; int8, 800 on 64 of 4096 x 4096 191 / 182.  Weights that
// the caches still hold from the last time are faster read as usual: 84 MB of fp8 18.6 / 22.0, 67 MB of int4 21.3 / 21.6; 134 MB of
// int4 39.3 / 37.2, 126 MB of fp4 33.3 / 31.2.  With row chunks that share their weights 256 rows of 8 experts, int8: 456 / 501; fp4,
// 512 rows on 64 of 7168 x 2048 at a skew of 1, without / with in every tile of one row block / with for experts of one tile: GEMV op 105 / 111 /
// 102, GEMM op 105 / 112 / 99.  bf16, whose lines are read in halves: 485 / 586; GK_QUAD gains nothing (int4, 16 rows each on 256 experts 476 / 470, fp4 unevenly routed 540 / 540).
constexpr int64_t NT_MIN_BYTES = 96 << 20;
int nontemporal_rows(const moe_grouped_args* a, GroupedKernel k) {
    const bool pair = k == GroupedKernel::TILES_PAIR;
    const bool small = k == GroupedKernel::TILES_PAIR_SMALL || k == GroupedKernel::TILES_PAIR_EXACT || k == GroupedKernel::TILES_PAIR_EXACT16;
    const bool byte = a->format == MOE_FMT_INT8 || a->format == MOE_FMT_FP8_REF, four_bit = a->format == MOE_FMT_INT4 || a->format == MOE_FMT_FP4_REF;
    if (!(pair || small) || !(byte || four_bit)) return 0;
    if (std::min(a->M, a->G) * (a->K * a->N >> (byte ? 0 : 1)) < NT_MIN_BYTES) return 0;
    return 16 * nt_mt_max(pair ? GK_PAIR : GK_PAIR_SMALL);
}

static GemmParams gemm_params(const moe_grouped_args* a, GroupedKernel kind) {
    GemmParams P;
    P.x = static_cast<const uint16_t*>(a->x);
    P.w = static_cast<const uint8_t*>(a->weight);
    P.scale = a->scale;
    P.offset = static_cast<const uint16_t*>(a->offset);
    P.gl = a->group_list;
    P.y = static_cast<uint16_t*>(a->y);
    P.M = a->M; P.K = (int)a->K; P.N = (int)a->N; P.G = (int)a->G; P.scale_rows = (int)a->scale_rows;
    P.epilogue = a->epilogue;
    P.nt_rows = nontemporal_rows(a, kind);
    P.slot = -1;
    P.stamp = 0;
    P.table_mode = 0;
    P.scale_div = scale_row_divider(a->K, a->scale_rows);
    return P;
}

int launch_tiles(const moe_grouped_args* a, GroupedKernel kind, hipStream_t stream) {
    const GemmParams P = gemm_params(a, kind);
    switch (kind) {
        case GroupedKernel::TILES_PAIR:
            switch (a->format) {
                case MOE_FMT_FP8_REF: return launch_gemm_kind<MOE_FMT_FP8_REF, GK_PAIR>(P, a, stream);
                case MOE_FMT_INT8: return launch_gemm_kind<MOE_FMT_INT8, GK_PAIR>(P, a, stream);
                case MOE_FMT_FP4_B32: return launch_gemm_kind<MOE_FMT_FP4_B32, GK_PAIR>(P, a, stream);
                case MOE_FMT_FP4_B16: return launch_gemm_kind<MOE_FMT_FP4_B16, GK_PAIR>(P, a, stream);
                default: return MOE_ERR_BAD_FORMAT;
            }
        case GroupedKernel::TILES_FP4_K:
            switch (a->format) {
                case MOE_FMT_FP4_B32: return launch_gemm_kind<MOE_FMT_FP4_B32, GK_FP4_K>(P, a, stream);
                case MOE_FMT_FP4_B16: return launch_gemm_kind<MOE_FMT_FP4_B16, GK_FP4_K>(P, a, stream);
                default: return MOE_ERR_BAD_FORMAT;
            }
        case GroupedKernel::TILES_PAIR_SMALL:
            switch (a->format) {
                case MOE_FMT_FP4_REF: return launch_gemm_kind<MOE_FMT_FP4_REF, GK_PAIR_SMALL>(P, a, stream);
                case MOE_FMT_INT4: return launch_gemm_kind<MOE_FMT_INT4, GK_PAIR_SMALL>(P, a, stream);
                default: return MOE_ERR_BAD_FORMAT;
            }
        case GroupedKernel::TILES_QUAD:
            switch (a->format) {
                case MOE_FMT_FP4_REF: return launch_gemm_kind<MOE_FMT_FP4_REF, GK_QUAD>(P, a, stream);
                case MOE_FMT_FP8_REF: return launch_gemm_kind<MOE_FMT_FP8_REF, GK_QUAD>(P, a, stream);
                case MOE_FMT_INT8: return launch_gemm_kind<MOE_FMT_INT8, GK_QUAD>(P, a, stream);
                case MOE_FMT_INT4: return launch_gemm_kind<MOE_FMT_INT4, GK_QUAD>(P, a, stream);
                default: return MOE_ERR_BAD_FORMAT;
            }
        case GroupedKernel::TILES_PAIR_EXACT:
            switch (a->format) {
                case MOE_FMT_FP4_REF: return launch_gemm_kind<MOE_FMT_FP4_REF, GK_PAIR_EXACT>(P, a, stream);
                case MOE_FMT_FP8_REF: return launch_gemm_kind<MOE_FMT_FP8_REF, GK_PAIR_EXACT>(P, a, stream);
                case MOE_FMT_INT4: return launch_gemm_kind<MOE_FMT_INT4, GK_PAIR_EXACT>(P, a, stream);
                default: return MOE_ERR_BAD_FORMAT;
            }
        case GroupedKernel::TILES_PAIR_EXACT16:
            return a->format == MOE_FMT_FP4_REF ? launch_gemm_kind<MOE_FMT_FP4_REF, GK_PAIR_EXACT16>(P, a, stream) : MOE_ERR_BAD_FORMAT;
        case GroupedKernel::TILES_BF16:
            return a->format == MOE_FMT_BF16 ? launch_gemm_kind<MOE_FMT_BF16, GK_BF16>(P, a, stream) : MOE_ERR_BAD_FORMAT;
        case GroupedKernel::TILES_BF16_128:
            return a->format == MOE_FMT_BF16 ? launch_gemm_kind<MOE_FMT_BF16, GK_BF16_128>(P, a, stream) : MOE_ERR_BAD_FORMAT;
        default: return MOE_ERR_BAD_FORMAT;
    }
}

}  // namespace moe
