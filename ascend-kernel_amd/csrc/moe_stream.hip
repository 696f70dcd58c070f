// Grouped GEMV / GEMM of a few rows on the N-contiguous containers (reference fp4 and fp8, int4, int8) for launches that
// leave most of the chip idle when a workgroup walks all of K: a token or two, few experts, few columns.
//
// Such a launch is bound by latency: a 256-column tile of the kernels in moe_gemm.hip walks K = 7168 in 112 dependent steps
// (a barrier each), and 8 rows of 8 experts with N = 512 make 16 of those tiles for 256 CUs.  Here a workgroup takes 16 T
// columns (32, 64 or 128) of one expert and its wavefronts split K between them: each streams its own range into registers,
// a few 32-k steps ahead, without LDS or barriers, and the partial sums meet once in LDS.  That case (18 MB of fp4 weights and
// scales): 47.6 -> 9.6 us, int4 48 -> 12.6, fp8 70 -> 16; two tokens on 256 experts of 7168 x 2048: int4 49 -> 33 us.
// What bounds it now: the launch, group_list and one step's latency are about 6 us; then the wait for the loads of a few wavefronts per
// SIMD (by counters 57 % of their cycles in that case, 33 % issuing: about 1.5 vector instructions per weight, 1.75 in 32-column strips of
// fp4, 2.5 with what a wavefront does before and after its 28 steps).
//
// MFMA: v_mfma_f32_16x16x32_bf16, x rows in A, weights in B.  Lane (i, q) = (lane & 15, lane >> 4) loads, of each of the 8 k
// rows 8 q + [0, 8) of a step, the dword (T = 8 and bytes: two) with its columns T i + [0, T): the 8 values of one column are
// its B fragment of MFMA t, column T i + t, so nothing crosses lanes.  The reference's pre-shuffled fp4 tile holds 8 k rows
// of 8 columns as 32 contiguous bytes.
//
// Arithmetic: ROUNDW that of the grouped GEMM op (weights rounded to bf16), else that of the GEMV op (weights not rounded:
// the fragments hold the codes, a scale group's sums are multiplied by its fp32 scale), as in gemm_tile_pair.
#include <type_traits>

#include "moe_device.h"
#include "moe_internal.h"
#include "scale_group.h"

namespace moe {

constexpr int ST_WAVES = 8;      // wavefronts per workgroup, each a share of K
constexpr int ST_ROWS = 16;      // x rows per pass over the weights

struct StreamParams {
    const uint16_t* x;
    const uint8_t* w;
    const void* scale;
    const uint16_t* offset;
    const int64_t* gl;
    uint16_t* y;
    int64_t M;
    int K, N, G, scale_rows;
    int epilogue;
    ScaleRowDivider scale_div;   // int4: the scale row of a 32-k step
};

typedef __amdgpu_buffer_rsrc_t rsrc_t;
static __device__ __forceinline__ rsrc_t slab(const void* p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (uint32_t)bytes, 0x00020000);
}
static __device__ __forceinline__ f32x4_t mfma(const u32x4_t& a, const u32x4_t& b, const f32x4_t& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// 4-bit codes, two columns a lane: the four lanes of a quad use a byte each of the same dwords.  A lane that loads all 8 rows of its
// dword loads four times what it uses, which takes the CU's vector memory path (64 bytes a cycle) four times as long (counters, together
// with the gathering of bytes below: lookups in the vector cache 1.29 / 0.83 M, address unit busy 6.6 / 5.4 k cycles, 3.2 / 2.5 vector
// instructions per weight).  So each lane of a quad loads two rows, and a 4 x 4 byte transpose over the quad (two DPP moves and two
// v_perm per dword) gives every lane its byte of all eight.  us, without / with: 8 single rows of 7168 x 512, fp4 GEMV op 10.5 / 9.6,
// GEMM op 11.2 / 10.5, int4 14.5 / 12.9; 192 rows on 8 experts of 4096 x 1024, fp4 15.1 / 13.4.  (Six or eight steps in flight instead of
// four in the registers that this frees: 0 to 2 % faster with fp4 and K = 7168, 2 to 11 % slower otherwise.  16 wavefronts: 0.88 to 1.02 times.)
template <int FMT, int T>
constexpr bool stream_quad() { return T == 2 && (FMT == MOE_FMT_FP4_REF || FMT == MOE_FMT_INT4); }

// Two int4 codes, the low or the high bytes of h, as fp32: a nibble read as e4m3 is q / 512, and the scaled conversion takes that back.
// (With 512 in the weight's scale instead, scales of 2^119 and more would leave the range of fp32; with -8 times the scale only those do for
// which the weight of code 0 does.)
template <bool HIGH>
static __device__ __forceinline__ f32x2_t int4_codes(uint32_t h) {
    return __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(h, 512.f, HIGH);
}

template <int FMT, int T>
struct StreamStep {   // what a wavefront holds of one 32-k step
    // k row j: the dword that holds this lane's columns; 8 columns of bytes: r[2 j] and r[2 j + 1]; stream_quad: lane l of a quad
    // holds the quad's dwords of rows 2 l and 2 l + 1
    uint32_t r[stream_quad<FMT, T>() ? 2 : T == 8 && (FMT == MOE_FMT_INT8 || FMT == MOE_FMT_FP8_REF) ? 16 : 8];
    u32x4_t x;
    uint32_t s[T / 2], s2[T / 2];   // scales of the T columns (fp8: s[0]); s2: fp4 without rounding, the second 16 k's
};

// STACK (fp4 without rounding, at most 8 rows): fragment row r < 8 of x keeps the first 16 k of x row r, row 8 + r the last
// 16 k, so one MFMA serves both scales of its 32 k (see gemm_tile_pair)
template <int FMT, bool ROUNDW, int T, bool STACK>
static __device__ __forceinline__ void stream_rows(const StreamParams& P, float* red, int g, int64_t row0, int mg, int n0) {
    constexpr bool FP4 = FMT == MOE_FMT_FP4_REF, F8 = FMT == MOE_FMT_FP8_REF, I8 = FMT == MOE_FMT_INT8, I4 = FMT == MOE_FMT_INT4;
    constexpr bool B8 = F8 || I8;
    constexpr int ST_COLS = 16 * T;
    constexpr bool QUAD = stream_quad<FMT, T>();
    constexpr bool TWO = FP4 && !ROUNDW && !STACK;   // two MFMAs per 32 k and column, one per scale
    // steps in flight (6, or 3 for 128 columns, change nothing; three where a fourth does not fit 128 registers)
    constexpr int D = FP4 && !ROUNDW && T == 4 ? 3 : 4;
    const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int steps = P.K >> 5;
    const int s0 = steps * wave / ST_WAVES, s1 = steps * (wave + 1) / ST_WAVES;
    const int64_t KN = (int64_t)P.K * P.N;
    const rsrc_t rw = slab(P.w + g * (B8 ? KN : KN >> 1), B8 ? KN : KN >> 1);
    const rsrc_t rx = slab(P.x + row0 * P.K, (int64_t)mg * P.K * 2);
    const rsrc_t rs = F8 ? slab(static_cast<const float*>(P.scale) + (int64_t)g * (P.K >> 7) * (P.N >> 7), (int64_t)(P.K >> 7) * (P.N >> 7) * 4)
                         : slab(static_cast<const uint16_t*>(P.scale) + (int64_t)g * P.scale_rows * P.N, (int64_t)P.scale_rows * P.N * 2);
    // x row of this lane's fragment row (rows past the last one lie outside the resource and read as zeros); STACK: lanes
    // whose half of k the fragment row does not keep are sent outside
    const int vx = STACK ? ((i >> 3) == (q >> 1) ? (i & 7) * P.K * 2 + q * 16 : 0x40000000) : i * P.K * 2 + q * 16;
    const int row_bytes = B8 ? P.N : P.N >> 1;
    const int col = n0 + T * i;   // this lane's first column
    const int ql = lane & 3;   // QUAD: which two of the 8 k rows this lane loads
    const int vw = FP4  ? (QUAD ? 8 * ql : 0) + (32 * (q & 1) + 8 * (q >> 1) + ((col >> 5) & 7)) * row_bytes + ((col >> 8) << 7) + 32 * ((col >> 3) & 3)
                   : B8 ? 8 * q * row_bytes + (col & ~3)
                        : (8 * q + (QUAD ? 2 * ql : 0)) * row_bytes + ((col >> 3) << 2);
    // QUAD: byte l of the dwords v of the quad's four lanes, in lane l
    const uint32_t quad_sel1 = ql & 1 ? 0x03070105u : 0x06020400u, quad_sel2 = ql & 2 ? 0x03020706u : 0x05040100u;
    auto quad_transpose = [&](uint32_t v) {
        const uint32_t h = __builtin_amdgcn_perm((uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, true), v, quad_sel1);      // lane l ^ 1
        return __builtin_amdgcn_perm((uint32_t)__builtin_amdgcn_mov_dpp((int)h, 0x4e, 0xf, 0xf, true), h, quad_sel2);   // lane l ^ 2
    };
    const int vs = FP4 && !TWO ? (q >> 1) * (P.N * 2) + col * 2 : col * 2;
    const uint32_t byte0 = B8 ? col & 3 : (col & 7) >> 1;   // the byte of a dword this lane's columns start at

    float ch_s[T], ch_o[T];
    if constexpr (I8) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
            ch_s[t] = bf16_bits_to_f32(static_cast<const uint16_t*>(P.scale)[(int64_t)g * P.N + col + t]);
            ch_o[t] = bf16_bits_to_f32(P.offset[(int64_t)g * P.N + col + t]);
        }
    }
    auto load_scales = [&](uint32_t (&d)[T / 2], int so) {
        if constexpr (T == 8) {
            const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rs, vs, so, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) d[e] = v[e];
        } else if constexpr (T == 4) {
            const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(rs, vs, so, 0);
            d[0] = v[0];
            d[1] = v[1];
        } else {
            d[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, vs, so, 0);
        }
    };

    auto load = [&](StreamStep<FMT, T>& d, int s) {
        d.x = __builtin_amdgcn_raw_buffer_load_b128(rx, vx, s * 64, 0);
        if constexpr (FP4) {
            const int so = ((s >> 1) * 64 + (s & 1) * 16) * row_bytes;
            if constexpr (QUAD) {
                const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(rw, vw, so, 0);
                d.r[0] = v[0];
                d.r[1] = v[1];
            } else {
                const u32x4_t lo = __builtin_amdgcn_raw_buffer_load_b128(rw, vw, so, 0);
                const u32x4_t hi = __builtin_amdgcn_raw_buffer_load_b128(rw, vw + 16, so, 0);
#pragma unroll
                for (int j = 0; j < 4; ++j) { d.r[j] = lo[j]; d.r[4 + j] = hi[j]; }
            }
            load_scales(d.s, 2 * s * (P.N * 2));
            if constexpr (TWO) load_scales(d.s2, (2 * s + 1) * (P.N * 2));
        } else {
#pragma unroll
            for (int j = 0; j < (QUAD ? 2 : 8); ++j) {
                if constexpr (B8 && T == 8) {
                    const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(rw, vw, (32 * s + j) * row_bytes, 0);
                    d.r[2 * j] = v[0];
                    d.r[2 * j + 1] = v[1];
                } else {
                    d.r[j] = __builtin_amdgcn_raw_buffer_load_b32(rw, vw, (32 * s + j) * row_bytes, 0);
                }
            }
            if constexpr (I4)
                load_scales(d.s, (int)scale_row(P.scale_div, (uint32_t)s) * (P.N * 2));
            if constexpr (F8) d.s[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, 0, ((s >> 2) * (P.N >> 7) + (n0 >> 7)) * 4, 0);
        }
    };

    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = zero;

    bool f8_plain = true;
    auto consume = [&](const StreamStep<FMT, T>& d) {
        // the two codes of byte `byte` of word
        auto fp4_pair = [](uint32_t word, int byte, float s) {
            switch (byte) {
                case 0: return ROUNDW ? e2m1_pair_scaled_bf16<0>(word, s) : __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, 1.f, 0));
                case 1: return ROUNDW ? e2m1_pair_scaled_bf16<1>(word, s) : __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, 1.f, 1));
                case 2: return ROUNDW ? e2m1_pair_scaled_bf16<2>(word, s) : __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, 1.f, 2));
                default: return ROUNDW ? e2m1_pair_scaled_bf16<3>(word, s) : __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, 1.f, 3));
            }
        };
        auto scale_of = [](const uint32_t (&s)[T / 2], int t) { return (t & 1) ? bf16_hi(s[t >> 1]) : bf16_lo(s[t >> 1]); };
        f32x4_t start = zero;
        if constexpr (I4 && !ROUNDW) {   // the fragments hold q: every product starts from -8 sum_k x
            const u32x4_t m8 = {0xc100c100u, 0xc100c100u, 0xc100c100u, 0xc100c100u};
            start = mfma(d.x, m8, zero);
        }
        u32x4_t xlo, xhi;
        if constexpr (TWO) {
            const uint32_t keep = q < 2 ? 0xffffffffu : 0u;
#pragma unroll
            for (int j = 0; j < 4; ++j) { xlo[j] = d.x[j] & keep; xhi[j] = d.x[j] & ~keep; }
        }
        const float f8s = F8 ? __uint_as_float(d.s[0]) * 256.f : 0.f;
        constexpr int TH = T < 4 ? T : 4;   // columns at a time
#pragma unroll
        for (int t0 = 0; t0 < T; t0 += TH) {
            u32x4_t bf[TH];
            float sc[TH];
#pragma unroll
            for (int t = 0; t < TH; ++t) sc[t] = F8 ? f8s : I8 ? 1.f : scale_of(d.s, t0 + t);
            const uint32_t b0 = T == 8 ? (B8 ? 0u : t0 >> 1) : byte0;
            // fp4, two or four columns: the lane's bytes of even and of odd k rows are gathered first, two or four row pairs to a dword
            // (QUAD: from the quad's lanes), and only they are paired up, the nibbles of two rows in a byte.  (Pairing whole dwords and
            // shifting took 28 instructions for 16 or 32 weights, this takes 12.)
            uint32_t even_col[2] = {0u, 0u}, odd_col[2] = {0u, 0u};   // T == 4: of row pairs 0 and 1, 2 and 3
            uint32_t even_rows = 0u, odd_rows = 0u;                   // QUAD: the lane's bytes of rows 0, 2, 4, 6 and 1, 3, 5, 7
            if constexpr (QUAD) {
                even_rows = quad_transpose(d.r[0]);
                odd_rows = quad_transpose(d.r[1]);
            }
            if constexpr (FP4 && T < 8) {
                auto pair_up = [&](uint32_t even, uint32_t odd, int e) {
                    const uint32_t m = 0x0f0f0f0fu;
                    even_col[e] = (even & m) | ((odd << 4) & ~m);
                    odd_col[e] = ((even >> 4) & m) | (odd & ~m);
                };
                if constexpr (QUAD) {
                    pair_up(even_rows, odd_rows, 0);
                } else {
                    const uint32_t sel = b0 | ((b0 + 1u) << 8) | ((4u + b0) << 16) | ((b0 + 5u) << 24);
                    pair_up(__builtin_amdgcn_perm(d.r[2], d.r[0], sel), __builtin_amdgcn_perm(d.r[3], d.r[1], sel), 0);
                    pair_up(__builtin_amdgcn_perm(d.r[6], d.r[4], sel), __builtin_amdgcn_perm(d.r[7], d.r[5], sel), 1);
                }
            }
            // int4, two columns: (even row, odd row) per byte, row pairs 0 and 1, 2 and 3; a nibble read as e4m3 is q / 512
            uint32_t quad_q[2][2] = {{0u, 0u}, {0u, 0u}};   // [even, odd column][row pairs]
            if constexpr (I4 && QUAD) {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint32_t u = __builtin_amdgcn_perm(odd_rows, even_rows, e ? 0x07030602u : 0x05010400u);
                    quad_q[0][e] = u & 0x0f0f0f0fu;
                    quad_q[1][e] = (u >> 4) & 0x0f0f0f0fu;
                }
            }
            // fp8 by the hardware's conversions, unless one of the wavefront's codes has turned out to be one that they make NaN of
            // (see decode_f8_plain in moe_gemm.hip).  us, without / with: 192 rows on 8 experts of 4096 x 2048 24.5 / 22.4, 16 single
            // rows of 7168 x 2048 49.7 / 47.1; random bytes 1 to 2 % slower.  In 32-column
            // strips, and those with the GEMV op's arithmetic, the two decodes side by side do not fit the registers.
            bool decoded = false;
            if constexpr (F8 && ROUNDW && T >= 4) {
                if (f8_plain) {
                    uint32_t seen_nan = 0u;
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        const uint32_t a = T == 8 ? d.r[4 * p + (t0 >> 2)] : d.r[2 * p], b = T == 8 ? d.r[4 * p + 2 + (t0 >> 2)] : d.r[2 * p + 1];
                        const float s = __uint_as_float(d.s[0]);
                        const f32x2_t a01 = __builtin_amdgcn_cvt_pk_f32_fp8(a, false), a23 = __builtin_amdgcn_cvt_pk_f32_fp8(a, true);
                        const f32x2_t b01 = __builtin_amdgcn_cvt_pk_f32_fp8(b, false), b23 = __builtin_amdgcn_cvt_pk_f32_fp8(b, true);
                        bf[0][p] = pack_bf16_rne(a01[0] * s, b01[0] * s);
                        bf[1][p] = pack_bf16_rne(a01[1] * s, b01[1] * s);
                        bf[2][p] = pack_bf16_rne(a23[0] * s, b23[0] * s);
                        bf[3][p] = pack_bf16_rne(a23[1] * s, b23[1] * s);
                        asm("v_pk_maximum3_f16 %0, %1, %2, %0" : "+v"(seen_nan) : "v"(bf[0][p]), "v"(bf[1][p]));
                        asm("v_pk_maximum3_f16 %0, %1, %2, %0" : "+v"(seen_nan) : "v"(bf[2][p]), "v"(bf[3][p]));
                    }
                    asm("v_pk_maximum3_f16 %0, %0, %0, %0 op_sel:[0,1,0] op_sel_hi:[0,1,0]" : "+v"(seen_nan));   // both halves
                    f8_plain = !__any(__builtin_isnan(__builtin_bit_cast(_Float16, (uint16_t)seen_nan)));
                    decoded = f8_plain;
                }
            }
            if constexpr (F8 && ROUNDW) {
                // Through fp16 (see e4m3_ref_pair_over_256).  PAIR: the 2^8 that this leaves out goes into the fp16 pairs, not into the block scale, which
                // from 2^120 on it would take out of the range of fp32.  32-column strips, which wait for their loads, pay nothing for
                // the half instruction per weight (8 single rows of 7168 x 512 15.7 / 15.6 us); the others 2 % with random codes, so they
                // look at the scale.
                auto through_fp16 = [&](auto PAIR) __attribute__((always_inline)) {
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        const uint32_t a = T == 8 ? d.r[4 * p + (t0 >> 2)] : d.r[2 * p], b = T == 8 ? d.r[4 * p + 2 + (t0 >> 2)] : d.r[2 * p + 1];
#pragma unroll
                        for (int t = 0; t < TH; ++t) {
                            const uint32_t at = T >= 4 ? (uint32_t)t : b0 + t;
                            const uint32_t sel8 = at | 0x0c00u | ((4u + at) << 16) | 0x0c000000u;   // [a.byte, 0, b.byte, 0]
                            uint32_t h2 = e4m3_ref_pair_over_256_fp16(__builtin_amdgcn_perm(b, a, sel8));
                            if constexpr (PAIR) h2 = fp16_pair_times_256(h2);
                            const float s = PAIR ? __uint_as_float(d.s[0]) : f8s;
                            float nz = -0.0f;
                            asm volatile("" : "+v"(nz));   // kept in a register: not an inline constant
                            bf[t][p] = pack_bf16_rne(fp16_lo_times(h2, s, nz), fp16_hi_times(h2, s, nz));
                        }
                    }
                };
                if (T < 4)
                    through_fp16(std::true_type{});
                else if (!decoded) {
                    if (((uint32_t)__builtin_amdgcn_readfirstlane((int)d.s[0]) & 0x7fffffffu) >= 0x7b800000u) [[unlikely]]   // 2^120
                        through_fp16(std::true_type{});
                    else
                        through_fp16(std::false_type{});
                }
            } else
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                // the dwords of k rows 2 p and 2 p + 1
                const uint32_t a = QUAD ? 0u : B8 && T == 8 ? d.r[4 * p + (t0 >> 2)] : d.r[2 * p], b = QUAD ? 0u : B8 && T == 8 ? d.r[4 * p + 2 + (t0 >> 2)] : d.r[2 * p + 1];
                if constexpr (I4 && QUAD) {
#pragma unroll
                    for (int t = 0; t < TH; ++t) {
                        const uint32_t h = quad_q[t][p >> 1];
                        if constexpr (ROUNDW) {
                            const f32x2_t f = p & 1 ? int4_codes<true>(h) : int4_codes<false>(h);
                            bf[t][p] = pack_bf16_rne(fmaf(f[0], sc[t], -8.f * sc[t]), fmaf(f[1], sc[t], -8.f * sc[t]));
                        } else {
                            bf[t][p] = __builtin_bit_cast(uint32_t, p & 1 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(h, 512.f, true)
                                                                          : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(h, 512.f, false));
                        }
                    }
                } else if constexpr (I4) {
                    // the lane's bytes of the two rows side by side, (a, b) per byte; a nibble read as e4m3 is q / 512
                    const uint32_t sel = b0 | ((4u + b0) << 8) | (T >= 4 ? ((b0 + 1u) << 16) | ((b0 + 5u) << 24) : 0x0c0c0000u);
                    const uint32_t u = __builtin_amdgcn_perm(b, a, sel);
                    const uint32_t h[2] = {u & 0x0f0f0f0fu, (u >> 4) & 0x0f0f0f0fu};   // even, odd columns
#pragma unroll
                    for (int t = 0; t < TH; ++t) {
                        if constexpr (ROUNDW) {
                            const f32x2_t f = t < 2 ? int4_codes<false>(h[t & 1]) : int4_codes<true>(h[t & 1]);
                            bf[t][p] = pack_bf16_rne(fmaf(f[0], sc[t], -8.f * sc[t]), fmaf(f[1], sc[t], -8.f * sc[t]));
                        } else {
                            bf[t][p] = __builtin_bit_cast(uint32_t, t < 2 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(h[t & 1], 512.f, false)
                                                                          : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(h[t & 1], 512.f, true));
                        }
                    }
                } else if constexpr (FP4 && T == 2) {
                    bf[0][p] = fp4_pair(even_col[0], p, sc[0]);
                    bf[1][p] = fp4_pair(odd_col[0], p, sc[1]);
                } else if constexpr (FP4 && T == 4) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) bf[t][p] = fp4_pair(t & 1 ? odd_col[p >> 1] : even_col[p >> 1], 2 * (p & 1) + (t >> 1), sc[t]);
                } else if constexpr (FP4) {
                    // nibbles of the two rows paired in a byte: even, odd columns
                    const uint32_t m = 0x0f0f0f0fu;
                    const uint32_t h[2] = {((a & m) | ((b << 4) & ~m)) >> (8 * b0), (((a >> 4) & m) | (b & ~m)) >> (8 * b0)};
#pragma unroll
                    for (int t = 0; t < TH; ++t) bf[t][p] = fp4_pair(h[t & 1], t >> 1, sc[t]);
                } else {
#pragma unroll
                    for (int t = 0; t < TH; ++t) {
                        const uint32_t at = T >= 4 ? (uint32_t)t : b0 + t;
                        if constexpr (F8) {
                            const uint32_t sel8 = at | 0x0c00u | ((4u + at) << 16) | 0x0c000000u;   // [a.byte, 0, b.byte, 0]
                            const uint32_t h2 = e4m3_ref_pair_over_256_fp16(__builtin_amdgcn_perm(b, a, sel8));
                            typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
                            const half2_t hv = __builtin_bit_cast(half2_t, h2);
                            bf[t][p] = pack_bf16_rne((float)hv[0], (float)hv[1]);
                        } else {
                            const float qa = (float)(int)(int8_t)(a >> (8 * at)), qb = (float)(int)(int8_t)(b >> (8 * at));
                            bf[t][p] = pack_bf16_rne(__fmul_rn(__fadd_rn(qa, ch_o[t0 + t]), ch_s[t0 + t]), __fmul_rn(__fadd_rn(qb, ch_o[t0 + t]), ch_s[t0 + t]));
                        }
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < TH; ++t) {
                f32x4_t& c = acc[t0 + t];
                if constexpr (ROUNDW) {
                    c = mfma(d.x, bf[t], c);
                } else if constexpr (TWO) {
                    const f32x4_t dl = mfma(xlo, bf[t], zero), dh = mfma(xhi, bf[t], zero);
                    const float s2 = scale_of(d.s2, t0 + t);
#pragma unroll
                    for (int e = 0; e < 4; ++e) c[e] = fmaf(dh[e], s2, fmaf(dl[e], sc[t], c[e]));
                } else {
                    const f32x4_t dd = mfma(d.x, bf[t], start);
#pragma unroll
                    for (int e = 0; e < 4; ++e) c[e] = fmaf(dd[e], sc[t], c[e]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);   // (or the scheduler decodes several steps at once, and spills)
        }
    };
    if (s0 < s1) {
        StreamStep<FMT, T> ring[D];
#pragma unroll
        for (int u = 0; u < D; ++u) load(ring[u], min(s0 + u, s1 - 1));
        int s = s0;
        for (; s + D < s1; s += D) {
#pragma unroll
            for (int u = 0; u < D; ++u) {
                consume(ring[u]);
                load(ring[u], min(s + u + D, s1 - 1));   // past the range: its last step again, from cache
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int u = 0; u < D; ++u)
            if (s + u < s1) {
                consume(ring[u]);
                __builtin_amdgcn_sched_barrier(0);
            }
    }
    if constexpr (STACK) {
        // lanes q and q + 2 hold the two scale groups' sums of the same rows
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[t][e] += __shfl_xor(acc[t][e], 32);
    }
    // partial sums [wavefront][row][column]; lane (i, q) holds rows 4 q + [0, 4) of its 8 columns
    const int rows4 = (mg + 3) & ~3;
    if (4 * q < mg) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float* d = red + ((wave * rows4 + 4 * q + e) * ST_COLS + T * i);
            if constexpr (T == 8) {
                reinterpret_cast<f32x4_t*>(d)[0] = f32x4_t{acc[0][e], acc[1][e], acc[2][e], acc[3][e]};
                reinterpret_cast<f32x4_t*>(d)[1] = f32x4_t{acc[4][e], acc[5][e], acc[6][e], acc[7][e]};
            } else if constexpr (T == 4)
                *reinterpret_cast<f32x4_t*>(d) = f32x4_t{acc[0][e], acc[1][e], acc[2][e], acc[3][e]};
            else
                *reinterpret_cast<f32x2_t*>(d) = f32x2_t{acc[0][e], acc[1][e]};
        }
    }
    __syncthreads();
    const bool swi = P.epilogue == MOE_EPILOGUE_SWIGLU;
    for (int idx = threadIdx.x; idx < mg * (ST_COLS / 4); idx += 64 * ST_WAVES) {
        const int row = idx / (ST_COLS / 4), c4 = idx % (ST_COLS / 4);
        f32x4_t v = zero;
#pragma unroll
        for (int w = 0; w < ST_WAVES; ++w) v += *reinterpret_cast<const f32x4_t*>(red + ((w * rows4 + row) * ST_COLS + 4 * c4));
        if (swi) {   // 4 columns are (gate, gate, up, up) of 2 output columns
            *reinterpret_cast<uint32_t*>(P.y + (row0 + row) * (int64_t)(P.N >> 1) + ((n0 + 4 * c4) >> 1)) =
                pack_bf16_rne(swiglu(v[0], v[2]), swiglu(v[1], v[3]));
        } else {
            u32x2_t o;
            o[0] = pack_bf16_rne(v[0], v[1]);
            o[1] = pack_bf16_rne(v[2], v[3]);
            *reinterpret_cast<u32x2_t*>(P.y + (row0 + row) * (int64_t)P.N + n0 + 4 * c4) = o;
        }
    }
}

// Columns whose weights (fp4: whose scales, the codes come in whole lines) share 128-byte cache lines.  The strips of
// such a group go to one XCD, one behind the other, so that its L2 fetches a line once: spread over the XCDs in launch
// order every strip fetched the whole lines (int4, 64-column strips, 32 experts of 7168 x 2048: 152 us).
template <int FMT>
constexpr int stream_line_cols(int T) { return FMT == MOE_FMT_INT4 ? 256 : FMT == MOE_FMT_FP4_REF && T < 8 ? 64 : 128; }

// Grid: groups of strips over `ranks` passes (16 rows of an expert), dealt to the XCDs (workgroup b runs on XCD b mod 8).
// Workgroup of rank r takes the r-th pass, the (r + ranks)-th and so on (the host's `ranks` covers them all at once); every
// wavefront finds it by itself, 256 experts per look at group_list (64 per look: 4 dependent reads for G = 256).  The passes of
// an expert run side by side, not one after the other in one workgroup: 192 rows of one expert make 12 of them.
template <int FMT, bool ROUNDW, int T>
__global__ __launch_bounds__(64 * ST_WAVES, T == 8 ? 2 : 4) void stream_kernel(StreamParams P, int ranks) {
    extern __shared__ float red[];
    const int lane = threadIdx.x & 63;
    constexpr int ST_COLS = 16 * T;
    constexpr int LINE = stream_line_cols<FMT>(T), S = LINE / ST_COLS;
    const int slot = blockIdx.x >> 3, group = (slot / S) * 8 + (blockIdx.x & 7), groups_n = P.N / LINE;
    if (group >= ranks * groups_n) return;
    const int n0 = (group % groups_n) * LINE + (slot % S) * ST_COLS;
    // expert and first row of the rank-th pass and the end of that expert's rows; how many passes there are
    int g = 0, r0 = 0, r1 = 0;
    auto find = [&](int rank) {
        constexpr int LOOK = 4;
        int seen = 0;
        for (int g0 = 0; g0 < P.G; g0 += 64 * LOOK) {
            int lo[LOOK], hi[LOOK];
#pragma unroll
            for (int c = 0; c < LOOK; ++c) {
                const int ge = g0 + 64 * c + lane;
                const int64_t first = ge > 0 && ge < P.G ? P.gl[ge - 1] : 0, last = ge < P.G ? P.gl[ge] : 0;
                lo[c] = (int)min(max(first, (int64_t)0), P.M);
                hi[c] = (int)min(max(last, (int64_t)0), P.M);
            }
#pragma unroll
            for (int c = 0; c < LOOK; ++c) {
                unsigned long long live = __ballot(hi[c] > lo[c]);
                int n = __popcll(live), at = 0, pass = 0;
                if (__ballot(hi[c] - lo[c] > ST_ROWS) == 0) {   // a pass each
                    if (rank >= seen && rank < seen + n) {
                        for (int k = rank - seen; k > 0; --k) live &= live - 1;
                        at = __builtin_ctzll(live);
                    }
                } else {
                    const int own = (max(hi[c] - lo[c], 0) + ST_ROWS - 1) / ST_ROWS;
                    int incl = own;
#pragma unroll
                    for (int off = 1; off < 64; off <<= 1) {
                        const int up = __shfl_up(incl, off, 64);
                        if (lane >= off) incl += up;
                    }
                    n = __builtin_amdgcn_readlane(incl, 63);
                    if (rank >= seen && rank < seen + n) {
                        at = __builtin_ctzll(__ballot(incl > rank - seen));
                        pass = rank - seen - __builtin_amdgcn_readlane(incl - own, at);
                    }
                }
                if (rank >= seen && rank < seen + n) {
                    g = g0 + 64 * c + at;
                    r0 = __builtin_amdgcn_readlane(lo[c], at) + pass * ST_ROWS;
                    r1 = __builtin_amdgcn_readlane(hi[c], at);
                }
                seen += n;
            }
        }
        return __builtin_amdgcn_readfirstlane(seen);
    };
    int rank = group / groups_n;
    const int passes = find(rank);
    while (rank < passes) {
        const int mg = min(ST_ROWS, r1 - r0);
        if constexpr (FMT == MOE_FMT_FP4_REF && !ROUNDW) {
            if (mg <= 8) stream_rows<FMT, ROUNDW, T, true>(P, red, g, r0, mg, n0);
            else stream_rows<FMT, ROUNDW, T, false>(P, red, g, r0, mg, n0);
        } else {
            stream_rows<FMT, ROUNDW, T, false>(P, red, g, r0, mg, n0);
        }
        rank += ranks;
        if (rank < passes) {
            __syncthreads();   // the partial sums are read
            find(rank);
        }
    }
}

template <int FMT, bool ROUNDW, int T>
static int launch_stream_kind(const moe_grouped_args* a, hipStream_t stream) {
    constexpr int ST_COLS = 16 * T;
    StreamParams P;
    P.x = static_cast<const uint16_t*>(a->x);
    P.w = static_cast<const uint8_t*>(a->weight);
    P.scale = a->scale;
    P.offset = static_cast<const uint16_t*>(a->offset);
    P.gl = a->group_list;
    P.y = static_cast<uint16_t*>(a->y);
    P.M = a->M; P.K = (int)a->K; P.N = (int)a->N; P.G = (int)a->G; P.scale_rows = (int)a->scale_rows;
    P.epilogue = a->epilogue;
    P.scale_div = scale_row_divider(a->K, a->scale_rows);
    const int rows = (int)min(a->M, (int64_t)ST_ROWS);
    const size_t lds = (size_t)ST_WAVES * ((rows + 3) & ~3) * ST_COLS * sizeof(float);
    static std::atomic<uint64_t> lds_set{0};
    if (const int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(&stream_kernel<FMT, ROUNDW, T>), ST_WAVES * ST_ROWS * ST_COLS * (int)sizeof(float), lds_set))
        return rc;
    // passes of 16 rows, at most: M rows over min(M, G) experts
    const int64_t ranks = (a->M + (ST_ROWS - 1) * min(a->M, a->G)) / ST_ROWS, groups = ranks * (a->N / stream_line_cols<FMT>(T));
    const int64_t grid = (groups + 7) / 8 * 8 * (stream_line_cols<FMT>(T) / ST_COLS);
    hipLaunchKernelGGL((stream_kernel<FMT, ROUNDW, T>), dim3((unsigned)grid), dim3(64 * ST_WAVES), lds, stream, P, (int)ranks);
    return hipGetLastError() == hipSuccess ? MOE_OK : MOE_ERR_LAUNCH;
}

template <int FMT, bool ROUNDW>
static int launch_stream_fmt(const moe_grouped_args* a, GroupedKernel width, hipStream_t stream) {
    switch (width) {
        case GroupedKernel::STRIPS_32: return launch_stream_kind<FMT, ROUNDW, 2>(a, stream);
        case GroupedKernel::STRIPS_64: return launch_stream_kind<FMT, ROUNDW, 4>(a, stream);
        default: return launch_stream_kind<FMT, ROUNDW, 8>(a, stream);
    }
}

int launch_strips(const moe_grouped_args* a, GroupedKernel width, bool gemm_rounding, hipStream_t stream) {
    switch (a->format) {
        case MOE_FMT_FP4_REF:
            return gemm_rounding ? launch_stream_fmt<MOE_FMT_FP4_REF, true>(a, width, stream) : launch_stream_fmt<MOE_FMT_FP4_REF, false>(a, width, stream);
        case MOE_FMT_FP8_REF:
            return gemm_rounding ? launch_stream_fmt<MOE_FMT_FP8_REF, true>(a, width, stream) : launch_stream_fmt<MOE_FMT_FP8_REF, false>(a, width, stream);
        case MOE_FMT_INT4:
            return gemm_rounding ? launch_stream_fmt<MOE_FMT_INT4, true>(a, width, stream) : launch_stream_fmt<MOE_FMT_INT4, false>(a, width, stream);
        case MOE_FMT_INT8: return gemm_rounding ? launch_stream_fmt<MOE_FMT_INT8, true>(a, width, stream) : MOE_ERR_BAD_FORMAT;
        default: return MOE_ERR_BAD_FORMAT;
    }
}

}  // namespace moe
