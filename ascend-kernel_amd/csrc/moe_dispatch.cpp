// Which kernel a grouped call gets, from its sizes alone (group_list stays on the device).  Every rule with what it was
// measured on; the launchers and the tests ask grouped_kernel.
#include <algorithm>

#include "moe_internal.h"

namespace moe {

// Columns the launch streams, at most: min(M, G) experts own rows
static int64_t columns(const moe_grouped_args* a) { return std::min(a->M, a->G) * a->N; }

// bf16 [N, K].  The vector kernel takes 4 rows of an expert per pass over its weights, the tile kernel up to 224, but only a
// workgroup per 256 columns (the two compute the same).  4 rows per expert, vector / tiles:
// 64 experts of 7168 x 2048 (512 tiles) 402 / 303 us, 16 of 7168 x 4096 (256) 208 / 162, 64 of 2048 x 1024 (256)
// 88 / 65, but 8 of 7168 x 4096 (128) 106 / 129, 8 of 7168 x 512 (16) 50 / 80; 2 rows, 512 tiles: 264 / 262.
// With the SwiGLU epilogue the line lies lower: an expert's passes are one chain in its workgroups, which is what unevenly
// routed rows wait for.  Vector / tiles in us at a routing skew (standard deviation of a per-expert bias of the logits) of 0.25
// and of 1, by rows per expert on average.  2 rows: 64 experts of 7168 x 2048 267 / 300 and 247 / 271, 64 of 2560 x 2048
// 108 / 128 and 112 / 112, 128 of 3072 x 1536 176 / 199 and 159 / 131; but with short rows of K, 128 of 1536 x 1536 116 / 108 and
// 108 / 65, 256 of 2048 x 2048 344 / 318 and 294 / 179, and at K = 4096, where the tiles start all over K, 128 of 4096 x 1536
// 268 / 245 and 221 / 164.  1 row: 256 of 2048 x 2048 216 / 233 and 158 / 138.  Up to 32 rows in all, few passes however
// they are routed, in few columns, 4 rows: 8 of 2048 x 2048 26 / 29 and 31 / 29, 8 of 7168 x 4096 111 / 130 and 125 / 130,
// but 8 of 3584 x 4096 63 / 47 and 71 / 47.
static bool bf16_vector_preferred(const moe_grouped_args* a) {
    if (a->epilogue != MOE_EPILOGUE_SWIGLU) return a->M <= (columns(a) >= 65536 ? 2 : 4) * a->G;
    if (a->M <= 32 && a->K >= 2048 && columns(a) <= (a->K >= 6144 ? 32768 : 16384)) return a->M <= 4 * a->G;
    return a->M <= (a->K <= 2048 || a->K == 4096 ? 1 : 2) * a->G;
}

// Tiles of at most 128 rows where tiles of 224, evenly filled, would be no more than half as many as the 256 CUs: an expert's
// rows then go to two CUs or more, whose workgroups share a weight slice in L2.  us, 176-row tiles of an earlier kernel / 224 / 128:
// 64 experts of 4096 x 512, 160 rows each (128 tiles) 115 / 117 / 88, unevenly routed (skew 0.5, see above) 114 / 120 / 99; 16 of
// 4096 x 2048, 160 rows 98 / 101 / 76, unevenly 97 / 100 / 97; 8 of 7168 x 2048, 160 rows 133 / 121 / 96; 8 of 4096 x 1024,
// 256 rows (64 tiles) 75 / 66 / 54; 75 rows, one tile either way, 116 / 89 / 91.  96 rows are as good with even routing, but unevenly
// routed they make a few tiles more than there are CUs (64 of 4096 x 512: 134 us); 64 rows lose (143).
static GroupedKernel bf16_tiles(const moe_grouped_args* a) {
    const int64_t experts = std::max(std::min(a->M, a->G), (int64_t)1), chunks = (a->M + BF16_ROWS * experts - 1) / (BF16_ROWS * experts);
    return 2 * experts * chunks * ((a->N + 255) / 256) <= 256 ? GroupedKernel::TILES_BF16_128 : GroupedKernel::TILES_BF16;
}

static GroupedKernel bf16_kernel(const moe_grouped_args* a, bool gemv_op) {
    if (bf16_vector_preferred(a)) return GroupedKernel::VECTOR;
    if (!gemv_op) return bf16_tiles(a);
    // The GEMV op takes sizes that the tiles do not, and with few columns the vector kernel stays ahead a little longer.
    // 64 experts of 7168 x 2048: 16 rows per expert 1225 -> 331 us on the tiles, 64 rows 4668 -> 405.  Few
    // columns: 6 rows per expert 77 / 81 us on 8 experts of 7168 x 512, 8 rows 93 / 81; 6 rows on 8 of 4096 x 2048 79 / 71.
    const bool fits = a->K % 64 == 0 && a->N % 256 == 0;
    return fits && (a->N * a->G >= 16384 || a->M > 6 * a->G) ? bf16_tiles(a) : GroupedKernel::VECTOR;
}

// fp4 [N, K/2].  The matrix-core GEMV kernel reads every weight row as contiguous runs, takes 16 rows of an expert per pass and
// has a variant with the GEMM's weight rounding.  An expert of more than 16 rows is passes in a row, so that the bound for the GEMM op,
// where tiles overtake it with balanced top-k routing, depends on the routing.  us, this kernel / tiles, fp4_b32, evenly routed,
// balanced top-k routing, skews of 0.25 and 1 (see bf16): 256 experts of 7168 x 2048, 4 rows per expert 389 / 519, 403 / 515, 386 / 508, 300 /
// 263, 8 rows 434 / 532, 467 / 533, 479 / 531, 590 / 321, 10 rows 470 / 534, 478 / 535, 537 / 539, 646 / 373, 12 rows 479 / 543, 532 / 543, 580
// / 542, 727 / 382; 64 of the same 8 rows 113 / 131, 127 / 131, 136 / 132, 158 / 126, 10 rows 120 / 132, 133 / 133, 145 / 137, 186 / 127.  Up to
// 65536 columns the tiles are one per CU, at best, and take longer: 8 of 4096 x 2048, 12 rows 22 / 37, 23 / 37, 34 / 38, 52 / 40.
// With the SwiGLU epilogue the line lies lower (skews 0.25 and 1): 256 of 2048 x 1024, 4 rows 61 / 78 and 74 / 47, 5 rows 71 / 79 and
// 88 / 48, 8 rows 79 / 81 and 131 / 60 (an expert of 109 rows is 7 passes in a row); 256 of 7168 x 2048, 4 rows 402 / 506 and 292 / 263, 8 rows
// 481 / 527 and 462 / 319.  Up to 64 rows in all, four passes at most: 8 of 4096 x 2048, 8 rows 22 / 37 against 37 / 37.
static bool fp4_rows_preferred(const moe_grouped_args* a) {
    if (a->epilogue != MOE_EPILOGUE_SWIGLU) return a->M <= (columns(a) <= 65536 ? 12 : 9) * a->G;
    return a->M <= (a->M <= 64 ? 8 : 5) * a->G;
}

// The same kernel where K is no multiple of 512 and its last iteration is not full, GEMV op (else the vector kernel).  us, the vector
// kernel / this one, fp4_b32 and fp4_b16: 8 rows, 1 to 8 experts, K = 1152: 8.0 / 5.5 and 8.8 / 6.7; 62 x 4 rows on 64 experts of 4736 x
// 768, skew 1: 196 / 46 and 212 / 59; 32 x 8 on 256 of 1920 x 2000: 131 / 63 and 146 / 83.  With 3 or 4 rows of an expert the vector kernel
// takes 1.4 times as long as with 1 or 2, this one as long.  Single rows, weights from HBM: the vector kernel is level or ahead where its steps
// of 2048 k are well filled against the 512 k of this one (K = 3456 to 4096, 5248 to 6144, 6784 to 8192, ...), and most with enough columns for
// requests to count: 8 rows on 8 of 64 experts, K = 6912, 2048 columns 31 / 39 and 41 / 44, 4096 columns 35 / 43 and 46 / 47, 512
// columns 26 / 25 and 36 / 30, one expert of 512 columns 20 / 24 and 27 / 29; K = 8064, 8193 to 32768 columns in all 0.73 and 0.88 times, K =
// 4736, up to 8192 columns 1.06 and 1.23 times.  So while experts with several rows are rare (4 tokens on 128 experts), and fp4_b16
// beyond 8192 columns only.
static bool fp4_rows_partial_gemv(const moe_grouped_args* a) {
    const int64_t steps = (a->K + 2047) / 2048, groups = (a->K + 511) / 512;
    const bool filled = a->K >= 3456 && 7 * steps <= 2 * groups, single_rows = a->M == 1 || 4 * a->M <= a->G;
    return !(filled && single_rows && columns(a) <= 32768 && (a->format == MOE_FMT_FP4_B32 || columns(a) > 8192));
}

// GEMM op, K no multiple of 512: the tiles take such a K as any other, so that the bounds by rows per expert lie lower, and go by the
// columns: few make a tile per CU at best, whose time hardly depends on its rows; with many, an expert of more than 16 rows is passes in
// a row here.  Tiles / this kernel, balanced top-k routing and skews of 0.25 and 1, median over K = 1152 to 7040 (fp4_b16 differs by
// 0.1): 32768 columns 12 rows per expert 1.2, 1.2 and 0.7; 65536 columns 4 rows 1.37, 1.39 and 1.41, 8 rows 1.32, 1.30 and
// 0.99, 10 rows 1.3, 1.0 and 0.8; 262144 columns 3 rows 1.39, 1.39 and 1.27, 4 rows 1.36, 1.34 and 1.11, 6 rows 1.30, 1.27 and 0.86,
// 12 rows 1.07, 0.99 and 0.52.
// Fewer rows than experts: the workgroups of experts without rows count beside a short K.  6 rows on 256 of 1280 x 7424 16.0 / 15.0, 12
// on 256 of 1280 x 4608 16.8 / 15.5, but 100 on 64 of 4480 x 1024 53 / 38.  (With the transposes that the GEMM op's form of this kernel had
// when the line was drawn: 17.6 / 21.9, 16.9 / 19.6 and 44 / 35.)
static bool fp4_rows_partial_gemm(const moe_grouped_args* a) {
    if (columns(a) <= 32768) return a->M <= 12 * a->G;
    return (a->K >= 4096 || a->M >= a->G) && a->M <= (columns(a) <= 65536 ? 4 : 3) * a->G;
}

// Tiles of K-contiguous fp4.  Two workgroups of 4 wavefronts per CU (TILES_FP4_K) are the better routine where a CU gets two tiles or
// more; a tile alone on its CU has half of the wavefronts there, and the 8-wavefront k-split routine is ahead.  us, TILES_FP4_K /
// TILES_PAIR, evenly routed, fp4_b32 and fp4_b16: 8 experts of 7168 x 2048 (64 tiles), 32 rows each 86 / 72 and 87 / 76, 64 rows 94 / 79
// and 98 / 85; 16 of 7168 x 4096 (256 tiles), 48 rows 1.12 and 1.06 times; 8 of 4480 x 7168, 128 rows 88 / 78 and 90 / 84; one
// expert of 7168 x 512, 128 rows 115 / 90 and 118 / 100; but 16 of 7168 x 4352 (272 tiles), 48 rows 0.88 and 0.88 times, and with 640 k 0.90
// and 0.88 times at 256 tiles (level at 1024 k; fp4_b16 0.94 at 1024, 1.01 at 1536 to 1792, 1.04 at 2048, but 0.90 to 0.94 with more
// than 100 rows at 1664).  Routing that leaves some experts more rows than a tile takes makes a
// few more tiles than CUs: 64 of 7168 x 1024 with 64 rows on average at a skew of 1, 159 / 167 and 162 / 183.  fp4_b16 with up to 16
// rows per expert and K an odd multiple of 128, whose rows of scales do not begin with 32 bytes: 0.92 to 0.96 times.
// TILES_FP4_K cuts an expert of 145 to 160 rows, one tile of TILES_PAIR, in two.  That is the faster way while the tiles do not fill
// the CUs (8 of 2048 x 1024, 152 rows: fp4_b16 35 / 44).  Beyond, it depends on how many experts have just that many.  152 rows on
// average, evenly routed, balanced top-k routing and at a skew of 0.25, TILES_FP4_K / TILES_PAIR: fp4_b32, 64 experts of 7168 x 4096 1.26,
// 0.98 and 0.93 times, 128 of 4096 x 2048 1.20, 1.00 and 0.88, but 128 of 2048 x 2048 1.15, 0.96 and 0.84; fp4_b16 1.17, 0.94 and 0.87
// on the first and 1.07, 0.92 and 0.81 on the last.
static int64_t fp4_tiles(const moe_grouped_args* a, int64_t rows) {
    const int64_t experts = std::max(std::min(a->M, a->G), (int64_t)1);
    return experts * ((a->M + rows * experts - 1) / (rows * experts)) * ((a->N + 255) / 256);
}

static GroupedKernel fp4_kcontiguous_tiles(const moe_grouped_args* a) {
    const bool b32 = a->format == MOE_FMT_FP4_B32;
    const int64_t quad = fp4_tiles(a, FP4_K_ROWS), pair = fp4_tiles(a, PAIR_ROWS);
    const bool pairs = quad == pair ? pair <= 256 && a->K >= (b32 ? 1024 : 2048) && (b32 || a->K % 256 == 0 || a->M > 16 * a->G)
                                    : quad > 256 && a->M <= PAIR_ROWS * a->G && b32 && a->K >= 4096;
    return pairs ? GroupedKernel::TILES_PAIR : GroupedKernel::TILES_FP4_K;
}

static GroupedKernel fp4_kcontiguous_kernel(const moe_grouped_args* a, bool gemv_op) {
    const bool whole = a->K % 512 == 0, partial = a->K >= FP4_ROWS_K_MIN && a->K % FP4_ROWS_K == 0;
    if (gemv_op) return whole || (partial && fp4_rows_partial_gemv(a)) ? GroupedKernel::FP4_ROWS : GroupedKernel::VECTOR;
    const bool rows = fp4_rows_preferred(a) && (whole || (partial && fp4_rows_partial_gemm(a)));
    return rows ? GroupedKernel::FP4_ROWS : fp4_kcontiguous_tiles(a);
}

// Strips for launches of up to 128 tiles of 256 columns, i.e. half of the CUs, and decode-like batches.  us, strips / tiles, 7168 x 2048,
// 1 and 4 rows per expert (skew 0.25): 16 experts (32768 columns) int4 34 / 58 and 36 / 59, fp4 29 / 52 and 31 / 52, fp8 46 / 64 and 48 / 64; 24
// (49152) int4 62 / 58 and 64 / 58, fp4 52 / 52 and 54 / 52, fp8 79 / 67 and 82 / 67; 32 (65536) int4 65 / 59, fp4 57 / 54, fp8 89 / 73.
// With 12 rows an expert of more than 16 is a second pass: 16 experts int4 63 / 61, fp4 53 / 55, fp8 77 / 65.  With up to 16384 columns
// twice as many rows: 192 rows on 8 experts of 4096 x 2048 at a skew of 0.5 int4 29 / 39, fp4 19 / 35, fp8 35 / 42, int8 34 / 43;
// all 192 owned by one expert int4 20 / 38, fp4 18 / 35, fp8 20 / 45, int8 21 / 45.  The passes are found by looking through group_list, 256
// experts at a time.
static bool strips_preferred(const moe_grouped_args* a) {
    return a->G <= 1024 && columns(a) <= 32768 && a->M <= (columns(a) <= 16384 ? 24 : 12) * a->G;
}

// The narrowest strips whose first passes leave every CU at most one workgroup (an expert with more rows than one pass takes
// has a workgroup per pass and strip, so there may be more).  Measured, 8 experts of K = 7168, 32 / 64 / 128 columns
// a strip: N = 512 (4096 columns in all) int4 12 / 16 / 25 us, fp4 10 / 13 / 23, fp8 15 / 16 / 24; N = 2048 (16384) int4 37 / 27 / 31, fp4 18 /
// 17 / 26, fp8 47 / 32 / 36; 16 experts of N = 2048 (32768) int4 68 / 49 / 34, fp4 31 / 30 / 29, fp8 88 / 59 / 46.
static GroupedKernel strip_width(const moe_grouped_args* a) {
    return columns(a) <= 8192 ? GroupedKernel::STRIPS_32 : columns(a) <= 16384 ? GroupedKernel::STRIPS_64 : GroupedKernel::STRIPS_128;
}

// GEMM op on the 4-bit containers: the small-stage kind (tiles of up to 32 rows, 8 wavefronts that split K, two workgroups per CU)
// against the prefill kind (up to 160 rows, 4 wavefronts).  us, prefill / small-stage kind:
//   12 rows per expert and fewer, always: 256 experts of 7168 x 2048, balanced top-k routing, 4 rows int4 428 / 369, fp4 409 / 380, 12 rows
//   455 / 393 and 452 / 410, at a skew of 0.5 (see bf16) 454 / 410 and 423 / 425.  Beyond, it depends on the routing, as an expert of many rows
//   is many passes over its weights: 16 rows, balanced int4 478 / 414, fp4 455 / 444, skew 0.5 473 / 446 and 446 / 450, skew 1 347 / 380 and
//   352 / 391 (12 rows at a skew of 1: 330 / 351 and 337 / 340).
//   Launches in which the prefill kind has a tile per CU at most, evenly routed: its 4 wavefronts are then alone there, and small tiles
//   are more and fill it, until they too are more than the CUs, which a short K does not make up for.  Times as fast, smallest / mean / largest
//   over 8 to 256 experts, K from 512, skews of 0 to 1.  Up to 128 tiles, int4: 32 rows 1.1 / 1.4 / 2.1, 40 rows 1.1 / 1.5 / 2.1, 48 rows 1.0 / 1.5 / 2.0
//   from K = 1024 on, but 0.9 at K = 512; fp4: 32 rows 1.1 / 1.4 / 2.1, 40 rows 1.0 / 1.4 / 2.1, 48 rows 0.96 / 1.4 / 2.0 from K = 1536 on, 0.9 and 0.8 at
//   K = 1024 and 512;
//   64 rows as low as 0.9 up to K = 2048.  129 to 192 tiles: 20 rows 1.0 / 1.3 / 1.9, 24 rows from K = 1536 on 1.15 / 1.4 / 1.95, at K = 1024 as low
//   as 0.9.  Up to 256 tiles, 24 rows: K = 3072 1.0 / 1.2 / 1.6, 7168 1.1 / 1.3 / 1.9; K = 2560 int4 1.0 / 1.2 / 1.5, fp4 as low as 0.92,
//   K = 1024 int4 0.94, fp4 0.85, K = 256 0.8 and 0.75.  K = 256 with fewer tiles: 0.95 to 1.2.
static bool small_tiles_preferred(const moe_grouped_args* a) {
    const int64_t tiles = std::min(a->M, a->G) * ((a->N + 255) / 256);
    const bool int4 = a->format == MOE_FMT_INT4;
    int rows = 12;
    if (a->K >= 512) {
        if (tiles <= 128)
            rows = a->K >= (int4 ? 1024 : 1536) ? 48 : 40;
        else if (tiles <= 192)
            rows = a->K >= 1536 ? 24 : 20;
        else if (tiles <= 256 && a->K >= (int4 ? 2560 : 3072))
            rows = 24;
    }
    return a->M <= rows * a->G;
}

static GroupedKernel n_contiguous_kernel(const moe_grouped_args* a, bool gemv_op) {
    if (strips_preferred(a)) return strip_width(a);
    // GEMV op, fp4: 16-row tiles, two workgroups per CU, in decode-like batches (on average at most 12 rows per expert); an expert with
    // more rows than that costs a pass over its weights per 16 rows.
    if (gemv_op) return a->M <= 12 * a->G && a->format == MOE_FMT_FP4_REF ? GroupedKernel::TILES_PAIR_EXACT16 : GroupedKernel::TILES_PAIR_EXACT;
    const bool four_bit = a->format == MOE_FMT_INT4 || a->format == MOE_FMT_FP4_REF;
    if (four_bit && small_tiles_preferred(a)) return GroupedKernel::TILES_PAIR_SMALL;
    // prefill: workgroups of 4 wavefronts without the k split, two per CU.  The 4-bit
    // ones always (256 experts of 128 rows, K = 7168, N = 4096: int4 1792 against 1905 us, fp4 1724 against 1867 us
    // with the k-split kind).  The one-byte ones, whose tiles move twice the bytes, when an expert has more rows than
    // one tile takes on average, so that its row chunks share a weight slice in L2: 8 experts of 512 rows, K = 4096,
    // N = 14336: int8 454 against 476 us, fp8 480 against 495 us; 64 experts of 512 rows at K = 7168, N = 4096: 1755
    // against 1870 us and 1872 against 1929 us; but with 128 rows per expert, every weight tile read once from HBM,
    // 1090 - 1110 against 1063 - 1098 us (int8) and 1125 - 1152 against 1088 - 1136 us (fp8) on 128 experts
    return four_bit || a->M > PAIR_ROWS * a->G ? GroupedKernel::TILES_QUAD : GroupedKernel::TILES_PAIR;
}

GroupedKernel grouped_kernel(const moe_grouped_args* a, bool gemv_op) {
    switch (a->format) {
        case MOE_FMT_BF16: return bf16_kernel(a, gemv_op);
        case MOE_FMT_FP4_B32:
        case MOE_FMT_FP4_B16: return fp4_kcontiguous_kernel(a, gemv_op);
        default: return n_contiguous_kernel(a, gemv_op);
    }
}

const char* grouped_kernel_name(GroupedKernel k) {
    switch (k) {
        case GroupedKernel::VECTOR: return "vector";
        case GroupedKernel::FP4_ROWS: return "fp4_rows";
        case GroupedKernel::STRIPS_32: return "strips_32";
        case GroupedKernel::STRIPS_64: return "strips_64";
        case GroupedKernel::STRIPS_128: return "strips_128";
        case GroupedKernel::TILES_PAIR: return "tiles_pair";
        case GroupedKernel::TILES_PAIR_EXACT: return "tiles_pair_exact";
        case GroupedKernel::TILES_PAIR_SMALL: return "tiles_pair_small";
        case GroupedKernel::TILES_PAIR_EXACT16: return "tiles_pair_exact16";
        case GroupedKernel::TILES_QUAD: return "tiles_quad";
        case GroupedKernel::TILES_FP4_K: return "tiles_fp4_k";
        case GroupedKernel::TILES_BF16: return "tiles_bf16";
        case GroupedKernel::TILES_BF16_128: return "tiles_bf16_128";
    }
    return nullptr;
}

int launch_grouped(const moe_grouped_args* a, bool gemv_op, hipStream_t stream) {
    const GroupedKernel k = grouped_kernel(a, gemv_op);
    switch (k) {
        case GroupedKernel::VECTOR: return launch_vector(a, stream);
        case GroupedKernel::FP4_ROWS: return launch_fp4_rows(a, !gemv_op, stream);
        case GroupedKernel::STRIPS_32:
        case GroupedKernel::STRIPS_64:
        case GroupedKernel::STRIPS_128: return launch_strips(a, k, !gemv_op, stream);
        default: return launch_tiles(a, k, stream);
    }
}

}  // namespace moe
