// Host-side declarations shared by the launchers and the C ABI.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>

#include "moe_gfx950.h"

namespace moe {
// Raises a kernel's dynamic LDS limit once per GPU (the attribute belongs to the kernel's image on the
// current device).  `done` is that kernel's bit mask of devices already set up: the only state the
// launchers keep.  A race repeats the same call.
inline int ensure_dynamic_lds(const void* kernel, int bytes, std::atomic<uint64_t>& done) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return MOE_ERR_NO_DEVICE;
    if (!((done.load(std::memory_order_acquire) >> dev) & 1u)) {
        if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return MOE_ERR_LAUNCH;
        done.fetch_or(uint64_t{1} << dev, std::memory_order_release);
    }
    return MOE_OK;
}

int launch_dequant_fp4_bf16(const moe_dequant_args* a, hipStream_t stream);
// The kernels of the two grouped ops.  TILES_PAIR_EXACT and TILES_PAIR_EXACT16 have the GEMV op's arithmetic (weights not
// rounded to bf16), the other TILES that of the GEMM op; STRIPS and FP4_ROWS come with either.
enum class GroupedKernel {
    VECTOR,               // K-contiguous containers without matrix cores (moe_gemv.hip)
    FP4_ROWS,             // K-contiguous fp4, 16 rows of an expert per pass (moe_gemv.hip)
    STRIPS_32, STRIPS_64, STRIPS_128,   // N-contiguous containers in strips of that many columns (moe_stream.hip)
    TILES_PAIR, TILES_PAIR_EXACT, TILES_PAIR_SMALL, TILES_PAIR_EXACT16, TILES_QUAD, TILES_FP4_K,   // kinds of moe_gemm.hip
    TILES_BF16, TILES_BF16_128   // tiles of up to BF16_ROWS, of up to 128 rows
};
constexpr int FP4_ROWS_K = 128, FP4_ROWS_K_MIN = 256;   // K of an FP4_ROWS call is a multiple and not less
constexpr int PAIR_ROWS = 160;    // rows of the largest tile of TILES_PAIR and TILES_QUAD
constexpr int FP4_K_ROWS = 144;   // of TILES_FP4_K
constexpr int BF16_ROWS = 224;    // rows of the largest bf16 tile
// the kernel of a valid call, by its sizes, format and epilogue (moe_dispatch.cpp)
GroupedKernel grouped_kernel(const moe_grouped_args* a, bool gemv_op);
const char* grouped_kernel_name(GroupedKernel k);
int launch_grouped(const moe_grouped_args* a, bool gemv_op, hipStream_t stream);
int launch_vector(const moe_grouped_args* a, hipStream_t stream);
// gemm_rounding: the arithmetic of the GEMM op
int launch_fp4_rows(const moe_grouped_args* a, bool gemm_rounding, hipStream_t stream);
int launch_strips(const moe_grouped_args* a, GroupedKernel width, bool gemm_rounding, hipStream_t stream);
int launch_tiles(const moe_grouped_args* a, GroupedKernel kind, hipStream_t stream);
// rows of the largest experts whose weights launch_tiles loads nontemporally, 0: of none
int nontemporal_rows(const moe_grouped_args* a, GroupedKernel kind);
// moves the grouped GEMM's launch number (which picks a launch's tile counter and stamp) by delta; returns the new number
int64_t gemm_shift_launch_number(int64_t delta);
int launch_prepack_fp4_ref(const moe_prepack_fp4_args* a, hipStream_t stream);
int launch_route(const moe_route_args* a, hipStream_t stream);
// the same with the workspace in the library's own static device array (a->workspace is ignored)
int launch_route_static(const moe_route_args* a, hipStream_t stream);
size_t route_workspace_bytes(const moe_route_args* a);
}  // namespace moe
