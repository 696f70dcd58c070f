"""GPU parity of the kernel for launches of few rows and columns (moe_stream.hip) in each of its strip widths: row counts on both
sides of its fragment halves and passes, a K shorter and longer than its wavefronts' pipelines, experts without rows in
front, between and behind, an epilogue, against the CPU oracle with the tolerances of helpers.py."""
import numpy as np
import pytest
import torch

import helpers as H
from test_gpu_tiles import _say, _swiglu

pytestmark = pytest.mark.gpu

COUNTS = [0, 1, 4, 5, 8, 9, 16, 17, 0]          # 9 experts: 9 N columns
WIDTHS = {32: 512, 64: 1536, 128: 2560}         # strip width -> N


@pytest.mark.parametrize("K", [128, 1152])       # 4 and 36 steps of 32 k for 8 wavefronts
@pytest.mark.parametrize("width", sorted(WIDTHS))
@pytest.mark.parametrize("fmt", ["fp4", "fp8", "int4", "int8"])
def test_strips(fmt, width, K):
    N = WIDTHS[width]
    case = H.make_case(fmt, len(COUNTS), K, N, np.cumsum(COUNTS), seed=K + width, extra_rows=2)
    used = int(case["group_list"][-1])
    for op in ("gemm",) if fmt == "int8" else ("gemm", "gemv"):
        assert H.kernel_of(case, op) == f"strips_{width}"
        _say(f"strips {op} {fmt} width={width} K={K}")
        got = H.run_cabi(case, H.upload(case), op)
        H.assert_close(got, H.oracle_out(case, gemv=op == "gemv"), rows=slice(0, used), what=f"{op} {fmt} width={width} K={K}")
        assert (got[used:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"
    _say(f"strips swiglu {fmt} width={width} K={K}")
    got, want = _swiglu(case)
    H.assert_close(got, want, rows=slice(0, used), what=f"swiglu {fmt} width={width} K={K}")


@pytest.mark.parametrize("group", [32, 64, 256])
def test_int4_scale_groups(group):
    case = H.make_case("int4", 4, 256, 256, np.cumsum([3, 0, 1, 2]), seed=group, group=group)
    for op in ("gemm", "gemv"):
        _say(f"strips int4 group={group} {op}")
        H.assert_close(H.run_cabi(case, H.upload(case), op), H.oracle_out(case, gemv=op == "gemv"), what=f"{op} group={group}")


@pytest.mark.parametrize("G,owners", [(300, (0, 63, 64, 255, 256, 299)), (1024, (1, 511, 512, 1023))])
def test_finds_the_experts_that_own_rows(G, owners):
    counts = np.zeros(G, dtype=np.int64)
    counts[list(owners)] = 2
    case = H.make_case("fp4", G, 64, 256, np.cumsum(counts), seed=G)
    _say(f"strips experts G={G}")
    H.assert_close(H.run_cabi(case, H.upload(case), "gemv"), H.oracle_out(case, gemv=True), what=f"G={G}")
    torch.cuda.synchronize()


@pytest.mark.parametrize("fmt", ["fp4", "int4"])
def test_passes_of_unevenly_owned_rows(fmt):
    """Experts of many passes between experts of one and of none, on both sides of a wavefront's 64 experts."""
    counts = np.zeros(300, dtype=np.int64)
    counts[[0, 2, 3, 63, 64, 256, 299]] = [33, 1, 16, 17, 38, 1, 20]
    case = H.make_case(fmt, len(counts), 256, 256, np.cumsum(counts), seed=5, extra_rows=1)
    used = int(case["group_list"][-1])
    assert H.kernel_of(case, "gemm") == H.kernel_of(case, "gemv") == "strips_128"
    for op in ("gemm", "gemv"):
        _say(f"strips passes {fmt} {op}")
        got = H.run_cabi(case, H.upload(case), op)
        H.assert_close(got, H.oracle_out(case, gemv=op == "gemv"), rows=slice(0, used), what=f"{op} {fmt}")
        assert (got[used:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"
