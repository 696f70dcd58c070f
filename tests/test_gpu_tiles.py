"""GPU parity of tile routines at the sizes where they change: row counts on both sides of each row-block boundary, the
shortest and uneven runs of their rings, against the CPU oracle with the tolerances of helpers.py (what two roundings to
bf16 of sums in different order give)."""
import sys

import numpy as np
import pytest
import torch

import helpers as H
import oracle

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _swiglu(case):
    """[M, N/2] of the fused epilogue on the GPU, and what the oracle's accumulators give."""
    import moe_gfx950 as mg

    dev = H.upload(case)
    M, K, N, G = case["M"], case["K"], case["N"], case["G"]
    y = torch.full((M, N // 2), 0x7FC0, dtype=torch.int16, device="cuda")
    p = lambda t: 0 if t is None else t.data_ptr()
    mg.grouped_gemm(mg.grouped_args(mg.format_from_compute_type(case["fmt"]), p(dev["x"]), p(dev["weight"]), p(dev["scale"]),
                                    p(dev["offset"]), p(dev["group_list"]), p(y), M, K, N, G, case["scale_rows"],
                                    epilogue=mg.EPILOGUE_SWIGLU), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    _, z = oracle.grouped_gemm(oracle.FMT_BY_NAME[case["fmt"]], case["x"], case["weight"], case["scale"], case["offset"],
                               case["group_list"], want_f32=True)
    want = oracle.swiglu_blocked16(z) if case["fmt"] in ("fp4_b32", "fp4_b16", "bf16") else oracle.swiglu_interleaved(z)
    return y.cpu().numpy().view(np.uint16), want


@pytest.mark.parametrize("epilogue", ["none", "swiglu"])
@pytest.mark.parametrize("K", [64, 128, 192, 448])   # 1, 2, 3 and 7 pairs of steps
@pytest.mark.parametrize("tile", [224, 128])
def test_bf16_row_blocks(tile, K, epilogue):
    """gemm_tile_bf16: every number of 32-row blocks from 1 to 7, the row before and after each, two and three chunks; and with
    so few column tiles that an expert's rows are cut into chunks of 128."""
    counts = [rows for b in (32, 64, 96, 128, 160, 192, 224) for rows in (b - 1, b, b + 1)] + [1, 16, 17, 449]
    counts += [0] * (129 - len(counts)) if tile == 224 else [257, 385]
    _say(f"bf16 row blocks K={K} epilogue={epilogue} tiles of {tile} rows")
    case = H.make_case("bf16", len(counts), K, 256, np.cumsum(counts), seed=K, extra_rows=3)
    assert H.kernel_of(case, "gemm", swiglu=epilogue == "swiglu") == {224: "tiles_bf16", 128: "tiles_bf16_128"}[tile]
    used = int(case["group_list"][-1])
    if epilogue == "swiglu":
        got, want = _swiglu(case)
    else:
        got, want = H.run_cabi(case, H.upload(case), "gemm"), H.oracle_out(case)
    H.assert_close(got, want, rows=slice(0, used), what=f"bf16 K={K} {epilogue}")
    assert (got[used:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"


@pytest.mark.parametrize("epilogue", ["none", "swiglu"])
@pytest.mark.parametrize("K", [2048, 4096])
def test_bf16_starts_all_over_k(K, epilogue):
    """With K a multiple of 2048 a column tile starts at a k pair of its own and goes round: one expert per start, from the
    first pair to the last two, tiles of one to three row blocks, experts without rows."""
    pairs = K // 64
    counts = [(33, 7, 0, 64, 1, 70)[g % 6] for g in range(pairs // 2 + 1)]
    _say(f"bf16 starts K={K} epilogue={epilogue}")
    case = H.make_case("bf16", len(counts), K, 256, np.cumsum(counts), seed=K, extra_rows=3)
    assert H.kernel_of(case, "gemm", swiglu=epilogue == "swiglu") == "tiles_bf16_128"
    used = int(case["group_list"][-1])
    if epilogue == "swiglu":
        got, want = _swiglu(case)
    else:
        got, want = H.run_cabi(case, H.upload(case), "gemm"), H.oracle_out(case)
    H.assert_close(got, want, rows=slice(0, used), what=f"bf16 starts K={K} {epilogue}")
    assert (got[used:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"


@pytest.mark.parametrize("K,N", [(192, 256), (160, 256), (128, 257), (128, 1024)])
def test_bf16_gemv_of_many_rows(K, N):
    """Sizes that the tile kernel takes over from the vector kernel, and those (K not a multiple of 64, a ragged N) that it does not."""
    counts = [0, 7, 1, 33, 250, 0, 4]
    case = H.make_case("bf16", len(counts), K, N, np.cumsum(counts), seed=K + N, extra_rows=2)
    _say(f"bf16 gemv of many rows K={K} N={N}")
    got, used = H.run_cabi(case, H.upload(case), "gemv"), sum(counts)
    H.assert_close(got, H.oracle_out(case, gemv=True), rows=slice(0, used), what=f"bf16 gemv K={K} N={N}")
    assert (got[used:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"


@pytest.mark.parametrize("epilogue", ["none", "swiglu"])
@pytest.mark.parametrize("K", [128, 256, 384, 896])   # 1, 2, 3 and 7 super-steps
@pytest.mark.parametrize("fmt", ["fp4_b32", "fp4_b16"])
def test_fp4_k_contiguous_row_blocks(fmt, K, epilogue):
    """gemm_tile_fp4_k: every number of 16-row blocks from 1 to 10, the row before and after each, two and three chunks, over
    two column tiles."""
    counts = [rows for b in range(16, 161, 16) for rows in (b - 1, b, b + 1)] + [1, 0, 321]
    _say(f"{fmt} row blocks K={K} epilogue={epilogue}")
    case = H.make_case(fmt, len(counts), K, 512, np.cumsum(counts), seed=K, extra_rows=3)
    assert H.kernel_of(case, "gemm", swiglu=epilogue == "swiglu") == "tiles_fp4_k"
    used = int(case["group_list"][-1])
    if epilogue == "swiglu":
        got, want = _swiglu(case)
    else:
        got, want = H.run_cabi(case, H.upload(case), "gemm"), H.oracle_out(case)
    H.assert_close(got, want, rows=slice(0, used), what=f"{fmt} K={K} {epilogue}")
    assert (got[used:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"


@pytest.mark.parametrize("epilogue", ["none", "swiglu"])
@pytest.mark.parametrize("K", [2048, 2176, 2432])   # 8, 8.5 and 9.5 super-blocks of scales of fp4_b32; 16, 17 and 19 of fp4_b16
@pytest.mark.parametrize("fmt", ["fp4_b32", "fp4_b16"])
def test_fp4_k_contiguous_pair_row_blocks(fmt, K, epilogue):
    """gemm_tile_pair on the K-contiguous fp4 containers (launches of few tiles): every number of 16-row blocks from 1 to 11, the
    row before and after each, two and three chunks, over two column tiles."""
    counts = [rows for b in range(16, 161, 16) for rows in (b - 1, b, b + 1)] + [1, 0, 321]
    _say(f"{fmt} pair row blocks K={K} epilogue={epilogue}")
    case = H.make_case(fmt, len(counts), K, 512, np.cumsum(counts), seed=K, extra_rows=3)
    assert H.kernel_of(case, "gemm", swiglu=epilogue == "swiglu") == "tiles_pair"
    used = int(case["group_list"][-1])
    if epilogue == "swiglu":
        got, want = _swiglu(case)
    else:
        got, want = H.run_cabi(case, H.upload(case), "gemm"), H.oracle_out(case)
    H.assert_close(got, want, rows=slice(0, used), what=f"{fmt} K={K} {epilogue}")
    assert (got[used:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"


@pytest.mark.parametrize("K,kernel", [(896, "tiles_fp4_k"), (2176, "tiles_pair")])
@pytest.mark.parametrize("fmt", ["fp4_b32", "fp4_b16"])
def test_fp4_k_contiguous_tiles_round_their_weights(fmt, K, kernel):
    """Both tile routines multiply weights rounded to bf16: few outputs differ from the oracle with that rounding (where the order
    of the sums moves one across a rounding boundary), a sizeable share from the oracle without it."""
    _say(f"{fmt} {kernel} rounding")
    case = H.make_case(fmt, 4, K, 512, [40, 90, 130, 200], seed=K)
    assert H.kernel_of(case, "gemm") == kernel
    got = H.run_cabi(case, H.upload(case), "gemm")
    own, other = (float(np.mean(got != H.oracle_out(case, gemv=g))) for g in (False, True))
    assert other > 0.03 and own < 0.25 * other, f"{own:.4f} of the outputs differ from rounded weights, {other:.4f} from un-rounded ones"


@pytest.mark.parametrize("fmt,G,N,kernel", [("int4", 600, 256, "tiles_quad"), ("fp4", 300, 512, "tiles_quad"), ("fp8", 300, 256, "tiles_pair"),
                                            ("int8", 511, 256, "tiles_pair"), ("fp4_b16", 300, 512, "tiles_fp4_k"),
                                            ("fp4_b16", 450, 256, "tiles_fp4_k"), ("bf16", 300, 256, "tiles_bf16")])
def test_order_of_experts(fmt, G, N, kernel):
    """Launches of more tiles than workgroups, too short for an order of their own (see test_long_launches_order_their_experts): more
    experts than a workgroup has threads, every number of 16-row blocks from 1 to 10, experts without rows."""
    some = [rows for b in range(16, 161, 16) for rows in (b - 1, b, b + 1)] + [0, 0, 1, 0, 330]
    counts = [some[(g * 17 + g // 35) % 35] for g in range(G)]
    _say(f"order of experts {fmt} G={G} N={N}")
    case = H.make_case(fmt, G, 128, N, np.cumsum(counts), seed=G, extra_rows=3)
    assert H.kernel_of(case, "gemm") == kernel
    used = int(case["group_list"][-1])
    got = H.run_cabi(case, H.upload(case), "gemm")
    H.assert_close(got, H.oracle_out(case), rows=slice(0, used), what=f"order of experts {fmt} G={G}")
    assert (got[used:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"


@pytest.mark.parametrize("K", [256, 384, 640, 768, 896, 1152, 1664, 3712, 7296])
@pytest.mark.parametrize("fmt", ["fp4_b32", "fp4_b16"])
def test_fp4_rows_of_a_partly_filled_last_step(fmt, K):
    """gemv_fp4_mfma_kernel where K is no multiple of 512: one to three groups of 128 k in the last step, the shortest K, chunks of
    x that end with a single group (1664, 3712 and 7296 with 16, 8 and 4 rows staged); both roundings, a ragged N, SwiGLU."""
    counts = [0, 1, 3, 4, 5, 8, 9, 16, 17]
    _say(f"{fmt} partly filled last step K={K}")
    for op, N in (("gemv", 141), ("gemm", 256), ("swiglu", 256)):
        used = sum(counts) if op != "swiglu" else 30
        case = H.make_case(fmt, 9, K, N, np.minimum(np.cumsum(counts), used), seed=K + N, extra_rows=2)
        assert H.kernel_of(case, "gemv" if op == "gemv" else "gemm", swiglu=op == "swiglu") == "fp4_rows"
        if op == "swiglu":
            got, want = _swiglu(case)
        else:
            got, want = H.run_cabi(case, H.upload(case), op), H.oracle_out(case, gemv=op == "gemv")
        H.assert_close(got, want, rows=slice(0, used), what=f"{fmt} {op} K={K}")
        assert (got[used:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"


@pytest.mark.parametrize("K", [3456, 6912])
@pytest.mark.parametrize("fmt", ["fp4_b32", "fp4_b16"])
def test_fp4_vector_kernel_on_single_rows(fmt, K):
    """gemv_kmajor_kernel on fp4 where gemv_fp4_mfma_kernel's last step would be partly filled: the last of its own steps and, beyond
    4096 k, the last chunk of x partly filled; experts with one and with five rows, a ragged N."""
    counts = [0, 1, 0, 0, 5, 0, 0, 1] + [0] * 24 + [1]
    _say(f"{fmt} vector kernel K={K}")
    case = H.make_case(fmt, len(counts), K, 1205, np.cumsum(counts), seed=K)
    assert H.kernel_of(case, "gemv") == "vector"
    H.assert_close(H.run_cabi(case, H.upload(case), "gemv"), H.oracle_out(case, gemv=True), what=f"{fmt} vector K={K}")


@pytest.mark.parametrize("fmt,G,K,N,kernel", [("int4", 600, 1024, 256, "tiles_quad"), ("fp4", 300, 1024, 512, "tiles_quad"),
                                              ("fp4_b32", 300, 1024, 512, "tiles_fp4_k"), ("fp4_b16", 300, 1024, 512, "tiles_fp4_k"),
                                              ("fp4_b16", 450, 1024, 256, "tiles_fp4_k"), ("int8", 511, 4096, 256, "tiles_pair"),
                                              ("fp8", 1100, 2048, 256, "tiles_pair")])
def test_long_launches_order_their_experts(fmt, G, K, N, kernel):
    """Launches of at least 1 << 19 tiles times k (tiles_pair: 3 << 20) take the experts with the largest tiles first: more experts than a
    workgroup has threads (two and three rounds of the sort, the last one partly filled), every number of 16-row blocks from 1 to 10,
    experts without rows; 450 fp4_b16 experts, for whose order LDS has no room.  No output depends on the order: the same bits as two
    launches of half of the experts each, which are too short for one."""
    import moe_gfx950 as mg

    limit = 3 << 20 if kernel == "tiles_pair" else 1 << 19
    some = [rows for b in range(16, 161, 16) for rows in (b - 1, b, b + 1)] + [0, 0, 1, 0, 330]
    counts = [some[(g * 17 + g // 35) % 35] for g in range(G)]
    _say(f"long launch {fmt} G={G} N={N}")
    gen = torch.Generator(device="cuda").manual_seed(G)
    weight = torch.randint(0, 64 if fmt == "fp8" else 256, (G, K * N // (1 if fmt in ("int8", "fp8") else 2)), dtype=torch.uint8, device="cuda", generator=gen)
    scales = {"int4": K // 128 * N, "fp4": K // 16 * N, "fp4_b32": K // 32 * N, "fp4_b16": K // 16 * N, "int8": N, "fp8": (K // 128) * (N // 128)}[fmt]
    scale = torch.rand(G, scales, device="cuda", generator=gen).mul_(0.05).to(torch.float32 if fmt == "fp8" else torch.bfloat16)
    offset = torch.randn(G, N, device="cuda", generator=gen).to(torch.bfloat16) if fmt == "int8" else None
    x = torch.randn(sum(counts), K, device="cuda", generator=gen).to(torch.bfloat16)

    def launch(g0, g1):
        """Experts [g0, g1) on their rows; tiles (at most) times k."""
        first, rows = sum(counts[:g0]), sum(counts[g0:g1])
        gl = torch.tensor(np.cumsum(counts[g0:g1]), device="cuda")
        y = torch.full((rows, N), 0x7FC0, dtype=torch.int16, device="cuda")
        args = mg.grouped_args(mg.format_from_compute_type(fmt), x[first:].data_ptr(), weight[g0:].data_ptr(), scale[g0:].data_ptr(),
                               0 if offset is None else offset[g0:].data_ptr(), gl.data_ptr(), y.data_ptr(), rows, K, N, g1 - g0,
                               {"int4": K // 128, "fp4": K // 16}.get(fmt, 1))
        assert mg.grouped_kernel(args, "gemm") == kernel
        mg.grouped_gemm(args, torch.cuda.current_stream().cuda_stream)
        return y, (rows // (144 if kernel == "tiles_fp4_k" else 160) + g1 - g0) * (N // 256) * K

    whole, work = launch(0, G)
    halves, works = zip(launch(0, G // 2), launch(G // 2, G))
    torch.cuda.synchronize()
    assert max(works) < limit <= work
    assert torch.equal(whole, torch.cat(halves)) and not bool((whole == 0x7FC0).any())


@pytest.mark.parametrize("K", [128, 256, 384, 512, 640, 896])   # 4, 8, 12, 16, 20 and 28 steps of 32 k
@pytest.mark.parametrize("fmt", ["int4", "fp4"])
def test_small_tiles_in_the_longer_ring(fmt, K):
    """GK_QUAD gives tiles of up to 48 rows six stages where a workgroup gets more than one tile: every row count up to two beyond."""
    counts = list(range(1, 51)) + [0, 48, 33, 16] + [17] * 12
    N = 2048
    _say(f"small tiles in the longer ring {fmt} K={K}")
    case = H.make_case(fmt, len(counts), K, N, np.cumsum(counts), seed=K, extra_rows=3)
    assert H.kernel_of(case, "gemm") == "tiles_quad"
    assert sum(c > 0 for c in counts) * (N // 256) > 512, "more tiles than workgroups"
    used = int(case["group_list"][-1])
    got = H.run_cabi(case, H.upload(case), "gemm")
    H.assert_close(got, H.oracle_out(case), rows=slice(0, used), what=f"{fmt} K={K}")
    assert (got[used:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"


# op, container, experts, K, N, kernel; the weights of all experts are 96 MiB or just under
NONTEMPORAL = [("gemm", "fp8", 48, 1024, 2048, "tiles_pair"), ("gemm", "int8", 48, 1024, 2048, "tiles_pair"), ("gemm", "int4", 96, 1024, 2048, "tiles_pair_small"),
               ("gemm", "fp4", 96, 1024, 2048, "tiles_pair_small"), ("gemv", "fp8", 48, 1024, 2048, "tiles_pair_exact"),
               ("gemv", "int4", 96, 1024, 2048, "tiles_pair_exact"), ("gemv", "fp4", 96, 1024, 2048, "tiles_pair_exact"),
               ("gemv", "fp4", 96, 1024, 2048, "tiles_pair_exact16")]


@pytest.mark.parametrize("spare", [0, 1])
@pytest.mark.parametrize("op,fmt,G,K,N,kernel", NONTEMPORAL)
def test_nontemporal_weights(op, fmt, G, K, N, kernel, spare):
    """Launches that read 96 MiB of weights load those of experts of one small tile nontemporally, smaller ones (here by an expert) do not: the
    row counts around each tile size, experts of several chunks."""
    _say(f"nontemporal weights {op} {fmt} {kernel} spare={spare}")
    counts = ([1, 8, 9, 15, 16, 17, 0, 31, 32, 33] if op == "gemv" or fmt in ("int4", "fp4") else [1, 16, 17, 33, 63, 64, 65, 161, 0, 80]) * G
    counts = counts[:G - spare]
    if kernel in ("tiles_pair_small", "tiles_pair_exact16"):   # 12 rows per expert at most, on average
        counts = [c if g % 3 else min(c, 1) for g, c in enumerate(counts)]
    case = H.make_case(fmt, len(counts), K, N, np.cumsum(counts), seed=G + spare, extra_rows=3)
    assert H.kernel_of(case, op) == kernel
    assert H.nontemporal_rows(case, op) == (0 if spare else 64 if kernel == "tiles_pair" else 16)
    used = int(case["group_list"][-1])
    got = H.run_cabi(case, H.upload(case), op)
    H.assert_close(got, H.oracle_out(case, gemv=op == "gemv"), rows=slice(0, used), what=f"{op} {fmt}")
    assert (got[used:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"


@pytest.mark.parametrize("epilogue", ["none", "swiglu"])
@pytest.mark.parametrize("fmt", ["int4", "fp4"])
@pytest.mark.parametrize("G,K,N,rows,kernel", [(8, 1600, 4096, 48, "tiles_pair_small"), (8, 1600, 4096, 49, "tiles_quad"), (8, 960, 4096, 40, "tiles_pair_small"),
                                               (8, 960, 4096, 48, "tiles_quad"), (12, 1600, 4096, 24, "tiles_pair_small"), (16, 1600, 4096, 24, "tiles_quad"),
                                               (8, 3136, 8192, 24, "tiles_pair_small"), (8, 3136, 8192, 25, "tiles_quad"), (17, 320, 4096, 13, "tiles_quad"),
                                               (8, 448, 4096, 13, "tiles_quad"), (1, 1600, 256, 48, "tiles_pair_small")])
def test_small_tiles_of_few_tile_launches(G, K, N, rows, kernel, fmt, epilogue):
    """The bounds by rows per expert, tiles and K between the small-stage and the prefill kind, unevenly owned: experts of many chunks."""
    counts = [rows] * G
    if G > 2:
        counts[0], counts[1] = 0, 2 * rows
    _say(f"{fmt} {kernel} {rows} rows on {G} experts {epilogue}")
    case = H.make_case(fmt, G, K, N, np.cumsum(counts), seed=rows, group=32)
    assert H.kernel_of(case, "gemm", swiglu=epilogue == "swiglu") == kernel
    if epilogue == "swiglu":
        got, want = _swiglu(case)
    else:
        got, want = H.run_cabi(case, H.upload(case), "gemm"), H.oracle_out(case)
    H.assert_close(got, want, what=f"{fmt} {kernel} {epilogue}")
