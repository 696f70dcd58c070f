"""Which kernel a grouped call gets, on both sides of every rule of the dispatch (host only)."""
import pytest

import helpers as H

N_CONTIG = ("fp4", "fp8", "int8", "int4")


def kernel(fmt, op, M, G, K, N, swiglu=False):
    scale_rows = {"fp4": K // 16, "int4": K // 32}.get(fmt, 1)
    return H.kernel_of(dict(fmt=fmt, M=M, K=K, N=N, G=G, scale_rows=scale_rows), op, swiglu)


@pytest.mark.parametrize("op", ["gemm", "gemv"])
@pytest.mark.parametrize("fmt", N_CONTIG)
def test_strips(fmt, op):
    if op == "gemv" and fmt == "int8":
        pytest.skip("the GEMV op has no such container")
    at = lambda M, G, N: kernel(fmt, op, M, G, 7168, N)   # noqa: E731
    assert at(8, 256, 512) == "strips_32"                              # a token with 8 experts
    assert (at(32, 32, 256), at(33, 33, 256)) == ("strips_32", "strips_64")      # 8192 columns
    assert (at(64, 64, 256), at(65, 65, 256)) == ("strips_64", "strips_128")     # 16384 columns
    assert at(128, 128, 256) == "strips_128" and at(129, 129, 256).startswith("tiles")   # 32768 columns
    assert at(24 * 8, 8, 2048) == "strips_64" and at(24 * 8 + 1, 8, 2048).startswith("tiles")
    assert at(12 * 16, 16, 2048) == "strips_128" and at(12 * 16 + 1, 16, 2048).startswith("tiles")
    assert at(4, 1024, 256) == "strips_32" and at(4, 1025, 256).startswith("tiles")


def test_tiles_of_the_n_contiguous_containers():
    rows = {r: {f: kernel(f, "gemm", r * 64, 64, 7168, 2048) for f in N_CONTIG} for r in (12, 13, 160, 161)}
    assert rows[12] == dict(fp4="tiles_pair_small", int4="tiles_pair_small", fp8="tiles_pair", int8="tiles_pair")
    assert rows[13] == rows[160] == dict(fp4="tiles_quad", int4="tiles_quad", fp8="tiles_pair", int8="tiles_pair")
    assert rows[161] == dict.fromkeys(N_CONTIG, "tiles_quad")
    rows = {r: {f: kernel(f, "gemv", r * 64, 64, 7168, 2048) for f in ("fp4", "int4", "fp8")} for r in (12, 13)}
    assert rows[12] == dict(fp4="tiles_pair_exact16", int4="tiles_pair_exact", fp8="tiles_pair_exact")
    assert rows[13] == dict.fromkeys(("fp4", "int4", "fp8"), "tiles_pair_exact")


@pytest.mark.parametrize("fmt", ["int4", "fp4"])
def test_small_tiles_of_few_tile_launches(fmt):
    """Rows per expert up to which the small-stage kind is taken: no more than are ahead of the prefill kind at that K and number of tiles."""
    def bound(G, N, K):
        names = [kernel(fmt, "gemm", r * G, G, K, N) for r in range(13, 50)]
        assert names == sorted(names) and set(names) <= {"tiles_pair_small", "tiles_quad"}
        return 12 + names.count("tiles_pair_small")

    for G, N in ((8, 4096), (128, 256), (33, 768)):     # up to 128 tiles
        K = {"int4": 1024, "fp4": 1536}[fmt]
        assert [bound(G, N, k) for k in (448, 512, K - 64, K, 7168)] == [12, 40, 40, 48, 48]
    for G, N in ((12, 4096), (129, 256), (64, 768)):    # up to 192
        assert [bound(G, N, K) for K in (448, 512, 1472, 1536, 7168)] == [12, 20, 20, 24, 24]
    K = {"int4": 2560, "fp4": 3072}[fmt]
    for G, N in ((16, 4096), (256, 256), (193, 256)):   # up to 256
        assert [bound(G, N, k) for k in (512, 1024, K - 64, K, 7168)] == [12, 12, 12, 24, 24]
    assert [bound(257, 256, k) for k in (512, 7168)] == [12, 12]
    # fewer rows than experts: 12 per expert at least
    assert kernel(fmt, "gemm", 1000, 2000, 1024, 4096) == "tiles_pair_small"


def test_nontemporal_weights():
    """Experts of one tile (of 4 row blocks on GK_PAIR, of one on the small-stage kinds) where the experts that may own rows have 96 MiB."""
    def rows(fmt, op, M, G, K, N):
        case = dict(fmt=fmt, M=M, K=K, N=N, G=G, scale_rows={"fp4": K // 16, "int4": K // 32}.get(fmt, 1))
        return H.kernel_of(case, op), H.nontemporal_rows(case, op)

    for fmt, op, M, kernel, most in (("fp8", "gemm", 1600, "tiles_pair", 64), ("int8", "gemm", 1600, "tiles_pair", 64), ("int4", "gemm", 600, "tiles_pair_small", 16),
                                     ("fp4", "gemm", 600, "tiles_pair_small", 16), ("fp8", "gemv", 600, "tiles_pair_exact", 16), ("int4", "gemv", 600, "tiles_pair_exact", 16),
                                     ("fp4", "gemv", 1600, "tiles_pair_exact", 16), ("fp4", "gemv", 600, "tiles_pair_exact16", 16),
                                     ("int4", "gemm", 1600, "tiles_quad", 0), ("fp4", "gemm", 1600, "tiles_quad", 0)):
        N = 2048 if fmt in ("fp8", "int8") else 4096   # 1.5 MiB an expert
        assert rows(fmt, op, M, 64, 768, N) == (kernel, most)
        assert rows(fmt, op, M, 64, 704 if fmt != "fp8" else 640, N) == (kernel, 0)
        assert (rows(fmt, op, 64, 256, 768, N)[1], rows(fmt, op, 63, 256, 768, N)[1]) == (rows(fmt, op, 64, 64, 768, N)[1], 0)   # 64 or 63 experts own rows
    assert rows("int8", "gemm", 161 * 64, 64, 7168, 4096) == ("tiles_quad", 0)
    for fmt in ("fp4_b32", "fp4_b16", "bf16"):
        assert rows(fmt, "gemm", 1600, 64, 7168, 4096)[1] == 0


@pytest.mark.parametrize("fmt", ["fp4_b32", "fp4_b16"])
def test_k_contiguous_fp4(fmt):
    at = lambda op, r, K, swiglu=False: kernel(fmt, op, r * 64, 64, K, 2048, swiglu)   # noqa: E731
    assert (at("gemv", 1, 7168), at("gemv", 100, 7168), at("gemv", 1, 7168 + 32)) == ("fp4_rows", "fp4_rows", "vector")
    assert (at("gemm", 9, 7168), at("gemm", 10, 7168), at("gemm", 5, 7168 + 128)) == ("fp4_rows", "tiles_fp4_k", "tiles_fp4_k")
    # up to 65536 columns, 12 rows per expert
    wide = lambda r, G, N: kernel(fmt, "gemm", r * G, G, 7168, N)   # noqa: E731
    assert (wide(12, 32, 2048), wide(13, 32, 2048), wide(12, 32, 2304), wide(9, 32, 2304)) == ("fp4_rows", "tiles_pair", "tiles_fp4_k", "fp4_rows")
    # with SwiGLU, 5 rows per expert; 8 with up to 64 rows in all
    assert (at("gemm", 5, 7168, True), at("gemm", 6, 7168, True)) == ("fp4_rows", "tiles_fp4_k")
    few = lambda M, G: kernel(fmt, "gemm", M, G, 4096, 2048, True)   # noqa: E731
    assert (few(64, 8), few(65, 8)) == ("fp4_rows", "tiles_pair")
    assert (few(32, 4), few(33, 4)) == ("fp4_rows", "tiles_pair")


@pytest.mark.parametrize("K", [640, 1152, 3328, 6912, 7040])
@pytest.mark.parametrize("fmt", ["fp4_b32", "fp4_b16"])
def test_k_contiguous_fp4_gemm_of_a_partly_filled_last_step(fmt, K):
    rows = lambda M, G, N, swiglu=False: kernel(fmt, "gemm", M, G, K, N, swiglu) == "fp4_rows"   # noqa: E731
    # rows per expert by the columns over all experts that own rows
    for G, N, bound in ((16, 2048, 12), (16, 2304, 4), (32, 2048, 4), (32, 2304, 3), (256, 3584, 3)):
        assert (rows(bound * G, G, N), rows(bound * G + 1, G, N)) == (True, False)
    # fewer rows than experts
    assert (rows(16, 256, 2048), rows(16, 256, 2304), rows(255, 256, 512)) == (True, K >= 4096, K >= 4096)
    # with SwiGLU not more than elsewhere: 5, or 8 with up to 64 rows in all
    assert (rows(5 * 16, 16, 2048, True), rows(5 * 16 + 1, 16, 2048, True)) == (True, False)
    assert (rows(64, 8, 2048, True), rows(65, 8, 2048, True)) == (True, False)
    assert (rows(3 * 32, 32, 2304, True), rows(3 * 32 + 1, 32, 2304, True)) == (True, False)


@pytest.mark.parametrize("fmt", ["fp4_b32", "fp4_b16"])
def test_k_contiguous_fp4_gemv_of_a_partly_filled_last_step(fmt):
    vector = lambda M, G, K, N: kernel(fmt, "gemv", M, G, K, N) == "vector"   # noqa: E731
    b32 = fmt == "fp4_b32"
    # well filled steps of the vector kernel
    assert [K for K in range(2176, 8192, 128) if K % 512 and vector(8, 64, K, 2048)] == [
        K for lo, hi in ((3456, 4096), (5248, 6144), (6784, 8192)) for K in range(lo, hi, 128) if K % 512]
    # few rows for the number of experts
    assert (vector(16, 64, 6912, 2048), vector(17, 64, 6912, 1024), vector(1, 1, 6912, 16384), vector(2, 2, 6912, 8192)) == (True, False, True, False)
    # columns
    assert (vector(16, 64, 6912, 512), vector(16, 64, 6912, 513)) == (b32, True)
    assert (vector(16, 64, 6912, 2048), vector(16, 64, 6912, 2049)) == (True, False)


def test_k_contiguous_fp4_shortest_k():
    # the shortest K of the rows kernel is two groups of 128
    for fmt in ("fp4_b32", "fp4_b16"):
        assert (kernel(fmt, "gemm", 8, 8, 128, 512), kernel(fmt, "gemm", 8, 8, 256, 512)) == ("tiles_fp4_k", "fp4_rows")
        assert (kernel(fmt, "gemv", 8, 8, 128, 512), kernel(fmt, "gemv", 8, 8, 256, 512)) == ("vector", "fp4_rows")


@pytest.mark.parametrize("fmt", ["fp4_b32", "fp4_b16"])
def test_k_contiguous_fp4_tiles(fmt):
    tiles = lambda r, G, K, N: kernel(fmt, "gemm", r * G, G, K, N)   # noqa: E731
    k_min = {"fp4_b32": 1024, "fp4_b16": 2048}[fmt]
    # a tile per CU: 256 tiles, and from some length of K on
    for r in (13, 144, 161, 288):
        chunks = -(-r // 160)
        assert (tiles(r, 16 // chunks, 7168, 4096), tiles(r, 16 // chunks, 7168, 4352)) == ("tiles_pair", "tiles_fp4_k")
        assert (tiles(r, 8, k_min, 1024), tiles(r, 8, k_min - 128, 1024)) == ("tiles_pair", "tiles_fp4_k")
    # fp4_b16, few rows, K an odd multiple of 128
    assert (tiles(16, 8, 7168 - 128, 1024), tiles(17, 8, 7168 - 128, 1024), tiles(16, 8, 7168 - 256, 1024)) == (
        "tiles_pair" if fmt == "fp4_b32" else "tiles_fp4_k", "tiles_pair", "tiles_pair")
    # 145 to 160 rows per expert: in two while that does not fill the CUs, beyond, in one on fp4_b32 with a long K
    assert (tiles(145, 8, 7168, 4096), tiles(160, 8, 7168, 4096)) == ("tiles_fp4_k", "tiles_fp4_k")
    large = "tiles_pair" if fmt == "fp4_b32" else "tiles_fp4_k"
    assert (tiles(145, 16, 4096, 4096), tiles(160, 64, 4096, 4096), tiles(160, 64, 4096 - 128, 4096)) == (large, large, "tiles_fp4_k")
    assert (tiles(144, 64, 4096, 4096), tiles(161, 64, 4096, 4096), tiles(320, 64, 4096, 4096)) == ("tiles_fp4_k",) * 3


def test_bf16():
    at = lambda op, M, G, N, K=7168: kernel("bf16", op, M, G, K, N)   # noqa: E731
    for op in ("gemm", "gemv"):
        assert (at(op, 2 * 64, 64, 2048), at(op, 2 * 64 + 1, 64, 2048)) == ("vector", "tiles_bf16")
    assert (at("gemm", 4 * 8, 8, 4096), at("gemm", 4 * 8 + 1, 8, 4096)) == ("vector", "tiles_bf16_128")
    assert (at("gemv", 6 * 8, 8, 512), at("gemv", 6 * 8 + 1, 8, 512)) == ("vector", "tiles_bf16_128")
    # up to 128 tiles of 224 rows
    for op in ("gemm", "gemv"):
        assert (at(op, 224 * 64, 64, 512), at(op, 224 * 64 + 1, 64, 512)) == ("tiles_bf16_128", "tiles_bf16")
        assert (at(op, 1000, 64, 512), at(op, 1000, 64, 768), at(op, 1000, 129, 256)) == ("tiles_bf16_128", "tiles_bf16", "tiles_bf16")
    # with SwiGLU
    swi = lambda M, G, N, K: kernel("bf16", "gemm", M, G, K, N, True)   # noqa: E731
    for K in (1024, 2048, 4096):
        assert (swi(256, 256, 2048, K), swi(257, 256, 2048, K)) == ("vector", "tiles_bf16")
    for K in (2112, 3072, 6144, 7168):
        assert (swi(512, 256, 2048, K), swi(513, 256, 2048, K)) == ("vector", "tiles_bf16")
    # up to 32 rows in all
    assert (swi(32, 8, 2048, 2048), swi(32, 8, 2304, 2048), swi(32, 8, 2048, 1984)) == ("vector", "tiles_bf16_128", "tiles_bf16_128")
    assert (swi(32, 8, 4096, 6144), swi(32, 8, 4352, 6144), swi(32, 8, 4096, 6080)) == ("vector", "tiles_bf16", "tiles_bf16_128")
    assert (swi(28, 7, 2048, 4096), swi(29, 7, 2048, 4096), swi(33, 9, 1024, 4096)) == ("vector", "tiles_bf16_128", "tiles_bf16_128")
    # sizes that the tiles do not take
    assert at("gemv", 1000, 8, 2049) == at("gemv", 1000, 8, 2048, K=7168 + 32) == "vector"


def test_not_a_valid_call():
    with pytest.raises(ValueError):
        kernel("int8", "gemv", 4, 4, 256, 256)
    with pytest.raises(ValueError):
        kernel("bf16", "gemm", 4, 4, 256, 100)
