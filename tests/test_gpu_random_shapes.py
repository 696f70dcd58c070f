"""Seeded random sweep of shapes, group lists and batch sizes through both grouped ops and every
weight format, against the oracle: decode batches (at most 4 rows per expert on average), batches around the 16-row block
size, and prefill, with empty experts and single rows.  With up to 7 experts and 768 columns the first two are strips on the
N-contiguous containers; test_random_decode_tiles draws sizes beyond those."""
import sys
import zlib

import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu

K_STEP = {"fp4": 64, "fp8": 128, "int8": 64, "int4": 128, "fp4_b32": 128, "bf16": 64, "fp4_b16": 128}


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _random_counts(rng, G, regime):
    if regime == "decode":        # M <= 4 G
        c = rng.integers(0, 5, G)
    elif regime == "mid":         # around the 16-row block size: both sides of the GEMV / GEMM kernel dispatch bound (12 G)
        c = rng.choice([0, 1, 5, 8, 15, 16, 17, 19], G)
    elif regime == "small_tile":  # 20 G < M <= 24 G: two row blocks of 16 (the last strips of few columns; bf16: one block of 32)
        c = np.full(G, 22) + rng.integers(-1, 2, G)
    else:                         # prefill: ragged, up to a few row blocks, some empty experts
        c = rng.choice([0, 3, 31, 33, 64, 100, 161, 200], G)
    if c.sum() == 0:
        c[rng.integers(0, G)] = 1
    return c


@pytest.mark.parametrize("regime", ["decode", "mid", "small_tile", "prefill"])
@pytest.mark.parametrize("fmt", H.FORMATS)
def test_random_gemm(fmt, regime):
    seed = zlib.crc32(f"rand-gemm/{fmt}/{regime}".encode())
    rng = np.random.default_rng(seed)
    for rep in range(2):
        G = int(rng.integers(1, 8))
        K = int(rng.integers(1, 9)) * K_STEP[fmt] * (4 if rep else 1)      # the second draw is a multiple of 512 for the 128-step formats
        N = int(rng.integers(1, 4)) * 256
        counts = _random_counts(rng, G, regime)
        gl = list(np.cumsum(counts))
        _say(f"random gemm fmt={fmt} regime={regime} G={G} K={K} N={N} counts={list(counts)}")
        group = 128 if K % 128 == 0 else 64
        case = H.make_case(fmt, G, K, N, gl, seed=seed % 1000 + rep, extra_rows=int(rng.integers(0, 3)), group=group)
        got = H.run_cabi(case, H.upload(case), "gemm")
        H.assert_close(got, H.oracle_out(case), rows=slice(0, gl[-1]), what=f"{fmt}/{regime}/{rep}")
        assert (got[gl[-1]:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"


@pytest.mark.parametrize("regime", ["decode", "mid"])
@pytest.mark.parametrize("fmt", H.GEMV_FORMATS)
def test_random_gemv(fmt, regime):
    seed = zlib.crc32(f"rand-gemv/{fmt}/{regime}".encode())
    rng = np.random.default_rng(seed)
    k_major = fmt in ("fp4_b32", "bf16", "fp4_b16")
    for rep in range(2):
        G = int(rng.integers(1, 8))
        K = int(rng.integers(1, 9)) * (32 if k_major and rep == 0 else K_STEP[fmt] * (4 if rep else 1))
        N = int(rng.integers(1, 700)) if k_major else int(rng.integers(1, 4)) * 256
        counts = _random_counts(rng, G, regime)
        gl = list(np.cumsum(counts))
        _say(f"random gemv fmt={fmt} regime={regime} G={G} K={K} N={N} counts={list(counts)}")
        group = 128 if K % 128 == 0 else 64
        case = H.make_case(fmt, G, K, N, gl, seed=seed % 1000 + rep, extra_rows=int(rng.integers(0, 3)), group=group)
        got = H.run_cabi(case, H.upload(case), "gemv")
        H.assert_close(got, H.oracle_out(case, gemv=True), rows=slice(0, gl[-1]), what=f"gemv {fmt}/{regime}/{rep}")
        assert (got[gl[-1]:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"


@pytest.mark.parametrize("op", ["gemm", "gemv"])
@pytest.mark.parametrize("fmt", ["fp4", "fp8", "int8", "int4"])
def test_random_decode_tiles(fmt, op):
    """Decode-sized batches of the N-contiguous containers in more columns than strips take."""
    if op == "gemv" and fmt not in H.GEMV_FORMATS:
        pytest.skip("the GEMV op has no such container")
    seed = zlib.crc32(f"rand-tiles/{fmt}/{op}".encode())
    rng = np.random.default_rng(seed)
    for regime in ("decode", "mid"):
        G = int(rng.integers(20, 32))
        K = int(rng.integers(1, 5)) * K_STEP[fmt]
        N = 2048 + 128 * int(rng.integers(0, 3)) if fmt == "fp8" else 2048 + 256 * int(rng.integers(0, 2))
        counts = np.maximum(_random_counts(rng, G, regime), rng.permutation(np.arange(G) < 17))   # 17 rows at least
        gl = list(np.cumsum(counts))
        _say(f"random tiles {op} fmt={fmt} regime={regime} G={G} K={K} N={N} counts={list(counts)}")
        case = H.make_case(fmt, G, K, N, gl, seed=seed % 1000, extra_rows=int(rng.integers(0, 3)), group=128 if K % 128 == 0 else 64)
        assert H.kernel_of(case, op).startswith("tiles")
        got = H.run_cabi(case, H.upload(case), op)
        H.assert_close(got, H.oracle_out(case, gemv=op == "gemv"), rows=slice(0, gl[-1]), what=f"tiles {op} {fmt}/{regime}")
        assert (got[gl[-1]:] == 0x7FC0).all(), "rows beyond group_list[-1] were written"
