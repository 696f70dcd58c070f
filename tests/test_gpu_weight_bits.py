"""The weights that the GEMM op multiplies by, bit for bit: rows of x with a single 1 make y the rounded weights themselves, over
every code and scales of most of the range (int4 and fp8: up to its ends), on every kernel that decodes the container."""
import sys

import numpy as np
import pytest
import torch

import helpers as H
import oracle
from test_gpu_tiles import _swiglu

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _scales(rng, shape, lo, hi):
    """bf16 bits of both signs, magnitudes from 2^lo to 2^hi."""
    e = rng.integers(lo + 127, hi + 127, shape)
    return ((rng.integers(0, 2, shape) << 15) | (e << 7) | rng.integers(0, 128, shape)).astype(np.uint16)


def _unit_rows(case, rng):
    """x of zeros with a 1 per row: every k in turn, in any order."""
    M, K = case["M"], case["K"]
    at = np.resize(rng.permutation(K), M)
    x = np.zeros((M, K), np.uint16)
    x[np.arange(M), at] = 0x3F80
    case["x"] = x
    return at


def _check(case, at, kernel):
    assert H.kernel_of(case, "gemm") == kernel
    got = oracle.bf16_bits_to_f32(H.run_cabi(case, H.upload(case), "gemm"))
    lo = 0
    for g, hi in enumerate(case["group_list"]):
        w = oracle.expand_weight(oracle.FMT_BY_NAME[case["fmt"]], case["weight"], case["scale"], case["offset"], g, True)
        want = w.reshape(case["K"], case["N"])[at[lo:hi]]
        assert np.array_equal(got[lo:hi], want), f"{case['fmt']} {kernel} expert {g}"
        lo = hi


# kernel, experts, K, N, rows per expert
INT4 = [("strips_32", 4, 256, 512, 16), ("strips_64", 6, 256, 2048, 16), ("strips_128", 10, 256, 2048, 12),
        ("tiles_pair_small", 20, 256, 2048, 12), ("tiles_quad", 2, 256, 256, 256), ("tiles_quad", 20, 256, 2048, 145)]


@pytest.mark.parametrize("kernel,G,K,N,rows", INT4)
def test_int4(kernel, G, K, N, rows):
    _say(f"int4 weight bits {kernel}")
    rng = np.random.default_rng(G + N)
    case = H.make_case("int4", G, K, N, np.arange(1, G + 1) * rows, seed=G, group=32)
    case["scale"] = _scales(rng, case["scale"].shape, -110, 117)
    _check(case, _unit_rows(case, rng), kernel)


# ... and the longer ring of tiles_quad (more than 512 tiles, up to 48 rows), nontemporal loads of tiles_pair_small (96 MiB of weights)
INT4_EXTREME = INT4 + [("tiles_quad", 128, 256, 2048, 13), ("tiles_quad", 70, 256, 2048, 40), ("tiles_pair_small", 96, 1024, 2048, 12)]


@pytest.mark.parametrize("kernel,G,K,N,rows", INT4_EXTREME)
def test_int4_extreme_scales(kernel, G, K, N, rows):
    """Scales up to 2^125, beyond which code 0 itself is out of range, and down to the least subnormal: in all columns of some experts, in
    a few groups of others, among ordinary ones (the tiles compute a tile with a scale of 2^117.98 and more twice)."""
    _say(f"int4 weight bits, extreme scales, {kernel}")
    rng = np.random.default_rng(G + N + 1)
    case = H.make_case("int4", G, K, N, np.arange(1, G + 1) * rows, seed=G, group=32)
    case["scale"] = _scales(rng, case["scale"].shape, -10, 10)
    large, small = _scales(rng, case["scale"].shape, 115, 125), _scales(rng, case["scale"].shape, -127, -110)
    for g in range(G):
        pick = [1.0, 0.002, 0.5, 1.0][g % 4]
        at = rng.random(case["scale"].shape[1:]) < pick
        case["scale"][g][at] = (small if g % 4 == 3 else large)[g][at]
    _check(case, _unit_rows(case, rng), kernel)


@pytest.mark.parametrize("epilogue", ["none", "swiglu"])
@pytest.mark.parametrize("kernel,G,N,rows", [("tiles_pair_small", 20, 2048, 12), ("tiles_quad", 4, 512, 170), ("tiles_quad", 80, 2048, 20)])
def test_int4_rows_that_are_no_number(kernel, G, N, rows, epilogue):
    """NaN and infinities in rows of x look to the tiles like scales out of the usual decode's range; without such a scale, and beside one,
    they stay in their rows."""
    _say(f"int4 {kernel} {epilogue}, x with NaN")
    rng = np.random.default_rng(rows)
    K = 256
    case = H.make_case("int4", G, K, N, np.arange(1, G + 1) * rows, seed=G)
    bad = rng.random(case["M"]) < 0.1
    case["x"][bad, rng.integers(0, K, bad.sum())] = rng.choice(np.array([0x7FC0, 0x7F80, 0xFF80], np.uint16), bad.sum())
    for g in range(0, G, 3):   # one column of a large scale, on zeros of x
        case["scale"][g, 0, int(rng.integers(0, N))] = (127 + 119) << 7
        case["x"][g * rows:(g + 1) * rows, :128] &= 0x8000
    case["x"][bad, 200] |= 0x7FC0
    assert H.kernel_of(case, "gemm", swiglu=epilogue == "swiglu") == kernel
    if epilogue == "swiglu":
        got, want = _swiglu(case)
    else:
        got, want = H.run_cabi(case, H.upload(case), "gemm"), H.oracle_out(case)
    H.assert_close(got, want, rows=~bad, what=f"{kernel} {epilogue}")
    assert not np.isfinite(oracle.bf16_bits_to_f32(got)[bad]).any()


# experts, K, rows per expert: 4, 8 and 16 staged rows, whole iterations of 512 k and one to three groups of 128 behind them, K on
# both sides of what is staged at a time (7168, 3584 and 1536)
@pytest.mark.parametrize("fmt", ["fp4_b32", "fp4_b16"])
@pytest.mark.parametrize("G,K,rows", [(64, 512, 4), (64, 640, 8), (64, 896, 12), (64, 1152, 3), (48, 1536, 12), (48, 1664, 12),
                                      (32, 2048, 12), (32, 3712, 8), (32, 4096, 7), (24, 7168, 4), (24, 7296, 4), (24, 7680, 4)])
def test_fp4_rows(fmt, G, K, rows):
    _say(f"{fmt} weight bits K={K}, {rows} rows")
    rng = np.random.default_rng(K)
    case = H.make_case(fmt, G, K, 256, np.arange(1, G + 1) * rows, seed=K)
    case["scale"] = _scales(rng, case["scale"].shape, -110, 117)
    _check(case, _unit_rows(case, rng), "fp4_rows")


# kernel, experts, K, N, rows per expert
FP8 = [("strips_32", 4, 256, 512, 16), ("strips_64", 6, 256, 2048, 16), ("strips_128", 10, 256, 2048, 12), ("tiles_pair", 20, 256, 2048, 40), ("tiles_pair", 4, 384, 384, 160),
       ("tiles_quad", 2, 256, 256, 256)]


@pytest.mark.parametrize("codes", ["without", "some", "all"])
@pytest.mark.parametrize("kernel,G,K,N,rows", FP8)
def test_fp8(kernel, G, K, N, rows, codes):
    """0x7F and 0xFF are +-480 here and NaN to the hardware's conversions: none of them, one in the middle of some experts, any."""
    _say(f"fp8 weight bits {kernel} 0x7F: {codes}")
    rng = np.random.default_rng(G + N)
    case = H.make_case("fp8", G, K, N, np.arange(1, G + 1) * rows, seed=G)
    if codes != "all":
        case["weight"][(case["weight"] & 0x7F) == 0x7F] ^= 1
    if codes == "some":
        for g in range(0, G, 2):
            case["weight"][g, rng.integers(0, K), rng.integers(0, N)] |= 0x7F
    e = rng.integers(-60, 40, case["scale"].shape)
    case["scale"] = (case["scale"] * np.exp2(e)).astype(np.float32)
    _check(case, _unit_rows(case, rng), kernel)


@pytest.mark.parametrize("kernel,G,K,N,rows", [("strips_32", 4, 2048, 512, 16), ("strips_64", 6, 2048, 2048, 16), ("strips_128", 10, 2048, 2048, 12),
                                               ("tiles_pair", 20, 1024, 2048, 40), ("tiles_pair", 48, 1024, 2048, 17), ("tiles_quad", 2, 1024, 256, 256),
                                               ("tiles_pair", 4, 512, 384, 160), ("tiles_quad", 4, 512, 384, 161)])
def test_fp8_extreme_scales(kernel, G, K, N, rows):
    """Block scales up to 2^127 beside codes 0x7F: a weight does not depend on its neighbours' codes.  0x7F stands in blocks with ordinary
    scales in front of the large ones (even experts) and in the blocks with the large scales (their columns overflow and are left out)."""
    _say(f"fp8 weight bits, extreme scales, {kernel}")
    rng = np.random.default_rng(G + N + 1)
    case = H.make_case("fp8", G, K, N, np.arange(1, G + 1) * rows, seed=G)
    w = case["weight"]
    w[(w & 0x7F) == 0x7F] ^= 1
    case["scale"][:] = np.exp2(rng.integers(-20, 20, case["scale"].shape)) * np.where(rng.random(case["scale"].shape) < 0.5, 1, -1)
    for kb in range(1, K // 128, 2):   # odd blocks of k: weights up to 1, scales up to 2^127
        at = slice(128 * kb, 128 * kb + 128)
        w[:, at] = (w[:, at] & 0x80) | (w[:, at] & 0x7F) % 0x39
        case["scale"][:, kb] = case["scale"][:, kb] * np.exp2(107.0)
    finite = np.ones((G, N), bool)
    for g in range(G):
        for n in range(int(rng.integers(0, 64)), N, 64):
            k = int(rng.integers(0, K // 256)) * 256
            if g % 2 == 0:
                w[g, k + int(rng.integers(0, 128)), n] |= 0x7F
            else:
                w[g, k + 128 + int(rng.integers(0, 128)), n] |= 0x7F
                finite[g, n] = False
    at = _unit_rows(case, rng)
    assert H.kernel_of(case, "gemm") == kernel
    got = oracle.bf16_bits_to_f32(H.run_cabi(case, H.upload(case), "gemm"))
    lo = 0
    for g, hi in enumerate(case["group_list"]):
        want = oracle.expand_weight(oracle.FMT_BY_NAME["fp8"], w, case["scale"], None, g, True).reshape(K, N)[at[lo:hi]]
        assert np.isfinite(want[:, finite[g]]).all()
        assert np.array_equal(got[lo:hi][:, finite[g]], want[:, finite[g]]), f"{kernel} expert {g}"
        lo = hi


@pytest.mark.parametrize("codes", ["without", "some", "all"])
@pytest.mark.parametrize("kernel,G,N,rows", [("tiles_pair_exact", 24, 2048, r) for r in (3, 16, 17, 40)]
                         + [("strips_32", 4, 512, 5), ("strips_64", 6, 2048, 16), ("strips_128", 10, 2048, 12)])
def test_fp8_gemv(kernel, G, N, rows, codes):
    """The same of the GEMV op, whose weights are not rounded: with scales of powers of two bf16 holds them."""
    _say(f"fp8 gemv weight bits {kernel}, {rows} rows, 0x7F: {codes}")
    rng = np.random.default_rng(rows)
    K = 256
    case = H.make_case("fp8", G, K, N, np.arange(1, G + 1) * rows, seed=rows)
    if codes != "all":
        case["weight"][(case["weight"] & 0x7F) == 0x7F] ^= 1
    if codes == "some":
        for g in range(0, G, 2):
            case["weight"][g, rng.integers(0, K), rng.integers(0, N)] |= 0x7F
    case["scale"] = np.exp2(rng.integers(-60, 40, case["scale"].shape)).astype(np.float32)
    at = _unit_rows(case, rng)
    assert H.kernel_of(case, "gemv") == kernel
    got, want = H.run_cabi(case, H.upload(case), "gemv"), H.oracle_out(case, gemv=True)
    assert np.array_equal(oracle.bf16_bits_to_f32(got), oracle.bf16_bits_to_f32(want)), at


# kernel, experts, K, N, rows per expert
FP4 = [("strips_32", 4, 256, 512, 16), ("strips_32", 2, 1088, 256, 5), ("strips_64", 6, 256, 2048, 16), ("strips_128", 10, 256, 2048, 12),
       ("tiles_pair_small", 20, 256, 2048, 12), ("tiles_quad", 2, 256, 256, 256)]


@pytest.mark.parametrize("kernel,G,K,N,rows", FP4)
def test_fp4(kernel, G, K, N, rows):
    _say(f"fp4 weight bits {kernel}")
    rng = np.random.default_rng(G + N)
    case = H.make_case("fp4", G, K, N, np.arange(1, G + 1) * rows, seed=G)
    case["scale"] = _scales(rng, case["scale"].shape, -110, 117)
    _check(case, _unit_rows(case, rng), kernel)


@pytest.mark.parametrize("rows", [1, 8, 9, 16])
@pytest.mark.parametrize("kernel,G,N", [("strips_32", 4, 512), ("strips_64", 6, 2048), ("strips_128", 10, 2048)])
def test_fp4_gemv_strips(kernel, G, N, rows):
    """The GEMV op's weights are not rounded: with scales of powers of two bf16 holds them."""
    _say(f"fp4 gemv weight bits {kernel}, {rows} rows")
    if rows > 12 and kernel == "strips_128":
        rows = 12
    rng = np.random.default_rng(G + rows)
    K = 256
    case = H.make_case("fp4", G, K, N, np.arange(1, G + 1) * rows, seed=rows)
    case["scale"] = ((rng.integers(-60, 60, case["scale"].shape) + 127) << 7).astype(np.uint16)
    at = _unit_rows(case, rng)
    assert H.kernel_of(case, "gemv") == kernel
    got, want = H.run_cabi(case, H.upload(case), "gemv"), H.oracle_out(case, gemv=True)
    assert np.array_equal(oracle.bf16_bits_to_f32(got), oracle.bf16_bits_to_f32(want)), at
