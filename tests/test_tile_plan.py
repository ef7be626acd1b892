"""The GEMM's tile choice (m5k_gemm_tile_plan; host only)."""

import ctypes
import random

import pytest

from m5kernels_amd import _lib, hip


def _plan(mode, m, n, k, aligned=True):
    return hip._tile_plan.__wrapped__(mode, m, n, k, 256, aligned, None)


def test_tile_by_shape():
    for mode in ("int8", "fp8"):
        assert _plan(mode, 1, 4096, 4096) == "decode"
        assert _plan(mode, 128, 4096, 4096) == "64-deep"
        assert _plan(mode, 256, 7168, 5376) == "64"
        assert _plan(mode, 512, 7168, 5376) == "128"
        assert _plan(mode, 4096, 4096, 16384) == "256"
    assert _plan("bf16", 128, 5376, 5120) == "64-deep"
    assert _plan("fp32", 128, 5376, 5120) == "256"


def test_rules_over_random_shapes():
    rng = random.Random(5)
    for _ in range(2000):
        m, n, k = (round(10 ** rng.uniform(0, 4.2)) for _ in range(3))
        for mode, size in (("int8", 1), ("fp8", 1), ("bf16", 2), ("fp16", 2)):
            tile = _plan(mode, m, n, k)
            assert tile != "decode" or m <= 32
            if mode != "int8" and k * size < 1024:
                assert tile == "256"  # one FP32 chain over K
            loose = _plan(mode, m, n, k, aligned=False)
            assert loose == "256" if mode == "fp8" else loose in ("64", "128")
        assert _plan("bf16", m, n, k) == _plan("fp16", m, n, k)


def test_a_forced_schedule_keeps_the_256_row_tiles():
    with hip.launch_override("plain"):
        assert _plan("int8", 1, 4096, 4096) == "256"
    assert _plan("int8", 1, 4096, 4096) == "decode"


def test_argument_checks():
    lib, tile, splits = _lib.load(), ctypes.c_int(0), ctypes.c_int(0)
    out = ctypes.byref(tile), ctypes.byref(splits)
    assert lib.m5k_gemm_tile_plan(_lib.I8, 4, 4, 4, 256, 1, 1, *out) == 0
    assert lib.m5k_gemm_tile_plan(_lib.I8, 0, 4, 4, 256, 1, 1, *out) == 1
    assert lib.m5k_gemm_tile_plan(_lib.I8, 4, 4, 4, 0, 1, 1, *out) == 1
    assert lib.m5k_gemm_tile_plan(_lib.I32, 4, 4, 4, 256, 1, 1, *out) == 1
    assert lib.m5k_gemm_tile_plan(_lib.I8, 4, 4, 4, 256, 1, 65, *out) == 1
    assert lib.m5k_gemm_tile_plan(_lib.BF16, 4, 4, 4, 256, 1, 2, *out) == 1
    assert lib.m5k_gemm_tile_plan(_lib.I8, 4, 4, 4, 256, 1, 1, None, None) == 1


def test_a_long_k_splits_where_decode_would_leave_cus_idle():
    # 30 x 2048 x 16384: 128 decode workgroups of 32 rows took 24 us, K ranges of ring tiles 14 us.
    assert hip._tile_plan.__wrapped__("int8", 30, 2048, 16384, 256, True, None, 16) != "decode"
    assert hip._tile_plan.__wrapped__("int8", 1, 4096, 4096, 256, True, None, 4) == "decode"


def test_one_round_of_half_tiles_is_not_given_up_for_two_rounds_of_small_ones():
    # 84 tiles of 256 x 256, as 168 halves in one round: BF16 256 x 21504 x 4096 55.5 us against 70.0 us on
    # 336 tiles of 128 x 128, INT8 256 x 21504 x 5376 39.9 us against 49.8 us.
    for m in (200, 256):
        assert _plan("bf16", m, 21504, 4096) == "256" and _plan("bf16", m, 21504, 5376) == "256"
        assert _plan("int8", m, 21504, 5376) == "256" and _plan("fp8", m, 21504, 5376) == "256"
    # One round of small tiles stays ahead (BF16 128 x 21504 x 4096: 36.8 us against 50.4 us), and two rounds where
    # the weight is larger than the Infinity Cache (BF16 400 x 16384 x 14336: 253.7 us against 285.2 us).
    assert _plan("bf16", 128, 21504, 4096) == "128" and _plan("int8", 128, 21504, 5376) == "128"
    assert _plan("bf16", 400, 16384, 14336) == "128"
