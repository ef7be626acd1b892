"""The split entry points' launches (m5k_gemm_split_plan; host only, no GPU): up to the count that a
call names by default, that count where it is forced."""

import ctypes
import random

import pytest
import torch

from m5kernels_amd import _lib, hip
from m5kernels_amd.harness import cli

SHAPES = [(128, 7168, 5376), (4096, 5376, 5376), (4096, 4096, 16384), (1024, 4096, 4096), (128, 4096, 16384)]


def _whole_ranges(k, splits, stage):
    """Ranges that are not empty when ceil(k / stage) stages are dealt out evenly over `splits`."""
    stages = -(-k // stage)
    return -(-stages // -(-stages // splits))


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_each_tuner_count_is_the_count_that_runs(m, n, k, monkeypatch):
    """Every launch of the tuner that names a count runs that many K ranges: at the time of the call into
    the library, its plan under the thread's settings says so."""
    seen = []

    def call(name, *args):
        if name == "m5k_gemm_set_schedule":
            return real_call(name, *args)
        if name == "m5k_gemm_i8_splitk":
            seen.append((args[14], hip.split_plan("int8", m, n, k, args[14])))

    real_call = _lib.call
    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(_lib, "device_tensor", lambda t, name: t.contiguous())
    monkeypatch.setattr(_lib, "stream_of", lambda t: None)
    monkeypatch.setattr(hip, "_cu_count", lambda device: 256)
    a, b = torch.zeros((m, k), dtype=torch.int8), torch.zeros((n, k), dtype=torch.int8)
    kw = dict(a_scales=torch.ones(m), b_scales=torch.ones(n), output_dtype=torch.bfloat16)
    launches = [launch for launch in cli.launch_space({"m": m, "n": n, "k": k}, "int8") if launch.splits]
    assert launches
    for launch in launches + [cli.Launch(None, s) for s in (2, 3, 16)]:
        seen.clear()
        with launch.active():
            hip.gemm(a, b, "int8", **kw)
        (asked, (tile, ranges)), = seen
        stage = 256 if tile == "64-deep" else 128
        assert asked == launch.splits and ranges == _whole_ranges(k, launch.splits, stage) > 1
        assert launch.schedule is None or tile.startswith("256")
    assert not _lib.load().m5k_gemm_schedule_state() & 64  # the setting ends with the call


def test_by_default_the_count_is_a_bound():
    for m, n, k in SHAPES:
        for splits in (2, 8, 64):
            assert 1 <= hip.split_plan("int8", m, n, k, splits)[1] <= splits
    assert hip.split_plan("int8", 128, 7168, 5376, 2) == ("64-deep", 1)
    assert hip.split_plan("int8", 900, 5376, 14336, 3) == ("256", 3)
    assert hip.split_plan("fp8", 16, 5120, 7168, 14)[1] > 1


def test_rules_over_random_shapes():
    rng = random.Random(9)
    for _ in range(2000):
        m, n = (round(10 ** rng.uniform(0, 4)) for _ in range(2))
        k, splits = 128 * round(10 ** rng.uniform(0, 2.3)), rng.randint(1, 64)
        for mode in ("int8", "fp8"):
            tile, ranges = hip.split_plan(mode, m, n, k, splits)
            assert 1 <= ranges <= splits and (ranges == 1 or tile != "decode")
            if ranges == 1:
                assert tile == hip._tile_plan.__wrapped__(mode, m, n, k, 256, True, None)
            with hip.exact_splits():
                tile, ranges = hip.split_plan(mode, m, n, k, splits)
                if ranges > 1:
                    wide = tile == "64-deep" or (mode == "fp8" and tile in ("64", "128"))
                    assert ranges == _whole_ranges(k, splits, 256 if wide else 128)
                else:
                    assert splits == 1 or _whole_ranges(k, splits, 128) == 1
                with hip.launch_override("plain"):
                    tile, ranges = hip.split_plan(mode, m, n, k, splits)
                    assert tile in ("256", "256x128") and ranges == _whole_ranges(k, splits, 128)


def test_settings_nest_and_are_thread_local():
    import threading

    state = _lib.load().m5k_gemm_schedule_state
    with hip.exact_splits():
        with hip.exact_splits():
            pass
        seen = []
        t = threading.Thread(target=lambda: seen.append(state() & 64))
        t.start()
        t.join()
        assert state() & 64 and seen == [0]
    assert not state() & 64


def test_argument_checks():
    lib, tile, ranges = _lib.load(), ctypes.c_int(0), ctypes.c_int(0)
    out = ctypes.byref(tile), ctypes.byref(ranges)
    assert lib.m5k_gemm_split_plan(_lib.I8, 4, 4, 4, 256, 1, *out) == 0
    assert lib.m5k_gemm_split_plan(_lib.U8, 4, 4, 128, 256, 64, *out) == 0
    assert lib.m5k_gemm_split_plan(_lib.BF16, 4, 4, 4, 256, 1, *out) == 1
    assert lib.m5k_gemm_split_plan(_lib.I8, 4, 0, 4, 256, 1, *out) == 1
    assert lib.m5k_gemm_split_plan(_lib.I8, 4, 4, 4, 0, 1, *out) == 1
    assert lib.m5k_gemm_split_plan(_lib.I8, 4, 4, 4, 256, 0, *out) == 1
    assert lib.m5k_gemm_split_plan(_lib.I8, 4, 4, 4, 256, 65, *out) == 1
    assert lib.m5k_gemm_split_plan(_lib.I8, 4, 4, 4, 256, 1, None, None) == 1
