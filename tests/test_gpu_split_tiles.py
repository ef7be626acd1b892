"""K ranges on every tile that the split entry points have, with every epilogue: INT8 bit for bit against
the unsplit launch and the oracle, FP8 against the float64 product.  Each case asserts first, through the
library's plan, that the tile and the number of ranges that it names are what runs."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import bits_of, np_of
from m5kernels_amd import _lib, gemm, hip, quantize
from oracle import reference as ref

pytestmark = pytest.mark.gpu

# (m, n, k, ranges): K ends in a partial stage (INT8) and the last range is shorter than the others or
# not; N % 4 != 0 takes the one-column form of the second pass, the others its four-column form.
INT8 = {
    "128": [(513, 768, 5392, 5), (65, 4095, 5376, 5), (700, 1000, 4112, 3)],
    "64": [(200, 1536, 4112, 3), (1, 17, 2064, 2), (5, 4095, 8320, 5)],
    "64-deep": [(1, 64, 4112, 3), (33, 130, 8336, 4), (65, 17, 4096, 2)],
    "256x128": [(1, 17, 1168, 2), (300, 520, 2064, 5), (257, 64, 1152, 3)],
    "256": [(257, 4095, 1168, 5), (513, 4096, 1152, 3)],
}
FP8 = {
    "128": [(513, 768, 5376, 5), (65, 4095, 5376, 5)],
    "64": [(200, 1536, 5376, 3), (1, 17, 2176, 2)],
    "64-deep": [(1, 64, 4096, 3), (65, 17, 4096, 2)],
    "256x128": [(1, 17, 1152, 2), (300, 520, 2176, 5)],
    "256": [(257, 4095, 1152, 5), (513, 4096, 1152, 3)],
}


def _cases(table):
    return [pytest.param(tile, *shape, id=f"{tile}-{'x'.join(map(str, shape))}") for tile, shapes in table.items()
            for shape in shapes]


def _schedule(tile):
    return "plain" if tile.startswith("256") else None


def _runs(mode, tile, m, n, k, ranges):
    print(f"case {mode} {tile} m={m} n={n} k={k} ranges={ranges}", flush=True)
    with hip.exact_splits(), hip.launch_override(_schedule(tile)):
        assert hip.split_plan(mode, m, n, k, ranges) == (tile, ranges)


@pytest.mark.parametrize("tile,m,n,k,ranges", _cases(INT8))
def test_int8_ranges_bit_exact(tile, m, n, k, ranges, device):
    _runs("int8", tile, m, n, k, ranges)
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    a, b = (torch.randint(-127, 128, (r, k), generator=g, dtype=torch.int8).to(device) for r in (m, n))
    sa, sb = ((torch.rand(r, generator=g) * 0.01 + 1e-3).to(device) for r in (m, n))
    rows = (torch.arange(m, dtype=torch.int32) % 3).to(device)
    res = torch.randn((m, n), generator=g).bfloat16().to(device)
    tables = torch.randn((3, n), generator=g).to(device)
    gates = tables.bfloat16()
    bf = torch.bfloat16
    for extra in (dict(output_dtype=bf), dict(output_dtype=torch.float16), dict(),
                  dict(bias=tables[0].clone(), output_dtype=bf), dict(bias=tables[1].clone()),
                  dict(bias=tables, bias_row_map=rows, output_dtype=torch.float16),
                  dict(residual=res, gate=gates[0].clone(), output_dtype=bf),
                  dict(residual=res, gate=gates, gate_row_map=rows, output_dtype=bf)):
        with hip.launch_override(_schedule(tile), ranges):
            got = gemm(a, b, "int8", a_scales=sa, b_scales=sb, **extra)
        with hip.launch_override("plain", 1):
            want = gemm(a, b, "int8", a_scales=sa, b_scales=sb, **extra)
        assert torch.equal(got, want), sorted(extra)
        if len(extra) == 1 and extra.get("output_dtype") is bf:
            few = sorted({0, m // 2, m - 1})
            expected = ref.c_i8_epilogue(ref.c_gemm_i8_acc(np_of(a[few]), np_of(b)), np_of(sa[few]), np_of(sb))
            np.testing.assert_array_equal(bits_of(got[few]), expected)


def _f8_split(a, b, sa, sb, ranges, out):
    (m, k), n = a.shape, b.shape[0]
    c = torch.empty((m, n), dtype=out, device=a.device)
    ws = torch.full((ranges, m, n), float("nan"), device=a.device)  # stale contents must not leak
    with hip.exact_splits():
        _lib.call("m5k_gemm_f8_splitk", _lib.ptr(a), _lib.ptr(b), m, n, k, _lib.ptr(sa), _lib.ptr(sb), _lib.ptr(c),
                  _lib.dtype_code(c), ranges, _lib.ptr(ws), ws.numel(), _lib.stream_of(a))
    assert not ws.isnan().any()  # every range wrote all of its sums
    return c


@pytest.mark.parametrize("tile,m,n,k,ranges", _cases(FP8))
def test_fp8_ranges_against_float64(tile, m, n, k, ranges, device):
    """The FP8 linear's 1e-4 rel-L2 bar, and no more error than the unsplit 256-row launch leaves (1.1:
    both are rounding noise).  BF16 outputs are the rounded FP32 ones; FP16 ones may differ by one step:
    the GPU multiplies by the last scale and converts to FP16 in one instruction, rounding once where
    FP32 and then FP16 round twice."""
    _runs("fp8", tile, m, n, k, ranges)
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    (a, sa), (b, sb) = (quantize(torch.randn((r, k), generator=g).to(device), "fp8") for r in (m, n))
    exact = (a.view(torch.float8_e4m3fn).double() * sa.double()[:, None]) @ (
        b.view(torch.float8_e4m3fn).double() * sb.double()[:, None]).T
    with hip.launch_override(_schedule(tile)):
        y = _f8_split(a, b, sa, sb, ranges, torch.float32)
        assert torch.equal(_f8_split(a, b, sa, sb, ranges, torch.bfloat16), y.bfloat16())
        half = _f8_split(a, b, sa, sb, ranges, torch.float16)
        # The same sign on both sides: the rest of the code counts FP16 steps.
        steps = (half.view(torch.int16).int() & 0x7FFF) - (y.half().view(torch.int16).int() & 0x7FFF)
        assert int(steps.abs().max()) <= 1
        assert torch.equal(_f8_split(a, b, sa, sb, ranges, torch.float32), y)  # deterministic
    with hip.launch_override("plain"):
        plain = gemm(a, b, "fp8", a_scales=sa, b_scales=sb)
    error, error_plain = ((t.double() - exact).norm() / exact.norm() for t in (y, plain))
    assert error < 1e-4 and error <= 1.1 * error_plain
