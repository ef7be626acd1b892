"""The small GEMM tiles (128 x 128, 64 x 64, decode) at their edges: INT8 bit-exact against the
oracle, float modes within the FP32 dot-product bound of the float64 product, and the unaligned
loader at every residue of K and base address."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import bits_of, np_of
from m5kernels_amd import gemm, hip, projection_qk_rope, projection_qkv_rope, qk_norm_rope, quantize
from oracle import reference as ref

pytestmark = pytest.mark.gpu

# (m, n, k) per tile: one row past and one short of a tile, K of an odd and an even number of
# stages, a ragged last line (K = 16 mod 128), a single line.
TILED = {
    "decode": [(1, 4096, 128), (16, 4095, 1040), (17, 1024, 4096), (32, 17, 1168), (5, 16, 2048)],
    "64": [(300, 520, 1024), (257, 4096, 1168), (193, 7104, 1024)],
    "64-deep": [(64, 64, 16384), (65, 127, 8336), (33, 4096, 5376), (128, 5377, 5120)],
    "128": [(512, 7168, 5376), (513, 6400, 1168), (128, 21376, 2176)],
}
CASES = [(tile, *shape) for tile, shapes in TILED.items() for shape in shapes]


def _int8(g, m, n, k, device):
    a = torch.randint(-127, 128, (m, k), generator=g, dtype=torch.int8).to(device)
    b = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int8).to(device)
    return a, b, (torch.rand(m, generator=g) * 0.01 + 1e-3).to(device), (torch.rand(n, generator=g) * 0.01 + 1e-3).to(device)


def _sampled(m):
    return sorted({0, m // 2, m - 1, min(m - 1, 15), min(m - 1, 16), min(m - 1, 64), min(m - 1, 127), min(m - 1, 128)})


@pytest.mark.parametrize("tile,m,n,k", CASES)
def test_int8_tiles_bit_exact_vs_oracle(tile, m, n, k, device):
    print(f"case {tile} m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    a, b, sa, sb = _int8(g, m, n, k, device)
    assert hip.tile_plan("int8", a, b) == tile
    y = gemm(a, b, "int8", a_scales=sa, b_scales=sb, output_dtype=torch.bfloat16)
    rows = _sampled(m)
    expected = ref.c_i8_epilogue(ref.c_gemm_i8_acc(np_of(a[rows]), np_of(b)), np_of(sa[rows]), np_of(sb))
    np.testing.assert_array_equal(bits_of(y[rows]), expected)
    # Every row against the forced 256-row tiles, with the epilogues that read row maps.
    rmap = (torch.arange(m, dtype=torch.int32) % 3).to(device)
    kw = [dict(bias=torch.randn((3, n), generator=g).to(device), bias_row_map=rmap, output_dtype=torch.float16),
          dict(bias=torch.randn((n,), generator=g).to(device), output_dtype=torch.float32),
          dict(residual=torch.randn((m, n), generator=g).bfloat16().to(device),
               gate=torch.randn((3, n), generator=g).bfloat16().to(device), gate_row_map=rmap,
               output_dtype=torch.bfloat16)]
    for extra in kw:
        got = gemm(a, b, "int8", a_scales=sa, b_scales=sb, **extra)
        with hip.launch_override("plain"):
            want = gemm(a, b, "int8", a_scales=sa, b_scales=sb, **extra)
        assert torch.equal(got, want), sorted(extra)


@pytest.mark.parametrize("mode", ["bf16", "fp16", "fp8"])
@pytest.mark.parametrize("tile,m,n,k", CASES)
def test_float_tiles_within_the_dot_product_bound(tile, m, n, k, mode, device):
    """FP32 output against the float64 product of the operands the kernel sees; any order of K
    products and sums stays within K 2^-24 sum |a b| (1.01 for the second-order terms).  FP8's MFMA
    sums 128 products per instruction in a fixed-point register aligned to the largest, which that
    bound does not describe: it keeps the 1e-4 rel-L2 bar of the FP8 linear's other tests, at every
    tile, and no more error than the 256-row tiles leave on the same operands (1.1: both are rounding
    noise)."""
    k = -(-k // 128) * 128 if mode == "fp8" else k
    print(f"case {tile} m={m} n={n} k={k} {mode}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    a = torch.randn((m, k), generator=g).to(device)
    b = torch.randn((n, k), generator=g).to(device)
    kw = {}
    if mode == "fp8":
        (a, sa), (b, sb) = quantize(a, "fp8"), quantize(b, "fp8")
        kw = dict(a_scales=sa, b_scales=sb)
        af = a.view(torch.float8_e4m3fn).double() * sa.double()[:, None]
        bf = b.view(torch.float8_e4m3fn).double() * sb.double()[:, None]
    else:
        dt = torch.bfloat16 if mode == "bf16" else torch.float16
        a, b = a.to(dt), b.to(dt)
        af, bf = a.double(), b.double()
    y = gemm(a, b, mode, **kw).double()
    exact = af @ bf.T
    if mode == "fp8":
        with hip.launch_override("plain"):
            plain = gemm(a, b, mode, **kw).double()
        error, error_plain = ((t - exact).norm() / exact.norm() for t in (y, plain))
        assert error < 1e-4 and error <= 1.1 * error_plain
    else:
        assert torch.all((y - exact).abs() <= (k + 4) * 2.0**-24 * 1.01 * (af.abs() @ bf.abs().T))
    assert torch.equal(gemm(a, b, mode, **kw).double(), y)  # deterministic


@pytest.mark.parametrize("k", [1, 15, 17, 127, 129, 1000, 1023, 4099])
@pytest.mark.parametrize("m,n", [(1, 33), (65, 130), (300, 520)])
def test_unaligned_rows_bit_exact(m, n, k, device):
    print(f"case m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    a, b, sa, sb = _int8(g, m, n, k, device)
    y = gemm(a, b, "int8", a_scales=sa, b_scales=sb, output_dtype=torch.bfloat16)
    np.testing.assert_array_equal(bits_of(y), ref.c_i8_epilogue(ref.c_gemm_i8_acc(np_of(a), np_of(b)), np_of(sa), np_of(sb)))
    x, w = torch.randn((m, k), generator=g).bfloat16().to(device), torch.randn((n, k), generator=g).bfloat16().to(device)
    exact, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    assert torch.all((gemm(x, w, "bf16").double() - exact).abs() <= (k + 4) * 2.0**-24 * 1.01 * size)


@pytest.mark.parametrize("k", [65, 100, 127])
@pytest.mark.parametrize("m,n", [(2305, 6017), (4096, 4096)])
def test_unaligned_rows_of_one_stage_over_many_tiles(m, n, k, device):
    """256-row tiles there, a partial tile on both sides.  |sum a b| <= 127 * 127 * 127 < 2^24, so the FP32
    product of the codes is exact, and the epilogue is its FP32 sequence."""
    print(f"case m={m} n={n} k={k}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    a, b, sa, sb = _int8(g, m, n, k, device)
    acc = a.float() @ b.float().T
    bias = torch.randn((n,), generator=g).to(device)
    res = torch.randn((m, n), generator=g).bfloat16().to(device)
    scaled = (acc * sa[:, None]) * sb
    kw = dict(a_scales=sa, b_scales=sb)
    assert torch.equal(gemm(a, b, "int8", **kw), scaled)
    assert torch.equal(gemm(a, b, "int8", output_dtype=torch.bfloat16, **kw), scaled.bfloat16())
    assert torch.equal(gemm(a, b, "int8", bias=bias, **kw), scaled + bias)
    gated = gemm(a, b, "int8", residual=res, gate=bias.bfloat16(), output_dtype=torch.bfloat16, **kw)
    assert torch.equal(gated, (res.float() + scaled.bfloat16().float() * bias.bfloat16().float()).bfloat16())


@pytest.mark.parametrize("offset", [1, 2, 7, 8, 15])
def test_unaligned_bases_bit_exact(offset, device):
    """16-byte rows whose first byte is not 16-byte aligned (a view into a larger buffer); the last
    row ends at the buffer's last byte."""
    m, n, k = 70, 150, 512
    g = torch.Generator(device="cpu").manual_seed(offset)
    fa = torch.randint(-127, 128, (offset + m * k,), generator=g, dtype=torch.int8).to(device)
    fb = torch.randint(-127, 128, (offset + n * k,), generator=g, dtype=torch.int8).to(device)
    a, b = fa[offset:].view(m, k), fb[offset:].view(n, k)
    sa, sb = torch.ones(m, device=device), torch.ones(n, device=device)
    y = gemm(a, b, "int8", a_scales=sa, b_scales=sb)
    expected = ref.c_gemm_i8_acc(np_of(a), np_of(b)).astype(np.float32)
    np.testing.assert_array_equal(np_of(y), expected)


@pytest.mark.parametrize("mode", ["int8", "bf16"])
@pytest.mark.parametrize("m,heads,k", [(128, 56, 1024), (130, 40, 1536), (1, 2, 2048), (40, 3, 1032), (300, 20, 1001)])
def test_qk_and_qkv_equal_staged(mode, m, heads, k, device):
    """Each route of the Q/K and Q/K/V projections (one-head ring tiles, the staged form, unaligned
    rows) gives the plain GEMM's projection through the staged postprocess, bit for bit."""
    print(f"case m={m} heads={heads} k={k} {mode}", flush=True)
    g = torch.Generator(device="cpu").manual_seed(m + heads + k)
    x = torch.randn((m, k), generator=g).bfloat16().to(device)
    w = (torch.randn((heads * 384, k), generator=g) * 0.05).bfloat16().to(device)
    qg, kg = ((1 + 0.1 * torch.randn(128, generator=g)).bfloat16().to(device) for _ in range(2))
    cos, sin = (torch.randn((m, 48), generator=g).bfloat16().to(device) for _ in range(2))
    a, b, skw, qkw, gkw = x, w, {}, {}, {}
    if mode == "int8":
        (a, sa), (b, sb) = quantize(x, "int8"), quantize(w, "int8")
        gkw = dict(a_scales=sa, b_scales=sb)
        skw, qkw = dict(a_scales=sa, b_scales=sb), dict(a_scales=sa, w_scales=sb)
    proj = gemm(a, b, mode, output_dtype=torch.bfloat16, **gkw)
    assert torch.equal(projection_qk_rope(a, b, qg, cos, sin, mode, **skw), qk_norm_rope(proj, qg, cos, sin))
    q, kk, v = projection_qkv_rope(a, b, qg, kg, cos, sin, mode, **qkw)
    blocks = proj.view(m, heads, 3, 128)
    for stream, (out, gamma) in enumerate(((q, qg), (kk, kg))):
        flat = blocks[:, :, stream].reshape(m, heads * 128)
        assert torch.equal(out, qk_norm_rope(flat, gamma, cos, sin, epsilon=1e-6)), stream
    assert torch.equal(v, blocks[:, :, 2].permute(1, 0, 2).contiguous())
