"""Unrotated RMS quantization (block 1): rows held in registers (K % 8 == 0, K from 640, FP32 512, to
16384) against the element-by-element kernel, which the same row with one zero appended takes."""

import pytest
import torch

from m5kernels_amd import rms_quantize

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k", [8, 16, 504, 512, 632, 640, 2040, 2048, 2056, 5376, 8200, 16376, 16384])
def test_register_rows_equal_the_general_kernel(dtype, k, device):
    g = torch.Generator(device="cpu").manual_seed(k)
    x = torch.randn((7, k), generator=g).to(dtype)
    x[1] = 0
    x[2, ::5] *= 50
    x[3, k // 2] = float("inf")
    x[4, k - 1] = float("nan")
    x[5] = torch.finfo(dtype).max * torch.sign(x[5])
    x = x.to(device)
    gamma = (1 + 0.1 * torch.randn(k, generator=g)).to(device)
    signs = (torch.randint(0, 2, (k,), generator=g, dtype=torch.int8) * 2 - 1).to(device)
    pad = lambda t, v: torch.cat([t, torch.full((*t.shape[:-1], 1), v, dtype=t.dtype, device=device)], -1)  # noqa: E731
    eps = 1e-5
    q, s = rms_quantize(x, gamma, signs, 1, epsilon=eps)
    qg, sg = rms_quantize(pad(x, 0), pad(gamma, 1), pad(signs, 1), 1, epsilon=eps)
    assert torch.equal(q, qg[:, :k])  # folded codes do not depend on the statistics
    # The appended zero divides the mean square by k + 1; the FP32 sums' order is each kernel's own
    # (k additions of non-negative terms: k 2^-24 relative at most, halved by the square root).
    rows = torch.tensor([0, 1, 2, 6], device=device)
    ss = x[rows].double().square().sum(1)
    ratio = torch.sqrt((ss / k + eps) / (ss / (k + 1) + eps))
    ratio[1] = 1.0  # a zero row's scale is 1
    torch.testing.assert_close(s[rows].double() * ratio, sg[rows].double(), rtol=k * 2.0**-24 + 2e-7, atol=0)
    # Not folded: codes of the normalized row, within one code of each other.
    qn, _ = rms_quantize(x, gamma, signs, 1, fold_scale=False, epsilon=eps)
    qw, _ = rms_quantize(pad(x, 0), pad(gamma, 1), pad(signs, 1), 1, fold_scale=False, epsilon=eps)
    assert int((qn[rows].int() - qw[rows, :k].int()).abs().max()) <= 1
