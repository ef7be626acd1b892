"""shift_split_condition reads 16-bit operands as they are for up to 8 conditioning rows: the bias
has the bits of FP32 copies of the same operands, at vector and odd K, for every table dtype."""

import pytest
import torch

from m5kernels_amd import shift_split_condition

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3, 8])
@pytest.mark.parametrize("n,k", [(1, 8), (33, 257), (1000, 5376)])
@pytest.mark.parametrize("operand", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("table", [torch.bfloat16, torch.float16, torch.float32])
def test_16_bit_operands_equal_fp32_copies(rows, n, k, operand, table, device):
    g = torch.Generator(device="cpu").manual_seed(rows + n + k)
    gamma = torch.randn((k,), generator=g).to(table).to(device)
    scale = torch.randn((rows, k), generator=g).to(table).to(device)
    shift = torch.randn((rows, k), generator=g).to(operand).to(device)
    w = torch.randn((n, k), generator=g).to(operand).to(device)
    combined, bias = shift_split_condition(gamma, scale, shift, w)
    assert torch.equal(combined, gamma.float() * (1 + scale.float()))
    wide = shift_split_condition(gamma, scale, shift.float(), w.float())
    mixed = shift_split_condition(gamma, scale, shift.float(), w)
    assert torch.equal(bias, wide[1]) and torch.equal(bias, mixed[1])
    exact, size = shift.double() @ w.double().T, shift.double().abs() @ w.double().abs().T
    assert torch.all((bias.double() - exact).abs() <= (k + 1) * 2.0**-24 * 1.01 * size)
