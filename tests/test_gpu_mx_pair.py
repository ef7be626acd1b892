"""MXINT8 operands expanded to BF16 in one launch, against one launch each and the exact values."""

import pytest
import torch

from m5kernels_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1, 1, 32), (1, 3, 96), (33, 5, 2048), (4, 257, 64)])
def test_pair_expansion_equals_single(m, n, k, device):
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    q = [torch.randint(-127, 128, (r, k), generator=g, dtype=torch.int8).to(device) for r in (m, n)]
    e = [torch.randint(100, 150, (r, k // 32), generator=g, dtype=torch.uint8).to(device) for r in (m, n)]
    one = [torch.empty((r, k), dtype=torch.bfloat16, device=device) for r in (m, n)]
    two = [torch.full((r, k), float("nan"), dtype=torch.bfloat16, device=device) for r in (m, n)]
    st = _lib.stream_of(q[0])
    for i, r in enumerate((m, n)):
        _lib.call("m5k_mxint8_to_bf16", _lib.ptr(q[i]), _lib.ptr(e[i]), r, k, _lib.ptr(one[i]), st)
    _lib.call("m5k_mxint8_pair_to_bf16", _lib.ptr(q[0]), _lib.ptr(e[0]), m, _lib.ptr(q[1]), _lib.ptr(e[1]), n, k,
              _lib.ptr(two[0]), _lib.ptr(two[1]), st)
    for i in range(2):
        assert torch.equal(one[i], two[i])
        want = q[i].double().view(-1, k // 32, 32) * torch.exp2(e[i].double() - 127)[:, :, None]
        assert torch.equal(one[i].double(), want.view(-1, k))
