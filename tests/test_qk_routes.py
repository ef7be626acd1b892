"""Which route the Q/K and Q/K/V projections take (host only; the sizes alone decide)."""

import pytest
import torch

from m5kernels_amd import hip, qk_rope


@pytest.fixture(autouse=True)
def cus(monkeypatch):
    monkeypatch.setattr(hip, "_cu_count", lambda device: 256)


def _staged(m, n, k, mode="int8", **kw):
    dt = torch.int8 if mode == "int8" else torch.bfloat16
    return qk_rope._staged(torch.zeros((m, k), dtype=dt), torch.zeros((1, k), dtype=dt).expand(n, k), mode, **kw)


@pytest.mark.parametrize("m,n,k", [(768, 10752, 1024), (512, 15360, 1024), (400, 15360, 16384), (256, 21504, 1024),
                                   (200, 21504, 5376), (768, 6144, 1024), (4096, 21504, 5376)])
def test_the_grouped_projection_stays_fused_on_256_row_tiles(m, n, k):
    assert hip._tile_plan.__wrapped__("int8", m, n, k, 256, True, (None, (None,) * 3)) == "256"
    assert not _staged(m, n, k, grouped=True) and not _staged(m, n, k, "bf16", grouped=True)


def test_small_tiles_are_staged_and_one_head_tiles_are_not():
    for grouped in (False, True):
        assert _staged(1, 4608, 4096, grouped=grouped) and _staged(64, 6144, 5376, grouped=grouped)
        assert not _staged(128, 21504, 5376, grouped=grouped)  # 128 x 128
        assert not _staged(4096, 6144, 4096, grouped=grouped)


def test_a_single_projection_follows_the_gemms_k_ranges():
    assert hip.splitk_plan(1024, 5376, 14336) > 1
    assert _staged(1024, 5376, 14336) and not _staged(1024, 5376, 14336, "bf16")
