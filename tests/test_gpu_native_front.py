"""The native front of quantize() and gemm() against the Python one, over the forms that both take:
the same outputs, and the Python front's errors where the call is refused."""

import pytest
import torch

from m5kernels_amd import gemm, hip, quantize

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.fixture
def fronts(monkeypatch):
    """Run a call through both fronts and compare; says whether the native one took it."""
    assert hip._fast is not None, "m5k_fast.so is missing: build the package"

    def both(call, native):
        taken = []

        class Spy:
            @staticmethod
            def gemm(*args):
                taken.append(hip_fast.gemm(*args))
                return taken[-1]

            @staticmethod
            def quantize(*args):
                taken.append(hip_fast.quantize(*args))
                return taken[-1]

        hip_fast = hip._fast
        results = []
        for front in (Spy, None):
            monkeypatch.setattr(hip, "_fast", front)
            try:
                results.append(call())
            except Exception as e:  # noqa: BLE001 - compared below
                results.append((type(e), str(e)))
            monkeypatch.setattr(hip, "_fast", hip_fast)
        first, second = results
        assert (bool(taken) and taken[-1] is not None) == native
        for x, y in zip(first if isinstance(first, tuple) else (first,), second if isinstance(second, tuple) else (second,)):
            if isinstance(x, torch.Tensor):
                assert x.dtype == y.dtype and x.shape == y.shape and x.device == y.device and x.is_contiguous()
                assert torch.equal(x, y)
            else:
                assert x == y
        return first

    return both


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("mode", ["int8", "fp8"])
def test_quantize_forms(mode, dtype, fronts, device):
    x = torch.randn(37, 96, device=device).to(dtype)
    fronts(lambda: quantize(x, mode), True)
    fronts(lambda: quantize(x[:, 3:4].contiguous(), mode), True)
    fronts(lambda: quantize(x.requires_grad_(), mode), True)
    x = x.detach()
    fronts(lambda: quantize(x.T, mode), False)  # strided: copied by the Python front
    fronts(lambda: quantize(x[:, ::2], mode), False)
    fronts(lambda: quantize(x[0], mode), False)  # not a matrix: refused
    fronts(lambda: quantize(x[:0], mode), False)
    fronts(lambda: quantize(x.int(), mode), False)
    fronts(lambda: quantize(x, "int9"), False)
    fronts(lambda: quantize(x.cpu(), mode), False)
    fronts(lambda: quantize(x, "mxint8"), False)


@pytest.mark.parametrize("m,n,k", [(1, 4096, 4096), (128, 768, 5376), (300, 520, 1000), (5, 33, 128)])
def test_gemm_forms(m, n, k, fronts, device):
    g = torch.Generator(device="cpu").manual_seed(m + n + k)
    x, w = torch.randn((m, k), generator=g).to(BF).to(device), torch.randn((n, k), generator=g).to(BF).to(device)
    rows = (torch.arange(m, dtype=torch.int32) % 3).to(device)
    table, vec = torch.randn((3, n), generator=g).to(device), torch.randn((n,), generator=g).to(device)
    res = torch.randn((m, n), generator=g).to(BF).to(device)
    for mode in ("int8", "fp8") if k % 128 == 0 else ("int8",):
        (a, sa), (b, sb) = quantize(x, mode), quantize(w, mode)
        kw = dict(a_scales=sa, b_scales=sb)
        for out in (None, BF, torch.float16, torch.float32):
            fronts(lambda: gemm(a, b, mode, output_dtype=out, **kw), True)
        fronts(lambda: gemm(a, b, mode, output_dtype=torch.float64, **kw), False)
        fronts(lambda: gemm(a, b, mode), False)  # scales required
        fronts(lambda: gemm(a, b, mode, a_scales=sa[:-1], b_scales=sb), False)
        fronts(lambda: gemm(a, b, mode, a_scales=sa.double(), b_scales=sb), False)
        fronts(lambda: gemm(a, b.T, mode, **kw), False)
        fronts(lambda: gemm(a, b.T.contiguous().T, mode, **kw), False)  # strided operand: copied
        fronts(lambda: gemm(a, b[:, :-1], mode, **kw), False)
        fronts(lambda: gemm(a, b, mode, (16, 64, 4), **kw), False)  # malformed tile
        fronts(lambda: gemm(a, b, mode, (16, 64, 4, 1), **kw), False)
        if mode == "int8":
            fronts(lambda: gemm(a, b, mode, bias=vec, **kw), True)
            fronts(lambda: gemm(a, b, mode, bias=table, bias_row_map=rows, output_dtype=torch.float16, **kw), True)
            fronts(lambda: gemm(a, b, mode, bias=table, **kw), False)
            fronts(lambda: gemm(a, b, mode, bias=vec, bias_row_map=rows, **kw), False)
            fronts(lambda: gemm(a, b, mode, bias_row_map=rows, **kw), False)
            fronts(lambda: gemm(a, b, mode, bias=vec.to(BF), **kw), False)
            fronts(lambda: gemm(a, b, mode, residual=res, gate=vec.to(BF), output_dtype=BF, **kw), True)
            fronts(lambda: gemm(a, b, mode, residual=res, gate=table.to(BF), gate_row_map=rows, output_dtype=BF, **kw), True)
            fronts(lambda: gemm(a, b, mode, residual=res, gate=table.to(BF), gate_row_map=rows.long(), output_dtype=BF, **kw),
                   False)
            fronts(lambda: gemm(a, b, mode, residual=res, gate=vec.to(BF), **kw), False)  # needs an explicit BF16
            fronts(lambda: gemm(a, b, mode, residual=res, output_dtype=BF, **kw), False)
            fronts(lambda: gemm(a, b, mode, residual=res, gate=vec.to(BF), bias=vec, output_dtype=BF, **kw), False)
        else:
            fronts(lambda: gemm(a, b, mode, bias=vec, **kw), False)
    for mode, dt in (("bf16", BF), ("fp16", torch.float16)):
        a, b = x.to(dt), w.to(dt)
        fronts(lambda: gemm(a, b, mode, output_dtype=BF), True)
        fronts(lambda: gemm(a, b, mode), True)
        fronts(lambda: gemm(a, b.float(), mode), False)
        fronts(lambda: gemm(a, b, mode, residual=res, gate=vec.to(BF), output_dtype=BF), mode == "bf16")
    fronts(lambda: gemm(x.float(), w.float(), "fp32"), False)
    fronts(lambda: gemm(x, w, "int7"), False)


def test_overrides_and_streams(fronts, monkeypatch, device):
    g = torch.Generator(device="cpu").manual_seed(1)
    a, b = (torch.randint(-127, 128, (r, 512), generator=g, dtype=torch.int8).to(device) for r in (40, 70))
    kw = dict(a_scales=torch.ones(40, device=device), b_scales=torch.ones(70, device=device))
    for schedule, splits in (("plain", None), (None, 2)):
        with hip.launch_override(schedule, splits):
            fronts(lambda: gemm(a, b, "int8", **kw), False)
    monkeypatch.setenv("M5K_GEMM_SCHEDULE", "mixed")
    fronts(lambda: gemm(a, b, "int8", **kw), False)
    monkeypatch.delenv("M5K_GEMM_SCHEDULE")
    monkeypatch.setenv("M5K_GEMM_MIXED_TILES", "0")
    fronts(lambda: gemm(a, b, "int8", **kw), True)
    side = torch.cuda.Stream(device=device)
    side.wait_stream(torch.cuda.current_stream(device))
    with torch.cuda.stream(side):
        y = gemm(a, b, "int8", **kw)
    side.synchronize()
    assert torch.equal(y, gemm(a, b, "int8", **kw))


def test_vmap_wrappers_go_to_the_python_front(fronts, device):
    x = torch.randn(2, 4, 64, device=device).to(BF)

    def call():
        return torch.vmap(lambda t: quantize(t, "int8")[0])(x)

    with pytest.raises(Exception):
        call()  # refused there, as before: a batched wrapper has no storage to read


def test_graph_capture_replays(device):
    """quantize + gemm under capture, replayed with new inputs and eager work between replays."""
    x = torch.randn(16, 1024, device=device).to(BF)
    w, ws = quantize(torch.randn(512, 1024, device=device).to(BF), "int8")

    def step():
        q, s = quantize(x, "int8")
        return gemm(q, w, "int8", a_scales=s, b_scales=ws, output_dtype=BF)

    step()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream(device=device)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        y = step()
    for i in range(3):
        x.copy_(torch.randn(16, 1024, device=device))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, step())
        torch.cuda.synchronize()
