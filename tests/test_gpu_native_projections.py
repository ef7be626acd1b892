"""The native front of the Q/K and Q/K/V projections against the Python one, over the forms that both
take: the same outputs on every route, and the Python front's errors where the call is refused."""

import pytest
import torch

from m5kernels_amd import hip, projection_qk_rope, projection_qkv_rope, quantize

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.fixture
def fronts(monkeypatch):
    """Run a call through both fronts and compare; says whether the native one took it."""
    native_front = hip._fast
    assert native_front is not None, "m5k_fast.so is missing: build the package"

    def both(call, native):
        taken = []

        class Spy:
            quantize, gemm = staticmethod(native_front.quantize), staticmethod(native_front.gemm)

            @staticmethod
            def qk(*args):
                taken.append(native_front.qk(*args))
                return taken[-1]

            @staticmethod
            def qkv(*args):
                taken.append(native_front.qkv(*args))
                return taken[-1]

        results = []
        for front in (Spy, None):
            monkeypatch.setattr(hip, "_fast", front)
            try:
                r = call()
                results.append(r if isinstance(r, tuple) else (r,))
            except Exception as e:  # noqa: BLE001 - compared below
                results.append((type(e), str(e)))
            monkeypatch.setattr(hip, "_fast", native_front)
        assert (bool(taken) and taken[-1] is not None) == native
        assert len(results[0]) == len(results[1])
        for x, y in zip(*results):
            if isinstance(x, torch.Tensor):
                assert x.dtype == y.dtype and x.shape == y.shape and x.device == y.device and x.is_contiguous()
                assert torch.equal(x, y)
            else:
                assert x == y

    return both


def _inputs(mode, m, heads, k, half, device):
    g = torch.Generator(device="cpu").manual_seed(m + heads + k)
    x = torch.randn((m, k), generator=g).to(BF).to(device)
    w = (torch.randn((heads * 384, k), generator=g) * 0.05).to(BF).to(device)
    gamma, k_gamma = ((1 + 0.1 * torch.randn(128, generator=g)).to(BF).to(device) for _ in range(2))
    cos, sin = (torch.randn((m, half), generator=g).to(BF).to(device) for _ in range(2))
    if mode == "bf16":
        return x, w, gamma, k_gamma, cos, sin, {}, {}
    (a, sa), (b, sb) = quantize(x, "int8"), quantize(w, "int8")
    return a, b, gamma, k_gamma, cos, sin, dict(a_scales=sa, b_scales=sb), dict(a_scales=sa, w_scales=sb)


# Decode, 64 x 64 tiles, K ranges, one-head tiles, 256-row tiles, unaligned rows.
SIZES = [(1, 4, 4096), (97, 12, 1280), (128, 2, 5376), (128, 56, 1024), (256, 56, 1024), (700, 19, 1024), (40, 3, 1000),
         (5, 2, 1001)]


@pytest.mark.parametrize("mode", ["int8", "bf16"])
@pytest.mark.parametrize("m,heads,k", SIZES)
def test_routes_agree(mode, m, heads, k, fronts, device):
    print(f"case {mode} m={m} heads={heads} k={k}", flush=True)
    for half in (64, 48, 5):
        a, b, gamma, k_gamma, cos, sin, skw, qkw = _inputs(mode, m, heads, k, half, device)
        fronts(lambda: projection_qk_rope(a, b, gamma, cos, sin, mode, **skw), True)
        fronts(lambda: projection_qk_rope(a, b, gamma, cos, sin, mode, epsilon=1e-6, **skw), True)
        fronts(lambda: projection_qkv_rope(a, b, gamma, k_gamma, cos, sin, mode, **qkw), True)


@pytest.mark.parametrize("mode", ["int8", "bf16"])
def test_other_forms_are_the_python_fronts(mode, fronts, monkeypatch, device):
    m, heads, k = 33, 2, 256
    a, b, gamma, k_gamma, cos, sin, skw, qkw = _inputs(mode, m, heads, k, 64, device)

    def qk(native, a=a, b=b, gamma=gamma, cos=cos, sin=sin, mode=mode, skw=skw, **kw):
        fronts(lambda: projection_qk_rope(a, b, gamma, cos, sin, mode, **skw, **kw), native)

    def qkv(native, a=a, b=b, gamma=gamma, k_gamma=k_gamma, cos=cos, sin=sin, mode=mode, qkw=qkw, **kw):
        fronts(lambda: projection_qkv_rope(a, b, gamma, k_gamma, cos, sin, mode, **qkw, **kw), native)

    wide = torch.randn(m, 128, device=device).to(BF)
    shifted = torch.ones(129, device=device, dtype=BF)[1:]  # 2-byte aligned: copied
    for call in (qk, qkv):
        call(True)
        call(False, epsilon=1)  # an integer is accepted
        for bad in (0.0, -1e-5, float("inf"), float("nan"), 1e-60, 1e60, "1e-5", True):
            call(False, epsilon=bad)
        call(False, mode="fp8")
        call(False, a=a.T.contiguous().T)  # strided: copied
        call(False, cos=wide[:, ::2], sin=wide[:, 1::2])
        call(False, cos=wide, sin=wide)  # wider than half a head
        call(False, cos=cos[:-1], sin=sin[:-1])
        call(False, cos=cos[:, :1], sin=sin)
        call(False, cos=cos.float(), sin=sin.float())
        call(False, gamma=gamma[:-1])
        call(False, gamma=gamma.float())
        call(False, gamma=shifted)
        call(False, a=a[:, :-1])
        call(False, a=a[:0])
        call(False, b=b[:-1])
        call(False, a=a.cpu(), b=b.cpu())
        call(False, a=a[0])
    qk(False, tile=(32, 128, 4, 1))  # equal, but checked as any given tile
    qk(False, tile=(31, 128, 4, 1))
    qkv(False, k_gamma=k_gamma[:-1])
    qkv(False, k_gamma=shifted)
    if mode == "int8":
        qk(False, skw=dict(a_scales=skw["a_scales"]))
        qk(False, skw=dict(a_scales=skw["a_scales"][:-1], b_scales=skw["b_scales"]))
        qkv(False, qkw=dict(a_scales=qkw["a_scales"].double(), w_scales=qkw["w_scales"]))
    else:
        ones = torch.ones(m, device=device)
        qk(False, skw=dict(a_scales=ones, b_scales=torch.ones(768, device=device)))
        qkv(False, qkw=dict(a_scales=ones, w_scales=torch.ones(768, device=device)))
    for schedule, splits in (("plain", None), (None, 2)):
        with hip.launch_override(schedule, splits):
            qk(False)
            qkv(False)
    monkeypatch.setenv("M5K_GEMM_SCHEDULE", "mixed")
    qk(False)
    monkeypatch.delenv("M5K_GEMM_SCHEDULE")
    monkeypatch.setenv("M5K_GEMM_MIXED_TILES", "0")
    qk(True)
    qkv(True)


@pytest.mark.parametrize("m,heads,k", [(97, 12, 1280), (128, 2, 5376), (256, 56, 1024)])
def test_streams_and_graph_replays(m, heads, k, device):
    """Staged, with K ranges, and fused: on a side stream, and captured, replayed with new inputs and eager
    work between replays."""
    a, b, gamma, k_gamma, cos, sin, _, qkw = _inputs("int8", m, heads, k, 64, device)

    def step():
        return projection_qkv_rope(a, b, gamma, k_gamma, cos, sin, "int8", **qkw)

    want, side = step(), torch.cuda.Stream(device=device)
    side.wait_stream(torch.cuda.current_stream(device))
    with torch.cuda.stream(side):
        got = step()
    side.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(got, want))
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        y = step()
    for i in range(3):
        a.copy_(torch.randint(-127, 128, a.shape, device=device, dtype=torch.int8))
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(p, q) for p, q in zip(y, step()))
        torch.cuda.synchronize()
