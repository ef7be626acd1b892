"""Performance cases of the quantized projection path, each through the package's public entry points.

One case is one step of a transformer block as a program runs it: the activation preparation
(quantize, rotate, normalize + modulate) followed by the projection it feeds, on weights that
were quantized once.  The widths are the ones that the repository's benchmark, harness and tests
use (4096 and 16384; 5376, 7168, 14336 and 5120), the token counts run from one token to the
9914 of a long video prompt, and the ragged family takes any size.

``listed`` names the cases, ``draw`` gives others of the same ranges, ``prepare`` makes what a
program holds before the call, ``run`` is one pass, ``work`` the bytes and operations that a pass
cannot do without, ``exact`` the same pass in 64 bits in plain torch.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parent.parent / "m5-max-kernels_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import m5kernels_amd as m5  # noqa: E402

BF16 = torch.bfloat16
_DTYPES = {"bf16": BF16, "fp16": torch.float16, "fp32": torch.float32}
_HEAD = 128
_MAX_FLOPS = 2 * 4096 * 4096 * 16384  # of the largest listed case


def listed():
    return [
        # One decoded token through an attention projection: launches and host work count.
        dict(name="int8_m1_q", kind="linear", mode="int8", m=1, n=4096, k=4096, block=0, epilogue="none", out="bf16"),
        # A short prompt (128 tokens, the harness's shortest) through FFN-down with the block's
        # residual update in the epilogue.
        dict(name="int8_m128_ffn_down_gated", kind="linear", mode="int8", m=128, n=5376, k=14336, block=0,
             epilogue="gated", out="bf16"),
        # The benchmark's headline: FFN-down of 4096 tokens, quantization included.
        dict(name="int8_m4096_ffn_down", kind="linear", mode="int8", m=4096, n=4096, k=16384, block=0,
             epilogue="none", out="bf16"),
        # Odd sizes of a non-standard model: rows of codes that are no multiple of 16 bytes, a ragged
        # last tile on both sides, a per-row bias table and FP16 output.
        dict(name="int8_m300_ragged", kind="linear", mode="int8", m=300, n=520, k=1000, block=0,
             epilogue="bias_table", out="fp16"),
        # FFN-up of a middle-sized prompt in FP8.
        dict(name="fp8_m1024_ffn_up", kind="linear", mode="fp8", m=1024, n=14336, k=5376, block=0, epilogue="none",
             out="bf16"),
        # The text embedding of a short prompt, which stays in BF16.
        dict(name="bf16_m128_text_in", kind="linear", mode="bf16", m=128, n=5376, k=5120, block=0, epilogue="none",
             out="bf16"),
        # Block-scaled INT8 (32-element blocks) on a middle-sized prompt.
        dict(name="mxint8_m1024_q", kind="linear", mode="mxint8", m=1024, n=4096, k=4096, block=0, epilogue="none",
             out="bf16"),
        # Residual update + AdaLN + Hadamard + INT8 preparation, then the Q projection: the ordinary
        # attention input of a 4096-token step.
        dict(name="gated_adaln_m4096_q", kind="adaln", m=4096, n=7168, k=5376, block=256, norm="rms", gated=True,
             tables=0),
        # Q (or K) projection with per-head RMSNorm and RoPE over a long video prompt, on rotated codes.
        dict(name="qk_rope_m9914", kind="qk", mode="int8", m=9914, n=4096, k=4096, block=256, rope_half=64),
        # Grouped Q/K/V projection of a short prompt.
        dict(name="qkv_rope_m128", kind="qkv", mode="int8", m=128, n=21504, k=5376, block=0, rope_half=48),
        # Norm-shift-split: the conditioning tables of one diffusion step and the projection that uses them.
        dict(name="shift_split_m2048_q", kind="shift", m=2048, n=7168, k=5376, block=256, tables=1),
        # RMS-quantized projection without rotation.
        dict(name="rms_m512_q", kind="rms", m=512, n=7168, k=5376, block=1, fold=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["ragged", "adaln", "adaln", "qk", "qkv", "shift", "rms"])
    widths = [1024, 2048, 4096, 5120, 5376, 7168, 8192, 14336, 16384]
    m, n, k = _log_int(rng, 1, 9914), rng.choice(widths), rng.choice(widths)
    if rng.random() < 0.3:  # widths off the usual ones; K stays a multiple of 256 for the rotations
        n, k = _log_int(rng, 32, 16384), 256 * _log_int(rng, 1, 64)
    if kind == "ragged":
        m, n, k = _log_int(rng, 1, 640), _log_int(rng, 17, 1600), _log_int(rng, 65, 5000)
        return dict(kind="linear", mode="int8", m=m, n=n, k=k, block=0,
                    epilogue=rng.choice(["none", "bias", "bias_table", "gated"]), out=rng.choice(["bf16", "fp16"]))
    if kind in ("qk", "qkv"):
        n = 384 * _log_int(rng, 2, 56) if kind == "qkv" else 128 * _log_int(rng, 2, 56)
    # The 16-bit products run at half the 8-bit rate: half the work at most.
    mode = {"linear": rng.choice(["int8", "int8", "fp8", "bf16", "fp16", "mxint8"]),
            "qk": rng.choice(["int8", "int8", "bf16"]), "qkv": rng.choice(["int8", "int8", "bf16"])}.get(kind, "int8")
    most = _MAX_FLOPS * (1.0 if mode in ("int8", "fp8") else 0.5)
    while 2.0 * m * n * k > most:
        m = m // 2 + 1
    if kind == "linear":
        epilogue, block, out = "none", 0, "bf16"
        if mode == "int8":
            epilogue = rng.choice(["none", "none", "bias", "bias_table", "gated", "gated_table"])
            block = rng.choice([0, 0, 128, 256])
            out = "bf16" if epilogue.startswith("gated") else rng.choice(["bf16", "bf16", "fp16", "fp32"])
        return dict(kind=kind, mode=mode, m=m, n=n, k=k, block=block, epilogue=epilogue, out=out)
    if kind == "adaln":
        return dict(kind=kind, m=m, n=n, k=k, block=rng.choice([128, 256]), norm=rng.choice(["rms", "rms", "layer"]),
                    gated=rng.random() < 0.5, tables=rng.choice([0, 3]))
    if kind == "qk" or kind == "qkv":
        return dict(kind=kind, mode=mode, m=m, n=n, k=k, block=rng.choice([0, 256]) if mode == "int8" else 0,
                    rope_half=rng.choice([48, 64]))
    if kind == "shift":
        return dict(kind=kind, m=m, n=n, k=k, block=256, tables=1)
    return dict(kind="rms", m=m, n=n, k=k, block=rng.choice([1, 256]), fold=rng.random() < 0.7)


# ---- inputs ---------------------------------------------------------------------------------


def _randn(g, *shape, std=1.0, dtype=BF16):
    t = torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)
    return (t if std == 1.0 else t.mul_(std)).to(dtype)


def _activations(g, m, k, dtype=BF16):
    """Normal values, with one channel in 128 ten times as large: a transformer's activations."""
    x = torch.randn(m, k, generator=g, device="cuda", dtype=torch.float32)
    x[:, 5::128] *= 10.0
    return x.to(dtype)


def _signs(g, k):
    return torch.randint(0, 2, (k,), generator=g, device="cuda", dtype=torch.int8) * 2 - 1


def _raw(case, seed):
    """Every input of the case before any quantization, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    m, n, k, kind = case["m"], case["n"], case["k"], case["kind"]
    mode = case.get("mode", "int8")
    act = torch.float16 if mode == "fp16" else BF16
    r = {"x": _activations(g, m, k, act), "w": _randn(g, n, k, std=1.0 / math.sqrt(k), dtype=act)}
    if case.get("block", 0) > 1 or kind in ("shift", "rms"):
        r["signs"] = _signs(g, k)
    if kind == "linear":
        epilogue = case["epilogue"]
        if epilogue.startswith("bias"):
            r["bias"] = _randn(g, *((3, n) if epilogue == "bias_table" else (n,)), std=0.1, dtype=torch.float32)
        if epilogue.startswith("gated"):
            r["residual"] = _randn(g, m, n)
            r["gate"] = _randn(g, *((3, n) if epilogue == "gated_table" else (n,)), std=0.2)
        if epilogue.endswith("table"):
            r["map"] = torch.randint(0, 3, (m,), generator=g, device="cuda", dtype=torch.int32)
    if kind in ("adaln", "shift", "rms"):
        p = case.get("tables", 0)
        rows = (p, k) if kind == "adaln" and p else (k,)
        r["gamma"] = (1.0 + _randn(g, k, std=0.1, dtype=torch.float32)).to(BF16)
        if kind == "rms":
            r["gamma"] = r["gamma"].float()
        else:
            r["scale"], r["shift"] = _randn(g, *rows, std=0.2), _randn(g, *rows, std=0.1)
        if kind == "adaln" and p:
            r["map"] = torch.randint(0, p, (m,), generator=g, device="cuda", dtype=torch.int32)
        if case.get("gated"):
            r["branch"], r["gate"] = _randn(g, m, k), _randn(g, k, std=0.2)
    if kind in ("qk", "qkv"):
        half = case["rope_half"]
        r["gamma"] = (1.0 + _randn(g, _HEAD, std=0.1, dtype=torch.float32)).to(BF16)
        r["k_gamma"] = (1.0 + _randn(g, _HEAD, std=0.1, dtype=torch.float32)).to(BF16)
        pos = torch.arange(m, device="cuda", dtype=torch.float64)[:, None]
        inv = 10000.0 ** (-torch.arange(half, device="cuda", dtype=torch.float64) / half)
        r["cos"], r["sin"] = (pos * inv).cos().to(BF16), (pos * inv).sin().to(BF16)
    return r


def prepare(case, seed):
    """Activations and tables on the GPU, and the weight as the program keeps it: rotated where the
    projection takes rotated codes, quantized once."""
    s = _raw(case, seed)
    s["case"] = dict(case)
    w, mode, block = s["w"], case.get("mode", "int8"), case.get("block", 0)
    if mode in ("int8", "fp8", "mxint8"):
        if block > 1:
            s["wq"], s["ws"] = m5.rotate_quantize(w, block, s["signs"])
        elif case["kind"] == "rms":  # the signs belong to the activation's rotation, the weight takes them too
            s["wq"], s["ws"] = m5.quantize(w * s["signs"].to(w.dtype), mode)
        else:
            s["wq"], s["ws"] = m5.quantize(w, mode)
        if case["kind"] != "shift":
            del s["w"]
    return s


# ---- one pass --------------------------------------------------------------------------------


def run(s):
    return _RUN[s["case"]["kind"]](s, s["case"])


def _run_linear(s, c):
    mode, out = c["mode"], _DTYPES[c["out"]]
    if mode in ("bf16", "fp16"):
        return m5.gemm(s["x"], s["w"], mode, output_dtype=out)
    q, qs = m5.rotate_quantize(s["x"], c["block"], s["signs"]) if c["block"] else m5.quantize(s["x"], mode)
    extra = {}
    if "bias" in s:
        extra = dict(bias=s["bias"], bias_row_map=s.get("map"))
    elif "residual" in s:
        extra = dict(residual=s["residual"], gate=s["gate"], gate_row_map=s.get("map"))
    return m5.gemm(q, s["wq"], mode, a_scales=qs, b_scales=s["ws"], output_dtype=out, **extra)


def _run_adaln(s, c):
    common = dict(norm=c["norm"], row_map=s.get("map"))
    if c["gated"]:
        q, qs, r_next = m5.fused_gated_residual_norm_hadamard_quantize(
            s["x"], s["branch"], s["gate"], s["gamma"], s["scale"], s["shift"], s["signs"], c["block"], **common)
    else:
        q, qs = m5.fused_norm_hadamard_quantize(s["x"], s["gamma"], s["scale"], s["shift"], s["signs"], c["block"],
                                                **common)
        r_next = None
    y = m5.gemm(q, s["wq"], "int8", a_scales=qs, b_scales=s["ws"], output_dtype=BF16)
    return {"y": y, "r_next": r_next}


def _run_qk(s, c):
    if c["mode"] == "bf16":
        return m5.projection_qk_rope(s["x"], s["w"], s["gamma"], s["cos"], s["sin"], "bf16", epsilon=1e-6)
    q, qs = m5.rotate_quantize(s["x"], c["block"], s["signs"]) if c["block"] else m5.quantize(s["x"], "int8")
    return m5.projection_qk_rope(q, s["wq"], s["gamma"], s["cos"], s["sin"], "int8", a_scales=qs, b_scales=s["ws"],
                                 epsilon=1e-6)


def _run_qkv(s, c):
    tables = (s["gamma"], s["k_gamma"], s["cos"], s["sin"])
    if c["mode"] == "bf16":
        return m5.projection_qkv_rope(s["x"], s["w"], *tables, "bf16")
    q, qs = m5.rotate_quantize(s["x"], c["block"], s["signs"]) if c["block"] else m5.quantize(s["x"], "int8")
    return m5.projection_qkv_rope(q, s["wq"], *tables, "int8", a_scales=qs, w_scales=s["ws"])


def _run_shift(s, c):
    combined, bias = m5.shift_split_condition(s["gamma"], s["scale"], s["shift"], s["w"])
    y = m5.norm_shift_split_gemm(s["x"], s["wq"], s["ws"], s["signs"], combined, bias, c["block"])
    return {"combined": combined, "bias": bias, "y": y}


def _run_rms(s, c):
    q, qs = m5.rms_quantize(s["x"], s["gamma"], s["signs"], c["block"], fold_scale=c["fold"])
    return m5.gemm(q, s["wq"], "int8", a_scales=qs, b_scales=s["ws"], output_dtype=BF16)


_RUN = {"linear": _run_linear, "adaln": _run_adaln, "qk": _run_qk, "qkv": _run_qkv, "shift": _run_shift,
        "rms": _run_rms}


# ---- what a pass cannot do without --------------------------------------------------------------


def work(case):
    m, n, k, kind, mode = case["m"], case["n"], case["k"], case["kind"], case.get("mode", "int8")
    flops = 2.0 * m * n * k
    read = 2 * m * k  # 16-bit activations
    read += {"int8": n * k + 4 * n, "fp8": n * k + 4 * n, "mxint8": n * k + n * k // 32}.get(mode, 2 * n * k)
    written = m * n * {"fp32": 4}.get(case.get("out", "bf16"), 2)
    if case.get("epilogue", "none").startswith("gated"):
        read += 2 * m * n
    if case.get("gated"):  # the branch in, the updated residual out
        read += 2 * m * k
        written += 2 * m * k
    if kind in ("qk", "qkv"):
        read += 4 * m * case["rope_half"]
    if kind == "shift":  # the original weight for the bias row, and the tables out
        read += 2 * n * k
        written += 4 * n + 4 * k
        flops += 2.0 * n * k
    return {"bytes": float(read + written), "flops": flops}


def tolerance(case):
    kind, mode = case["kind"], case.get("mode", "int8")
    if kind == "linear" and mode == "int8":
        # Codes, scales and INT32 sums are pinned bit for bit, and the FP32 epilogue's order too.
        return "exact"
    if kind == "linear":
        # FP32 sums in another order move a 16-bit result by one step now and then: 1e-4 measured over
        # K 1024 to 16384, the largest single difference one BF16 step (0.0078).
        return {"rel": 4e-4, "max": 2e-2}
    # A row statistic summed in another order moves a few codes, and a 16-bit result, by one step:
    # 3e-4 measured against the 64-bit pass with the same BF16 boundaries, 0.012 for a single value.
    return {"rel": 1.2e-3, "max": 4e-2}


# ---- the same pass in 64 bits --------------------------------------------------------------------


def _rotate64(x, block):
    if block <= 1:
        return x
    h = torch.ones(1, 1, dtype=torch.float64, device=x.device)
    while h.shape[0] < block:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return ((x.reshape(-1, block) @ h) / math.sqrt(block)).reshape(x.shape)


def _codes64(x, mode):
    """(dequantized codes' integers or E4M3 values, scale [rows]) of symmetric per-row quantization."""
    if mode == "mxint8":
        b = x.reshape(x.shape[0], -1, 32)
        peak = b.abs().amax(2, keepdim=True)
        e = torch.where(peak == 0, torch.zeros_like(peak),
                        (torch.floor(torch.log2(peak.clamp_min(1e-300)).float().double()) - 6).clamp(-127, 127))
        unit = ((e.long() + 1023) << 52).view(torch.float64)  # 2**e, exact: ties are common in 16-bit inputs
        return (torch.round(b / unit).clamp(-127, 127) * unit).reshape(x.shape), None
    peak = x.abs().amax(1, keepdim=True)
    top = 448.0 if mode == "fp8" else 127.0
    scale = torch.where(peak == 0, torch.ones_like(peak), peak / top)
    z = (x * top / peak.clamp_min(1e-300)).clamp(-top, top)  # half the peak is a tie, 63.5, and stays one
    if mode == "fp8":
        return z.float().to(torch.float8_e4m3fn).double(), scale[:, 0]
    return torch.round(z), scale[:, 0]


def _bf(x):
    """A documented BF16 boundary of the path."""
    return x.float().to(BF16).double()


def _product(q, qs, wq, ws):
    y = q @ wq.T
    return y if qs is None else y * qs[:, None] * ws[None, :]


def _norm_rope64(p, gamma, cos, sin, half, eps):
    """[M, heads, 128] BF16 projection -> [heads, M, 128]."""
    u = p / torch.sqrt((p * p).mean(2, keepdim=True) + eps) * gamma.double()
    c, s = cos.double()[:, None, :], sin.double()[:, None, :]
    lo, hi = u[..., :half], u[..., half:2 * half]
    return torch.cat([lo * c - hi * s, hi * c + lo * s, u[..., 2 * half:]], 2).transpose(0, 1).contiguous()


def exact(case, seed):
    r = _raw(case, seed)
    m, n, kind, mode, block = case["m"], case["n"], case["kind"], case.get("mode", "int8"), case.get("block", 0)
    x, w = r["x"].double(), r["w"].double()
    signs = r["signs"].double() if "signs" in r else None
    if kind == "linear" and mode in ("bf16", "fp16"):
        return x @ w.T
    if mode == "bf16":
        wq = ws = None
    else:
        wq, ws = _codes64(w if signs is None else _rotate64(w * signs, block), mode)
    if kind == "linear":
        q, qs = _codes64(_rotate64(x * signs, block) if block else x, mode)
        y = _product(q, qs, wq, ws)
        if "bias" in r:
            y = y + (r["bias"].double()[r["map"].long()] if "map" in r else r["bias"].double())
        if "residual" in r:
            gate = r["gate"].double()[r["map"].long()] if "map" in r else r["gate"].double()
            y = r["residual"].double() + _bf(y) * gate
        return y
    if kind in ("qk", "qkv"):
        if mode == "bf16":
            p = _bf(x @ w.T)
        else:
            q, qs = _codes64(_rotate64(x * signs, block) if block else x, mode)
            p = _bf(_product(q, qs, wq, ws))
        rope = (r["cos"], r["sin"], case["rope_half"], 1e-6)
        if kind == "qk":
            return _norm_rope64(p.reshape(m, n // _HEAD, _HEAD), r["gamma"], *rope)
        p = p.reshape(m, n // (3 * _HEAD), 3, _HEAD)
        return (_norm_rope64(p[:, :, 0], r["gamma"], *rope), _norm_rope64(p[:, :, 1], r["k_gamma"], *rope),
                p[:, :, 2].transpose(0, 1).contiguous())
    if kind == "adaln":
        r_next = _bf(x + r["branch"].double() * r["gate"].double()) if case["gated"] else None
        v = x if r_next is None else r_next
        if case["norm"] == "layer":
            v = v - v.mean(1, keepdim=True)
        scale, shift = r["scale"].double(), r["shift"].double()
        if "map" in r:
            scale, shift = scale[r["map"].long()], shift[r["map"].long()]
        v = v / torch.sqrt((v * v).mean(1, keepdim=True) + 1e-5) * r["gamma"].double()
        q, qs = _codes64(_rotate64(_bf(v * (1.0 + scale) + shift) * signs, block), "int8")
        return {"y": _product(q, qs, wq, ws), "r_next": r_next}
    gamma = r["gamma"].double()
    combined = bias = None
    if kind == "shift":
        gamma = combined = gamma * (1.0 + r["scale"].double())
        bias = w @ r["shift"].double()
    inv = 1.0 / torch.sqrt((x * x).mean(1) + 1e-5)
    z = _rotate64(x * gamma * signs, block)
    peak = z.abs().amax(1)
    q = torch.round(z * 127.0 / peak[:, None])
    y = _product(q, peak * inv / 127.0, wq, ws)
    return y if kind == "rms" else {"combined": combined, "bias": bias, "y": y + bias}
