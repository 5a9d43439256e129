"""What the performance of this framework is measured on.

The cases are the work its callers have it do, through the public entry points
of the `GPU` class, `DiTBlock` and `optimizer_step`: group-quantized linears
from the small layers of a character GPT (rows of 128) to those of a large
decoder (4096 x 14336), at one row (decode) up to 8192 rows (prefill), forward
and backward, int8, int4 and fp32 weights, both math modes, with sizes that are
no multiple of any tile among them; the looped DiT block, forward and as a
training step; and the optimizer's update with its re-quantization.

listed() names the cases; draw() gives others of the same ranges.
"""
from __future__ import annotations

import importlib.util
import math
import os
import random
import sys

import torch

PKG_DIR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "diffusion-gpt-metal_amd")


def _package():
    if "dgm_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "dgm_amd", os.path.join(PKG_DIR, "__init__.py"), submodule_search_locations=[PKG_DIR])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["dgm_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["dgm_amd"]


# ---- the cases --------------------------------------------------------------


def _linear(name, passes, bits, M, N, K, G, math_mode="fp32", bias=False):
    c = {"kind": "linear", "passes": passes, "bits": bits, "M": M, "N": N, "K": K, "G": G, "math": math_mode,
         "bias": bias}
    return dict(c, name=name) if name else c


def _dit(name, train, B, T, C, F, H, bits=8, loops=4, G=32):
    c = {"kind": "dit", "train": train, "B": B, "T": T, "C": C, "F": F, "H": H, "bits": bits, "loops": loops, "G": G}
    return dict(c, name=name) if name else c


def _optimizer(name, bits, rows, cols, G):
    c = {"kind": "optimizer", "bits": bits, "rows": rows, "cols": cols, "G": G}
    return dict(c, name=name) if name else c


def listed():
    return [
        # The MLP up-projection of the small int8 character GPT (batch 16,
        # block 64, width 128, group 8) in one training step: forward with
        # bias, bias gradient, dX and dW.
        _linear("gpt_mlp_step_int8", "step", 8, 1024, 512, 128, 8, bias=True),
        # The DiT's down-projection (8 x 64 tokens, 768 -> 192) in one int4
        # training step.
        _linear("dit_mlp_step_int4", "step", 4, 512, 192, 768, 32),
        # One generated token through a large decoder's up-projection.
        _linear("decode_int4_one_row", "forward", 4, 1, 14336, 4096, 128),
        # A batch of 24 sequences, one token each, through its int8
        # down-projection.
        _linear("decode_int8_batch24", "forward", 8, 24, 4096, 14336, 128),
        # A 2048-token prompt in the default math mode.
        _linear("prefill_int4_2048", "forward", 4, 2048, 14336, 4096, 128),
        # A prompt whose length, width and output are no multiple of a tile,
        # int8 weights with a bias, groups of 32.
        _linear("prefill_int8_ragged", "forward", 8, 517, 4100, 4128, 32, bias=True),
        # The reduced-precision mode on a long prompt.
        _linear("prefill_int4_8192_bf16", "forward", 4, 8192, 14336, 4096, 128, "bf16"),
        # dX and the accumulated dW of a large int8 linear under training.
        _linear("backward_int8_2048", "backward", 8, 2048, 4096, 4096, 128),
        # A training step of an fp32 linear (no quantization): 32 stories of
        # 384 tokens.
        _linear("step_fp32_12288", "step", 32, 12288, 1536, 384, 8),
        # The photos DiT's block: one denoising step's forward.
        _dit("dit_block_forward", False, 8, 64, 192, 768, 4),
        # A wider DiT block on 256 tokens per picture: one training step.
        _dit("dit_block_train_wide", True, 4, 256, 512, 2048, 8),
        # The optimizer's update of an int4 up-projection, an int8 square one
        # and a norm, with the squared-gradient sums and the re-quantization.
        _optimizer("optimizer_int4", 4, 14336, 4096, 128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step):
    """Log-uniform in [lo, hi], two in three times a multiple of step."""
    v = _log(rng, lo, hi)
    return max(step, v // step * step) if rng.random() < 0.67 else v


def draw(rng):
    kind = rng.choice(["small", "decode", "prefill", "prefill", "backward", "backward", "bf16", "fp32", "dit",
                       "optimizer"])
    bits = rng.choice([4, 8])
    if kind == "dit":
        H, D = rng.choice([(4, 48), (4, 64), (6, 64), (8, 64), (8, 48)])
        T = rng.choice([16, 64, 128, 256])
        B = max(1, min(16, 1024 // T // rng.choice([1, 2])))
        C = H * D
        return _dit(None, rng.random() < 0.5, B, T, C, 4 * C, H, bits, rng.choice([2, 3, 4]))
    if kind == "optimizer":
        G = rng.choice([32, 64, 128])
        return _optimizer(None, bits, _log(rng, 256, 14336), G * _log(rng, 4, 4096 // G), G)
    if kind == "small":     # the small models' linears
        G = rng.choice([8, 16, 32])
        return _linear(None, rng.choice(["forward", "step"]), bits, _size(rng, 65, 1024, 64), _size(rng, 32, 1024, 32),
                       G * _log(rng, 4, 768 // G), G, bias=rng.random() < 0.5)
    if kind == "fp32":      # linears that are not quantized
        return _linear(None, rng.choice(["forward", "step"]), 32, _size(rng, 128, 12288, 64), _size(rng, 64, 1536, 32),
                       _size(rng, 64, 512, 32), 8, bias=rng.random() < 0.5)
    G = rng.choice([32, 64, 128])
    if kind == "decode":
        N, K = rng.choice([(14336, 4096), (4096, 14336), (4096, 4096), (1024, 4096), (6144, 4096)])
        return _linear(None, "forward", bits, _log(rng, 1, 64), N, K, G, rng.choice(["fp32", "bf16"]))
    if kind == "bf16":
        return _linear(None, "forward", bits, _size(rng, 128, 8192, 128), _size(rng, 512, 14336, 128),
                       G * _log(rng, 512 // G, 4096 // G), G, "bf16", bias=rng.random() < 0.5)
    if kind == "prefill":
        return _linear(None, "forward", bits, _size(rng, 65, 2048, 64), _size(rng, 512, 14336, 64),
                       G * _log(rng, 512 // G, 4096 // G), G, bias=rng.random() < 0.5)
    return _linear(None, "backward", bits, _size(rng, 128, 2048, 64), _size(rng, 512, 4096, 64),
                   G * _log(rng, 512 // G, 4096 // G), G)


# ---- inputs -----------------------------------------------------------------

_CONTEXT = {}


def _context(math_mode="fp32"):
    """The program's GPU contexts, one for each math mode it uses."""
    if math_mode not in _CONTEXT:
        dgm = _package()
        stream = torch.cuda.Stream()
        gpu = dgm.GPU(stream=stream)
        gpu.set_math(dgm.DGM_MATH_BF16 if math_mode == "bf16" else dgm.DGM_MATH_FP32)
        _CONTEXT[math_mode] = (gpu, stream)
    return _CONTEXT[math_mode]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _activations(g, M, K):
    """N(0, 1) rows in which one channel in 256 is ten times as large, as the
    inputs of a trained model's linears are."""
    x = torch.randn(M, K, generator=g, device="cuda")
    big = torch.rand(K, generator=g, device="cuda") < 1.0 / 256
    return x * torch.where(big, 10.0, 1.0)


def _gradients(g, M, N):
    """Small values whose size differs from token to token (a factor of e)."""
    return torch.randn(M, N, generator=g, device="cuda") * (
        1e-3 * torch.exp(torch.randn(M, 1, generator=g, device="cuda")))


def _linear_inputs(case, seed):
    g = _gen(seed)
    M, N, K = case["M"], case["N"], case["K"]
    t = {"w": torch.randn(N, K, generator=g, device="cuda") * 0.02, "x": _activations(g, M, K)}
    t["bias"] = torch.randn(N, generator=g, device="cuda") * 0.1 if case["bias"] else None
    if case["passes"] != "forward":
        t["dy"] = _gradients(g, M, N)
    return t


DIT_NORMS = ("n1", "n1b", "n2", "n2b", "nf")


def _dit_inputs(case, seed):
    g = _gen(seed)
    C, F, D = case["C"], case["F"], case["C"] // case["H"]
    shapes = {"wq": (C, C), "wk": (D, C), "wv": (D, C), "wo": (C, C), "wgate": (F, C), "wup": (F, C), "wdown": (C, F)}
    w = {n: torch.randn(*s, generator=g, device="cuda") * (1.0 / math.sqrt(s[1])) for n, s in shapes.items()}
    for n in DIT_NORMS:
        w[n] = 1.0 + 0.1 * torch.randn(C, generator=g, device="cuda")
    rows = case["B"] * case["T"]
    x = torch.randn(rows, C, generator=g, device="cuda")
    gx = torch.randn(rows, C, generator=g, device="cuda") * 1e-3
    return w, x, gx


OPT = dict(lr=3e-4, wd=0.1, clip=1.0, step_index=100)


def _optimizer_shapes(case):
    """(name, rows, cols, quantized, decay, bits): the case's matrix, a smaller int8 one and a norm."""
    r, c, G = case["rows"], case["cols"], case["G"]
    return [("up", r, c, True, True, case["bits"]), ("square", max(1, r // 4), c, True, True, 8),
            ("norm", 1, c, False, False, 32)]


def _optimizer_inputs(case, seed):
    g = _gen(seed)
    out = []
    for _, r, c, _, _, _ in _optimizer_shapes(case):
        n = r * c
        # A gradient norm below the clip, moments of the same size.
        std = 0.4 / math.sqrt(case["rows"] * case["cols"] * 1.5)
        out.append((torch.randn(n, generator=g, device="cuda") * 0.02, torch.randn(n, generator=g, device="cuda") * std,
                    torch.randn(n, generator=g, device="cuda") * std,
                    torch.rand(n, generator=g, device="cuda") * std * std))
    return out


def prepare(case, seed):
    dgm = _package()
    if case["kind"] == "linear":
        gpu, _ = _context(case["math"])
        bits, M, N, K, G = (case[k] for k in ("bits", "M", "N", "K", "G"))
        t = _linear_inputs(case, seed)
        st = {"gpu": gpu, "case": case, "q": None, "s": None, "y": torch.empty(M, N, device="cuda")}
        st.update(t)
        if case["passes"] != "forward":
            st.update(dx=torch.empty(M, K, device="cuda"), dw=torch.zeros(N, K, device="cuda"),
                      db=torch.zeros(N, device="cuda"))
        if bits != 32:
            st["q"] = torch.empty(N * K // (2 if bits == 4 else 1), dtype=torch.uint8 if bits == 4 else torch.int8,
                                  device="cuda")
            st["s"] = torch.empty(N * (K // G), device="cuda")
            torch.cuda.synchronize()
            gpu.begin()
            gpu.quantize(t["w"], st["q"], st["s"], N, K, bits, G)
            gpu.end()
            st["w"] = None
        torch.cuda.synchronize()
        gpu.begin()     # one region holds a step's many calls
        return st
    gpu, stream = _context()
    if case["kind"] == "dit":
        w, x, gx = _dit_inputs(case, seed)
        torch.cuda.synchronize()
        cfg = dgm.DiTConfig(B=case["B"], T=case["T"], C=case["C"], F=case["F"], H=case["H"], D=case["C"] // case["H"],
                            loops=case["loops"], group=case["G"], bits=case["bits"])
        block = dgm.DiTBlock(gpu, cfg, w)
        st = {"gpu": gpu, "stream": stream, "case": case, "block": block, "x0": x, "x": torch.empty_like(x)}
        if case["train"]:
            block.zero_grads()
            st.update(gx0=gx, gx=torch.empty_like(gx))
        torch.cuda.synchronize()
        gpu.begin()
        return st
    params = []
    for (name, r, c, quantized, decay, bits), (w, g, m, v) in zip(_optimizer_shapes(case),
                                                                  _optimizer_inputs(case, seed)):
        p = dgm.Param(name, r, c, quantized, decay, bits, case["G"])
        p.w, p.g, p.m, p.v = w, g, m, v
        params.append(p)
    torch.cuda.synchronize()
    return {"gpu": gpu, "case": case, "params": params, "sumsq": torch.zeros(len(params), device="cuda")}


# ---- one pass ---------------------------------------------------------------


def run(st):
    case, gpu = st["case"], st["gpu"]
    if case["kind"] == "linear":
        bits, M, N, K, G, passes = (case[k] for k in ("bits", "M", "N", "K", "G", "passes"))
        out = {}
        if passes != "backward":
            gpu.gemmNT(bits, st["w"], st["q"], st["s"], st["x"], st["bias"], st["y"], M, N, K, G)
            out["y"] = st["y"]
        if passes != "forward":
            if case["bias"]:
                gpu.biasGrad(st["dy"], st["db"], M, N)
                out["db"] = st["db"]
            gpu.gemmBwd(bits, st["w"], st["q"], st["s"], st["dy"], st["x"], st["dx"], st["dw"], M, N, K, G,
                        accumulate=passes == "backward")
            out.update(dx=st["dx"], dw=st["dw"])
        return out
    if case["kind"] == "dit":
        block, n = st["block"], st["x0"].numel()
        if not case["train"]:
            gpu.copy(st["x0"], st["x"], n)
            block.forward(st["x"])
            return {"x": st["x"]}
        with torch.cuda.stream(st["stream"]):
            block.zero_grads()
        gpu.copy(st["x0"], st["x"], n)
        gpu.copy(st["gx0"], st["gx"], n)
        block.forward_train(st["x"])
        block.backward(st["gx"])
        return {"x": st["x"], "gx": st["gx"], "grads": dict(block.grads)}
    norm = _package().optimizer_step(gpu, st["params"], OPT["lr"], OPT["wd"], OPT["clip"], OPT["step_index"],
                                     sumsq=st["sumsq"])
    out = {"norm": norm}
    for p in st["params"]:
        out[p.name] = {"w": p.w, "m": p.m, "v": p.v}
        if p.quantized:
            out[p.name].update(q=p.q, scale=p.scale)
    return out


# ---- what a pass cannot do without, and how exact it is ------------------------


def _weight_bytes(bits, n, G):
    return n * 4.0 if bits == 32 else n * bits / 8.0 + n / G * 4.0


def work(case):
    if case["kind"] == "linear":
        M, N, K = (float(case[k]) for k in ("M", "N", "K"))
        w = _weight_bytes(case["bits"], N * K, case["G"])
        b = f = 0.0
        if case["passes"] != "backward":
            b += w + 4 * (M * K + M * N + (N if case["bias"] else 0))
            f += 2 * M * N * K
        if case["passes"] != "forward":
            # dY, X and the weights in; dX and dW out (dW in too where it accumulates).
            acc = 2 if case["passes"] == "backward" else 1
            b += w + 4 * (M * N + M * K + M * K + acc * N * K + (N if case["bias"] else 0))
            f += 4 * M * N * K
        return {"bytes": b, "flops": f}
    if case["kind"] == "dit":
        M, T, C, F, L = (float(case[k]) for k in ("T", "T", "C", "F", "loops"))
        M *= case["B"]
        D = C / case["H"]
        wn = 2 * C * C + 2 * D * C + 3 * C * F
        fwd = L * (2 * M * wn + 4 * M * T * C)
        w = _weight_bytes(case["bits"], wn, case["G"]) + 20 * C
        if not case["train"]:
            return {"bytes": w + 8 * M * C, "flops": fwd}
        # Every loop's activations that the backward needs are written and read once.
        acts = L * 4 * M * (8 * C + 2 * D + 3 * F) + L * 4 * case["B"] * case["H"] * T * T
        return {"bytes": 2 * w + 4 * wn + 16 * M * C + 2 * acts, "flops": 3 * fwd}
    b = f = 0.0
    for _, r, c, quantized, _, bits in _optimizer_shapes(case):
        n = float(r * c)
        # The clip needs the norm of all gradients before the update: g is read twice.
        b += n * (4 * 8) + (_weight_bytes(bits, n, case["G"]) if quantized else 0)
        f += 14 * n
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["kind"] == "linear":
        if case["math"] == "bf16":
            return {"rel": 1e-2, "max": 5e-2}
        # Sums of up to 14336 fp32 products: 1e-7 to 7e-7 in the 2-norm.
        return {"rel": 4e-6, "max": 2e-4}
    if case["kind"] == "dit":
        # Up to four loops of seven linears, five norms and a softmax.
        return {"rel": 2e-5, "max": 2e-3}
    # A sum of squares in another order moves nothing here (no clip); w, m and
    # v are a few fp32 operations each. A code may move where w / s is a tie.
    return {"rel": 1e-6, "max": 1e-4, "differ": 1e-5}


# ---- the same in 64 bits ------------------------------------------------------


def _dequantized(w, bits, G):
    """The weights that the codes and scales of w stand for, in 64 bits."""
    if bits == 32:
        return w.double()
    N, K = w.shape
    qmax = 7.0 if bits == 4 else 127.0
    grp = w.reshape(N, K // G, G)
    # A tensor divisor: torch divides by a number through its reciprocal, which rounds otherwise.
    top = grp.abs().amax(dim=2, keepdim=True)
    s = torch.clamp(top / torch.full_like(top, qmax), min=1e-8)
    codes = torch.clamp(torch.round(grp / s), -qmax, qmax)
    return (codes.double() * s.double()).reshape(N, K)


def _exact_linear(case, seed):
    t = _linear_inputs(case, seed)
    wd, x = _dequantized(t["w"], case["bits"], case["G"]), t["x"].double()
    out = {}
    if case["passes"] != "backward":
        out["y"] = x @ wd.T
        if case["bias"]:
            out["y"] += t["bias"].double()
    if case["passes"] != "forward":
        dy = t["dy"].double()
        if case["bias"]:
            out["db"] = dy.sum(0)
        out.update(dx=dy @ wd, dw=dy.T.contiguous() @ x)
    return out


def _exact_dit(case, seed):
    w32, x, gx = _dit_inputs(case, seed)
    B, T, C, F, H, L = (case[k] for k in ("B", "T", "C", "F", "H", "loops"))
    D, eps, mix = C // H, 1e-6, 0.5
    w = {n: (t.double() if n in DIT_NORMS else _dequantized(t, case["bits"], case["G"])) for n, t in w32.items()}
    # The tables are inputs of the block, made on the host in 32 bits.
    cos, sin = (torch.from_numpy(t.reshape(T, D)).cuda().double() for t in _rope(T, D))
    x = x.double()
    if case["train"]:
        for t in (*w.values(), x):
            t.requires_grad_(True)

    def rms(v, n):
        return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + eps) * n

    def rope(v):
        half = D // 2
        rot = torch.cat([-v[..., half:], v[..., :half]], dim=-1)
        return v * cos[:, None, :] + rot * sin[:, None, :]

    xi, v0 = x, None
    for loop in range(L):
        ln1 = rms(xi, w["n1"])
        q = rope((ln1 @ w["wq"].T).reshape(B, T, H, D)).transpose(1, 2)
        k = rope((ln1 @ w["wk"].T).reshape(B, T, 1, D)).transpose(1, 2)
        v = (ln1 @ w["wv"].T).reshape(B, T, 1, D).transpose(1, 2)
        if loop == 0:
            v0 = v
        else:
            v = (1.0 - mix) * v + mix * v0
        k, v = (t.expand(B, H, T, D).contiguous() for t in (k, v))
        p = torch.softmax(q.contiguous() @ k.transpose(-1, -2).contiguous() / math.sqrt(D), dim=-1)
        av = (p @ v).transpose(1, 2).reshape(B * T, C)
        mid = xi + rms(av @ w["wo"].T, w["n1b"])
        ln2 = rms(mid, w["n2"])
        z = ln2 @ w["wgate"].T
        mlp = (z * torch.sigmoid(z) * (ln2 @ w["wup"].T)) @ w["wdown"].T
        xi = rms(mid + rms(mlp, w["n2b"]), w["nf"])
    if not case["train"]:
        return {"x": xi}
    xi.backward(gx.double())
    return {"x": xi.detach(), "gx": x.grad, "grads": {n: t.grad.reshape(-1) for n, t in w.items()}}


def _rope(T, D, theta=1e4):
    import numpy as np
    f = np.float32
    inv = np.power(f(theta), -(np.arange(0, D, 2, dtype=f) / f(D)), dtype=f)
    ang = np.arange(T, dtype=f)[:, None] * inv[None, :]
    return np.tile(np.cos(ang), (1, 2)), np.tile(np.sin(ang), (1, 2))


def _exact_optimizer(case, seed):
    b1, b2, eps = 0.9, 0.95, 1e-8
    inputs = _optimizer_inputs(case, seed)
    bc1, bc2 = 1 / (1 - b1 ** OPT["step_index"]), 1 / (1 - b2 ** OPT["step_index"])
    out = {"norm": float(sum(g.double().square().sum() for _, g, _, _ in inputs).sqrt())}
    for (name, r, c, quantized, decay, bits), (w, g, m, v) in zip(_optimizer_shapes(case), inputs):
        w, g, m, v = (t.double() for t in (w, g, m, v))
        m = b1 * m + (1 - b1) * g
        v = b2 * v + (1 - b2) * g * g
        w = w - OPT["lr"] * (m * bc1 / ((v * bc2).sqrt() + eps) + (OPT["wd"] if decay else 0.0) * w)
        out[name] = {"w": w, "m": m, "v": v}
        if quantized:
            s = w.reshape(r * (c // case["G"]), case["G"]).abs().amax(1) / (7.0 if bits == 4 else 127.0)
            out[name].update(q=None, scale=torch.clamp(s, min=1e-8))
    return out


def exact(case, seed):
    if case["kind"] == "linear":
        return _exact_linear(case, seed)
    return _exact_dit(case, seed) if case["kind"] == "dit" else _exact_optimizer(case, seed)


if __name__ == "__main__":
    for c in listed() + [draw(random.Random(s)) for s in range(6)]:
        print(c, work(c), tolerance(c))
