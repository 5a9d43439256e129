"""The DiT block where a linear is a large product (csrc/gemm_planes.hip: gate and
up from 7 * 2^27 products on, the backward's linears from 11 * 2^26), against
float64 autograd: forward, training forward and backward at the edges of the row
kernels (512 and 1024 columns), on both attention kernels (heads whose keys and
values take more than half of the LDS, T = 256 with D = 64, and less), with int8,
int4 and fp32 weights. The operand pieces lie in the caller's workspace: the
context allocates nothing, a captured forward gives the eager bits, and a workspace
without that room runs on the fp32 kernels."""
from __future__ import annotations

import math

import numpy as np
import pytest

from conftest import from_dev, rel_err

pytestmark = pytest.mark.gpu

CFGS = [   # B, T, C, F, H, bits, group, loops
    (1, 256, 768, 2560, 12, 8, 32, 2),     # row kernel of 16 columns a lane; 16-wave attention
    (2, 256, 512, 1792, 8, 4, 32, 2),      # gate and up on their line, 8 columns a lane
    (8, 64, 320, 2880, 5, 32, 8, 2),       # 4-wave attention, fp32 weights
    (1, 144, 1024, 3264, 16, 8, 64, 1),    # the widest row; rows that are no multiple of a tile
]


def _reference(dgm, cfg, blk, w, x, gx):
    """xs[loops], dL/dxs[0] and the parameters' gradients in float64."""
    import torch
    B, T, C, H, D = cfg.B, cfg.T, cfg.C, cfg.H, cfg.D
    ws = {}
    for n, (N, K) in cfg.linear_shapes().items():
        if cfg.bits == 32:
            ws[n] = w[n].double().reshape(N, K).clone()
            continue
        q = blk.codes[n]
        codes = q.view(torch.int8).double() if cfg.bits == 8 else torch.stack(
            [(q << 4).view(torch.int8) >> 4, q.view(torch.int8) >> 4], dim=1).reshape(-1).double()
        ws[n] = (codes.reshape(N, K // cfg.group, cfg.group) * blk.scales[n].double().reshape(N, -1, 1)).reshape(N, K)
    for n in dgm.DIT_NORMS:
        ws[n] = w[n].double().clone()
    x = x.double().clone()
    for t in (*ws.values(), x):
        t.requires_grad_(True)
    cos, sin = blk.cos.double().reshape(T, D), blk.sin.double().reshape(T, D)

    def rms(v, n):
        return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + cfg.eps) * ws[n]

    def rope(v):
        rot = torch.cat([-v[..., D // 2:], v[..., :D // 2]], dim=-1)
        return v * cos[:, None, :] + rot * sin[:, None, :]
    xi, v0 = x, None
    for loop in range(cfg.loops):
        ln1 = rms(xi, "n1")
        q = rope((ln1 @ ws["wq"].T).reshape(B, T, H, D)).transpose(1, 2)
        k = rope((ln1 @ ws["wk"].T).reshape(B, T, 1, D)).transpose(1, 2)
        v = (ln1 @ ws["wv"].T).reshape(B, T, 1, D).transpose(1, 2)
        if loop == 0:
            v0 = v
        else:
            v = (1.0 - cfg.mix) * v + cfg.mix * v0
        k, v = (t.expand(B, H, T, D).contiguous() for t in (k, v))
        p = torch.softmax(q.contiguous() @ k.transpose(-1, -2).contiguous() / math.sqrt(D), dim=-1)
        av = (p @ v).transpose(1, 2).reshape(B * T, C)
        mid = xi + rms(av @ ws["wo"].T, "n1b")
        ln2 = rms(mid, "n2")
        z = ln2 @ ws["wgate"].T
        mlp = (z * torch.sigmoid(z) * (ln2 @ ws["wup"].T)) @ ws["wdown"].T
        xi = rms(mid + rms(mlp, "n2b"), "nf")
    xi.backward(gx.double())
    return xi.detach(), x.grad, {n: t.grad for n, t in ws.items()}


def _block(dgm, gpu, cfg, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = {n: torch.randn(N * K, generator=g, device="cuda") / math.sqrt(K) for n, (N, K) in cfg.linear_shapes().items()}
    for n in dgm.DIT_NORMS:
        w[n] = 1.0 + 0.1 * torch.randn(cfg.C, generator=g, device="cuda")
    x = torch.randn(cfg.B * cfg.T, cfg.C, generator=g, device="cuda")
    gx = torch.randn(cfg.B * cfg.T, cfg.C, generator=g, device="cuda") * 1e-2
    torch.cuda.synchronize()
    return dgm.DiTBlock(gpu, cfg, w), w, x, gx


@pytest.mark.parametrize("B,T,C,F,H,bits,group,loops", CFGS)
def test_large_block(dgm, torch_cuda, B, T, C, F, H, bits, group, loops):
    torch = torch_cuda
    cfg = dgm.DiTConfig(B=B, T=T, C=C, F=F, H=H, D=C // H, loops=loops, group=group, bits=bits)
    st = torch.cuda.Stream()
    gpu = dgm.GPU(stream=st)
    try:
        blk, w, x0, gx0 = _block(dgm, gpu, cfg, C + F)
        blk.zero_grads()
        xf, xt, gx = x0.clone(), x0.clone(), gx0.clone()
        torch.cuda.synchronize()
        gpu.begin()
        blk.forward(xf)
        blk.forward_train(xt)
        blk.backward(gx)
        gpu.end()
        assert gpu.workspaceBytes() == 0
        ref, rgx, rg = _reference(dgm, cfg, blk, w, x0, gx0)
        errs = {"x": rel_err(from_dev(xf), ref.cpu()), "x train": rel_err(from_dev(xt), ref.cpu()),
                "gx": rel_err(from_dev(gx), rgx.cpu())}
        errs.update({n: rel_err(from_dev(blk.grads[n]), t.reshape(-1).cpu()) for n, t in rg.items()})
        assert all(e <= 1e-5 for e in errs.values()), errs
        # Captured: the same kernels in the same workspace, so the same bits.
        xc = x0.clone()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st):
            gpu.begin()
            blk.forward(xc)
        for _ in range(3):
            xc.copy_(x0)
            torch.cuda.synchronize()
            with torch.cuda.stream(st):
                graph.replay()
            st.synchronize()
            assert torch.equal(xc, xf)
            xe = x0.clone()
            torch.cuda.synchronize()
            gpu.begin()
            blk.forward(xe)
            gpu.end()
            assert torch.equal(xe, xf)
        del graph
    finally:
        torch.cuda.synchronize()
        gpu.close()


def test_workspace_without_room_for_pieces(dgm, gpu, torch_cuda):
    """The sizes of the pieces before these are still enough."""
    torch = torch_cuda
    from dgm_amd.dit import _ws_sizes
    B, T, C, F, H, bits, group, loops = CFGS[1]
    cfg = dgm.DiTConfig(B=B, T=T, C=C, F=F, H=H, D=C // H, loops=loops, group=group, bits=bits)
    blk, _, x0, _ = _block(dgm, gpu, cfg, 9)
    x1, x2 = x0.clone(), x0.clone()
    gpu.begin()
    blk.forward(x1)
    gpu.end()
    least = sum((n + 63) & ~63 for _, n in _ws_sizes(cfg))
    assert least < blk.ws_floats
    behind = blk.ws[least:].clone()
    blk.ws_floats = least
    blk.ws[least:] = 7.0
    torch.cuda.synchronize()
    gpu.begin()
    blk.forward(x2)
    gpu.end()
    assert bool((blk.ws[least:] == 7.0).all()) and behind.numel() > 0
    assert not torch.equal(x1, x2) and rel_err(from_dev(x1), from_dev(x2)) <= 1e-5
