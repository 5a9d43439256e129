"""Decode forwards whose groups lie inside a block of the f16 kernel
(csrc/gemm_decode.hip): groups of 32, and int4 groups of 64, at the edges of its
row tiles, intervals (the last one not whole), column blocks and slices of K, and
on both sides of where it is taken. The reference is the float64 product of the
same operands. Bound per element, against the row's and column's 2-norms |a| |b|,
which no partial sum exceeds: 2 roundings of a split element, 8 of a group's
partial (two pieces, one each 8 products), 2 of the fold of each of K / 32
groups, 16 for the sums of waves and slices: (26 + K / 16) * 2^-24 |a| |b|."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import from_dev

pytestmark = pytest.mark.gpu


def _operands(gpu, bits, M, N, K, G, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K, generator=g, device="cuda")
    x *= torch.where(torch.rand(K, generator=g, device="cuda") < 1 / 256, 100.0, 1.0)
    w = torch.randn(N, K, generator=g, device="cuda") * 0.02
    bias = torch.randn(N, generator=g, device="cuda")
    q = torch.empty(N * K // (2 if bits == 4 else 1), dtype=torch.uint8, device="cuda")
    s = torch.empty(N * (K // G), device="cuda")
    torch.cuda.synchronize()
    gpu.begin()
    gpu.quantize(w, q, s, N, K, bits, G)
    gpu.end()
    if bits == 8:
        codes = q.view(torch.int8).double()
    else:
        codes = torch.stack([(q << 4).view(torch.int8) >> 4, q.view(torch.int8) >> 4], dim=1).reshape(-1).double()
    wd = (codes.reshape(N, K // G, G) * s.double().reshape(N, K // G, 1)).reshape(N, K)
    return x, bias, q, s, wd


def _within(y, ref, x, wd, K):
    bound = (26 + K / 16) * 2.0 ** -24 * x.double().norm(dim=1)[:, None] * wd.norm(dim=1)[None, :]
    return bool(((y.double() - ref).abs() <= bound + ref.abs() * 2.0 ** -24).all())


SHAPES = [   # bits, M, N, K, G
    (4, 1, 70, 2304, 32), (4, 16, 64, 2048, 64), (4, 17, 130, 4352, 32), (4, 32, 1, 14336, 64),
    (4, 33, 2050, 2560, 32), (4, 64, 1030, 14336, 32), (4, 48, 4100, 4096, 64), (4, 5, 16500, 1024, 32),
    (8, 1, 70, 2176, 32), (8, 16, 64, 2048, 32), (8, 31, 130, 4224, 32), (8, 64, 1030, 14336, 32),
    (8, 49, 2050, 2432, 32), (8, 20, 16500, 1152, 32), (8, 64, 1000, 2048, 32), (4, 16, 1000, 1792, 32),
]


@pytest.mark.parametrize("math", ["fp32", "bf16"])
@pytest.mark.parametrize("bits,M,N,K,G", SHAPES)
def test_groups(dgm, gpu, math, bits, M, N, K, G):
    import torch
    x, bias, q, s, wd = _operands(gpu, bits, M, N, K, G, M + N)
    ref = x.double() @ wd.T + bias.double()
    ys = [torch.full((M, N), float("nan"), device="cuda") for _ in range(3)]
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    a, b = dgm.GPU(stream=st), dgm.GPU(stream=st)
    try:
        for c in (a, b):
            c.set_math(dgm.DGM_MATH_FP32 if math == "fp32" else dgm.DGM_MATH_BF16)
        a.begin()
        a.gemmNT(bits, None, q, s, x, bias, ys[0], M, N, K, G)
        a.gemmNT_noalloc(bits, None, q, s, x, bias, ys[1], M, N, K, G)
        a.end()
        graph = torch.cuda.CUDAGraph()   # a context without staging: the kernels that need none
        with torch.cuda.graph(graph, stream=st):
            b.begin()
            b.gemmNT(bits, None, q, s, x, bias, ys[2], M, N, K, G)
        for _ in range(2):
            ys[2].zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(st):
                graph.replay()
            st.synchronize()
            assert b.workspaceBytes() == 0 and _within(ys[2], ref, x, wd, K)
        del graph
        for y in ys[:2]:
            assert _within(y, ref, x, wd, K)
        if a.workspaceBytes() <= dgm.DGM_NOALLOC_SCRATCH_BYTES:
            assert np.array_equal(from_dev(ys[0]).view(np.uint32), from_dev(ys[1]).view(np.uint32))
    finally:
        torch.cuda.synchronize()
        a.close()
        b.close()


@pytest.mark.parametrize("bits,M,N,K,G", [(4, 20, 100, 2048, 32), (8, 3, 100, 2048, 32), (4, 40, 2100, 2048, 64)])
def test_values(gpu, bits, M, N, K, G):
    """Infinities and NaN land where the products put them; rows of very
    different size keep their own precision; unaligned scales give the product."""
    import torch
    x, bias, q, s, wd = _operands(gpu, bits, M, N, K, G, 5)
    x *= torch.exp2(torch.randint(-90, 60, (M, 1), device="cuda").float())
    x[0, 5], x[1, 40], x[2, 77], x[2, 9] = float("inf"), float("nan"), -float("inf"), float("inf")
    so = torch.zeros(s.numel() + 1, device="cuda")
    so[1:] = s
    ys = [torch.zeros(M, N, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    gpu.begin()
    gpu.gemmNT(bits, None, q, s, x, None, ys[0], M, N, K, G)
    gpu.gemmNT(bits, None, q, so[1:], x, None, ys[1], M, N, K, G)
    gpu.end()
    # Row by row: a product that is all zeros but for the codes' own.
    ref = torch.stack([(x[m].double()[None, :] * wd).sum(dim=1) for m in range(M)])
    for y in ys:
        assert torch.equal(torch.isnan(y), torch.isnan(ref))
        inf = torch.isinf(ref)
        assert torch.equal(torch.isinf(y), inf) and torch.equal(y[inf].double(), ref[inf])
        assert _within(y[3:], ref[3:], x[3:], wd, K) if M > 3 else True


@pytest.mark.parametrize("bits,M,N,K,G", [(4, 20, 100, 2048, 32), (8, 3, 2100, 2048, 32), (4, 40, 2100, 2048, 64),
                                          (8, 64, 1100, 4096, 32)])
@pytest.mark.parametrize("ratio", [1e4, 1e6, 1e8, 1e9, 1e12, 1e30])
def test_outlier_channels_against_zeros(gpu, bits, M, N, K, G, ratio):
    """One channel of each block far above the others meets weights of zero: the
    others are the whole product. Each is held to 2^-20 of itself, or its row is
    computed in fp32: 2^-19 of the result's 2-norm, the sums' 5e-7 within that."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, generator=g, device="cuda")
    w = torch.randn(N, K, generator=g, device="cuda") * 0.02
    x[:, 7::64] *= ratio
    w[:, 7::64] = 0
    q = torch.empty(N * K // (2 if bits == 4 else 1), dtype=torch.uint8, device="cuda")
    s = torch.empty(N * (K // G), device="cuda")
    y = torch.empty(M, N, device="cuda")
    bias = torch.randn(N, generator=g, device="cuda")
    torch.cuda.synchronize()
    gpu.begin()
    gpu.quantize(w, q, s, N, K, bits, G)
    gpu.gemmNT(bits, None, q, s, x, bias, y, M, N, K, G)
    gpu.end()
    codes = q.view(torch.int8).double() if bits == 8 else torch.stack(
        [(q << 4).view(torch.int8) >> 4, q.view(torch.int8) >> 4], dim=1).reshape(-1).double()
    wd = (codes.reshape(N, K // G, G) * s.double().reshape(N, K // G, 1)).reshape(N, K)
    ref = x.double() @ wd.T + bias.double()
    err = float((y.double() - ref).norm() / ref.norm())
    assert err <= 2.0 ** -19, err


@pytest.mark.parametrize("bits,G", [(4, 32), (4, 64), (8, 32)])
def test_sums_of_codes_beyond_fp32(gpu, bits, G):
    """A sum of codes * x over a group may pass fp32's largest number where the
    scale brings the result back: the result is finite."""
    import torch
    M, N, K = 18, 200, 2048
    x, bias, q, s, wd = _operands(gpu, bits, M, N, K, G, 8)
    x[:9] *= 1e35
    y = torch.empty(M, N, device="cuda")
    torch.cuda.synchronize()
    gpu.begin()
    gpu.gemmNT(bits, None, q, s, x, bias, y, M, N, K, G)
    gpu.end()
    ref = x.double() @ wd.T + bias.double()
    assert float(ref.abs().max()) < 3.4e38 and torch.isfinite(y).all()
    assert _within(y, ref, x, wd, K)
