"""The large products on split operands (csrc/gemm_planes.hip): forward, dX and dW.

Sizes sit at the edges of its tiles (128 and 256 rows), stages (16 and 32 of
the contraction) and parts (tiles cut along the contraction), on both sides of
where each is taken. The reference is the float64 product of
the same operands. Bound per element, against the row's and column's 2-norms
|a| |b| (every element of a split operand is within 2^-23 of its value and the
product of the low pieces within 2^-22 at worst, mostly a quarter of both, and a
sum of n products, rounded once per 8, is within n/8 * 2^-24 of |a| |b| at
worst): (2 + n / 8) * 2^-24 |a| |b|.
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inputs(gpu, bits, M, N, K, G, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K, generator=g, device="cuda")
    dy = torch.randn(M, N, generator=g, device="cuda") * 1e-3
    w = torch.randn(N, K, generator=g, device="cuda") * 0.02
    bias = torch.randn(N, generator=g, device="cuda")
    if bits == 32:
        return x, dy, w, None, None, w.double(), bias
    q = torch.empty(N * K // (2 if bits == 4 else 1), dtype=torch.uint8, device="cuda")
    s = torch.empty(N * (K // G), device="cuda")
    torch.cuda.synchronize()
    gpu.begin()
    gpu.quantize(w, q, s, N, K, bits, G)
    gpu.end()
    if bits == 8:
        codes = q.view(torch.int8).double()
    else:
        lo, hi = (q << 4).view(torch.int8) >> 4, q.view(torch.int8) >> 4
        codes = torch.stack([lo, hi], dim=1).reshape(-1).double()
    wd = (codes.reshape(N, K // G, G) * s.double().reshape(N, K // G, 1)).reshape(N, K)
    return x, dy, w, q, s, wd, bias


def _within(got, ref, a, b, n):
    """got against ref = a b^T (a [R, n], b [C, n]), where ref is finite."""
    import torch
    bound = (2 + n / 8) * 2.0 ** -24 * a.norm(dim=1)[:, None] * b.norm(dim=1)[None, :] + 2.0 ** -149
    return bool(((got.double() - ref).abs() <= bound + ref.abs() * 2.0 ** -24).all()) and torch.isfinite(got).all()


SHAPES = [   # bits, M, N, K, G
    (8, 1024, 1024, 1024, 8),       # groups smaller than a stage
    (4, 1025, 1023, 1024, 32),      # one row above a tile, one column below
    (4, 129, 8191, 1024, 64),       # a last tile of one row; odd N
    (32, 1537, 385, 2040, 8),       # a contraction that is no multiple of a stage
    (8, 130, 2050, 4100, 10),       # groups of 10: no vector loads
    (4, 128, 14336, 1026, 18),      # odd row bytes for int4
    (8, 517, 640, 4128, 32),        # few tiles: cut along the contraction
    (4, 2048, 4352, 256, 128),      # whole tiles and a cut last round
    (8, 1000, 1029, 960, 96),       # groups of three stages, an odd number of tiles cut
    (4, 300, 3000, 1056, 32),       # an odd number of stages
    (8, 65, 2700, 4288, 32),        # fewest rows; all three just above their lines
    (32, 67, 2305, 4000, 8),        # forward above its line for a long contraction, dX and dW below theirs
    (4, 641, 1504, 768, 32),        # dX and dW above their line, forward below its
    (8, 96, 8192, 960, 96),         # between those two lines, few rows
]


@pytest.mark.parametrize("bits,M,N,K,G", SHAPES)
def test_products(gpu, bits, M, N, K, G):
    import torch
    x, dy, w, q, s, wd, bias = _inputs(gpu, bits, M, N, K, G, M + N)
    y, dx = (torch.full(sh, float("nan"), device="cuda") for sh in ((M, N), (M, K)))
    dw0 = torch.randn(N, K, device="cuda")
    dw, acc = torch.full((N, K), float("nan"), device="cuda"), dw0.clone()
    torch.cuda.synchronize()
    gpu.begin()
    gpu.gemmNT(bits, w, q, s, x, bias, y, M, N, K, G)
    gpu.gemmDX(bits, w, q, s, dy, dx, M, N, K, G)
    gpu.gemmDW(dy, x, dw, M, N, K)
    gpu.gemmDWAcc(dy, x, acc, M, N, K)
    gpu.end()
    xd, dyd = x.double(), dy.double()
    assert _within(y, xd @ wd.T + bias.double(), xd, wd, K)
    assert _within(dx, dyd @ wd, dyd, wd.T.contiguous(), N)
    ref = dyd.T.contiguous() @ xd
    assert _within(dw, ref, dyd.T.contiguous(), xd.T.contiguous(), M)
    assert _within(acc, ref + dw0.double(), dyd.T.contiguous(), xd.T.contiguous(), M)
    # gemmBwd is the two calls, bitwise.
    dx2, dw2 = torch.empty_like(dx), torch.empty_like(dw)
    gpu.begin()
    gpu.gemmBwd(bits, w, q, s, dy, x, dx2, dw2, M, N, K, G)
    gpu.end()
    assert torch.equal(dx, dx2) and torch.equal(dw, dw2)


@pytest.mark.parametrize("bits,M,N,K,G", [(4, 1024, 1024, 1024, 32), (8, 1000, 1024, 1024, 64), (8, 1024, 1024, 1024, 8),
                                          (32, 1024, 1024, 1024, 8)])
def test_unaligned_buffers(gpu, bits, M, N, K, G):
    """Operands that start 4 bytes past a 16-byte boundary: the split reads
    them element by element, with the same products."""
    import torch
    x, dy, w, q, s, _, _ = _inputs(gpu, bits, M, N, K, G, 3)

    def off(t):
        if t is None:
            return None
        n = 4 // t.element_size()
        raw = torch.zeros(t.numel() + n, dtype=t.dtype, device="cuda")
        raw[n:] = t.reshape(-1)
        return raw[n:]
    outs = []
    for a in ((x, dy, w, q, s), tuple(off(t) for t in (x, dy, w, q, s))):
        y, dx, dw = (torch.full(sh, float("nan"), device="cuda") for sh in ((M, N), (M, K), (N, K)))
        torch.cuda.synchronize()
        gpu.begin()
        gpu.gemmNT(bits, a[2], a[3], a[4], a[0], None, y, M, N, K, G)
        gpu.gemmBwd(bits, a[2], a[3], a[4], a[1], a[0], dx, dw, M, N, K, G)
        gpu.end()
        outs.append((y, dx, dw))
    for a, b in zip(*outs):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("kind", ["nonfinite", "token", "rows", "tiny", "zeros"])
def test_values(gpu, kind):
    """Infinities and NaN land where the products of the operands put them;
    rows of very different size each keep their own precision."""
    import torch
    bits, M, N, K, G = 4, 1030, 1000, 1024, 32
    x, dy, w, q, s, wd, _ = _inputs(gpu, bits, M, N, K, G, 5)
    if kind == "nonfinite":
        x[3, 5], x[7, 9], x[11, 2], dy[4, 6], dy[1029, 999] = float("inf"), -float("inf"), float("nan"), float("inf"), \
            float("nan")
    elif kind == "token":      # a token whose gradients overflowed: every row of dW
        dy[517], x[13] = float("nan"), float("inf")
    elif kind == "rows":
        x *= torch.exp2(torch.randint(-60, 60, (M, 1), device="cuda").float())
        dy *= torch.exp2(torch.randint(-30, 30, (1, N), device="cuda").float())
    elif kind == "tiny":
        x *= 1e-38
        dy *= 1e-6
    else:
        x[5], x[:, 3], dy[8], dy[:, 2] = 0, 0, 0, 0
    y, dx, dw = (torch.full(sh, 7.0, device="cuda") for sh in ((M, N), (M, K), (N, K)))
    torch.cuda.synchronize()
    gpu.begin()
    gpu.gemmNT(bits, w, q, s, x, None, y, M, N, K, G)
    gpu.gemmBwd(bits, w, q, s, dy, x, dx, dw, M, N, K, G)
    gpu.end()
    xd, dyd = x.double(), dy.double()
    for got, a, b, n in ((y, xd, wd, K), (dx, dyd, wd.T.contiguous(), N),
                         (dw, dyd.T.contiguous(), xd.T.contiguous(), M)):
        ref = a @ b.T
        if kind in ("nonfinite", "token"):
            assert torch.equal(torch.isnan(got), torch.isnan(ref))
            inf = torch.isinf(ref)
            assert torch.equal(torch.isinf(got), inf) and torch.equal(got[inf].double(), ref[inf])
            assert not torch.isfinite(ref).all()
            ra, cb = torch.isfinite(a).all(1), torch.isfinite(b).all(1)
            got, ref, a, b = got[ra][:, cb], ref[ra][:, cb], a[ra], b[cb]
        if kind == "tiny":      # results below 2^-126 keep an absolute 2^-149
            assert bool(((got.double() - ref).abs() <= (2 + n / 8) * 2.0 ** -24 * a.norm(dim=1)[:, None] *
                         b.norm(dim=1)[None, :] + 2.0 ** -148).all())
        else:
            assert _within(got, ref, a, b, n)


# 2-norm of the error over that of the result where an element far below its
# row's largest carries the sum. It is held to 2^-20 of itself (or its row goes to
# the fp32 kernel): 2^-19 for one such operand with the product of the low pieces,
# 2^-18 for two, the sums' own 5e-7 within that.
FAR_ONE, FAR_BOTH = 2.0 ** -19, 2.0 ** -18


@pytest.mark.parametrize("bits,G", [(4, 32), (8, 8), (32, 8)])
@pytest.mark.parametrize("ratio", [1e4, 1e6, 1e8, 1e9, 1e12, 1e30])
def test_outlier_channel_against_zeros(gpu, bits, G, ratio):
    """One channel of X (one output of dY) far above the others meets weights of
    zero: the others are the whole product and keep their precision."""
    import torch
    M, N, K = 512, 1536, 1024
    g = torch.Generator(device="cuda").manual_seed(3)
    x, dy = torch.randn(M, K, generator=g, device="cuda"), torch.randn(M, N, generator=g, device="cuda")
    w = torch.randn(N, K, generator=g, device="cuda") * 0.02
    x[:, 100] *= ratio
    dy[:, 7] *= ratio
    w[:, 100] = 0
    w[7] = 0
    q = s = None
    wd = w.double()
    if bits != 32:
        q = torch.empty(N * K // (2 if bits == 4 else 1), dtype=torch.uint8, device="cuda")
        s = torch.empty(N * (K // G), device="cuda")
        torch.cuda.synchronize()
        gpu.begin()
        gpu.quantize(w, q, s, N, K, bits, G)
        gpu.end()
        codes = q.view(torch.int8).double() if bits == 8 else torch.stack(
            [(q << 4).view(torch.int8) >> 4, q.view(torch.int8) >> 4], dim=1).reshape(-1).double()
        wd = (codes.reshape(N, K // G, G) * s.double().reshape(N, K // G, 1)).reshape(N, K)
    y, dx = torch.empty(M, N, device="cuda"), torch.empty(M, K, device="cuda")
    torch.cuda.synchronize()
    gpu.begin()
    gpu.gemmNT(bits, w, q, s, x, None, y, M, N, K, G)
    gpu.gemmDX(bits, w, q, s, dy, dx, M, N, K, G)
    gpu.end()
    for got, ref in ((y, x.double() @ wd.T), (dx, dy.double() @ wd)):
        err = float((got.double() - ref).norm() / ref.norm())
        assert err <= FAR_ONE, err


@pytest.mark.parametrize("nonzero", [2, 15, 17, 200])
def test_rows_of_mostly_zeros(gpu, nonzero):
    """Zeros are not counted among the elements that a few small ones may hide in:
    one huge element and a few others, the huge one against zeros."""
    import torch
    M, N, K = 512, 1700, 1003
    g = torch.Generator(device="cuda").manual_seed(nonzero)
    x, w = torch.zeros(M, K, device="cuda"), torch.randn(N, K, generator=g, device="cuda")
    for i in range(1, nonzero):
        x[torch.arange(M, device="cuda"), torch.randint(1, K, (M,), generator=g, device="cuda")] = 1.0 + i / 7
    x[:, 0] = 1e12
    w[:, 0] = 0
    y = torch.empty(M, N, device="cuda")
    torch.cuda.synchronize()
    gpu.begin()
    gpu.gemmNT(32, w, None, None, x, None, y, M, N, K, 8)
    gpu.end()
    ref = x.double() @ w.double().T
    err = float((y.double() - ref).norm() / ref.norm())
    assert err <= FAR_ONE, err


@pytest.mark.parametrize("spread", [8, 16, 24, 40, 60])
def test_tokens_scaled_against_each_other(gpu, spread):
    """Tokens whose X is 2^s as large and whose dY is 2^-s: every product of dW
    matters alike, however far the elements lie below their column's largest."""
    import torch
    M, N, K = 1024, 1024, 1024
    g = torch.Generator(device="cuda").manual_seed(spread)
    x, dy = torch.randn(M, K, generator=g, device="cuda"), torch.randn(M, N, generator=g, device="cuda")
    f = torch.exp2(torch.randint(0, spread + 1, (M, 1), generator=g, device="cuda").float())
    x, dy = x * f, dy / f
    dw = torch.empty(N, K, device="cuda")
    torch.cuda.synchronize()
    gpu.begin()
    gpu.gemmDW(dy, x, dw, M, N, K)
    gpu.end()
    ref = dy.double().T.contiguous() @ x.double()
    err = float((dw.double() - ref).norm() / ref.norm())
    assert err <= FAR_BOTH, err


@pytest.mark.parametrize("bits,G", [(4, 32), (8, 8), (32, 8)])
@pytest.mark.parametrize("spread", [16, 24, 60])
def test_outputs_scaled_against_each_other(gpu, bits, G, spread):
    """The same along the contraction of dX: rows of W 2^s as large (their
    codes' scales, for quantized weights), outputs of dY 2^-s."""
    import torch
    M, N, K = 512, 1536, 1024
    g = torch.Generator(device="cuda").manual_seed(spread)
    f = torch.exp2(torch.randint(0, spread + 1, (N,), generator=g, device="cuda").float())
    w = torch.randn(N, K, generator=g, device="cuda") * f[:, None]
    dy = torch.randn(M, N, generator=g, device="cuda") / f
    q = s = None
    wd = w.double()
    if bits != 32:
        q = torch.empty(N * K // (2 if bits == 4 else 1), dtype=torch.uint8, device="cuda")
        s = torch.empty(N * (K // G), device="cuda")
        torch.cuda.synchronize()
        gpu.begin()
        gpu.quantize(w, q, s, N, K, bits, G)
        gpu.end()
        codes = q.view(torch.int8).double() if bits == 8 else torch.stack(
            [(q << 4).view(torch.int8) >> 4, q.view(torch.int8) >> 4], dim=1).reshape(-1).double()
        wd = (codes.reshape(N, K // G, G) * s.double().reshape(N, K // G, 1)).reshape(N, K)
    dx = torch.empty(M, K, device="cuda")
    torch.cuda.synchronize()
    gpu.begin()
    gpu.gemmDX(bits, w, q, s, dy, dx, M, N, K, G)
    gpu.end()
    ref = dy.double() @ wd
    err = float((dx.double() - ref).norm() / ref.norm())
    assert err <= FAR_BOTH, err


def test_buffer_capture_and_streams(dgm, gpu, torch_cuda):
    """Calls that alternate between two streams give the same product; a
    captured call, dgm_gemmNT_noalloc and a context that reserved less than
    the planes take the kernels that stage nothing, and nothing is allocated."""
    torch = torch_cuda
    bits, M, N, K, G = 8, 1024, 2048, 1024, 32
    x, _, w, q, s, wd, _ = _inputs(gpu, bits, M, N, K, G, 9)
    ref = x.double() @ wd.T
    st = [torch.cuda.Stream(), torch.cuda.Stream()]
    ys = [torch.zeros(M, N, device="cuda") for _ in range(8)]
    torch.cuda.synchronize()
    g = dgm.GPU(stream=st[0])
    try:
        assert g.workspaceBytes() == 0
        g.reserve(64 << 20)
        held = g.workspaceBytes()
        g.begin()
        for i, y in enumerate(ys):      # each stream's call uses the one plane buffer
            g.set_stream(st[i % 2])
            g.gemmNT(bits, w, q, s, x, None, y, M, N, K, G)
        g.end()
        torch.cuda.synchronize()
        assert g.workspaceBytes() == held
        for y in ys:
            assert _within(y, ref, x.double(), wd, K) and torch.equal(y, ys[0])
        g.set_stream(st[0])
        yc = torch.zeros(M, N, device="cuda")
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st[0]):
            g.begin()
            g.gemmNT(bits, w, q, s, x, None, yc, M, N, K, G)
        for _ in range(3):
            yc.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(st[0]):
                graph.replay()
            g.begin()
            g.gemmNT(bits, w, q, s, x, None, ys[0], M, N, K, G)
            g.end()
            st[0].synchronize()
            assert _within(yc, ref, x.double(), wd, K)
        yn = torch.zeros(M, N, device="cuda")
        torch.cuda.synchronize()
        g.begin()
        g.gemmNT_noalloc(bits, w, q, s, x, None, yn, M, N, K, G)
        g.end()
        assert torch.equal(yn, yc)
        assert g.workspaceBytes() == held
        small = dgm.GPU(stream=st[0])
        small.reserve(2 * M * K)     # less than the pieces
        held = small.workspaceBytes()
        ys[1].zero_()
        torch.cuda.synchronize()
        small.begin()
        small.gemmNT(bits, w, q, s, x, None, ys[1], M, N, K, G)
        small.end()
        assert torch.equal(ys[1], yc) and not torch.equal(ys[0], yc) and small.workspaceBytes() == held
        small.close()
        del graph
    finally:
        torch.cuda.synchronize()
        g.close()


@pytest.mark.parametrize("mib", [1, 5, 8, 20, 24, 64])
@pytest.mark.parametrize("bits,M,N,K,G", [(8, 2048, 256, 2048, 32), (4, 1024, 1024, 1024, 32), (32, 2048, 384, 1024, 8)])
def test_pair_under_a_reserve(dgm, torch_cuda, mib, bits, M, N, K, G):
    """gemmBwd is bitwise the two calls also where the reserve holds the pieces
    of neither product, of one, of each but not of both, or of both."""
    torch = torch_cuda
    c = dgm.GPU(stream=torch.cuda.current_stream())
    try:
        x, dy, w, q, s, _, _ = _inputs(c, bits, M, N, K, G, 4)
        c.reserve(mib << 20)
        outs = [[torch.zeros(sh, device="cuda") for sh in ((M, K), (N, K))] for _ in range(2)]
        torch.cuda.synchronize()
        c.begin()
        c.gemmDX(bits, w, q, s, dy, outs[0][0], M, N, K, G)
        c.gemmDW(dy, x, outs[0][1], M, N, K)
        c.gemmBwd(bits, w, q, s, dy, x, *outs[1], M, N, K, G)
        c.end()
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    finally:
        c.close()


def test_buffer_doubles(dgm, torch_cuda):
    """The buffer of the pieces at least doubles when it grows, as the workspace
    does, so that what it keeps until the context goes is less than what it
    uses, however many sizes a program runs through."""
    torch = torch_cuda
    c = dgm.GPU(stream=torch.cuda.current_stream())
    try:
        sizes = []
        for M in (32768, 33792, 34816):
            x, w = torch.ones(M, 4096, device="cuda"), torch.ones(2048, 4096, device="cuda")
            y = torch.empty(M, 2048, device="cuda")
            torch.cuda.synchronize()
            c.begin()
            c.gemmNT(32, w, None, None, x, None, y, M, 2048, 4096, 8)
            c.end()
            assert bool((y == 4096).all())
            sizes.append(c.workspaceBytes())
        assert sizes[0] > 256 << 20 and sizes[1] >= 2 * sizes[0] and sizes[2] == sizes[1]
    finally:
        c.close()


def test_codes_of_one_plane_take_half(dgm, torch_cuda):
    """A forward whose codes are kept as one plane takes 2 bytes for each, not the
    4 of two planes (scales and X come to less than another byte here)."""
    torch = torch_cuda
    M, N, K, G = 128, 14336, 4096, 128
    c = dgm.GPU(stream=torch.cuda.current_stream())
    try:
        x, _, w, q, s, wd, _ = _inputs(c, 4, M, N, K, G, 2)
        y = torch.empty(M, N, device="cuda")
        torch.cuda.synchronize()
        c.begin()
        c.gemmNT(4, w, q, s, x, None, y, M, N, K, G)
        c.end()
        assert _within(y, x.double() @ wd.T, x.double(), wd, K)
        assert c.workspaceBytes() < 3 * N * K
    finally:
        c.close()


def test_time_of_nonfinite(dgm, torch_cuda):
    """A token of NaN gradients flags every row of dW and one of dX. The call
    then takes what the fp32 MFMA kernels take for all of it (a context whose
    reserve leaves no room for the pieces runs those), not a multiple: less
    than three times that."""
    torch = torch_cuda
    M, N, K, G = 2048, 2048, 2048, 32
    st = torch.cuda.Stream()
    a, b = dgm.GPU(stream=st), dgm.GPU(stream=st)
    try:
        x, dy, w, q, s, _, _ = _inputs(a, 8, M, N, K, G, 21)
        dx, dw = torch.empty(M, K, device="cuda"), torch.empty(N, K, device="cuda")
        dy[100] = float("nan")
        b.reserve(1 << 20)
        torch.cuda.synchronize()

        def us(g):
            times = []
            for _ in range(4):
                e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
                g.begin()
                e[0].record(st)
                g.gemmBwd(8, w, q, s, dy, x, dx, dw, M, N, K, G)
                e[1].record(st)
                g.end()
                times.append(e[0].elapsed_time(e[1]) * 1e3)
            return min(times[1:])
        fp32 = us(b)
        assert torch.isnan(dw).all()
        dw.zero_()
        torch.cuda.synchronize()
        pieces = us(a)
        assert torch.isnan(dw).all() and int(torch.isnan(dx).sum()) == K
        print(f"fp32 kernels {fp32:.0f} us, pieces with a NaN token {pieces:.0f} us")
        assert pieces < 3 * fp32
    finally:
        torch.cuda.synchronize()
        a.close()
        b.close()
