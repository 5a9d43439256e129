"""Decode forwards of 17 to 64 rows whose K is cut over workgroups
(csrc/gemm_decode.hip): few columns, long K, at the edges of its slices (a last
interval that is not whole, an odd number of intervals, a column block past N,
groups that straddle slices), against the float64 product at the mode's bar.
Where the staging fits the static scratch, dgm_gemmNT_noalloc gives the same
bits; a context whose reserve has no room for the slices' sums keeps K whole."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import from_dev, rel_err, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("math", ["fp32", "bf16"])
@pytest.mark.parametrize("bits,M,N,K,G", [(8, 17, 1000, 14336, 128), (8, 64, 130, 4096 + 1536, 64),
                                          (4, 33, 64, 7 * 4096 + 768, 128), (4, 24, 2050, 8192, 1024),
                                          (8, 40, 4096, 6144, 512)])
def test_sliced_decode(dgm, gpu, orc, math, bits, M, N, K, G):
    import torch
    rng = np.random.default_rng(M + N)
    x = rng.standard_normal(M * K).astype(np.float32)
    q = torch.zeros(N * K // (2 if bits == 4 else 1), dtype=torch.uint8 if bits == 4 else torch.int8, device="cuda")
    s = torch.zeros(N * (K // G), device="cuda")
    bias = rng.standard_normal(N).astype(np.float32)
    gpu.begin()
    gpu.quantize(to_dev((rng.standard_normal(N * K) * 0.02).astype(np.float32)), q, s, N, K, bits, G)
    gpu.end()
    wd = orc.dequant(from_dev(q), from_dev(s), N, K, G, bits).reshape(N, K).astype(np.float64)
    ref = x.reshape(M, K).astype(np.float64) @ wd.T + bias
    xd, bd = to_dev(x), to_dev(bias)
    ys = [torch.full((M * N,), float("nan"), device="cuda") for _ in range(3)]
    mode = dgm.DGM_MATH_FP32 if math == "fp32" else dgm.DGM_MATH_BF16
    cut, whole = (dgm.GPU(stream=torch.cuda.current_stream()) for _ in range(2))
    try:
        whole.reserve(260 * K + 512)     # the pieces, but not the sums of the slices
        held = whole.workspaceBytes()
        for c in (cut, whole):
            c.set_math(mode)
            c.begin()
        cut.gemmNT(bits, None, q, s, xd, bd, ys[0], M, N, K, G)
        whole.gemmNT(bits, None, q, s, xd, bd, ys[1], M, N, K, G)
        cut.gemmNT_noalloc(bits, None, q, s, xd, bd, ys[2], M, N, K, G)
        cut.end()
        whole.end()
        assert whole.workspaceBytes() == held
        for y in ys:
            assert rel_err(from_dev(y).reshape(M, N), ref) <= (1e-5 if math == "fp32" else 1e-2)
        if cut.workspaceBytes() <= dgm.DGM_NOALLOC_SCRATCH_BYTES:
            assert np.array_equal(from_dev(ys[0]).view(np.uint32), from_dev(ys[2]).view(np.uint32))
    finally:
        cut.close()
        whole.close()
