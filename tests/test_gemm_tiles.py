"""The tiled GEMMs at the edges of their tiles, against float64 products: the
256x256 ping-pong kernel on Q4_K (q4k_gemm_pp.hip: partial row and column
tiles, unaligned widths, K splits; its sets and one super-block per row in
test_prefill.py), the half-block and eight-wave kernels, and the 128x128 and
256x256 kernels on widened weights (proj_gemm.hip: one stage, ring remainders,
K splits, bias, narrow outputs of Q4_K)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import to_dev
from test_gemv_any import Q4K, Q6K, Q8_0, weight

pytestmark = pytest.mark.gpu

BF16, F32 = 2, 3
# Both operands are rounded to f16 (2^-12 relative each, random): about 3e-4 of
# the products' norm, and per element 5 sigma of that (6 over 1e7 elements).
TOL = 6e-4


def any_weight(rt, orc, fmt, n, k, seed):
    if fmt in (Q4K, Q6K, Q8_0):
        return weight(rt, orc, fmt, n, k, seed)
    w = (np.random.default_rng(seed).normal(size=(n, k)) * 0.02).astype(np.float32)
    if fmt == F32:
        return w, w.astype(np.float64)
    bits = (w.view(np.uint32) >> 16).astype(np.uint16)
    return bits, (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


@pytest.mark.parametrize("fmt,m,n,k,with_bias", [
    (Q4K, 1300, 6001, 1024, False), (Q4K, 1537, 5120, 256, True), (Q4K, 2305, 3000, 512, False),
    (Q4K, 1100, 1500, 10240, True), (Q4K, 1400, 259, 3584, True), (Q4K, 600, 10241, 768, False),
    (Q4K, 1847, 2146, 3840, True), (Q4K, 601, 4378, 5632, False),
    (BF16, 9, 130, 64, True), (BF16, 129, 127, 128, True), (BF16, 400, 260, 192, False), (BF16, 700, 1021, 4160, True),
    (BF16, 4100, 2050, 320, True), (F32, 1000, 3001, 256, True), (F32, 130, 514, 2048, False),
    (Q6K, 1500, 300, 4608, True), (Q8_0, 2600, 3100, 448, True),
])
def test_tiled_gemm_matches_float64(rt, orc, dev, fmt, m, n, k, with_bias):
    import torch
    w, w64 = any_weight(rt, orc, fmt, n, k, seed=m + n)
    rng = np.random.default_rng(k)
    x = rng.normal(size=(m, k)).astype(np.float32)
    x[m // 2] *= np.float32(2.0 ** 40)
    bias = rng.normal(size=n).astype(np.float32) if with_bias else None
    out = torch.full((m * n + 256,), -7.0, dtype=torch.float32, device=dev)
    xd, wd = to_dev(x, dev), to_dev(w.view(np.int16) if fmt == BF16 else w, dev)
    rt.qlinear_forward(fmt, wd, xd, out, m, n, k, bias=None if bias is None else to_dev(bias, dev))
    torch.cuda.synchronize()
    assert bool((out[m * n:] == -7.0).all())
    got = out[:m * n].view(m, n).double()
    x64, wt = xd.double(), to_dev(w64, dev).T.contiguous()
    ref = x64 @ wt
    mag = torch.sqrt((x64 * x64) @ (wt * wt)) + 1e-30
    if bias is not None:
        ref = ref + to_dev(bias, dev).double()
        mag = mag + 1e-3 * to_dev(bias, dev).double().abs()
    err = (got - ref).abs() / mag
    assert float(err.max()) < 6 * TOL, float(err.max())
    rows = torch.linalg.norm((got - ref) / mag, dim=1) / np.sqrt(n)
    assert float(rows.max()) < 2 * TOL and float(rows.mean()) < TOL
