"""The few-row GEMM (rows_gemm.hip) through rt_qlinear_forward and
rt_q4k_gemm_bf16, against float64 products of the oracle's dequantisers: edges
of its row and column tiles, K splits, bias, and weights whose block scales
rise and vanish along a row."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2, to_dev
from test_gemv_any import Q4K, Q6K, Q8_0, weight

pytestmark = pytest.mark.gpu

# Both operands are rounded to f16 (2^-12 relative each, random): about 3e-4 of
# the products' norm, and per element 5 sigma of that.
TOL = 6e-4


def forward(rt, dev, fmt, w, x, n, k, bias=None, bf16=False):
    import torch
    m = x.shape[0]
    out = torch.full((m * n + 64,), -7.0, dtype=torch.float32, device=dev)
    if bf16:
        rt.q4k_gemm(to_dev(x, dev).to(torch.bfloat16), to_dev(w, dev), out, m, n, k)
    else:
        rt.qlinear_forward(fmt, to_dev(w, dev), to_dev(x, dev), out, m, n, k,
                           bias=None if bias is None else to_dev(bias, dev))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.all(got[m * n:] == -7.0)
    return got[:m * n].reshape(m, n)


def check(got, x, w64, bias=0.0):
    ref = x.astype(np.float64) @ w64.T + bias
    mag = np.sqrt((x.astype(np.float64) ** 2) @ (w64 ** 2).T) + np.abs(bias) * 1e-3 + 1e-30
    assert np.max(np.abs(got - ref) / mag) < 5 * TOL
    assert np.linalg.norm(got - ref) / np.linalg.norm(mag) < TOL


@pytest.mark.parametrize("fmt,m,n,k,with_bias", [
    (Q4K, 1, 1, 256, True), (Q4K, 9, 31, 768, False), (Q4K, 32, 10241, 256, True), (Q4K, 33, 2049, 2304, False),
    (Q4K, 65, 6146, 1280, True), (Q4K, 40, 260, 8192, True), (Q4K, 384, 96, 512, False), (Q4K, 385, 96, 512, True),
    (Q6K, 1, 33, 256, True), (Q6K, 40, 70, 4096, True), (Q6K, 100, 1025, 768, False), (Q6K, 384, 40, 1280, True),
    (Q8_0, 2, 31, 64, True), (Q8_0, 33, 130, 192, False), (Q8_0, 40, 36, 4160, True), (Q8_0, 300, 1153, 1152, False),
])
def test_rows_gemm_matches_float64(rt, orc, dev, fmt, m, n, k, with_bias):
    rng = np.random.default_rng(m + n + k)
    w, w64 = weight(rt, orc, fmt, n, k, seed=n + k)
    x = rng.normal(size=(m, k)).astype(np.float32)
    bias = rng.normal(size=n).astype(np.float32) if with_bias else None
    check(forward(rt, dev, fmt, w, x, n, k, bias), x, w64, 0.0 if bias is None else bias.astype(np.float64))
    if fmt == Q4K and not with_bias:
        import torch
        xb = torch.from_numpy(x).to(torch.bfloat16).float().numpy()
        check(forward(rt, dev, fmt, w, xb, n, k, bf16=True), xb, w64)


def test_rows_gemm_rescales_along_k(rt, orc, dev):
    """Q4_K columns whose blocks grow by 2^20 in all, start with zero blocks, or
    are zero throughout: each wave's exponent follows its blocks; rows of A at
    2^100, 2^-100 and zero; a NaN stays in its row."""
    m, n, k = 37, 70, 4096
    w = orc.synth_q4k(3, n, k).reshape(n, k // 256, 144).copy()
    d = np.array([2.0 ** (-14 + 1.3 * b) for b in range(16)], np.float16).view(np.uint16)
    for r in range(n):
        for b in range(16):
            scale = d[b if r % 3 else 15 - b]
            w[r, b, 0:2] = np.array([scale], np.uint16).view(np.uint8)
            w[r, b, 2:4] = np.array([scale], np.uint16).view(np.uint8)
    w[5, :7, 0:4] = 0
    w[6, :, 0:4] = 0
    w64 = orc.q4k_dequant(w.reshape(-1), n, k).reshape(n, k).astype(np.float64)
    x = np.random.default_rng(4).normal(size=(m, k)).astype(np.float32)
    x[1] *= np.float32(2.0 ** 80)
    x[2] *= np.float32(2.0 ** -100)
    x[3] = 0.0
    got = forward(rt, dev, Q4K, w.reshape(-1), x, n, k)
    for r in (0, 1, 2, 36):
        check(got[r:r + 1], x[r:r + 1], w64)
    assert np.all(got[3] == 0.0) and np.all(got[:, 6] == 0.0)
    x[7, 9] = np.nan
    got = forward(rt, dev, Q4K, w.reshape(-1), x, n, k)
    assert np.all(np.isnan(got[7])) and np.all(np.isfinite(np.delete(got, 7, axis=0)))
    a = forward(rt, dev, Q4K, w.reshape(-1), x, n, k)
    assert np.array_equal(a, got, equal_nan=True)
