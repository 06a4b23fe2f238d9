"""f32 and bf16 weights times a few activation rows (k_gemv_rows): every split
of K over waves, row remainders of weights and activations, the shortest K,
against float64."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import to_dev

pytestmark = pytest.mark.gpu

BF16, F32 = 2, 3


@pytest.mark.parametrize("fmt", [BF16, F32])
@pytest.mark.parametrize("m,n,k", [
    (1, 1, 8), (2, 3, 520), (3, 5, 4096), (4, 349, 5696), (5, 64, 1032), (6, 1023, 2048), (7, 2561, 4104),
    (8, 8193, 1024), (9, 131, 1096), (1, 40001, 640), (17, 9000, 200),
])
def test_few_rows_match_float64(rt, dev, fmt, m, n, k):
    import torch
    rng = np.random.default_rng(n + k)
    w = rng.normal(size=(n, k)).astype(np.float32)
    bits = w
    if fmt == BF16:
        bits = (w.view(np.uint32) >> 16).astype(np.uint16)
        w = (bits.astype(np.uint32) << 16).view(np.float32)
        bits = bits.view(np.int16)
    x = rng.normal(size=(m, k)).astype(np.float32)
    bias = rng.normal(size=n).astype(np.float32) if n % 2 else None
    out = torch.full((m * n + 64,), -7.0, dtype=torch.float32, device=dev)
    xd, wd = to_dev(x, dev), to_dev(w, dev)
    rt.qlinear_forward(fmt, to_dev(bits, dev), xd, out, m, n, k, bias=None if bias is None else to_dev(bias, dev))
    torch.cuda.synchronize()
    assert bool((out[m * n:] == -7.0).all())
    ref = xd.double() @ wd.double().T
    mag = xd.double().abs() @ wd.double().abs().T
    if bias is not None:
        ref, mag = ref + to_dev(bias, dev).double(), mag + to_dev(bias, dev).double().abs()
    # per lane at most 8 * ceil(K / 512) + 4 chained additions, six of the wave,
    # sixteen of the split and the bias: each rounds to 2^-24 of at most mag
    steps = 8 * -(-k // 512) + 4 + 6 + 16 + 1
    err = (out[:m * n].view(m, n).double() - ref).abs() / mag
    assert float(err.max()) < steps * 2.0 ** -24
