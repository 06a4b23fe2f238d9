"""The any-K Q4_K / Q6_K / Q8_0 GEMV (gemv_any.hip) against float64 products
of the oracle's dequantisers: row lengths and row counts at the edges of its
workgroup shapes, and non-finite activations."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2, to_dev
from test_kquant import synth_q6k, synth_q8_0

pytestmark = pytest.mark.gpu

Q4K, Q6K, Q8_0 = 1, 4, 5


def weight(rt, orc, fmt, n, k, seed):
    """(device bytes, float64 values [n, k])."""
    rng = np.random.default_rng(seed)
    if fmt == Q4K:
        w = orc.synth_q4k(seed, n, k)
        return w, orc.q4k_dequant(w, n, k).reshape(n, k).astype(np.float64)
    if fmt == Q6K:
        w = synth_q6k(rng, n * k // 256)
        return rt.q6k_repack(w), orc.q6k_dequant(w, n * k).reshape(n, k).astype(np.float64)
    w = synth_q8_0(rng, n * k // 32)
    return rt.q8_0_repack(w), orc.q8_0_dequant(w, n * k).reshape(n, k).astype(np.float64)


def gemv(rt, dev, fmt, w, x, n, k):
    import torch
    y = torch.full((n + 64,), -7.0, dtype=torch.float32, device=dev)  # 64 words past the end must stay
    call = {Q4K: rt.q4k_gemv, Q6K: rt.q6k_gemv, Q8_0: rt.q8_0_gemv}[fmt]
    call(to_dev(w, dev), to_dev(x, dev), y, n, k)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.all(got[n:] == -7.0)
    return got[:n]


# The smallest and longest rows the kernel takes and the first one past it
# (the wave-per-row kernel), rows of odd slot counts, one row, row counts one
# off a workgroup's, and counts that take 1, 2 and 4 rows per thread.
@pytest.mark.parametrize("fmt,n,k", [
    (Q4K, 1, 768), (Q4K, 229, 3328), (Q4K, 3841, 3840), (Q4K, 10753, 1280), (Q4K, 193, 15360), (Q4K, 65, 16384),
    (Q4K, 33, 16640),
    (Q6K, 1, 256), (Q6K, 1151, 6912), (Q6K, 9001, 768), (Q6K, 385, 12288), (Q6K, 50, 16384), (Q6K, 9, 16640),
    (Q8_0, 3, 32), (Q8_0, 515, 96), (Q8_0, 6913, 1152), (Q8_0, 1000, 9024), (Q8_0, 40, 16384), (Q8_0, 21, 16416),
])
def test_gemv_any_matches_float64(rt, orc, dev, fmt, n, k):
    w, w64 = weight(rt, orc, fmt, n, k, seed=n + k)
    x = (np.random.default_rng(k).normal(size=k) * np.exp(0.5 * np.random.default_rng(n).normal(size=k))).astype(np.float32)
    x[k // 2] = 0.0
    ref = w64 @ x.astype(np.float64)
    got = gemv(rt, dev, fmt, w, x, n, k)
    # Error of a row: the products' magnitudes times a few f32 roundings (the
    # last digit is 2^-23 of a chunk's bound, at most 2^3 the typical |x|);
    # Q4_K's scaled codes and mins cancel, so both parts count.
    mag = np.sqrt(((np.abs(w64) + (np.abs(w64).max() if fmt == Q4K else 0)) ** 2) @ (x.astype(np.float64) ** 2)) + 1e-30
    assert np.max(np.abs(got - ref) / mag) < 4e-6
    assert rel_l2(got, ref) < 2e-6


@pytest.mark.parametrize("fmt,k", [(Q4K, 1280), (Q6K, 1280), (Q8_0, 1152)])
def test_gemv_any_keeps_non_finite_values(rt, orc, dev, fmt, k):
    """A NaN makes every row NaN; an infinity makes a row non-finite, its
    sign the weight's, and not a number where the weight is zero."""
    n = 70
    w, w64 = weight(rt, orc, fmt, n, k, seed=5)
    x = np.random.default_rng(1).normal(size=k).astype(np.float32)
    x[77] = np.nan
    assert np.all(np.isnan(gemv(rt, dev, fmt, w, x, n, k)))
    x[77] = -np.inf
    got = gemv(rt, dev, fmt, w, x, n, k)
    assert not np.any(np.isfinite(got))
    if fmt != Q4K:  # Q4_K: scale * inf - min * inf, not a number in f32 either
        live = w64[:, 77] != 0
        assert np.array_equal(np.sign(got[live]), -np.sign(w64[live, 77])) and np.all(np.isnan(got[~live]))
    for big in (1e33, 1e-28):  # near both ends of the exponent range
        x[77] = 0.5
        xs = (x * np.float32(big)).astype(np.float32)
        assert rel_l2(gemv(rt, dev, fmt, w, xs, n, k), w64 @ xs.astype(np.float64)) < 2e-6


def q4k_parts(w, n, k):
    """float64 scale * code and min of every weight, [n, k] each: the two sums of
    the reference's integer trick (autograd2.rs:1671-1698)."""
    b = w.reshape(n, k // 256, 144)
    d = b[:, :, 0:2].copy().view(np.float16)[..., 0].astype(np.float64)
    dm = b[:, :, 2:4].copy().view(np.float16)[..., 0].astype(np.float64)
    sc, qs = b[:, :, 4:16].astype(np.int64), b[:, :, 16:].reshape(n, -1, 4, 32)
    sv = np.concatenate([sc[..., 0:4] & 63, (sc[..., 8:12] & 15) | (sc[..., 0:4] >> 6) << 4], -1)
    mv = np.concatenate([sc[..., 4:8] & 63, (sc[..., 8:12] >> 4) | (sc[..., 4:8] >> 6) << 4], -1)
    q = np.stack([qs & 15, qs >> 4], 3).reshape(n, -1, 8, 32).astype(np.float64)
    s, m = (d[..., None] * sv)[..., None], (dm[..., None] * mv)[..., None]
    return (q * s).reshape(n, k), np.broadcast_to(m, q.shape).reshape(n, k)


def q4k_bound(w, x, n, k):
    """What f32 products and sums may differ by: the longest chain of roundings
    from a product to the result (8 of a quarter sub-block, 2 + 2 + 1 to the
    slot, k / 1024 + 4 over the slots, sum x and the last store), 2^-24 each, of
    the sum of the magnitudes that meet in it."""
    sq, m = q4k_parts(w, n, k)
    return (8 + 5 + -(-k // 1024) + 4 + 2) * 2.0 ** -24 * ((np.abs(sq) + np.abs(m)) @ np.abs(x.astype(np.float64)))


@pytest.mark.parametrize("n,k", [(70, 768), (600, 3840), (4000, 1280)])
def test_gemv_any_q4k_keeps_small_activations(rt, orc, dev, n, k):
    """A channel 2^20 times the others, its weights and its sub-blocks' mins zero:
    the rest of its 64 activations keep all their bits."""
    big = 200  # super-block 0, chunk 3, sub-block 6
    w = orc.synth_q4k(9, n, k).reshape(n, k // 256, 144).copy()
    w[:, 0, 16 + 32 * 3 + big - 192] &= 0xF0  # code of the channel
    w[:, 0, 12 + 2] &= 0x0F  # the min of sub-block 6: low bits ...
    w[:, 0, 8 + 2] &= 0x3F   # ... and high bits
    w = w.reshape(-1)
    w64 = orc.q4k_dequant(w, n, k).reshape(n, k).astype(np.float64)
    assert np.all(w64[:, big] == 0.0)
    x = np.random.default_rng(k).normal(size=k).astype(np.float32)
    x[big] = 2.0 ** 20
    got = gemv(rt, dev, Q4K, w, x, n, k)
    rest = x.copy()
    rest[big] = 0.0
    assert np.all(np.abs(got - w64 @ x.astype(np.float64)) <= q4k_bound(w, rest, n, k))


def test_gemv_any_q4k_top_of_the_range(rt, orc, dev):
    """Activations whose products with the codes overflow, and the weight's own
    products do not: finite, and as exact."""
    n, k = 333, 1280
    w = orc.synth_q4k(11, n, k).reshape(-1, 144).copy()
    w[:, 0:4] = (w[:, 0:4].copy().view(np.float16) / np.float16(256)).view(np.uint8)
    w = w.reshape(-1)
    w64 = orc.q4k_dequant(w, n, k).reshape(n, k).astype(np.float64)
    assert np.abs(w64).max() < 0.9
    x = np.random.default_rng(2).normal(size=k).astype(np.float32)
    for at in ([77], [500, 501, 1270]):
        for big in (2e36, 3.3e38):
            y = x.copy()
            y[at] = np.float32(big) / len(at)
            got = gemv(rt, dev, Q4K, w, y, n, k)
            assert np.all(np.abs(got - w64 @ y.astype(np.float64)) <= q4k_bound(w, y, n, k))


@pytest.mark.parametrize("fmt,n,k", [(Q6K, 333, 1280), (Q8_0, 333, 1120)])
def test_gemv_any_top_of_the_range(rt, orc, dev, fmt, n, k):
    """Finite activations up to the largest float, products within range: the
    digits' scale stays finite."""
    if fmt == Q6K:
        b, at, scale = synth_q6k(np.random.default_rng(12), n * k // 256).reshape(-1, 210), 208, 2.0 ** -9
    else:
        b, at, scale = synth_q8_0(np.random.default_rng(12), n * k // 32).reshape(-1, 34), 0, 2.0 ** -5
    b[:, at:at + 2] = (b[:, at:at + 2].copy().view(np.float16) * np.float16(scale)).view(np.uint8)
    w = (rt.q6k_repack if fmt == Q6K else rt.q8_0_repack)(b.reshape(-1))
    w64 = (orc.q6k_dequant if fmt == Q6K else orc.q8_0_dequant)(b.reshape(-1), n * k).reshape(n, k).astype(np.float64)
    assert 0 < np.abs(w64).max() < 0.9
    x = np.random.default_rng(2).normal(size=k).astype(np.float32)
    for at in ([77], [500, 501, 1000]):
        for big in (1.75e38, 3.3e38):
            y = x.copy()
            y[at] = np.float32(big) / len(at)
            ref = w64 @ y.astype(np.float64)
            got = gemv(rt, dev, fmt, w, y, n, k)
            assert np.all(np.isfinite(got))
            # 2^-30 of a chunk's largest x per product, and a few f32 roundings
            assert np.all(np.abs(got - ref) <= 16 * 2.0 ** -24 * (np.abs(w64) @ np.abs(y.astype(np.float64))) +
                          len(at) * 64 * 2.0 ** -30 * big)


@pytest.mark.parametrize("fmt,n,k", [(Q6K, 70, 1280), (Q6K, 9001, 768), (Q8_0, 70, 1120), (Q8_0, 7000, 1152)])
def test_gemv_any_wide_chunks(rt, orc, dev, fmt, n, k):
    """Chunks that four digits of one scale do not cover, in every workgroup
    shape: a channel 2^20 (and 2^8) times the others whose weights are zero, a
    chunk of small values beside it, and a vector below 2^-110.  The others keep
    f32 accuracy: 2^-24 of the sum of the magnitudes for each of 8 products of a
    chain, 2 and 1 to the slot, k / 1024 + 4 over the slots, and the store."""
    rng = np.random.default_rng(13)
    big = k - 40  # in Q8_0's half chunk at the end of 1120
    if fmt == Q6K:
        b = synth_q6k(rng, n * k // 256).reshape(n, k // 256, 210).copy()
        i = big % 256
        j, m, l = i // 128, i % 128 // 32, i % 32
        ql, qh = 64 * j + 32 * (m & 1) + l, 128 + 32 * j + l
        b[:, big // 256, ql] &= 0xF0 if m < 2 else 0x0F
        b[:, big // 256, qh] = b[:, big // 256, qh] & ~np.uint8(3 << 2 * m) | np.uint8(2 << 2 * m)  # code 32: zero
        w, w64 = rt.q6k_repack(b.reshape(-1)), orc.q6k_dequant(b.reshape(-1), n * k)
    else:
        b = synth_q8_0(rng, n * k // 32).reshape(n, k // 32, 34).copy()
        b[:, big // 32, 2 + big % 32] = 0
        w, w64 = rt.q8_0_repack(b.reshape(-1)), orc.q8_0_dequant(b.reshape(-1), n * k)
    w64 = w64.reshape(n, k).astype(np.float64)
    assert np.all(w64[:, big] == 0.0)
    x0 = rng.normal(size=k).astype(np.float32)
    steps = 8 + 2 + 1 + -(-k // 512) + 4 + 1
    for what in ("channel 2^20", "channel 2^8", "small chunk", "small vector"):
        x = x0.copy()
        if what.startswith("channel"):
            x[big] = 2.0 ** 20 if what.endswith("20") else 2.0 ** 8
        elif what == "small chunk":
            x[64:112] *= np.float32(2.0 ** -30)
        else:
            x *= np.float32(2.0 ** -112)
        rest = x.astype(np.float64)
        rest[big] = 0.0
        got = gemv(rt, dev, fmt, w, x, n, k)
        bound = steps * 2.0 ** -24 * (np.abs(w64) @ np.abs(rest)) + k * 2.0 ** -149
        assert np.all(np.abs(got - w64 @ x.astype(np.float64)) <= bound), what


def test_gemv_any_large_lds_from_two_threads(rt, orc, dev):
    """Rows whose staging needs more than 64 KB of LDS, of two lengths, launched by
    two host threads at once: neither takes the other's allowance away."""
    import threading
    import torch
    work = []
    for n, k in ((40, 16384), (64, 14336)):
        w, w64 = weight(rt, orc, Q6K, n, k, seed=k)
        x = np.random.default_rng(n).normal(size=k).astype(np.float32)
        work.append((to_dev(w, dev), to_dev(x, dev), torch.zeros(200, n, device=dev), n, k, w64 @ x.astype(np.float64)))
    errors = []

    def run(w, x, y, n, k, ref):
        try:
            stream = torch.cuda.Stream()
            for i in range(y.shape[0]):
                rt.q6k_gemv(w, x, y[i], n, k, stream=stream)
            stream.synchronize()
        except Exception as e:  # reported by the test's own thread
            errors.append(e)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=run, args=a) for a in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for _, _, y, _, _, ref in work:
        got = y.cpu().numpy()
        assert rel_l2(got[0], ref) < 2e-6 and np.array_equal(got, np.broadcast_to(got[0], got.shape))


def test_gemv_any_large_lds_captured(rt, orc, dev):
    """The first call of that length inside a capture; calls of a shorter length
    between the replays."""
    import torch
    n, k = 40, 16384
    w, w64 = weight(rt, orc, Q8_0, n, k, seed=1)
    ws, ws64 = weight(rt, orc, Q8_0, n, 16000, seed=2)
    x = np.random.default_rng(3).normal(size=k).astype(np.float32)
    wd, xd, y = to_dev(w, dev), to_dev(x, dev), torch.zeros(n, device=dev)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        rt.q8_0_gemv(wd, xd, y, n, k, stream=torch.cuda.current_stream())
    for _ in range(4):
        y.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert rel_l2(y.cpu().numpy(), w64 @ x.astype(np.float64)) < 2e-6
        assert rel_l2(gemv(rt, dev, Q8_0, ws, x[:16000], n, 16000), ws64 @ x[:16000].astype(np.float64)) < 2e-6
