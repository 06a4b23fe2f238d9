"""Performance cases of the Q4_K / BF16 decode path: what a program that runs
Gemma-3 and FLUX layers on quantised weights asks of the library, each through
the package's public calls.

A case is a dict of plain values; `op` names the call:

  gemv     one linear layer of one token (q4k_gemv, q6k_gemv, q8_0_gemv, bf16_gemv)
  linear   QLinear::forward of m rows with optional bias (qlinear_forward)
  gemm     the FLUX GEMM: bfloat16 rows times a Q4_K weight (q4k_gemm)
  decode   HipDecodeContext.decode_step: one token at position `ctx`
  verify   HipDecodeContext.decode_step_batch: m tokens from position `ctx`
  prefill  HipDecodeContext.prefill of `t` tokens

Weights are made as a quantiser leaves them: bell-shaped codes, scales of one
sign, minima near the middle of the codes' range, a standard deviation of
about 1/sqrt(k).  Everything is made from the seed on the GPU.
"""
from __future__ import annotations

import importlib.util
import math
import pathlib
import sys

import numpy as np
import torch

REPO = pathlib.Path(__file__).resolve().parents[1]
PKG_DIR = REPO / "rich-triplet_amd"


def _package():
    if "rich_triplet_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location("rich_triplet_amd", PKG_DIR / "__init__.py",
                                                      submodule_search_locations=[str(PKG_DIR)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["rich_triplet_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["rich_triplet_amd"]


DEV = "cuda:0"
FORMATS = {"q4k": 1, "bf16": 2, "f32": 3, "q6k": 4, "q8_0": 5}  # RT_LINEAR_*
BYTES_PER_WEIGHT = {"q4k": 144 / 256, "bf16": 2.0, "f32": 4.0, "q6k": 210 / 256, "q8_0": 34 / 32}
K_STEP = {"q4k": 256, "q6k": 256, "q8_0": 64, "bf16": 64, "f32": 64}

# Gemma-3-4B (Config4::gemma3_4b) and the widths of the gemma3_1b preset; the
# 1B's hidden width is not whole super-blocks, so its files hold Q8_0 there.
MODELS = {
    "4b": dict(hidden=2560, ffn=10240, n_q_heads=8, n_kv_heads=4, head_dim=256, sliding_window=1024, global_every=6),
    "1b": dict(hidden=1152, ffn=6912, n_q_heads=4, n_kv_heads=1, head_dim=256, sliding_window=512, global_every=6),
}
ROPE = dict(rope_theta_local=10000.0, rope_theta_global=1000000.0, rope_fs_local=1.0, rope_fs_global=0.125, eps=1e-6,
            attn_scale=1.0 / 16.0)
# Projection formats of a layer, by the file's quantisation.
LAYOUTS = {
    "q4_k_s": dict(q="q4k", k="q4k", v="q4k", o="q4k", gate="q4k", up="q4k", down="q4k"),
    "q4_k_m": dict(q="q4k", k="q4k", v="q6k", o="q4k", gate="q4k", up="q4k", down="q6k"),
    "q8_0": dict(q="q8_0", k="q8_0", v="q8_0", o="q4k", gate="q8_0", up="q8_0", down="q6k"),
}
VOCAB = 262144


def listed():
    return [
        # a token's smallest projection (Gemma-3-4B attention output): launch and latency
        dict(name="gemv_o_4b", op="gemv", fmt="q4k", n=2560, k=2048),
        # a token's FFN up projection at the widths of Gemma-3-12B
        dict(name="gemv_up_12b", op="gemv", fmt="q4k", n=15360, k=3840),
        # the Q6_K down projection of a Q4_K_M file
        dict(name="gemv_q6k_down_4b", op="gemv", fmt="q6k", n=2560, k=10240),
        # a short prompt (a chat turn of 40 tokens) through the FFN gate
        dict(name="linear_q4k_turn", op="linear", fmt="q4k", m=40, n=10240, k=2560, bias=False),
        # an ordinary prompt through a Q8_0 FFN at the 1B widths
        dict(name="linear_q8_0_prompt", op="linear", fmt="q8_0", m=300, n=6912, k=1152, bias=False),
        # a BF16 linear with bias over a thousand image and text tokens (FLUX attention projection)
        dict(name="linear_bf16_bias", op="linear", fmt="bf16", m=1000, n=3072, k=3072, bias=True),
        # the FFN gate of a 512-token prompt, bfloat16 rows
        dict(name="gemm_512", op="gemm", m=512, n=10240, k=2560),
        # the FLUX MLP-up GEMM at 1024x1024 images (4096 image + 512 text tokens)
        dict(name="gemm_flux_up", op="gemm", m=4608, n=12288, k=3072),
        # generation with Gemma-3-4B at a 4,000-token context: every layer and the tied lm_head
        dict(name="decode_4b", op="decode", model="4b", layout="q4_k_s", layers=34, vocab=VOCAB, ctx=4001),
        # generation with the 1B widths, a short chat
        dict(name="decode_1b", op="decode", model="1b", layout="q8_0", layers=26, vocab=VOCAB, ctx=700),
        # speculative verification of 5 tokens through one local/global period of a Q4_K_M file
        dict(name="verify_4b", op="verify", model="4b", layout="q4_k_m", layers=6, vocab=1000, m=5, ctx=1500),
        # a long prompt through one local/global period of Gemma-3-4B
        dict(name="prefill_4b", op="prefill", model="4b", layout="q4_k_s", layers=6, vocab=1000, t=4096, sliding=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _multiple(rng, lo, hi, step):
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    op = rng.choice(["gemv", "gemv", "linear", "linear", "linear", "gemm", "gemm", "decode", "verify", "prefill"])
    if op == "gemv":
        fmt = rng.choice(["q4k", "q4k", "q6k", "q8_0", "bf16"])
        return dict(op=op, fmt=fmt, n=_log(rng, 200, 40000), k=_multiple(rng, 512, 16384, K_STEP[fmt]))
    if op == "linear":
        fmt = rng.choice(["q4k", "q4k", "q6k", "q8_0", "bf16", "f32"])
        return dict(op=op, fmt=fmt, m=_log(rng, 1, 2000), n=_log(rng, 200, 12000),
                    k=_multiple(rng, 512, 12288, K_STEP[fmt]), bias=rng.random() < 0.3)
    if op == "gemm":
        return dict(op=op, m=_log(rng, 1, 4608), n=_log(rng, 200, 12288), k=_multiple(rng, 512, 3072, 256))
    model = rng.choice(["4b", "4b", "1b"])
    layout = "q8_0" if model == "1b" else rng.choice(["q4_k_s", "q4_k_m"])
    base = dict(op=op, model=model, layout=layout, layers=rng.choice([2, 4, 6]), vocab=1000 * rng.randint(1, 60))
    if op == "decode":
        return dict(base, ctx=_log(rng, 1, 8000))
    if op == "verify":
        return dict(base, m=rng.randint(2, 8), ctx=_log(rng, 1, 8000))
    return dict(base, t=_log(rng, 4, 4000), sliding=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed, *tag):
    h = int(seed) & 0x7FFFFFFF
    for t in tag:
        h = (h * 1000003 + int(t) + 1) & 0x7FFFFFFFFFFF
    return torch.Generator(device=DEV).manual_seed(h)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _ints(g, lo, hi, *shape):
    return torch.randint(lo, hi, shape, generator=g, device=DEV, dtype=torch.int32)


def _block_scale(g, nb, codes_std, k):
    """One f16 scale per block: a lognormal factor times what gives weights of
    standard deviation 1/sqrt(k) at codes of codes_std (scales included)."""
    return (torch.exp(0.2 * _randn(g, nb)) / (codes_std * math.sqrt(k))).to(torch.float16)


def _q4k(g, n, k):
    """(blocks, parts): 144-byte Q4_K blocks and the fields they hold."""
    nb = n * (k // 256)
    q = torch.round(7.5 + 2.7 * _randn(g, nb, 256)).clamp_(0, 15).to(torch.uint8)
    sv = _ints(g, 24, 64, nb, 8)
    mv = (sv + _ints(g, -2, 3, nb, 8)).clamp(0, 63)
    d = _block_scale(g, nb, 2.7 * 44.0, k)
    dmin = (7.5 * d.float()).to(torch.float16)
    out = torch.empty(nb, 144, dtype=torch.uint8, device=DEV)
    out[:, 0:2] = d.view(torch.uint8).view(nb, 2)
    out[:, 2:4] = dmin.view(torch.uint8).view(nb, 2)
    out[:, 4:8] = (sv[:, :4] | ((sv[:, 4:] >> 4) << 6)).to(torch.uint8)
    out[:, 8:12] = (mv[:, :4] | ((mv[:, 4:] >> 4) << 6)).to(torch.uint8)
    out[:, 12:16] = ((sv[:, 4:] & 15) | ((mv[:, 4:] & 15) << 4)).to(torch.uint8)
    c = q.view(nb, 4, 2, 32)
    out[:, 16:] = (c[:, :, 0] | (c[:, :, 1] << 4)).reshape(nb, 128)
    return out.view(-1), (q, sv, mv, d, dmin)


def _q6k(g, n, k):
    nb = n * (k // 256)
    q = torch.round(32.0 + 10.0 * _randn(g, nb, 256)).clamp_(0, 63).to(torch.uint8)
    sc = _ints(g, 40, 120, nb, 16) * (1 - 2 * _ints(g, 0, 2, nb, 16))
    d = _block_scale(g, nb, 10.0 * 83.0, k)
    c = q.view(nb, 2, 4, 32)  # half, quarter of the half, element
    lo, hi = c & 15, c >> 4
    ql = torch.cat([lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)], dim=2).reshape(nb, 128)
    qh = (hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)).reshape(nb, 64)
    planes = [ql.reshape(-1), qh.reshape(-1), sc.to(torch.int8).view(torch.uint8).reshape(-1), d.view(torch.uint8)]
    return torch.cat(planes), (q, sc, d)


def _q8_0(g, n, k):
    nb = n * (k // 32)
    q = torch.round(45.0 * _randn(g, nb, 32)).clamp_(-127, 127).to(torch.int8)
    d = _block_scale(g, nb, 45.0, k)
    return torch.cat([q.view(torch.uint8).reshape(-1), d.view(torch.uint8)]), (q, d)


def _weight(fmt, g, n, k):
    if fmt == "q4k":
        return _q4k(g, n, k)
    if fmt == "q6k":
        return _q6k(g, n, k)
    if fmt == "q8_0":
        return _q8_0(g, n, k)
    w = _randn(g, n, k) / math.sqrt(k)
    w = w.to(torch.bfloat16) if fmt == "bf16" else w
    return w, (w,)


def _weight64(fmt, parts, n, k):
    """The weight's values in 64 bits."""
    if fmt == "q4k":
        q, sv, mv, d, dmin = parts
        s = d.double()[:, None] * sv.double()
        m = dmin.double()[:, None] * mv.double()
        return (q.view(-1, 8, 32).double() * s[:, :, None] - m[:, :, None]).view(n, k)
    if fmt == "q6k":
        q, sc, d = parts
        s = d.double()[:, None] * sc.double()
        return ((q.view(-1, 16, 16).double() - 32.0) * s[:, :, None]).view(n, k)
    if fmt == "q8_0":
        q, d = parts
        return (q.double() * d.double()[:, None]).view(n, k)
    return parts[0].double()


def _layer_shapes(m):
    h, f, d = m["hidden"], m["ffn"], m["head_dim"]
    qd, kvd = m["n_q_heads"] * d, m["n_kv_heads"] * d
    return dict(q=(qd, h), k=(kvd, h), v=(kvd, h), o=(h, qd), gate=(f, h), up=(f, h), down=(h, f))


def _layer(case, seed, i):
    """Layer i: packed projections and norm vectors, and the projections' fields."""
    m, lay = MODELS[case["model"]], LAYOUTS[case["layout"]]
    packed, parts = {}, {}
    for j, (name, (n, k)) in enumerate(_layer_shapes(m).items()):
        packed[name], parts[name] = _weight(lay[name], _gen(seed, 10 + i, j), n, k)
    g = _gen(seed, 10 + i, 50)
    for name in ("in_norm", "post_attn_norm", "pre_ffn_norm", "post_ffn_norm"):
        packed[name] = 0.1 * _randn(g, m["hidden"])
    for name in ("q_norm", "k_norm"):
        packed[name] = 0.1 * _randn(g, m["head_dim"])
    return packed, parts


def _cache_rows(case, seed, i):
    """The K and V rows of the tokens before this call: normalised, rotated
    keys have components of about 1."""
    m = MODELS[case["model"]]
    g = _gen(seed, 10 + i, 60)
    kvd = m["n_kv_heads"] * m["head_dim"]
    return _randn(g, case["ctx"], kvd), _randn(g, case["ctx"], kvd)


def _embedding(case, seed):
    g = _gen(seed, 5)
    h = MODELS[case["model"]]["hidden"]
    e = torch.empty(case["vocab"], h, dtype=torch.bfloat16, device=DEV).normal_(0.0, 0.03, generator=g)
    return e, 0.1 * _randn(g, h)


def _tokens(case, seed):
    count = {"decode": 1, "verify": case.get("m"), "prefill": case.get("t")}[case["op"]]
    g = torch.Generator().manual_seed(int(seed) & 0x7FFFFFFF)
    return torch.randint(0, case["vocab"], (count,), generator=g).numpy().astype(np.int32)


def _activations(case, seed):
    """Rows as a norm or an activation leaves them: about N(0, 1), a few large channels."""
    m, k = case.get("m", 1), case["k"]
    g = _gen(seed, 2)
    gain = torch.exp(0.3 * _randn(g, k))
    return _randn(g, m, k) * gain


class _DeviceRows:
    """Rows of a context's K or V cache, as memory that torch can view; a view
    keeps this object, and so the context that owns the memory."""

    def __init__(self, ctx, ptr, shape):
        self.ctx = ctx
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f4", data=(ptr, False), version=2)


def _context(case, seed):
    rt = _package()
    m, op = MODELS[case["model"]], case["op"]
    first = 0 if op == "prefill" else case["ctx"]
    count = {"decode": 1, "verify": case.get("m"), "prefill": case.get("t")}[op]
    cfg = dict(m, n_layers=case["layers"], vocab=case["vocab"], **ROPE)
    ctx = rt.HipDecodeContext(cfg, first + count + 8)
    lay = {p: FORMATS[f] for p, f in LAYOUTS[case["layout"]].items()}
    kvd = m["n_kv_heads"] * m["head_dim"]
    for i in range(case["layers"]):
        packed, _ = _layer(case, seed, i)
        kv = _cache_rows(case, seed, i) if first else None
        torch.cuda.synchronize()  # the context works on its own stream
        ctx.set_layer(i, packed, formats=lay)
        if first:
            ctx.sync_kv_from_cpu(i, kv[0], kv[1], first)
    embed, final_norm = _embedding(case, seed)
    torch.cuda.synchronize()
    ctx.set_embed(embed, final_norm)
    rows = {}
    for i in range(case["layers"])[-31:]:  # the rows this call writes
        for name, p in zip("kv", ctx.kv_ptrs(i)):
            rows["%s%02d" % (name, i)] = torch.as_tensor(_DeviceRows(ctx, p + first * kvd * 4, (count, kvd)), device=DEV)
    ctx.synchronize()
    return dict(case=case, ctx=ctx, tokens=_tokens(case, seed), rows=rows)


def prepare(case, seed):
    rt = _package()
    if case["op"] in ("decode", "verify", "prefill"):
        return _context(case, seed)
    m, n, k = case.get("m", 1), case["n"], case["k"]
    w, _ = _weight(case.get("fmt", "q4k"), _gen(seed, 1), n, k)
    x = _activations(case, seed)
    state = dict(case=case, rt=rt, w=w, x=x.to(torch.bfloat16) if case["op"] == "gemm" else x,
                 y=torch.empty(m, n, device=DEV), bias=None)
    if case.get("bias"):
        state["bias"] = _randn(_gen(seed, 3), n)
    return state


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "decode":
        logits = state["ctx"].decode_step(int(state["tokens"][0]), case["ctx"])
        return dict(state["rows"], logits=logits)
    if op == "verify":
        logits = state["ctx"].decode_step_batch(state["tokens"], case["ctx"])
        return dict(state["rows"], logits=logits)
    if op == "prefill":
        logits = state["ctx"].prefill(state["tokens"], 0, mode=1 if case["sliding"] else 0)
        return dict(state["rows"], logits=logits)
    rt, w, x, y, n, k = state["rt"], state["w"], state["x"], state["y"], case["n"], case["k"]
    if op == "gemv":
        call = dict(q4k=rt.q4k_gemv, q6k=rt.q6k_gemv, q8_0=rt.q8_0_gemv, bf16=rt.bf16_gemv)[case["fmt"]]
        call(w, x, y, n, k)
    elif op == "linear":
        rt.qlinear_forward(FORMATS[case["fmt"]], w, x, y, case["m"], n, k, bias=state["bias"])
    else:
        rt.q4k_gemm(x, w, y, case["m"], n, k)
    return y


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _keys_seen(case, first, count, glob):
    """Sum over the call's rows of the keys each one attends to."""
    w = MODELS[case["model"]]["sliding_window"]
    total = 0
    for r in range(first, first + count):
        lo = 0
        if not glob:
            lo = max(0, r + 1 - w) if case["op"] != "prefill" or case["sliding"] else max(0, first + count - w)
        total += max(0, r + 1 - lo)
    return total


def work(case):
    op = case["op"]
    if op in ("gemv", "linear", "gemm"):
        m, n, k = case.get("m", 1), case["n"], case["k"]
        weight = n * k * BYTES_PER_WEIGHT[case.get("fmt", "q4k")]
        x = m * k * (2 if op == "gemm" else 4)
        return dict(bytes=weight + x + 4 * m * n + (4 * n if case.get("bias") else 0), flops=2.0 * m * n * k)
    m, lay = MODELS[case["model"]], LAYOUTS[case["layout"]]
    count = {"decode": 1, "verify": case.get("m"), "prefill": case.get("t")}[op]
    first = 0 if op == "prefill" else case["ctx"]
    logit_rows = 1 if op == "prefill" else count
    hd, kvd = m["n_q_heads"] * m["head_dim"], m["n_kv_heads"] * m["head_dim"]
    nbytes = case["vocab"] * m["hidden"] * 2 + logit_rows * case["vocab"] * 4
    flops = 2.0 * logit_rows * case["vocab"] * m["hidden"]
    for i in range(case["layers"]):
        glob = i % m["global_every"] == m["global_every"] - 1
        # after the last layer's K and V rows a prompt needs its last row only
        tail = 1 if op == "prefill" and i == case["layers"] - 1 else count
        for name, (n, k) in _layer_shapes(m).items():
            rows = count if name in ("k", "v") else tail
            nbytes += n * k * BYTES_PER_WEIGHT[lay[name]]
            flops += 2.0 * rows * n * k
        keys = _keys_seen(case, first, count, glob) if tail == count else _keys_seen(case, first + count - 1, 1, glob)
        flops += 4.0 * keys * hd
        seen = first + count if glob else min(first + count, m["sliding_window"] + count - 1)
        nbytes += 8 * seen * kvd  # K and V rows, each once
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    # About four times the error measured against exact():
    #   16-bit activation digits, exact integer dots      4.6e-5 (q4k), 3.8e-5 (q6k)
    #   f32 products and sums of unquantised weights      1e-7 to 2e-7
    #   f16 operands of the matrix cores, f32 sums        2.1e-4 (bfloat16 rows), 2.9e-4 (f32 rows)
    #   whole steps: one-token and verify layers 4e-4, prefill layers 8.2e-4, growing with depth
    op, fmt = case["op"], case.get("fmt")
    if op == "gemv":
        return {"rel": 2e-5 if fmt == "bf16" else 2e-4}
    if op == "linear" and case["m"] <= 8 and fmt in ("bf16", "f32"):
        return {"rel": 1e-5}
    if op in ("linear", "gemm"):
        return {"rel": 1.2e-3}
    return {"rel": 3.2e-3 if op == "prefill" else 1.6e-3}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _rms(x, gamma, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * (1.0 + gamma.double())


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _rope(x, pos, theta, fs):
    """NeoX rotation of x [rows, heads, d] at positions pos [rows]."""
    half = x.shape[-1] // 2
    inv = torch.pow(torch.tensor(theta, dtype=torch.float64, device=DEV),
                    -2.0 * torch.arange(half, dtype=torch.float64, device=DEV) / (2 * half))
    a = (pos.double() * fs)[:, None] * inv[None]
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * c - hi * s, lo * s + hi * c], -1)


def _model64(case, seed):
    m, op, eps = MODELS[case["model"]], case["op"], ROPE["eps"]
    lay, shapes = LAYOUTS[case["layout"]], _layer_shapes(m)
    nq, nkv, d, w = m["n_q_heads"], m["n_kv_heads"], m["head_dim"], m["sliding_window"]
    first = 0 if op == "prefill" else case["ctx"]
    tokens = torch.from_numpy(_tokens(case, seed)).long().to(DEV)
    count = tokens.numel()
    embed, final_norm = _embedding(case, seed)
    x = embed[tokens].double() * math.sqrt(m["hidden"])
    pos = torch.arange(first, first + count, device=DEV)
    keys = torch.arange(first + count, device=DEV)
    out = {}
    for i in range(case["layers"]):
        packed, parts = _layer(case, seed, i)

        def proj(name, v):
            return v @ _weight64(lay[name], parts[name], *shapes[name]).T

        glob = i % m["global_every"] == m["global_every"] - 1
        theta, fs = (ROPE["rope_theta_global"], ROPE["rope_fs_global"]) if glob else \
            (ROPE["rope_theta_local"], ROPE["rope_fs_local"])
        xn = _rms(x, packed["in_norm"], eps)
        q = _rope(_rms(proj("q", xn).view(count, nq, d), packed["q_norm"], eps), pos, theta, fs)
        kr = _rope(_rms(proj("k", xn).view(count, nkv, d), packed["k_norm"], eps), pos, theta, fs)
        vr = proj("v", xn).view(count, nkv, d)
        out["k%02d" % i], out["v%02d" % i] = kr.reshape(count, nkv * d), vr.reshape(count, nkv * d)
        if first:
            kc, vc = _cache_rows(case, seed, i)
            kr = torch.cat([kc.double().view(first, nkv, d), kr])
            vr = torch.cat([vc.double().view(first, nkv, d), vr])
        seen = keys[None, :] <= pos[:, None]
        if not glob:
            if op == "prefill" and not case["sliding"]:
                seen &= (keys >= count - w)[None, :]
            else:
                seen &= keys[None, :] > pos[:, None] - w
        att = torch.empty(count, nq, d, dtype=torch.float64, device=DEV)
        for hq in range(nq):
            hk = hq // (nq // nkv)
            s = (q[:, hq] @ kr[:, hk].T.contiguous()) * ROPE["attn_scale"]
            s = torch.softmax(s.masked_fill(~seen, -math.inf), -1)
            att[:, hq] = torch.nan_to_num(s, nan=0.0) @ vr[:, hk]  # a row that sees no key attends to nothing
        x = x + _rms(proj("o", att.view(count, nq * d)), packed["post_attn_norm"], eps)
        xn = _rms(x, packed["pre_ffn_norm"], eps)
        h = _gelu(proj("gate", xn)) * proj("up", xn)
        x = x + _rms(proj("down", h), packed["post_ffn_norm"], eps)
    last = x[-1:] if op == "prefill" else x
    xn = _rms(last, final_norm, eps)
    logits = torch.cat([xn @ e.double().T for e in embed.split(32768)], -1)
    out = {n: v for n, v in out.items() if int(n[1:]) >= case["layers"] - 31}
    out["logits"] = logits if op == "verify" else logits[0]
    return out


def exact(case, seed):
    if case["op"] in ("decode", "verify", "prefill"):
        return _model64(case, seed)
    fmt, n, k = case.get("fmt", "q4k"), case["n"], case["k"]
    _, parts = _weight(fmt, _gen(seed, 1), n, k)
    x = _activations(case, seed)
    x = x.to(torch.bfloat16) if case["op"] == "gemm" else x
    y = x.double() @ _weight64(fmt, parts, n, k).T
    return y + _randn(_gen(seed, 3), n).double() if case.get("bias") else y
