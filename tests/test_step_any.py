"""The decode step of shapes without fused templates (gemv_any.hip) against the
oracle, per mix of projection formats: sets that share a format (one launch
with the norm in front), a v of another format, and sets of mixed or BF16
formats behind a prologue of their own."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2
from test_kquant import apply_formats, mixed_ctx

pytestmark = pytest.mark.gpu

BF16, Q6K, Q8_0 = 2, 4, 5


# hidden 768: 24 Q8_0 slots per row (workgroups that hold rows of two
# matrices); hidden 3840 (Gemma-3-12B's): 1024-thread workgroups of q|k|v; ffn
# 15360: a down projection that stages more than 64 KB, captured
@pytest.mark.parametrize("hidden,ffn,heads,kv,plan", [
    (768, 1536, (4, 128), 2, {}),
    (768, 1536, (4, 128), 2, {p: Q6K for p in ("q", "k", "v", "o", "gate", "up", "down")}),
    (768, 1536, (4, 128), 2, {p: Q8_0 for p in ("q", "k", "v", "o", "gate", "up", "down")}),
    (768, 1536, (4, 128), 1, dict(v=Q6K, o=BF16, gate=Q8_0, down=Q8_0)),
    (768, 1536, (2, 256), 2, dict(q=BF16, k=BF16, v=BF16, gate=BF16, up=BF16, down=BF16)),
    (3840, 4096, (16, 256), 8, dict(v=Q6K, down=Q6K)),
    (768, 15360, (4, 128), 2, dict(down=Q6K)),
])
def test_step_any_matches_oracle(rt, orc, hidden, ffn, heads, kv, plan):
    from test_oracle import make_model
    cfg = dict(hidden=hidden, ffn=ffn, n_q_heads=heads[0], n_kv_heads=kv, head_dim=heads[1], n_layers=3, vocab=777,
               sliding_window=9, global_every=3, rope_theta_local=10000.0, rope_theta_global=1000000.0,
               rope_fs_local=1.0, rope_fs_global=0.125, eps=1e-6, attn_scale=1.0 / np.sqrt(heads[1]))
    pos, max_seq = 21, 40
    layers, embed, fnorm = make_model(orc, cfg, max_seq=max_seq, ctx=pos, seed=hidden + len(plan))
    dev_layers, fmts = apply_formats(orc, cfg, layers, {i: dict(plan) for i in range(3)}, seed=7)
    d = mixed_ctx(rt, cfg, dev_layers, fmts, embed, fnorm, pos, max_seq, layers)
    got = d.decode_step(19, pos)
    ref = orc.gemma3_decode_step(cfg, layers, embed, fnorm, token=19, pos=pos)
    # f32 products and sums on both sides: three layers of 1e-7 to 1e-6 each,
    # amplified where a sublayer's output nearly cancels before its post-norm
    # (these synthetic weights have a large mean)
    assert rel_l2(got, ref) < 1e-4, rel_l2(got, ref)
    d.set_graph(False)
    assert np.array_equal(d.decode_step(19, pos), got)
    d.close()


def test_verify_of_two_widths_at_once(rt, orc):
    """A context of hidden 3840, whose batched head stages 120 KB, verifies after
    one of hidden 768 was created: each gives its own steps' logits."""
    from test_oracle import make_model
    made = []
    for hidden, heads in ((3840, (16, 256)), (768, (4, 128))):
        cfg = dict(hidden=hidden, ffn=1536, n_q_heads=heads[0], n_kv_heads=4, head_dim=heads[1], n_layers=1, vocab=777,
                   sliding_window=9, global_every=2, rope_theta_local=10000.0, rope_theta_global=1000000.0,
                   rope_fs_local=1.0, rope_fs_global=0.125, eps=1e-6, attn_scale=1.0 / np.sqrt(heads[1]))
        layers, embed, fnorm = make_model(orc, cfg, max_seq=24, ctx=5, seed=hidden)
        made.append((cfg, layers, embed, fnorm, mixed_ctx(rt, cfg, layers, [[1] * 7], embed, fnorm, 5, 24, layers)))
    for cfg, layers, embed, fnorm, d in made:
        got = d.decode_step_batch([3, 4, 5], 5)
        for i, t in enumerate((3, 4, 5)):
            ref = orc.gemma3_decode_step(cfg, layers, embed, fnorm, token=t, pos=5 + i)
            assert rel_l2(got[i], ref) < 1e-3
        d.close()
