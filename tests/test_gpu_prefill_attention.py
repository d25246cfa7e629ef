"""The batched attention where the masking changes from stage to stage: key
halves that every query of a wave sees whole (no masking), the diagonal, a
ragged last stage and a ragged last query tile, at head_dim 64, 32 and 48, in
both forms (one and two key groups).  Sampled rows of a batch against the
oracle at their positions (logits within the end-to-end bar)."""
import numpy as np
import pytest

from purebee_amd import synth
from purebee_amd.native import TYPE_Q8_0
from tests.test_gpu_prefill import LOGIT_TOL, make_pair, tiny

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_heads,n_kv", [(8, 2), (16, 4), (10, 2)])
@pytest.mark.parametrize("start,n", [(0, 130), (64, 64), (190, 129), (31, 33)])
@pytest.mark.parametrize("groups", ["1", "2"])
def test_masked_and_whole_stages(ctx, monkeypatch, n_heads, n_kv, start, n, groups):
    print(f"[case] attention stages heads {n_heads}/{n_kv} start {start} n {n} groups {groups}",
          flush=True)
    monkeypatch.setenv("PBX_PREFILL_ATTN_GROUPS", groups)
    cfg = tiny(TYPE_Q8_0, TYPE_Q8_0, dim=480 if n_heads == 10 else 512, hidden_dim=256, n_heads=n_heads, n_kv_heads=n_kv,
               max_seq=384)
    model, ref, cfg = make_pair(ctx, cfg, 700 + start + n_heads)
    toks = [int(t) for t in synth.random_tokens(701 + n, start + n, cfg["vocab_size"])]
    if start:
        model.forward(toks[:start], 0, want_logits=False)
    logits, _ = model.forward_batch(toks[start:], start)
    picked = sorted({0, 1, 31, 32, n // 2, n - 2, n - 1})
    worst, done = 0.0, 0
    for t in picked:
        r = ref.forward(toks[done:start + t + 1], done)
        done = start + t + 1
        worst = max(worst, float(np.abs(logits[t] - r).max()))
    print(f"  worst max-abs {worst:.2e}")
    assert worst <= LOGIT_TOL
    model.free()
    ref.close()
