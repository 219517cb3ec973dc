"""Prefill attention where its LDS score rows end: 1008 keys are the most that
leave room for the padding between rows, 1009 to 1024 go without it, and 1025
would not fit. One layer, so the logits hang on the last query's attention alone:
at most 1 ulp, as the double sums run in another order than the oracle's."""
import numpy as np
import pytest

import oracle as O
import uq

pytestmark = pytest.mark.gpu


def ordered(a):
    a = a.view(np.int32).astype(np.int64)
    return np.where(a < 0, -(a & 0x7FFFFFFF), a)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("n", [15, 16, 1007, 1008, 1009, 1024])
def test_score_row_edges(gpu, head_dim, n):
    cfg = dict(layers=1, dim=256, hidden=512, heads=256 // head_dim, kv_heads=128 // head_dim, head_dim=head_dim,
               vocab=1000, max_seq=1040, eps=1e-6, theta=1e6)
    t = uq.synth_qwen2(cfg, 31)
    g, o = uq.Qwen2Model(cfg, t), O.Model(cfg, {k: v[3] for k, v in t.items()})
    toks = uq.synth_tokens(n, n, cfg["vocab"])
    nxt = g.prefill(toks)
    rc, onxt, olg = o.prefill(toks, want_logits=True)
    assert rc == 0 and nxt == onxt
    assert np.abs(ordered(g.logits()) - ordered(olg)).max() <= 1
    if n == 1024:
        with pytest.raises(uq.UqError):
            g.prefill(uq.synth_tokens(1, 1025, cfg["vocab"]))
