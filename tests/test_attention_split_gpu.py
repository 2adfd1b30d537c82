"""The split decode attention (attn_rope_split_k and attn_rope_split_vec_k,
attn_combine_k) against the oracle where its tiles and ranges end: 1 to 65 cached positions (a wave of 16
with none, one and all of its positions, the second tile of 64), 4100 (ranges
of two tiles), grouped heads of every size up to 8 and one, head_dim 64, 128
and 256.  The prompt goes through the token-by-token path up to 70 positions,
so every length is checked; TIGHT_TOL (2e-5 normwise)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import TIGHT_TOL, normwise_err
from test_decode_gpu import SMALL, build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("embed,heads,kv", [(256, 4, 2), (448, 7, 1), (512, 8, 1), (512, 4, 2), (1024, 8, 1), (1024, 8, 8),
                                            (1024, 4, 1), (2048, 16, 16), (4096, 16, 16)])
def test_every_length(rinf, synth, oracle, ctx, embed, heads, kv):
    cfg = dict(SMALL, embed_dim=embed, n_heads=heads, n_kv_heads=kv, n_layers=1)
    dev, ref, _ = build(rinf, synth, oracle, ctx, cfg, "q8_0", 31, 80)
    dev.set_attention_path(2)
    logits = np.zeros(cfg["vocab_size"], np.float32)
    for pos in range(70):
        tok = (pos * 37 + 5) % cfg["vocab_size"]
        dev.forward(tok, pos, logits)
        assert normwise_err(logits, ref.forward(tok, pos)) <= TIGHT_TOL, pos
    # a shorter conversation over the same cache: rows past it hold old values
    dev.reset()
    dev2, ref2, _ = build(rinf, synth, oracle, ctx, cfg, "q8_0", 31, 80)
    dev2.close()
    for pos in range(5):
        tok = (pos * 91 + 1) % cfg["vocab_size"]
        dev.forward(tok, pos, logits)
        assert normwise_err(logits, ref2.forward(tok, pos)) <= TIGHT_TOL, pos
    dev.close()


def test_ranges_of_two_tiles(rinf, synth, oracle, ctx):
    cfg = dict(SMALL, embed_dim=128, n_heads=2, n_kv_heads=1, hidden_dim=128, n_layers=1, vocab_size=300)
    n = 4100
    dev, ref, _ = build(rinf, synth, oracle, ctx, cfg, "q8_0", 33, n + 40)
    prompt = np.random.default_rng(5).integers(0, 300, n)
    dev.prefill(prompt)
    for pos, tok in enumerate(prompt):
        ref.forward(int(tok), pos)
    logits = np.zeros(300, np.float32)
    for i in range(30):
        dev.forward(i, n + i, logits)
        assert normwise_err(logits, ref.forward(i, n + i)) <= TIGHT_TOL, i
    dev.close()


@pytest.mark.parametrize("embed,heads,kv,mix,most", [(384, 6, 2, "q4_k_m", 288), (384, 3, 1, "q4_k_m", 320),
                                                     (512, 2, 1, "f16", 480)])
def test_where_the_split_begins(rinf, synth, oracle, ctx, embed, heads, kv, mix, most):
    """A wo that takes no two ranges (rows of 1.5 blocks, F16): one workgroup per
    head up to the length where the split is as fast, which grows with the head
    size."""
    cfg = dict(SMALL, embed_dim=embed, n_heads=heads, n_kv_heads=kv, n_layers=1)
    dev, _, _ = build(rinf, synth, oracle, ctx, cfg, mix, 35, most + 8)
    prompt = np.arange(most + 1) * 37 % cfg["vocab_size"]
    got = {}
    for path in (0, 1, 2):
        dev.reset()
        dev.prefill(prompt[:most - 1])
        dev.set_attention_path(path)
        for pos in (most - 1, most):
            logits = np.zeros(cfg["vocab_size"], np.float32)
            dev.forward(int(prompt[pos]), pos, logits)
            got[path, pos + 1] = logits.tobytes()
        dev.set_attention_path(0)
    assert got[1, most] != got[2, most] and got[1, most + 1] != got[2, most + 1]
    assert got[0, most] == got[1, most] and got[0, most + 1] == got[2, most + 1]
    dev.close()


def test_ranges_of_many_groups(rinf, synth, oracle, ctx):
    """One workgroup per head and kv head, 16 of them: 16 ranges each, of two tiles
    beyond 1024 positions."""
    cfg = dict(SMALL, embed_dim=1024, n_heads=16, n_kv_heads=16, hidden_dim=256, n_layers=1, vocab_size=300)
    n = 1020
    dev, ref, _ = build(rinf, synth, oracle, ctx, cfg, "q8_0", 34, n + 40)
    prompt = np.random.default_rng(6).integers(0, 300, n)
    dev.prefill(prompt)
    for pos, tok in enumerate(prompt):
        ref.forward(int(tok), pos)
    logits = np.zeros(300, np.float32)
    for i in range(30):
        dev.forward(i, n + i, logits)
        assert normwise_err(logits, ref.forward(i, n + i)) <= TIGHT_TOL, i
    dev.close()


@pytest.mark.parametrize("embed,heads,kv,most", [(1280, 5, 1, 1280), (256, 2, 2, 832), (1024, 4, 1, 2560)])
def test_where_the_vector_units_end(rinf, synth, oracle, ctx, embed, heads, kv, most):
    """Across the length at which attn_rope_split_vec_k (head_dim 256, and 128 with a
    kv head per head) gives way to attn_rope_split_k."""
    cfg = dict(SMALL, embed_dim=embed, n_heads=heads, n_kv_heads=kv, hidden_dim=256, n_layers=1, vocab_size=300)
    n = most - 8
    dev, ref, _ = build(rinf, synth, oracle, ctx, cfg, "q8_0", 36, n + 20)
    prompt = np.random.default_rng(7).integers(0, 300, n)
    dev.prefill(prompt)
    for pos, tok in enumerate(prompt):
        ref.forward(int(tok), pos)
    logits = np.zeros(300, np.float32)
    for i in range(20):
        dev.forward(i, n + i, logits)
        assert normwise_err(logits, ref.forward(i, n + i)) <= TIGHT_TOL, i
    dev.close()
