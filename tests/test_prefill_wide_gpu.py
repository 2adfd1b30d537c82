"""GPU parity of the wide batched prefill (prompts of more than 64 tokens,
rust-inference_amd/csrc/qg_prefill_wide.hip) against the oracle's
token-by-token forward pass, where its tiles end: prompts around 64 and 128
tokens, matrices of fewer rows than a tile and of rows that no tile divides,
rows that start in the middle of a block (cols % 256 == 128), every head size,
a prompt that takes two wide chunks, and one that continues a cache.  The
greedy steps after the prompt read every cached position.  Tolerance: TIGHT_TOL
(2e-5 normwise, conftest.py)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import TIGHT_TOL, normwise_err
from test_decode_gpu import SMALL, build
from test_prefill_gpu import prefill_and_compare

pytestmark = pytest.mark.gpu

HALF = dict(SMALL, embed_dim=384, n_heads=6, n_kv_heads=2, hidden_dim=640)       # rows of 1.5 and 2.5 blocks
HD128 = dict(SMALL, embed_dim=512, n_heads=4, n_kv_heads=1, hidden_dim=768)
HD256 = dict(SMALL, embed_dim=1024, n_heads=4, n_kv_heads=2, hidden_dim=1280)


@pytest.mark.parametrize("mix", ["q4_k_m", "q5_k", "q8_0", "q5_k_m"])
@pytest.mark.parametrize("n", [65, 128, 129])
def test_tiles(rinf, synth, oracle, ctx, mix, n):
    e0, errs, _ = prefill_and_compare(rinf, synth, oracle, ctx, SMALL, mix, n, n, 4, 192)
    assert e0 <= TIGHT_TOL and max(errs) <= TIGHT_TOL, (e0, errs)


@pytest.mark.parametrize("cfg,mix,n", [(HALF, "q4_k_m", 130), (HALF, "q5_k_m", 193), (HALF, "q8_0", 70),
                                       (HD128, "q4_k_m", 300), (HD256, "q5_k_m", 97), (HD256, "q8_0", 257)])
def test_shapes(rinf, synth, oracle, ctx, cfg, mix, n):
    e0, errs, _ = prefill_and_compare(rinf, synth, oracle, ctx, cfg, mix, n, n, 4, 320)
    assert e0 <= TIGHT_TOL and max(errs) <= TIGHT_TOL, (e0, errs)


def test_two_chunks_and_continued(rinf, synth, oracle, ctx):
    e0, errs, _ = prefill_and_compare(rinf, synth, oracle, ctx, SMALL, "q4_k_m", 7, 1100, 3, 1200)
    e1, errs1, _ = prefill_and_compare(rinf, synth, oracle, ctx, SMALL, "q5_k_m", 8, 300, 3, 400, split=81)
    assert max([e0, e1] + errs + errs1) <= TIGHT_TOL, (e0, errs, e1, errs1)


@pytest.mark.parametrize("mix,embed,hd,hidden,n", [
    ("q4_k_m", 256, 64, 4864, 66), ("q4_k_m", 256, 64, 8192, 70), ("q5_k", 256, 64, 8320, 66),
    ("q8_0", 256, 64, 18944, 130), ("q4_k_m", 256, 64, 20480, 66), ("q8_0", 256, 64, 20608, 66),
    ("q4_k_m", 256, 64, 32768, 66), ("q4_k_m", 4352, 256, 256, 66), ("q4_k_m", 256, 64, 32896, 66)])
def test_long_rows(rinf, synth, oracle, ctx, mix, embed, hd, hidden, n):
    """Rows of x in each number of pieces per thread (up to 4096, 8192, 20480 and
    32768 elements), at and beside the lines; beyond the last, 64-token chunks."""
    cfg = dict(SMALL, n_layers=1, embed_dim=embed, n_heads=embed // hd, n_kv_heads=1, hidden_dim=hidden)
    e0, errs, _ = prefill_and_compare(rinf, synth, oracle, ctx, cfg, mix, 6, n, 2, 160)
    assert e0 <= TIGHT_TOL and max(errs) <= TIGHT_TOL, (e0, errs)


class Edited:
    """synth with gen_model's tensors changed by `edit`."""

    def __init__(self, synth, edit):
        self.synth, self.edit = synth, edit

    def gen_model(self, cfg, mix, seed):
        t = self.synth.gen_model(cfg, mix, seed)
        self.edit(t)
        return t


# byte offsets of the f16 scales (d, and dmin) of a block, elements and bytes of one
SCALES = {8: ((0,), 32, 34), 12: ((0, 2), 256, 144), 13: ((0, 2), 256, 176), 14: ((208,), 256, 210)}


def scale_blocks(mat, first, last, factor):
    """The scales of the blocks that hold the flat elements first .. last - 1."""
    raw, dtype, _, _ = mat
    offsets, be, bb = SCALES[dtype]
    blocks = raw.reshape(-1, bb)[first // be:-(-last // be)]
    for o in offsets:
        f = np.ascontiguousarray(blocks[:, o:o + 2]).view(np.float16)
        blocks[:, o:o + 2] = (f.astype(np.float32) * factor).astype(np.float16).view(np.uint8)


@pytest.mark.parametrize("cfg,mix", [(dict(SMALL, hidden_dim=1024), "q4_k_m"), (dict(SMALL, hidden_dim=1024), "q5_k"),
                                     (dict(SMALL, hidden_dim=1024), "q8_0"), (HALF, "q4_k_m")])
def test_outlier(rinf, synth, oracle, ctx, cfg, mix):
    """One activation 2^40 times the others (row 4 of gate and up 2^20 times the
    rest) that no output depends on (its 256-element group's weights in down
    are zero): the other groups keep their 22 bits, as in the 64-token chunks.
    Under a scale common to the token they would vanish."""
    def edit(t):
        for layer in range(cfg["n_layers"]):
            for slot in ("gate", "up"):
                scale_blocks(t["mats"][slot, layer], 4 * cfg["embed_dim"], 5 * cfg["embed_dim"], 2.0 ** 20)
            raw, dtype, rows, cols = t["mats"]["down", layer]
            for r in range(rows):
                if dtype == 14:                   # a scale byte per 16 elements
                    f = np.arange(r * cols, r * cols + 256, 16)
                    raw.reshape(-1, 210)[f // 256, 192 + f % 256 // 16] = 0
                else:
                    scale_blocks(t["mats"]["down", layer], r * cols, r * cols + 256, 0.0)

    for seed in (1, 2, 3):
        e0, errs, _ = prefill_and_compare(rinf, Edited(synth, edit), oracle, ctx, cfg, mix, seed, 70 + seed, 4, 96)
        assert e0 <= TIGHT_TOL and max(errs) <= TIGHT_TOL, (seed, e0, errs)


@pytest.mark.parametrize("n", [64, 65])
def test_q6_k_products_are_exact(rinf, synth, oracle, ctx, n):
    """Q6_K values of 12 bits (scale -127, code 1: d 3937) against x of two f16
    pieces, hi + 0.125 each, that sum to zero: v is zero, and only if every
    product of a piece of x with a piece of the weight is formed (the low
    pieces' with the weight's last bit sum to 32 d of 64 million).  wo spreads v
    with alternating signs, so logits other than the all-equal h's show it."""
    cfg = dict(SMALL, n_layers=1, norm_eps=0.0)
    E, V = cfg["embed_dim"], cfg["vocab_size"]
    x = np.where(np.arange(E) % 2 == 0, 1000.125, -999.875)
    x[0:32:2] -= 2.0
    assert x.sum() == 0

    def edit(t):
        for slot in ("wq", "wk", "wv", "gate", "up", "down"):
            scale_blocks(t["mats"][slot, 0], 0, int(np.prod(t["mats"][slot, 0][2:])), 0.0)
        emb = t["mats"]["token_embd", 0]
        t["mats"]["token_embd", 0] = (np.ones(V * E, np.float32).view(np.uint8), 0, V, E)
        wv = t["mats"]["wv", 0][0].reshape(-1, 210)
        wv[:, :128], wv[:, 128:192], wv[:, 192:208] = 0x11, 0, 0x81
        wv[:, 208:210] = np.array([256.0], np.float16).view(np.uint8)
        wo = t["mats"]["wo", 0][0].reshape(E, 144)                  # one block a row: d = +-2^-6, codes 1, mins 0
        wo[:, 0:2] = np.where(np.arange(E) % 2 == 0, 2.0 ** -6, -2.0 ** -6).astype(np.float16).view(np.uint8).reshape(E, 2)
        wo[:, 2:4], wo[:, 4:8], wo[:, 8:12], wo[:, 12:16], wo[:, 16:] = 0, 1, 0, 1, 0x11
        assert emb[2:] == (V, E)
        t["vecs"]["attn_norm", 0] = x.astype(np.float32)
        for b in ("bq", "bk", "bv"):
            t["vecs"][b, 0][:] = 0

    dev, _, _ = build(rinf, Edited(synth, edit), oracle, ctx, cfg, "q4_k_m", 21, 96)
    logits = np.zeros(V, np.float32)
    dev.prefill(np.arange(n), logits)
    dev.close()
    t = synth.gen_model(cfg, "q4_k_m", 21)
    raw, dtype, rows, cols = t["mats"]["lm_head", 0]
    ref = oracle.mat_vec_mul(raw, dtype, rows, cols, t["vecs"]["final_norm", 0])
    err = normwise_err(logits, ref)
    assert err <= TIGHT_TOL, err


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_non_finite_x(rinf, synth, oracle, ctx, value):
    """A token whose embedding is not finite: the logits of every prompt that holds
    it are NaN where the oracle's are, and nothing of it stays for the next."""
    E, V, bad = SMALL["embed_dim"], SMALL["vocab_size"], 17
    emb = np.random.default_rng(4).standard_normal((V, E)).astype(np.float32)
    emb[bad, 5] = value

    def edit(t):
        t["mats"]["token_embd", 0] = (emb.view(np.uint8).reshape(-1), 0, V, E)

    dev, ref, _ = build(rinf, Edited(synth, edit), oracle, ctx, SMALL, "q4_k_m", 16, 200)
    logits = np.zeros(V, np.float32)
    rng = np.random.default_rng(16)
    for n, at in ((70, 69), (150, 3), (130, 64), (130, None)):
        prompt = rng.integers(bad + 1, V, n)
        if at is not None:
            prompt[at] = bad
        dev.reset()
        ref.reset()
        dev.prefill(prompt, logits)
        for pos, tok in enumerate(prompt):
            ref_l = ref.forward(int(tok), pos)
        assert np.array_equal(np.isnan(logits), np.isnan(ref_l)) and np.isnan(ref_l).all() == (at is not None)
    assert normwise_err(logits, ref_l) <= TIGHT_TOL
    dev.close()


def test_no_room_for_the_wide_buffers(rinf, synth, oracle, ctx):
    """Where the wide chunks' buffers cannot be allocated the prompt goes through
    64-token chunks; the next prompt finds room and takes the wide ones.  The
    context's last error stays the one of the call before them."""
    dev, ref, shared = build(rinf, synth, oracle, ctx, SMALL, "q4_k_m", 11, 400)
    prompt = np.random.default_rng(11).integers(0, SMALL["vocab_size"], 330)
    logits = np.zeros(SMALL["vocab_size"], np.float32)
    pos = 0
    with pytest.raises(rinf.QgemvError):
        dev.prefill([SMALL["vocab_size"]])
    last_error = ctx.lib.qg_last_error(ctx.h)
    for part, fail in ((prompt[:40], False), (prompt[40:190], True), (prompt[190:], False)):
        if fail:
            ctx.fail_allocations(1)
        dev.prefill(part, logits)
        ctx.fail_allocations(0)
        assert ctx.lib.qg_last_error(ctx.h) == last_error
        for tok in part:
            ref_l = ref.forward(int(tok), pos)
            pos += 1
        assert normwise_err(logits, ref_l) <= TIGHT_TOL, pos
    dev.close()
    if shared is not None:
        shared.free()


def test_every_failed_allocation(rinf, synth, oracle, ctx):
    """Each allocation of a prefill fails in turn.  Of the buffers every prefill
    needs: out of memory, nothing kept, and the next call starts over.  Of the
    wide chunks': the prompt goes through 64-token chunks, and the buffers
    before the failed one are given back."""
    cfg = dict(SMALL, n_layers=1)
    dev, ref, _ = build(rinf, synth, oracle, ctx, cfg, "q4_k_m", 12, 96)
    prompt = np.random.default_rng(12).integers(0, cfg["vocab_size"], 70)
    for pos, tok in enumerate(prompt):
        ref_l = ref.forward(int(tok), pos)
    logits = np.zeros(cfg["vocab_size"], np.float32)

    def attempt(skip):
        dev.reset()
        logits[:] = 0
        ctx.fail_allocations(1, skip)
        try:
            dev.prefill(prompt, logits)
        finally:
            ctx.fail_allocations(0)
        assert normwise_err(logits, ref_l) <= TIGHT_TOL, skip

    failed = 0
    for skip in range(64):
        try:
            attempt(skip)
            break
        except rinf.QgemvError as e:
            assert e.status == 6, e
            failed += 1
            assert dev.seq_len == 0
    assert failed >= 12                           # qg_model.hip, pf_alloc
    held = dev.resident_bytes()
    for skip in range(64):                        # wide_alloc, until all of them go through
        attempt(skip)
        if dev.resident_bytes() != held:
            break
    assert 1 <= skip < 63
    dev.close()


def test_buffers_follow_the_prompts(rinf, synth, oracle, ctx):
    """The wide chunks' buffers are as long as the prompts so far need and not as
    long as the cache, and fit the layers' matrices as they are: V apart from Q
    and K (Q6_K, Q4_K), then, with another matrix in its slot, beside them in one
    launch of the first layer."""
    dev, ref, _ = build(rinf, synth, oracle, ctx, SMALL, "q4_k_m", 14, 1024)
    logits = np.zeros(SMALL["vocab_size"], np.float32)
    rng = np.random.default_rng(14)

    def run(n):
        prompt = rng.integers(0, SMALL["vocab_size"], n)
        dev.reset()
        ref.reset()
        dev.prefill(prompt, logits)
        for pos, tok in enumerate(prompt):
            ref_l = ref.forward(int(tok), pos)
        assert normwise_err(logits, ref_l) <= TIGHT_TOL, n
        return dev.resident_bytes()["total"]

    bytes_ = [run(n) for n in (20, 65, 300, 128, 900, 70)]
    narrow, short, middle, _, most, _ = bytes_
    assert narrow < short < middle < most and bytes_[3] == middle and bytes_[5] == most
    assert 4 * (short - narrow) < most - narrow
    kv, E = SMALL["n_kv_heads"] * 64, SMALL["embed_dim"]
    raw = synth.gen_weights(12, kv, E, 5)
    dev.set_matrix(rinf.M_WV, 0, raw, 12, kv, E)
    ref.set_mat("wv", 0, raw, 12, kv, E)
    for n in (130, 65, 400):
        run(n)
    dev.close()
