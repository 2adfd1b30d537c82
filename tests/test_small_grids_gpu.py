"""The paired [gate; up] and [Q;K] + V launches in the smaller workgroups they
take when there is about one row group per compute unit: row counts around
one group, one workgroup and one workgroup per unit, whole-block and
straddling rows.  Against the oracle's mat-vec of the normalised input, and the
decode step of a model of such shapes, within TIGHT_TOL (2e-5 normwise)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import TIGHT_TOL, normwise_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", ["Q4_K", "Q5_K", "Q8_0", "Q6_K"])
@pytest.mark.parametrize("half,cols", [(2, 256), (8, 896), (34, 896), (1024, 896), (2050, 512), (4864, 896), (5200, 2048)])
def test_glu(rinf, synth, oracle, ctx, t, half, cols):
    import torch
    dtype = rinf.TYPE_IDS[t]
    raw = synth.gen_weights(dtype, 2 * half, cols, half + cols)
    rng = np.random.default_rng(half)
    a, b = rng.standard_normal(cols).astype(np.float32), rng.standard_normal(cols).astype(np.float32)
    nw = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
    s = a.astype(np.float64) + b
    x = (s / np.sqrt(np.mean(s * s) + 1e-6) * nw).astype(np.float32)
    y = oracle.mat_vec_mul(raw, dtype, 2 * half, cols, x).astype(np.float64)
    ref = y[:half] / (1 + np.exp(-y[:half])) * y[half:]
    mat = ctx.upload(raw, dtype, 2 * half, cols)
    d = [torch.from_numpy(v).cuda() for v in (a, b, nw)]
    h, total = torch.zeros(half, device="cuda"), torch.zeros(cols, device="cuda")
    torch.cuda.synchronize()
    mat.matvec_norm_glu_dev(d[0], d[1], d[2], 1e-6, h, total)
    ctx.synchronize()
    assert normwise_err(h.cpu().numpy(), ref) <= TIGHT_TOL
    assert np.array_equal(total.cpu().numpy(), a + b)
    mat.free()


@pytest.mark.parametrize("embed,heads,kv,hidden", [(896, 14, 2, 4864), (1024, 16, 16, 256), (2048, 16, 2, 1280)])
def test_pair_in_decode(rinf, synth, oracle, ctx, embed, heads, kv, hidden):
    from test_decode_gpu import SMALL, build
    cfg = dict(SMALL, embed_dim=embed, n_heads=heads, n_kv_heads=kv, hidden_dim=hidden, n_layers=1)
    dev, ref, _ = build(rinf, synth, oracle, ctx, cfg, "q4_k_m", 3, 16)
    logits = np.zeros(cfg["vocab_size"], np.float32)
    for pos in range(6):
        dev.forward(pos * 7, pos, logits)
        assert normwise_err(logits, ref.forward(pos * 7, pos)) <= TIGHT_TOL, pos
    dev.close()
