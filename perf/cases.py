"""The work this library is used for, as cases that can be timed and compared.

Every case goes through the package's public entry points (``GpuContext``,
``DeviceMatrix``, ``DeviceModel``) on seeded random-init weights of the
architectures this repository names (Qwen2-0.5B, Qwen2-7B, Llama-3-8B):

* ``gemv``     plain mat-vecs of a few matrices of one shape (one per layer),
               vectors on the device; ``f32`` the same in the f32 precision
               mode;
* ``host``     the drop-in ``mat_vec_mul(weight bytes, x, out)`` with host
               arrays, as an inference engine that keeps its state on the host
               calls it;
* ``norm``     RMSNorm of the residual stream and a projection (the lm_head);
* ``glu``      RMSNorm, gate and up projections, silu(gate) * up;
* ``dequant``  a whole matrix to f32;
* ``prefill``  a prompt through a model's layers, the last token's logits;
* ``decode``   a prompt and then one token after the other (a chat turn).

The model cases have the widths of their architecture and few layers (the
small one has all of them), with the vocabulary cut by about as much, so that
the layers and the lm_head keep their shares of a token.
"""
from __future__ import annotations

import importlib.util
import pathlib
import sys

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent
PKG_NAME = "rust_inference_amd"


def _package():
    """rust-inference_amd/ (a hyphenated directory) as rust_inference_amd."""
    if PKG_NAME not in sys.modules:
        d = ROOT / "rust-inference_amd"
        spec = importlib.util.spec_from_file_location(PKG_NAME, d / "__init__.py",
                                                      submodule_search_locations=[str(d)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[PKG_NAME] = mod
        spec.loader.exec_module(mod)
    return sys.modules[PKG_NAME]


TYPES = {"F32": 0, "F16": 1, "Q4_0": 2, "Q5_0": 6, "Q8_0": 8, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14}
# (block elements, block bytes)
BLOCK = {"F32": (1, 4), "F16": (1, 2), "Q4_0": (32, 18), "Q5_0": (32, 22), "Q8_0": (32, 34),
         "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210)}

ARCH = {
    "qwen2-0.5b": dict(embed=896, heads=14, kv_heads=2, hidden=4864, base=1e6, eps=1e-6, tied=True),
    "qwen2-7b": dict(embed=3584, heads=28, kv_heads=4, hidden=18944, base=1e6, eps=1e-6, tied=False),
    "llama3-8b": dict(embed=4096, heads=32, kv_heads=8, hidden=14336, base=5e5, eps=1e-5, tied=False),
}
# quantization mixes: attn_v, ffn_down and the lm_head differ from the rest
MIXES = {
    "q4_k_m": dict(rest="Q4_K", wv="Q6_K", down="Q6_K", lm_head="Q6_K"),
    "q5_k_m": dict(rest="Q5_K", wv="Q6_K", down="Q6_K", lm_head="Q6_K"),
    "q5_k": dict(rest="Q5_K", lm_head="Q6_K"),
    "q8_0": dict(rest="Q8_0"),
}


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # the smallest call: one query projection of Qwen2-0.5B
        {"name": "gemv_q8_0_896x896", "kind": "gemv", "type": "Q8_0", "rows": 896, "cols": 896, "layers": 1},
        # the headline shape, the down projection of Llama-3-8B, of four layers
        {"name": "gemv_q4_k_4096x14336", "kind": "gemv", "type": "Q4_K", "rows": 4096, "cols": 14336, "layers": 4},
        # an unquantized tensor whose rows are no multiple of anything
        {"name": "gemv_f16_3001x2050", "kind": "gemv", "type": "F16", "rows": 3001, "cols": 2050, "layers": 2},
        # the f32 arithmetic option, for callers who need the reference's per-product rounding
        {"name": "f32_q4_k_4096x14336", "kind": "f32", "type": "Q4_K", "rows": 4096, "cols": 14336, "layers": 1},
        # the drop-in call from the host: Qwen2-7B's down projection
        {"name": "host_q6_k_3584x18944", "kind": "host", "type": "Q6_K", "rows": 3584, "cols": 18944},
        # final norm and lm_head of Qwen2-7B: the largest matrix
        {"name": "norm_q6_k_152064x3584", "kind": "norm", "type": "Q6_K", "rows": 152064, "cols": 3584},
        # the MLP's gate and up of Qwen2-7B (decode)
        {"name": "glu_q4_k_18944x3584", "kind": "glu", "type": "Q4_K", "rows": 18944, "cols": 3584},
        # a layer matrix handed to something that wants f32
        {"name": "dequant_q4_k_14336x4096", "kind": "dequant", "type": "Q4_K", "rows": 14336, "cols": 4096},
        # a short prompt (the benchmark's 64 tokens)
        {"name": "prefill_qwen2_7b_64", "kind": "prefill", "arch": "qwen2-7b", "mix": "q4_k_m", "layers": 2,
         "vocab": 10240, "prompt": 64},
        # a long prompt (a document), an odd number of tokens
        {"name": "prefill_llama3_8b_1001", "kind": "prefill", "arch": "llama3-8b", "mix": "q5_k_m", "layers": 2,
         "vocab": 10240, "prompt": 1001},
        # a short chat turn on the small model, all layers
        {"name": "decode_qwen2_0_5b_32_64", "kind": "decode", "arch": "qwen2-0.5b", "mix": "q4_k_m", "layers": 24,
         "vocab": 151936, "prompt": 32, "steps": 64},
        # a long conversation: 2000 cached tokens, then an answer of 256
        {"name": "decode_qwen2_7b_2000_256", "kind": "decode", "arch": "qwen2-7b", "mix": "q4_k_m", "layers": 2,
         "vocab": 10240, "prompt": 2000, "steps": 256},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _cols(rng, lo, hi, t):
    """A row length: whole superblocks mostly, else whole small blocks, else any."""
    c, r = _log(rng, lo, hi), rng.random()
    if r < 0.7:
        return max(256, c // 256 * 256)
    return max(32, c // 32 * 32) if r < 0.85 else c | 1


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemv", "f32", "host", "norm", "glu", "dequant", "prefill", "prefill",
                       "decode"])
    if kind in ("prefill", "decode"):
        arch = rng.choice(sorted(ARCH))
        c = {"kind": kind, "arch": arch, "mix": rng.choice(sorted(MIXES)),
             "layers": rng.choice([1, 2, 3, 6] if arch == "qwen2-0.5b" else [1, 2]),
             "vocab": _log(rng, 2000, 10240), "prompt": _log(rng, 1, 1000)}
        if kind == "decode":
            c["steps"] = _log(rng, 8, 128)
        return c
    quant = ["Q4_0", "Q5_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K"]
    t = rng.choice(quant + ["F16", "F32"] if kind in ("gemv", "dequant") else quant)
    if kind == "norm":
        return {"kind": kind, "type": t, "rows": _log(rng, 64, 40000), "cols": _log(rng, 2, 32) * 256 - 128 * rng.randrange(2)}
    if kind == "glu":
        return {"kind": kind, "type": t, "rows": _log(rng, 32, 2400) * 8, "cols": _log(rng, 2, 16) * 256}
    cols = _cols(rng, 96, 20000, t)
    most = (4 << 20) if cols % 32 else (100 << 20) if kind != "f32" else (40 << 20)       # elements
    rows = min(_log(rng, 32, 40000), max(16, most // cols))
    c = {"kind": kind, "type": t, "rows": rows, "cols": cols}
    if kind in ("gemv", "f32"):
        c["layers"] = rng.choice([1, 1, 2])
    return c


# ------------------------------------------------------------------ weights

def _blocks(t, rows, cols):
    return -(-(rows * cols) // BLOCK[t][0])


def _nbytes(t, rows, cols):
    return _blocks(t, rows, cols) * BLOCK[t][1]


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _weights(t, rows, cols, gen):
    """Raw GGUF bytes (on the GPU) of a random-init matrix: codes and sub-block
    scales uniform over their bits, values centred with standard deviation
    about 1/sqrt(cols)."""
    nb, bb, dev = _blocks(t, rows, cols), BLOCK[t][1], gen.device
    sigma = cols ** -0.5
    if t in ("F32", "F16"):
        w = torch.randn(nb, generator=gen, device=dev) * sigma
        return (w if t == "F32" else w.half()).view(torch.uint8).reshape(-1)
    raw = torch.randint(0, 256, (nb, bb), dtype=torch.uint8, generator=gen, device=dev)
    # a random sign per block cancels the mean that the unsigned codes leave
    d = torch.rand(nb, generator=gen, device=dev) * 0.5 + 0.75
    d = d * (torch.randint(0, 2, (nb,), generator=gen, device=dev) * 2 - 1) * sigma
    if t in ("Q4_K", "Q5_K"):
        mid, sd = (7.5, 4.61) if t == "Q4_K" else (15.5, 9.23)
        d = (d / (36.4 * sd)).half()
        sc = torch.randint(1, 64, (nb, 8), dtype=torch.uint8, generator=gen, device=dev)
        raw[:, 0:2] = _f16_bytes(d)
        raw[:, 2:4] = _f16_bytes(d.float() * mid)
        # the scales and the mins (equal here) in their 12-byte pack
        raw[:, 4:8] = (sc[:, 0:4] & 63) | ((sc[:, 4:8] >> 4) << 6)
        raw[:, 8:12] = raw[:, 4:8]
        raw[:, 12:16] = (sc[:, 4:8] & 15) | ((sc[:, 4:8] & 15) << 4)
    elif t == "Q6_K":
        raw[:, 208:210] = _f16_bytes(d / (73.9 * 18.5))
    else:
        raw[:, 0:2] = _f16_bytes(d / {"Q8_0": 73.9, "Q4_0": 4.61, "Q5_0": 9.23}[t])
    return raw.reshape(-1)


def _host(raw):
    return raw.cpu().numpy()


def _values(t, raw, n):
    """The first n values of a matrix's raw bytes (a uint8 tensor), in 64 bits."""
    bs, bb = BLOCK[t]
    if t == "F32":
        return raw.view(torch.float32)[:n].double()
    if t == "F16":
        return raw.view(torch.float16)[:n].double()
    b = raw.reshape(-1, bb)

    def half(o):
        return b[:, o:o + 2].contiguous().view(torch.float16).double()

    if t == "Q8_0":
        v = b[:, 2:34].contiguous().view(torch.int8).double() * half(0)
    elif t == "Q4_0":                                     # neighbours share a byte
        q = torch.stack([b[:, 2:18] & 15, b[:, 2:18] >> 4], 2).reshape(-1, 32)
        v = (q.double() - 8) * half(0)
    elif t == "Q5_0":                                     # the halves share a byte; bit i of qh is element i's fifth
        q = torch.cat([b[:, 6:22] & 15, b[:, 6:22] >> 4], 1)
        bit = torch.arange(32, device=raw.device)
        h = (b[:, 2:6][:, bit // 8] >> (bit % 8).to(torch.uint8)) & 1
        v = (q.double() + 16 * h.double() - 16) * half(0)
    elif t in ("Q4_K", "Q5_K"):
        p = b[:, 4:16]
        sc = torch.cat([p[:, 0:4] & 63, (p[:, 8:12] & 15) | ((p[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([p[:, 4:8] & 63, (p[:, 8:12] >> 4) | ((p[:, 4:8] >> 6) << 4)], 1)
        o = 16 if t == "Q4_K" else 48
        qs = b[:, o:o + 128].reshape(-1, 4, 32)           # 32 bytes: sub-block 2 j low, 2 j + 1 high
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        if t == "Q5_K":
            bit = torch.arange(8, dtype=torch.uint8, device=raw.device).reshape(1, 8, 1)
            q = q + 16 * ((b[:, 16:48].reshape(-1, 1, 32) >> bit) & 1).double()
        v = q * (half(0) * sc.double()).unsqueeze(2) - (half(2) * mn.double()).unsqueeze(2)
    else:                                                 # Q6_K: two halves of 128
        ql, qh = b[:, 0:128].reshape(-1, 2, 64), b[:, 128:192].reshape(-1, 2, 32)
        q = torch.stack([(ql[..., :32] & 15) | ((qh & 3) << 4), (ql[..., 32:] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[..., :32] >> 4) | (((qh >> 4) & 3) << 4), (ql[..., 32:] >> 4) | ((qh >> 6) << 4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = (q.double() - 32).reshape(-1, 16, 16) * (sc * half(208)).unsqueeze(2)
    return v.reshape(-1)[:n]


def _times(t, raw, rows, cols, x):
    """W x (x: [cols] or [cols, n]) in 64 bits, a run of rows at a time."""
    bs, bb = BLOCK[t]
    step = max(1, (64 << 20) // cols // 256) * 256        # rows that start on a block
    out = []
    for r in range(0, rows, step):
        n = min(step, rows - r) * cols
        o = r * cols // bs * bb
        out.append(_values(t, raw[o:o + -(-n // bs) * bb], n).reshape(-1, cols) @ x)
    return torch.cat(out)


# ------------------------------------------------------------------- state

_contexts = {}


def _context(f32=False):
    """The program's context (one per precision mode)."""
    if f32 not in _contexts:
        r = _package()
        c = r.GpuContext(0)
        if f32:
            c.set_precision(r.PRECISION_F32)
        _contexts[f32] = c
    return _contexts[f32]


class _Held:
    """A matrix, freed with the state that holds it."""

    def __init__(self, mat):
        self.mat = mat

    def __del__(self):
        if self.mat.ctx.h:
            self.mat.free()


class _Keyed:
    """Host weight bytes whose device copy goes with them."""

    def __init__(self, ctx, raw):
        self.ctx, self.raw = ctx, raw

    def __del__(self):
        if self.ctx.h:
            self.ctx.invalidate(self.raw)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _slots(case):
    """(slot, type, rows, cols) of a layer's matrices."""
    a, m = ARCH[case["arch"]], MIXES[case["mix"]]
    E, H, kv = a["embed"], a["hidden"], a["embed"] // a["heads"] * a["kv_heads"]
    shapes = {"wq": (E, E), "wk": (kv, E), "wv": (kv, E), "wo": (E, E), "gate": (H, E), "up": (H, E), "down": (E, H)}
    return [(s, m.get(s, m["rest"]), r, c) for s, (r, c) in shapes.items()]


def _model_parts(case, seed):
    """The model's raw matrices, vectors and token ids, from the seed alone."""
    a, m, gen = ARCH[case["arch"]], MIXES[case["mix"]], _gen(seed)
    E, V = a["embed"], case["vocab"]
    kv = E // a["heads"] * a["kv_heads"]

    def vec(n, mean):
        return torch.randn(n, generator=gen, device="cuda") * 0.02 + mean

    mats = {("token_embd", 0): (m["rest"], V, E, _weights(m["rest"], V, E, gen))}
    if not a["tied"]:
        t = m.get("lm_head", m["rest"])
        mats["lm_head", 0] = (t, V, E, _weights(t, V, E, gen))
    vecs = {("final_norm", 0): vec(E, 1.0)}
    for l in range(case["layers"]):
        for s, t, r, c in _slots(case):
            mats[s, l] = (t, r, c, _weights(t, r, c, gen))
        vecs["attn_norm", l], vecs["ffn_norm", l] = vec(E, 1.0), vec(E, 1.0)
        if case["arch"].startswith("qwen2"):
            vecs["bq", l], vecs["bk", l], vecs["bv", l] = vec(E, 0.0), vec(kv, 0.0), vec(kv, 0.0)
    n = case["prompt"] + case.get("steps", 0)
    return mats, vecs, torch.randint(0, V, (n,), generator=gen, device="cuda")


def prepare(case, seed):
    kind, r = case["kind"], _package()
    if kind in ("prefill", "decode"):
        a, ctx = ARCH[case["arch"]], _context()
        n = case["prompt"] + case.get("steps", 0)
        model = r.DeviceModel(ctx, a["embed"], case["layers"], a["heads"], a["kv_heads"], a["hidden"], case["vocab"],
                              n, a["base"], a["eps"])
        mats, vecs, tokens = _model_parts(case, seed)
        state = {"model": model, "shared": None}
        M = {"token_embd": r.M_TOKEN_EMBD, "lm_head": r.M_LM_HEAD, "wq": r.M_WQ, "wk": r.M_WK, "wv": r.M_WV,
             "wo": r.M_WO, "gate": r.M_GATE, "up": r.M_UP, "down": r.M_DOWN}
        V = {"final_norm": r.V_FINAL_NORM, "attn_norm": r.V_ATTN_NORM, "ffn_norm": r.V_FFN_NORM, "bq": r.V_BQ,
             "bk": r.V_BK, "bv": r.V_BV}
        for (s, l), (t, rows, cols, raw) in mats.items():
            if s == "token_embd" and a["tied"]:
                mat = ctx.upload(_host(raw), TYPES[t], rows, cols)
                model.share_matrix(r.M_TOKEN_EMBD, 0, mat)
                model.share_matrix(r.M_LM_HEAD, 0, mat)
                state["shared"] = mat
            else:
                model.set_matrix(M[s], l, _host(raw), TYPES[t], rows, cols)
        for (s, l), v in vecs.items():
            model.set_vector(V[s], l, v.cpu().numpy())
        state["held"] = _Turn(model, state["shared"])
        state["tokens"] = tokens.cpu().numpy().astype(np.uint32)
        state["prompt"] = state["tokens"][:case["prompt"]].copy()
        state["steps"] = [int(t) for t in state["tokens"][case["prompt"]:]]
        state["logits"] = np.zeros(case["vocab"], np.float32)
        state["last"] = np.zeros(case["vocab"], np.float32)
        return dict(state, kind=kind)

    t, rows, cols = case["type"], case["rows"], case["cols"]
    gen = _gen(seed)
    ctx = _context(kind == "f32")
    if kind == "host":
        raw = _host(_weights(t, rows, cols, gen))
        return {"kind": kind, "ctx": ctx, "raw": raw, "held": _Keyed(ctx, raw), "type": TYPES[t], "rows": rows,
                "cols": cols, "x": torch.randn(cols, generator=gen, device="cuda").cpu().numpy(),
                "y": np.zeros(rows, np.float32)}
    if kind == "glu":
        raw = torch.cat([_weights(t, rows, cols, gen), _weights(t, rows, cols, gen)])
        mat = ctx.upload(_host(raw), TYPES[t], 2 * rows, cols)
    elif kind in ("gemv", "f32"):
        mats = [ctx.upload(_host(_weights(t, rows, cols, gen)), TYPES[t], rows, cols) for _ in range(case["layers"])]
        x = torch.randn(cols, generator=gen, device="cuda")
        return {"kind": kind, "mats": mats, "held": [_Held(m) for m in mats], "x": x,
                "y": [torch.zeros(rows, device="cuda") for _ in mats]}
    else:
        mat = ctx.upload(_host(_weights(t, rows, cols, gen)), TYPES[t], rows, cols)
    state = {"kind": kind, "mat": mat, "held": _Held(mat)}
    if kind == "dequant":
        return dict(state, out=torch.zeros(rows, cols, device="cuda"))
    # the residual stream, what the last block adds to it, and the norm's weights
    return dict(state, a=torch.randn(cols, generator=gen, device="cuda"),
                b=torch.randn(cols, generator=gen, device="cuda") * 0.3,
                nw=torch.randn(cols, generator=gen, device="cuda") * 0.02 + 1,
                sum=torch.zeros(cols, device="cuda"), y=torch.zeros(rows, device="cuda"))


class _Turn:
    """A model and the embedding it shares, closed in that order."""

    def __init__(self, model, shared):
        self.model, self.shared = model, shared

    def __del__(self):
        self.model.close()
        if self.shared is not None and self.shared.ctx.h:
            self.shared.free()


def run(state):
    kind = state["kind"]
    if kind in ("gemv", "f32"):
        for mat, y in zip(state["mats"], state["y"]):
            mat.matvec_dev(state["x"], y)
        return state["y"]
    if kind == "host":
        state["ctx"].mat_vec_mul(state["raw"], state["type"], state["x"], state["y"], state["rows"], state["cols"])
        return state["y"]
    if kind == "norm":
        state["mat"].matvec_norm_dev(state["a"], state["b"], state["nw"], 1e-6, state["y"], state["sum"])
        return [state["y"], state["sum"]]
    if kind == "glu":
        state["mat"].matvec_norm_glu_dev(state["a"], state["b"], state["nw"], 1e-6, state["y"], state["sum"])
        return [state["y"], state["sum"]]
    if kind == "dequant":
        state["mat"].dequant_dev(state["out"])
        return state["out"]
    m, steps = state["model"], state["steps"]
    m.reset()
    m.prefill(state["prompt"], state["logits"])
    if kind == "prefill":
        return state["logits"]
    pos = len(state["prompt"])
    for i, token in enumerate(steps):
        m.forward(token, pos + i, state["last"] if i + 1 == len(steps) else None)
    return [state["logits"], state["last"]]


# ---------------------------------------------------------- work and limits

def work(case):
    kind = case["kind"]
    if kind not in ("prefill", "decode"):
        t, rows, cols = case["type"], case["rows"], case["cols"]
        n = 2 if kind == "glu" else case.get("layers", 1)
        w = n * _nbytes(t, rows, cols)
        if kind == "dequant":
            return {"bytes": w + 4 * rows * cols, "flops": 2 * rows * cols}
        vecs = cols + (rows if kind == "glu" else n * rows) + (3 * cols if kind in ("norm", "glu") else 0)
        return {"bytes": w + 4 * vecs, "flops": 2 * n * rows * cols}
    a, m = ARCH[case["arch"]], MIXES[case["mix"]]
    E, L, V, hd = a["embed"], case["layers"], case["vocab"], a["embed"] // a["heads"]
    kv = hd * a["kv_heads"]
    layer = sum(_nbytes(t, r, c) for _, t, r, c in _slots(case))
    params = sum(r * c for _, _, r, c in _slots(case))
    head = _nbytes(m["rest"] if a["tied"] else m.get("lm_head", m["rest"]), V, E)
    P, K = case["prompt"], case.get("steps", 0)
    seen = sum(range(P + 1, P + K + 1))                   # positions the steps attend to
    bytes_ = (1 + K) * (L * layer + head + 4 * V) + L * 8 * kv * (P + K + seen)
    flops = (P + K) * L * 2 * params + (1 + K) * 2 * V * E + L * 4 * E * (P * (P + 1) // 2 + seen)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "dequant":                                 # the reference's own f32 operations
        return "exact"
    # against 64 bits: 0.7e-7 to 4.5e-7 for one mat-vec (x in 22 bits, f32
    # sums), up to 1.2e-5 for a model's logits (rotary angles of 2000 positions
    # in f32); sums in another order differ by as much
    return {"rel": 5e-5 if kind in ("prefill", "decode") else 2e-6}


# ------------------------------------------------------------------- 64 bits

def _rms(x, w, eps):
    return x * (x.square().mean(-1, keepdim=True) + eps).rsqrt() * w


def _embedding(t, raw, cols, tokens):
    """Rows of the embedding as the reference's dequantize_row places them: a
    row that starts inside a block has its later blocks at whole-block columns."""
    bs, bb = BLOCK[t]
    nk = -(-cols // bs)
    start = tokens * cols
    out = torch.zeros(len(tokens), cols, dtype=torch.float64, device="cuda")
    for off in (start % bs).unique().tolist():
        rows = (start % bs == off).nonzero().flatten()
        at = (start[rows] // bs)[:, None] + torch.arange(nk, device="cuda")
        v = _values(t, raw.reshape(-1, bb)[at].reshape(-1), rows.numel() * nk * bs).reshape(-1, nk * bs)
        row = torch.zeros(rows.numel(), nk * bs, dtype=torch.float64, device="cuda")
        row[:, :bs - off] = v[:, off:bs]
        row[:, bs:] = v[:, bs:]
        out[rows] = row[:, :cols]
    return out


def _logits(case, seed):
    a = ARCH[case["arch"]]
    E, heads, eps = a["embed"], a["heads"], float(np.float32(a["eps"]))
    hd, rep = E // heads, heads // a["kv_heads"]
    mats, vecs, tokens = _model_parts(case, seed)

    def mul(key, x):                                      # [n, cols] -> [n, rows]
        t, rows, cols, raw = mats[key]
        return _times(t, raw, rows, cols, x.t().contiguous()).t().contiguous()

    t, _, _, raw = mats["token_embd", 0]
    h = _embedding(t, raw, E, tokens)
    n = len(tokens)
    # the rotary tables' angles are f32 products, as the reference's
    theta = np.float32(1) / np.power(np.float32(a["base"]), np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd))
    angle = torch.from_numpy((np.arange(n, dtype=np.float32)[:, None] * theta[None]).astype(np.float64)).cuda()
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    mask = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)

    def rope(x):
        x0, x1 = x[..., 0::2], x[..., 1::2]
        return torch.stack([x0 * cos - x1 * sin, x0 * sin + x1 * cos], -1).reshape(x.shape)

    for l in range(case["layers"]):
        x = _rms(h, vecs["attn_norm", l].double(), eps)
        q, k, v = (mul((s, l), x) + (vecs[b, l].double() if (b, l) in vecs else 0)
                   for s, b in (("wq", "bq"), ("wk", "bk"), ("wv", "bv")))
        q, k, v = rope(q.reshape(n, heads, hd)), rope(k.reshape(n, -1, hd)), v.reshape(n, -1, hd)
        o = torch.empty(n, heads, hd, dtype=torch.float64, device="cuda")
        for i in range(heads):
            s = q[:, i] @ k[:, i // rep].t().contiguous() * hd ** -0.5
            o[:, i] = torch.softmax(s.masked_fill_(mask, -torch.inf), -1) @ v[:, i // rep].contiguous()
        h = h + mul(("wo", l), o.reshape(n, E))
        x = _rms(h, vecs["ffn_norm", l].double(), eps)
        g = mul(("gate", l), x)
        h = h + mul(("down", l), g * torch.sigmoid(g) * mul(("up", l), x))
    head = ("token_embd", 0) if a["tied"] else ("lm_head", 0)
    at = [case["prompt"] - 1] + ([n - 1] if case["kind"] == "decode" else [])
    return mul(head, _rms(h[at], vecs["final_norm", 0].double(), eps)).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "decode"):
        y = _logits(case, seed)
        return y[0].copy() if kind == "prefill" else [y[0].copy(), y[1].copy()]
    t, rows, cols, gen = case["type"], case["rows"], case["cols"], _gen(seed)
    if kind == "host":
        raw = _weights(t, rows, cols, gen)
        x = torch.randn(cols, generator=gen, device="cuda").double()
        return _times(t, raw, rows, cols, x).cpu().numpy()
    if kind in ("gemv", "f32"):
        raws = [_weights(t, rows, cols, gen) for _ in range(case["layers"])]
        x = torch.randn(cols, generator=gen, device="cuda").double()
        return [_times(t, w, rows, cols, x) for w in raws]
    if kind == "dequant":
        return _values(t, _weights(t, rows, cols, gen), rows * cols).reshape(rows, cols)
    raws = [_weights(t, rows, cols, gen) for _ in range(2 if kind == "glu" else 1)]
    a = torch.randn(cols, generator=gen, device="cuda")
    b = torch.randn(cols, generator=gen, device="cuda") * 0.3
    nw = torch.randn(cols, generator=gen, device="cuda") * 0.02 + 1
    s = a.double() + b.double()
    x = _rms(s, nw.double(), float(np.float32(1e-6)))
    y = [_times(t, w, rows, cols, x) for w in raws]
    return [y[0] if kind == "norm" else y[0] * torch.sigmoid(y[0]) * y[1], s]
