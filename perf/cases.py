"""The calls that a program makes through this package, with their inputs, for timing.

Five kinds of case, each through a public entry point:

  host      Weight.matvec_into: one matvec from and to host buffers, as an engine that keeps
            its activations on the host calls it
  matvec    Weight.matvec_dev / matvec_multi_dev: p activation rows (1: a decode step; a few:
            a batch of requests or a short chat turn; hundreds: a prompt) against one or two
            weights
  ffn       swiglu_down_dev: a decode step's feed-forward block
  attend    KVCacheF16.attend_dev: one decode position over a filled cache, in both modes
  prefill, decode   LlamaDecoder: a whole prompt, and a run of decode steps after one

Weights are GGUF blocks whose fields follow those of matrices drawn N(0, 0.02); activations
are N(0, 1).  `exact` evaluates the same products in 64 bits from the same fields: the int8
activations are what the format defines (one float32 scale per 256 values), the sums are not.
"""
import math

import numpy as np
import torch

import gopherllm_amd as g
from gopherllm_amd import _lib
from gopherllm_amd.synth import LLAMA3_8B, build_decoder

TYPES = {"q4_0": 2, "q8_0": 8, "q4_k": 12, "q5_k": 13, "q6_k": 14}
BLOCK_BYTES = {"q4_0": 144, "q8_0": 272, "q4_k": 144, "q5_k": 176, "q6_k": 210}  # per 256 values
N_HEADS, N_KV, HEAD_DIM = 32, 8, 128


def listed():
    return [
        # the smallest call: a key projection with the activations on the host, where the
        # copies, the launch and the wait are what counts
        {"name": "host_key", "kind": "host", "type": "q4_k", "rows": 1024, "cols": 4096},
        # the feed-forward block of a decode step, three quarters of a layer's weights
        {"name": "decode_ffn", "kind": "ffn", "type": "q4_k", "dim": 4096, "hidden": 14336},
        # the logits of a decode step
        {"name": "vocab_head", "kind": "matvec", "type": "q6_k", "rows": 128256, "cols": 4096, "p": 1, "n": 1},
        # eight requests decoded together, gate projection
        {"name": "batch8_gate", "kind": "matvec", "type": "q4_k", "rows": 14336, "cols": 4096, "p": 8, "n": 1},
        # a few tokens against a down projection kept at higher precision
        {"name": "batch5_down", "kind": "matvec", "type": "q6_k", "rows": 4096, "cols": 14336, "p": 5, "n": 1},
        # a prompt chunk through gate and up, which share its activations
        {"name": "prompt_gate_up", "kind": "matvec", "type": "q4_k", "rows": 14336, "cols": 4096, "p": 512, "n": 2},
        # a ragged prompt through a down projection kept at higher precision
        {"name": "prompt_down", "kind": "matvec", "type": "q6_k", "rows": 4096, "cols": 14336, "p": 333, "n": 1},
        # a prompt chunk in an 8-bit model
        {"name": "prompt_q8", "kind": "matvec", "type": "q8_0", "rows": 14336, "cols": 4096, "p": 512, "n": 1},
        # decode attention with greedy parity, at an odd context
        {"name": "attend_exact", "kind": "attend", "ctx": 4001, "exact": True},
        # decode attention over a long context, in the fast mode
        {"name": "attend_split", "kind": "attend", "ctx": 32768, "exact": False},
        # a long prompt through some layers of an 8B-shaped model: projections, RoPE, causal
        # attention, SwiGLU, logits
        {"name": "model_prompt", "kind": "prefill", "layers": 4, "p": 3000},
        # decode steps of an 8B-shaped model after a 512-token prompt
        {"name": "model_decode", "kind": "decode", "layers": 32, "p": 512, "steps": 8},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "ffn", "matvec", "matvec", "matvec", "attend", "prefill", "decode"])
    types = ["q4_k", "q4_k", "q6_k", "q8_0", "q5_k", "q4_0"]
    if kind == "host":
        return {"kind": kind, "type": rng.choice(types), "rows": _logint(rng, 512, 8192),
                "cols": 256 * rng.randint(4, 32)}
    if kind == "ffn":
        dim = 256 * rng.randint(8, 20)
        return {"kind": kind, "type": rng.choice(["q4_k", "q6_k"]), "dim": dim,
                "hidden": 256 * rng.randint(2 * dim // 256, int(3.5 * dim) // 256)}
    if kind == "matvec":
        return {"kind": kind, "type": rng.choice(types), "rows": _logint(rng, 1000, 14336),
                "cols": 256 * _logint(rng, 6, 56), "p": _logint(rng, 1, 512), "n": 1}
    if kind == "attend":
        return {"kind": kind, "ctx": _logint(rng, 200, 32768), "exact": rng.random() < 0.7}
    if kind == "prefill":
        return {"kind": kind, "layers": rng.randint(2, 4), "p": _logint(rng, 17, 3000)}
    return {"kind": kind, "layers": rng.randint(8, 32), "p": _logint(rng, 100, 2000), "steps": 8}


# --- weights as GGUF blocks -------------------------------------------------


def _generator(seed, key):
    return torch.Generator(device="cuda").manual_seed(1_000_003 * int(seed) + key)


def _rand(gen, shape, lo, hi):
    return torch.randint(lo, hi + 1, shape, generator=gen, device="cuda", dtype=torch.uint8)


def _normal_codes(gen, rows, cols, mean, std, lo, hi):
    """Integers of a rounded normal distribution, cut to lo..hi."""
    v = torch.randn((rows, cols), generator=gen, device="cuda").mul_(std).add_(mean)
    return v.round_().clamp_(lo, hi).to(torch.int16 if lo < 0 else torch.uint8)


def _halves(gen, shape, about):
    """f16 block scales within 20 percent of `about`."""
    r = torch.rand(shape, generator=gen, device="cuda")
    return (about * (0.8 + 0.4 * r)).to(torch.float16)


def _fields(kind, rows, cols, gen):
    """The fields of a rows x cols weight with entries about N(0, 0.02)."""
    nb = cols // 256
    if kind in ("q4_k", "q5_k"):
        top = 15 if kind == "q4_k" else 31
        step = 0.0074 if kind == "q4_k" else 0.0037  # scale of one code
        return {"q": _normal_codes(gen, rows, cols, top / 2, top / 5.6, 0, top),
                "sc": _rand(gen, (rows, nb, 8), 40, 63), "m": _rand(gen, (rows, nb, 8), 40, 63),
                "d": _halves(gen, (rows, nb), step / 52), "dmin": _halves(gen, (rows, nb), step * top / 2 / 52)}
    if kind == "q6_k":
        sc = _rand(gen, (rows, nb, 16), 80, 127).to(torch.int16)
        sign = _rand(gen, (rows, nb, 16), 0, 1).to(torch.int16) * 2 - 1
        return {"q": _normal_codes(gen, rows, cols, 32, 11, 0, 63), "sc": sc * sign,
                "d": _halves(gen, (rows, nb), 0.0018 / 104)}
    if kind == "q8_0":
        return {"q": _normal_codes(gen, rows, cols, 0, 48, -127, 127), "d": _halves(gen, (rows, nb * 8), 0.00042)}
    return {"q": _normal_codes(gen, rows, cols, 8, 2.7, 0, 15), "d": _halves(gen, (rows, nb * 8), 0.0074)}


def _scale_bytes(sc, m):
    """The 12 bytes that hold eight 6-bit scales and eight 6-bit mins."""
    lo, hi = sc[..., :4], sc[..., 4:]
    mlo, mhi = m[..., :4], m[..., 4:]
    return torch.cat([lo | ((hi >> 4) << 6), mlo | ((mhi >> 4) << 6), (hi & 15) | ((mhi & 15) << 4)], -1)


def _bytes_of(h, shape):
    return h.contiguous().view(torch.uint8).view(shape)


def _pack(kind, f):
    """The fields as a GGUF tensor's bytes."""
    rows, cols = f["q"].shape
    nb = cols // 256
    if kind in ("q4_k", "q5_k"):
        q = f["q"].view(rows, nb, 4, 2, 32)
        parts = [_bytes_of(f["d"], (rows, nb, 2)), _bytes_of(f["dmin"], (rows, nb, 2)), _scale_bytes(f["sc"], f["m"])]
        if kind == "q5_k":
            qh = torch.zeros((rows, nb, 32), dtype=torch.uint8, device="cuda")
            for c in range(4):
                qh |= (q[:, :, c, 0] >> 4) << (2 * c)
                qh |= (q[:, :, c, 1] >> 4) << (2 * c + 1)
            parts.append(qh)
        parts.append(((q[:, :, :, 0] & 15) | ((q[:, :, :, 1] & 15) << 4)).reshape(rows, nb, 128))
    elif kind == "q6_k":
        q = f["q"].view(rows, nb, 2, 4, 32)
        ql = torch.cat([(q[:, :, :, 0] & 15) | ((q[:, :, :, 2] & 15) << 4),
                        (q[:, :, :, 1] & 15) | ((q[:, :, :, 3] & 15) << 4)], -1)
        qh = (q[:, :, :, 0] >> 4) | ((q[:, :, :, 1] >> 4) << 2) | ((q[:, :, :, 2] >> 4) << 4) | ((q[:, :, :, 3] >> 4) << 6)
        parts = [ql.reshape(rows, nb, 128), qh.reshape(rows, nb, 64),
                 f["sc"].to(torch.int8).view(torch.uint8), _bytes_of(f["d"], (rows, nb, 2))]
    elif kind == "q8_0":
        parts = [_bytes_of(f["d"], (rows, nb * 8, 2)), f["q"].to(torch.int8).view(torch.uint8).view(rows, nb * 8, 32)]
    else:
        q = f["q"].view(rows, nb * 8, 2, 16)
        parts = [_bytes_of(f["d"], (rows, nb * 8, 2)), q[:, :, 0] | (q[:, :, 1] << 4)]
    return torch.cat(parts, -1).reshape(-1)


def _weight(kind, rows, cols, seed, key):
    raw = _pack(kind, _fields(kind, rows, cols, _generator(seed, key)))
    w = g.Weight.from_device(raw, TYPES[kind], rows, cols)
    torch.cuda.synchronize()  # raw goes back to the allocator here
    return w


def _activations(p, cols, seed, key=99):
    return torch.randn((p, cols), generator=_generator(seed, key), device="cuda")


# --- the same products in 64 bits -------------------------------------------


def _q8k(x):
    """(q, scale) of the int8 activation format: one float32 scale per 256 values."""
    p, cols = x.shape
    v = x.float().view(p, cols // 256, 256)
    amax = v.abs().amax(-1, keepdim=True)
    one = amax.new_full((), 127.0)
    q = torch.where(amax > 0, (v * (one / amax)).round(), torch.zeros_like(v))
    return q.double().view(p, cols), (amax / one).double().expand_as(v).reshape(p, cols)


def _exact_matvec(kind, f, x):
    """x (p, cols) against the fields' weight: the codes meet the int8 activations, the
    format's offset (min, -32, -8) the activations as they are."""
    rows, cols = f["q"].shape
    q8, xs = _q8k(x)
    a = (q8 * xs).T.contiguous()
    xt = x.double().T.contiguous()
    out = torch.empty((x.shape[0], rows), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 26) // cols)
    for r in range(0, rows, step):
        e = {k: v[r:r + step].double() for k, v in f.items()}
        n = e["q"].shape[0]
        if kind in ("q4_k", "q5_k"):
            code = e["q"].view(n, -1, 8, 32) * (e["d"][..., None] * e["sc"])[..., None]
            off = -(e["dmin"][..., None] * e["m"])[..., None].expand_as(code)
        elif kind == "q6_k":
            s = (e["d"][..., None] * e["sc"])[..., None]
            code = e["q"].view(n, -1, 16, 16) * s
            off = (-32.0 * s).expand_as(code)
        else:
            s = e["d"][..., None]
            code = e["q"].view(n, -1, 32) * s
            off = (-8.0 * s).expand_as(code) if kind == "q4_0" else None
        y = code.reshape(n, cols) @ a
        if off is not None:
            y = y + off.reshape(n, cols) @ xt
        out[:, r:r + n] = y.T
    return out


def _silu_mul(gate, up):
    return gate / (1.0 + torch.exp(-gate)) * up


# --- cases ------------------------------------------------------------------


def _model(case, seed):
    cfg = dict(LLAMA3_8B, n_layers=case["layers"])
    return build_decoder(cfg, max_len=4096, seed=int(seed) + 1)


def _prompt(case, seed, n):
    rng = np.random.default_rng(int(seed) + 17)
    return rng.integers(0, LLAMA3_8B["vocab"], n, dtype=np.uint32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "host":
        return {"kind": kind, "w": _weight(case["type"], case["rows"], case["cols"], seed, 1),
                "x": _activations(1, case["cols"], seed)[0].cpu().numpy(), "out": np.empty(case["rows"], np.float32)}
    if kind == "ffn":
        dim, hidden = case["dim"], case["hidden"]
        return {"kind": kind, "gate": _weight(case["type"], hidden, dim, seed, 1),
                "up": _weight(case["type"], hidden, dim, seed, 2), "down": _weight(case["type"], dim, hidden, seed, 3),
                "x": _activations(1, dim, seed), "out": torch.empty((1, dim), device="cuda")}
    if kind == "matvec":
        ws = [_weight(case["type"], case["rows"], case["cols"], seed, 1 + i) for i in range(case["n"])]
        return {"kind": kind, "ws": ws, "x": _activations(case["p"], case["cols"], seed),
                "outs": [torch.empty((case["p"], case["rows"]), device="cuda") for _ in ws]}
    if kind == "attend":
        ctx, kvd = case["ctx"], N_KV * HEAD_DIM
        kv = g.KVCacheF16(1, kvd, kvd, ctx)
        k, v = _activations(ctx, kvd, seed, 5), _activations(ctx, kvd, seed, 6)
        for pos in range(ctx):
            kv.store_kv_dev(0, pos, k[pos], v[pos])
        torch.cuda.synchronize()
        return {"kind": kind, "kv": kv, "q": _activations(1, N_HEADS * HEAD_DIM, seed), "ctx": ctx,
                "mode": _lib.ATTN_EXACT if case["exact"] else _lib.ATTN_SPLITK,
                "out": torch.empty((1, N_HEADS * HEAD_DIM), device="cuda")}
    m = _model(case, seed)
    if kind == "prefill":
        return {"kind": kind, "m": m, "tokens": _prompt(case, seed, case["p"])}
    toks = _prompt(case, seed, case["p"] + case["steps"])
    m.prefill(toks[:case["p"]])
    return {"kind": kind, "m": m, "p": case["p"], "tokens": [int(t) for t in toks[case["p"]:]]}


def run(s):
    kind = s["kind"]
    if kind == "host":
        return s["w"].matvec_into(s["x"], s["out"])
    if kind == "ffn":
        return g.swiglu_down_dev(s["gate"], s["up"], s["down"], s["x"], s["out"])
    if kind == "matvec":
        if len(s["ws"]) == 1:
            return s["ws"][0].matvec_dev(s["x"], s["outs"][0])
        g.matvec_multi_dev(s["ws"], s["x"], s["outs"])
        return s["outs"]
    if kind == "attend":
        return s["kv"].attend_dev(0, s["q"], N_HEADS, N_KV, HEAD_DIM, 0, s["ctx"] - 1, HEAD_DIM ** -0.5, s["out"],
                                  mode=s["mode"])
    if kind == "prefill":
        first, logits = s["m"].prefill(s["tokens"], want_logits=True)
        return {"first": first, "logits": logits, "hidden": s["m"].hidden()}
    # the tokens a sampler on the host chose; each step's greedy token comes back beside them
    greedy = [s["m"].decode(t, s["p"] + i) for i, t in enumerate(s["tokens"])]
    return {"greedy": greedy, "hidden": s["m"].hidden()}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "decode"):
        return None
    if kind == "host":
        f = _fields(case["type"], case["rows"], case["cols"], _generator(seed, 1))
        return _exact_matvec(case["type"], f, _activations(1, case["cols"], seed))[0].cpu().numpy()
    if kind == "ffn":
        t, dim, hidden = case["type"], case["dim"], case["hidden"]
        x = _activations(1, dim, seed)
        gate = _exact_matvec(t, _fields(t, hidden, dim, _generator(seed, 1)), x)
        up = _exact_matvec(t, _fields(t, hidden, dim, _generator(seed, 2)), x)
        return _exact_matvec(t, _fields(t, dim, hidden, _generator(seed, 3)), _silu_mul(gate, up))
    if kind == "matvec":
        x = _activations(case["p"], case["cols"], seed)
        ys = [_exact_matvec(case["type"], _fields(case["type"], case["rows"], case["cols"], _generator(seed, 1 + i)), x)
              for i in range(case["n"])]
        return ys[0] if len(ys) == 1 else ys
    ctx = case["ctx"]
    k = _activations(ctx, N_KV * HEAD_DIM, seed, 5).half().double().view(ctx, N_KV, 1, HEAD_DIM)
    v = _activations(ctx, N_KV * HEAD_DIM, seed, 6).half().double().view(ctx, N_KV, HEAD_DIM)
    q = _activations(1, N_HEADS * HEAD_DIM, seed).double().view(1, N_KV, N_HEADS // N_KV, HEAD_DIM)
    w = ((k * q).sum(-1) * HEAD_DIM ** -0.5).softmax(0)  # (ctx, kv head, query head)
    return (w[..., None] * v[:, :, None]).sum(0).reshape(1, -1)


def _weight_bytes(kind, rows, cols):
    return rows * (cols // 256) * BLOCK_BYTES[kind]


def work(case):
    kind = case["kind"]
    if kind == "host":
        r, c = case["rows"], case["cols"]
        return {"bytes": _weight_bytes(case["type"], r, c) + 4 * (r + c), "flops": 2 * r * c}
    if kind == "ffn":
        d, h = case["dim"], case["hidden"]
        return {"bytes": 3 * _weight_bytes(case["type"], h, d) + 8 * d, "flops": 6 * d * h}
    if kind == "matvec":
        r, c, p, n = case["rows"], case["cols"], case["p"], case["n"]
        return {"bytes": n * _weight_bytes(case["type"], r, c) + 4 * p * (c + n * r), "flops": 2 * n * p * r * c}
    if kind == "attend":
        row = N_KV * HEAD_DIM * 2 * 2
        return {"bytes": case["ctx"] * row + 8 * N_HEADS * HEAD_DIM, "flops": 4 * case["ctx"] * N_HEADS * HEAD_DIM}
    c = LLAMA3_8B
    per_layer = c["dim"] * (2 * c["dim"] + 2 * N_KV * HEAD_DIM + 3 * c["hidden"])
    weights = case["layers"] * per_layer
    layer_bytes = weights // 256 * BLOCK_BYTES["q4_k"]
    head_bytes = c["vocab"] * c["dim"] // 256 * BLOCK_BYTES["q6_k"]
    kv_row = case["layers"] * N_KV * HEAD_DIM * 2 * 2
    pairs = case["layers"] * N_HEADS * HEAD_DIM * 4  # attention, per (token, position)
    p = case["p"]
    if kind == "prefill":
        return {"bytes": layer_bytes + head_bytes + p * kv_row + 4 * c["vocab"],
                "flops": 2 * p * weights + pairs * p * (p + 1) // 2 + 2 * c["vocab"] * c["dim"]}
    n = case["steps"]
    return {"bytes": n * (layer_bytes + head_bytes + p * kv_row),
            "flops": n * (2 * weights + pairs * p + 2 * c["vocab"] * c["dim"])}


def tolerance(case):
    """What sums of float32 in another order change; about four times what was seen between
    each path and its 64-bit form."""
    kind = case["kind"]
    if kind in ("prefill", "decode"):
        # Greedy tokens and hidden states are defined bit for bit.  No looser bound would tell a
        # right result from a wrong one: raising half of one norm's weights by their last bit
        # moves int8 roundings in every later layer, and with them the logits by 0.04 (two
        # layers) to 0.35 (32 layers) of their norm.
        return "exact"
    if kind == "ffn":
        # a few of the hidden values' int8 roundings fall the other way (7e-4 seen)
        return {"rel": 3e-3, "max": 2e-2}
    if kind == "attend":
        return {"rel": 8e-6, "max": 8e-5}  # 2e-6 seen
    return {"rel": 3e-6, "max": 3e-5}  # 6e-7 seen
