"""The framework's work as cases that can be timed: single operators, the sampler, the isolated recurrence, whole
decode steps and speculative rounds, and prompts, each through the public entry points of the `aqueduct` package.

A case is a dict of plain values; its "kind" says which part of the framework it runs:

  op          quantise activation rows and multiply them by one ggml weight matrix on the caller's stream: every
              projection of a model is such a call (1 column: plain decode; 2..8: a speculative verify; 9..64: a prompt
              chunk), in each weight type of the Q4_K_M mix, with and without the q8-fine activations
  recurrence  the Gated-DeltaNet recurrence of one verify batch with rollback to the kept rows
  sample      one logits row through the sampler (top-k / top-p / min-p), a draw, and the distribution it was drawn
              from: what proposing a draft takes
  decode      one plain greedy step of a model at some context, logits to the host
  round       one greedy speculative round of a model at some context
  prompt      a request's start: a new sequence state, its prompt, the logits of the last row (k = 0) or the first
              speculative round (k > 0)

Models are the 27B hybrid's shapes with random weights: all 64 layers ("layers": 64, vocabulary 248320), or one
interval of it ("layers": 4: three DeltaNet layers and one attention layer, every width as in the whole model,
vocabulary 32768), which is what a pass spends its time on without the length.
"""
import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "qwen-3.8-in-rust_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import aqueduct as aq  # noqa: E402

TYPES = {"q4_k": aq.Q4_K, "q5_k": aq.Q5_K, "q6_k": aq.Q6_K, "q8_0": aq.Q8_0, "q4_0": aq.Q4_0}
_ctx = _stream = None


def context():
    global _ctx
    if _ctx is None:
        _ctx = aq.Context(0)
    return _ctx


def stream():
    """The one stream a program queues its operators on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream.cuda_stream


def op(weight, rows, cols, n, fine=False):
    return {"kind": "op", "weight": weight, "rows": rows, "cols": cols, "n": n, "fine": fine}


def recurrence(nk, nv, d, t, keep):
    return {"kind": "recurrence", "nk": nk, "nv": nv, "d": d, "t": t, "keep": keep}


def sample(vocab, top_k, top_p, min_p, temperature):
    return {"kind": "sample", "vocab": vocab, "top_k": top_k, "top_p": top_p, "min_p": min_p,
            "temperature": temperature}


def decode(layers, context_len):
    return {"kind": "decode", "layers": layers, "context": context_len}


def spec_round(layers, context_len, k):
    return {"kind": "round", "layers": layers, "context": context_len, "k": k}


def prompt(layers, length, k):
    return {"kind": "prompt", "layers": layers, "length": length, "k": k}


def listed():
    return [
        # the smallest projection of a decode step (an output projection at one column): launch and latency count
        dict(op("q4_k", 5120, 6144, 1), name="matvec_q4k_5120x6144"),
        # the down projection over a --spec 3 verify batch
        dict(op("q6_k", 5120, 17408, 4), name="verify_q6k_5120x17408_n4"),
        # gate / up over a whole prompt chunk
        dict(op("q4_k", 17408, 5120, 64), name="prompt_q4k_17408x5120_n64"),
        # the down projection over a prompt's last, ragged chunk
        dict(op("q6_k", 5120, 17408, 37), name="prompt_q6k_5120x17408_n37"),
        # gate / up over a verify batch with the q8-fine activations
        dict(op("q4_k", 17408, 5120, 4, True), name="fine_q4k_17408x5120_n4"),
        # a layer's recurrence in a --spec 3 round that keeps two rows
        dict(recurrence(16, 48, 128, 4, 2), name="recurrence_48x128_t4"),
        # the usual chat sampling of one row of logits
        dict(sample(248320, 40, 0.95, 0.0, 0.8), name="sample_248320_top40"),
        # plain greedy decode of the whole model early in a conversation
        dict(decode(64, 64), name="decode_27b_at_64"),
        # greedy speculative decode of the whole model in a conversation of some length
        dict(spec_round(64, 1000, 3), name="round_27b_at_1000"),
        # the same on one interval of layers with a document in the context
        dict(spec_round(4, 8000, 3), name="round_block_at_8000"),
        # an ordinary prompt whose last chunk is ragged, plain decode to follow
        dict(prompt(4, 777, 0), name="prompt_block_777"),
        # a document as the prompt, speculative decode to follow
        dict(prompt(4, 5000, 3), name="prompt_block_5000_spec"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["op", "op", "op", "op", "recurrence", "sample", "decode", "round", "round", "prompt", "prompt"])
    if kind == "op":
        weight = rng.choice(["q4_k", "q4_k", "q6_k", "q6_k", "q5_k", "q8_0", "q4_0"])
        fine = weight in ("q4_k", "q5_k", "q6_k") and rng.random() < 0.2
        return op(weight, _log_int(rng, 300, 17408), 256 * _log_int(rng, 4, 68), _log_int(rng, 1, 64), fine)
    if kind == "recurrence":
        nk = rng.choice([4, 8, 16, 24])
        t = rng.randint(1, 8)
        return recurrence(nk, nk * rng.randint(1, 3), rng.choice([64, 128]), t, rng.randint(1, t))
    if kind == "sample":
        return sample(_log_int(rng, 4096, 248320), rng.choice([0, 20, 40, 100]), rng.choice([1.0, 0.95, 0.8]),
                      rng.choice([0.0, 0.05]), rng.choice([0.6, 0.8, 1.0]))
    if kind == "decode":
        return decode(4, _log_int(rng, 16, 8000))
    if kind == "round":
        return spec_round(4, _log_int(rng, 16, 8000), rng.choice([1, 2, 3, 3, 5, 7]))
    return prompt(4, _log_int(rng, 9, 4000), rng.choice([0, 0, 3]))


# ------------------------------------------------------------------------------------------------ weights, rows
def _codes(g, shape, mean, sigma, lo, hi):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return (x * sigma + mean).round_().clamp_(lo, hi).to(torch.int16)


def _f16_bytes(x):
    return x.to(torch.float16).view(torch.uint8).reshape(*x.shape, 2)


def _weight(case, seed):
    """(ggml bytes, values in float64) of a matrix with bell-shaped codes, as quantised weights have them."""
    t, rows, cols = case["weight"], case["rows"], case["cols"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    u8 = torch.uint8

    def uniform(shape, lo, hi):
        return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo

    if t in ("q8_0", "q4_0"):
        nb = cols // 32
        d = uniform((rows, nb), 4e-4, 6e-4) * (1.0 if t == "q8_0" else 16.0)
        if t == "q8_0":
            q = _codes(g, (rows, nb, 32), 0, 40, -127, 127)
            raw = torch.cat([_f16_bytes(d), q.to(torch.int8).view(u8)], -1)
        else:
            q = _codes(g, (rows, nb, 32), 8, 3, 0, 15)
            raw = torch.cat([_f16_bytes(d), (q[..., :16] | (q[..., 16:] << 4)).to(u8)], -1)
            q = q - 8
        return raw, lambda: (q.double() * d.to(torch.float16).double()[..., None]).reshape(rows, cols)
    nb = cols // 256
    if t == "q6_k":
        q = _codes(g, (rows, nb, 256), 32, 11, 0, 63)
        sc = (uniform((rows, nb, 16), 70, 127.9).floor() * torch.sign(uniform((rows, nb, 16), -1, 1) + 1e-9)).to(
            torch.int16)
        d = uniform((rows, nb), 1.5e-5, 2.5e-5)
        h = q.reshape(rows, nb, 2, 4, 32)  # half, quarter of it, position
        ql = torch.cat([(h[..., 0, :] & 15) | ((h[..., 2, :] & 15) << 4),
                        (h[..., 1, :] & 15) | ((h[..., 3, :] & 15) << 4)], -1).reshape(rows, nb, 128)
        qh = ((h[..., 0, :] >> 4) | ((h[..., 1, :] >> 4) << 2) | ((h[..., 2, :] >> 4) << 4) |
              ((h[..., 3, :] >> 4) << 6)).reshape(rows, nb, 64)
        raw = torch.cat([ql.to(u8), qh.to(u8), sc.to(torch.int8).view(u8), _f16_bytes(d)], -1)
        return raw, lambda: ((q.double() - 32).reshape(rows, nb, 16, 16) * sc.double()[..., None] *
                             d.to(torch.float16).double()[..., None, None]).reshape(rows, cols)
    top = 15 if t == "q4_k" else 31
    q = _codes(g, (rows, nb, 256), top / 2, top / 5, 0, top)
    sc = uniform((rows, nb, 8), 30, 63.9).floor().to(torch.int16)
    mn = uniform((rows, nb, 8), 30, 63.9).floor().to(torch.int16)
    d = uniform((rows, nb), 1.0e-4, 1.6e-4) * (15 / top)
    dmin = uniform((rows, nb), 0.8e-3, 1.2e-3)
    packed = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6),
                        (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)
    h = q.reshape(rows, nb, 4, 2, 32)  # pair of sub-blocks, which of the pair, position
    qs = ((h[..., 0, :] & 15) | ((h[..., 1, :] & 15) << 4)).reshape(rows, nb, 128)
    parts = [_f16_bytes(d), _f16_bytes(dmin), packed.to(u8)]
    if t == "q5_k":
        bits = torch.arange(8, device="cuda", dtype=torch.int16)[:, None]
        parts.append(((q.reshape(rows, nb, 8, 32) >> 4) << bits).sum(-2).to(u8))
    raw = torch.cat(parts + [qs.to(u8)], -1)

    def values():
        dd, dm = d.to(torch.float16).double(), dmin.to(torch.float16).double()
        v = q.double().reshape(rows, nb, 8, 32) * (sc.double() * dd[..., None])[..., None]
        return (v - (mn.double() * dm[..., None])[..., None]).reshape(rows, cols)

    return raw, values


def _rows(case, seed):
    """Activation rows as a norm gives them: about unit variance, a few channels far larger."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((case["n"], case["cols"]), dtype=np.float32)
    x[:, rng.integers(0, case["cols"], max(1, case["cols"] // 500))] *= 8.0
    return x


# ------------------------------------------------------------------------------------------------------ prepare
def _config(layers):
    cfg = aq.config_27b()
    if layers != cfg.n_layer:
        cfg.n_layer, cfg.vocab = layers, 32768
    return cfg


def _tokens(seed, n, vocab):
    return np.random.default_rng(seed).integers(0, vocab, n).astype(np.uint32)


def _buffer(t):
    """A torch tensor where the package takes one of its device buffers."""
    return SimpleNamespace(p=t.data_ptr())


def _prepare_op(case, seed):
    ctx, t = context(), TYPES[case["weight"]]
    raw, _ = _weight(case, seed)
    w = aq.Weight(ctx, t, case["rows"], case["cols"], raw.cpu().numpy().reshape(-1))
    a = aq.Act(ctx, case["cols"], case["n"])
    a.set(_rows(case, seed))
    y = torch.zeros(case["n"], case["rows"], device="cuda")
    torch.cuda.synchronize()
    return {"case": case, "w": w, "a": a, "y": y, "yb": _buffer(y), "type": t}


def _run_op(s):
    case = s["case"]
    handle = stream()
    if case["fine"]:
        with aq.q8_fine():
            aq.quantize_on(s["a"], s["type"], case["n"], handle)
            aq.matmul_on(context(), s["w"], s["a"], case["n"], s["yb"], handle)
    else:
        aq.quantize_on(s["a"], s["type"], case["n"], handle)
        aq.matmul_on(context(), s["w"], s["a"], case["n"], s["yb"], handle)
    return s["y"]


def _recurrence_inputs(case, seed):
    rng = np.random.default_rng(seed)
    nk, nv, d, t = case["nk"], case["nv"], case["d"], case["t"]

    def unit(*shape):
        x = rng.standard_normal(shape)
        return x / np.linalg.norm(x, axis=-1, keepdims=True)

    q, k = unit(t, nk, d) / math.sqrt(d), unit(t, nk, d)
    v = rng.standard_normal((t, nv, d))
    g = -rng.exponential(0.3, (t, nv))
    beta = 1.0 / (1.0 + np.exp(-rng.standard_normal((t, nv))))
    state = rng.standard_normal((nv, d, d)) * 0.3
    return [np.ascontiguousarray(x, dtype=np.float32) for x in (q, k, v, g, beta, state)]


def _prepare_recurrence(case, seed):
    dev = [torch.from_numpy(x).cuda() for x in _recurrence_inputs(case, seed)]
    out = torch.zeros(case["t"], case["nv"], case["d"], device="cuda")
    torch.cuda.synchronize()
    return {"case": case, "dev": dev, "buf": [_buffer(x) for x in dev], "out": out, "outb": _buffer(out)}


def _run_recurrence(s):
    c = s["case"]
    q, k, v, g, beta, state = s["buf"]
    aq.deltanet_verify_commit_dev(context(), c["nk"], c["nv"], c["d"], c["d"], c["t"], c["keep"], q, k, v, g, beta,
                                  state, s["outb"])
    return {"out": s["out"], "state": s["dev"][5]}


def _logits(case, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal(case["vocab"]) * 2.5).astype(np.float32)


def _prepare_sample(case, seed):
    logits = torch.from_numpy(_logits(case, seed)).cuda()
    dense = torch.zeros_like(logits)
    torch.cuda.synchronize()
    cfg = aq.sampler_config(case["temperature"], case["top_k"], case["top_p"], case["min_p"], seed)
    return {"sampler": aq.Sampler(context(), cfg, case["vocab"]), "logits": logits, "buf": _buffer(logits),
            "dense": dense, "denseb": _buffer(dense)}


def _run_sample(s):
    token = s["sampler"].sample(s["buf"])
    s["sampler"].write_dense(s["denseb"])
    return {"token": token, "probs": s["dense"]}


def _prepare_model(case, seed):
    cfg = _config(case["layers"])
    s = {"case": case, "model": aq.Model(context(), cfg, mix=aq.MIX_Q4_K_M, seed=seed)}
    if case["kind"] == "prompt":
        s["ids"] = _tokens(seed, case["length"], cfg.vocab)
        return s
    ids = _tokens(seed, case["context"], cfg.vocab)
    room = 4000 if case["layers"] > 4 else 16000  # positions for the tokens that repeated passes add
    s["state"] = aq.State(s["model"], case.get("k", 0), case["context"] + room)
    s["last"] = s["state"].spec_prefill(ids) if case["kind"] == "round" else s["state"].prefill(ids)
    return s


def _run_decode(s):
    s["last"], logits = s["state"].forward_token(s["last"], want_logits=True)
    return {"token": s["last"], "logits": logits}


def _round(state, x_p, k):
    m, emitted = state.spec_round(x_p)
    return emitted, {"accepted": m, "emitted": np.array(emitted, np.int64), "logits": state.logits_row(k)}


def _run_round(s):
    emitted, out = _round(s["state"], s["last"], s["case"]["k"])
    s["last"] = emitted[-1]
    return out


def _run_prompt(s):
    k, n = s["case"]["k"], len(s["ids"])
    state = aq.State(s["model"], k, n + 64)
    if k:
        out = _round(state, state.spec_prefill(s["ids"]), k)[1]
    else:
        token, logits = state.prefill(s["ids"], want_logits=True)
        out = {"token": token, "logits": logits}
    state.free()
    return out


def prepare(case, seed):
    return {"op": _prepare_op, "recurrence": _prepare_recurrence, "sample": _prepare_sample, "decode": _prepare_model,
            "round": _prepare_model, "prompt": _prepare_model}[case["kind"]](case, seed) | {"kind": case["kind"]}


def run(state):
    return {"op": _run_op, "recurrence": _run_recurrence, "sample": _run_sample, "decode": _run_decode,
            "round": _run_round, "prompt": _run_prompt}[state["kind"]](state)


# ------------------------------------------------------------------------------------------------------ bounds
def _model_work(case):
    """Weights once, the state and the cached rows once; two operations per weight and row."""
    cfg = _config(case["layers"])
    plan = aq.model_plan(cfg, aq.MIX_Q4_K_M, 1)
    mtp = "blk.%d." % cfg.n_layer
    size = {name: (sp.rows * aq.row_bytes(sp.ggml_type, sp.cols), sp.rows * sp.cols) for name, sp in plan}
    main = [v for n, v in size.items() if n.startswith("blk.") and not n.startswith(mtp)]
    draft = [v for n, v in size.items() if n.startswith(mtp)]
    head = size["output.weight"]
    n_att = cfg.n_layer // cfg.full_attention_interval
    n_dn = cfg.n_layer - n_att
    kv_row = 2 * cfg.n_head_kv * cfg.head_dim * 4
    rec = n_dn * cfg.dn_n_v_heads * cfg.dn_head_dim_k * cfg.dn_head_dim_v * 4

    def pass_flops(rows, ctx):
        return rows * (2 * sum(v[1] for v in main) + 8 * rec / 4 + n_att * 4 * cfg.n_head * cfg.head_dim * ctx)

    main_bytes, draft_bytes = sum(v[0] for v in main), sum(v[0] for v in draft)
    logits = cfg.vocab * 4

    def round_work(ctx, k):
        b = main_bytes + head[0] + (k + 1) * logits + 3 * rec + n_att * kv_row * ctx
        b += k * (draft_bytes + head[0] + kv_row * ctx)
        f = pass_flops(k + 1, ctx) + 2 * head[1] * (2 * k + 1) + 2 * k * sum(v[1] for v in draft)
        return b, f + k * 4 * cfg.n_head * cfg.head_dim * ctx

    if case["kind"] == "decode":
        ctx = case["context"]
        return (main_bytes + head[0] + logits + 2 * rec + n_att * kv_row * ctx, pass_flops(1, ctx) + 2 * head[1])
    if case["kind"] == "round":
        return round_work(case["context"], case["k"])
    n, k = case["length"], case["k"]
    b = main_bytes + head[0] + logits + rec + n_att * kv_row * n
    f = pass_flops(n, n / 2) + 2 * head[1]
    if k:
        rb, rf = round_work(n, k)
        b += rb + draft_bytes + kv_row * n
        f += rf + n * (2 * sum(v[1] for v in draft) + 4 * cfg.n_head * cfg.head_dim * n / 2)
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "op":
        r, c, n = case["rows"], case["cols"], case["n"]
        b, f = r * aq.row_bytes(TYPES[case["weight"]], c) + 4 * n * (c + r), 2 * r * c * n
    elif kind == "recurrence":
        t, d, nv = case["t"], case["d"], case["nv"]
        b = 4 * (2 * nv * d * d + t * (2 * case["nk"] * d + 2 * nv * d + 2 * nv))
        f = (t + case["keep"]) * nv * 7 * d * d
    elif kind == "sample":
        b, f = 4 * case["vocab"], 2 * case["vocab"]
    else:
        b, f = _model_work(case)
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    kind = case["kind"]
    if kind == "op":
        return {"rel": 2.5e-6}
    if kind == "recurrence":
        return {"rel": 1e-6}
    if kind == "sample":
        return {"rel": 1.5e-6, "differ": 0.01}
    # activations are quantised to 8 bits before every projection, so another order of a sum moves codes here and
    # there and the difference travels through the layers that follow (last-bit changes of one norm's weights move
    # the logits of four layers by 2.5e-2 and of all 64 by 0.12, the largest difference by 0.12 and 0.56 of their size)
    return {"rel": 0.03, "max": 0.5, "differ": 0.01}


# ------------------------------------------------------------------------------------------------------- exact
def _quantised(x, kind):
    """The rows' values after the 8-bit quantiser (part of the format, so its codes are made in 32 bits as it says):
    one scale per 256 values, or one 16-bit scale per 32."""
    n, cols = x.shape
    f = np.float32
    if kind == "q8_k":
        b = x.reshape(n, -1, 256)
        at = np.abs(b).argmax(-1)
        top = np.take_along_axis(b, at[..., None], -1)
        iscale = f(-127.0) / np.where(top == 0, f(1), top)
        q = np.where(top == 0, 0, np.minimum(127, np.rint(iscale * b)))
        d = np.where(top == 0, 0, f(1.0) / iscale)
    else:
        b = x.reshape(n, -1, 32)
        top = np.abs(b).max(-1, keepdims=True)
        d = top / f(127.0)
        inv = np.where(d == 0, f(0), f(1.0) / np.where(d == 0, f(1), d))
        v = (b * inv).astype(f)
        q = np.sign(v) * np.floor(np.abs(v).astype(np.float64) + 0.5)
        d = d.astype(np.float16)
    return (q.astype(np.float64) * d.astype(np.float64)).reshape(n, cols)


def _exact_op(case, seed):
    _, values = _weight(case, seed)
    kind = "q8_k" if case["weight"] in ("q4_k", "q5_k", "q6_k") and not case["fine"] else "q8_0"
    x = torch.from_numpy(_quantised(_rows(case, seed), kind)).cuda()
    return x @ values().T


def _exact_recurrence(case, seed):
    q, k, v, g, beta, state = (torch.from_numpy(x).double() for x in _recurrence_inputs(case, seed))
    heads = torch.arange(case["nv"]) % case["nk"]
    s, out, kept = state.clone(), [], None
    for i in range(case["t"]):
        qi, ki = q[i][heads], k[i][heads]
        s = s * torch.exp(g[i])[:, None, None]
        delta = (v[i] - (s * ki[:, :, None]).sum(1)) * beta[i][:, None]
        s = s + ki[:, :, None] * delta[:, None, :]
        out.append((s * qi[:, :, None]).sum(1))
        if i + 1 == case["keep"]:
            kept = s
    return {"out": torch.stack(out), "state": kept}


def _exact_sample(case, seed):
    x = _logits(case, seed).astype(np.float64)
    ids = np.lexsort((np.arange(x.size), -x))
    if case["top_k"]:
        ids = ids[: case["top_k"]]
    p = np.exp((x[ids] - x[ids[0]]) / float(np.float32(case["temperature"])))
    p /= p.sum()
    if case["top_p"] < 1:
        n = int(np.searchsorted(np.cumsum(p), float(np.float32(case["top_p"])))) + 1
        ids, p = ids[:n], p[:n]
    if case["min_p"] > 0:
        keep = p >= float(np.float32(case["min_p"])) * p[0]
        ids, p = ids[keep], p[keep]
    dense = np.zeros(case["vocab"])
    dense[ids] = p / p.sum()
    return {"token": None, "probs": dense}


def exact(case, seed):
    f = {"op": _exact_op, "recurrence": _exact_recurrence, "sample": _exact_sample}.get(case["kind"])
    return f(case, seed) if f else None
