"""The work that programs have this framework do, as cases that can be timed and checked.

A case is one layer, one operation over a long context, or one whole model call, through
the public entry points (``emprise_amd.HipBackend`` and ``emprise_amd.Model``):

  ffn        an FFN with its norm: one token (decode), a few (draft verification), a
             prompt or a prompt chunk
  recurrent  one Gated DeltaNet block, one token
  delta      the Gated DeltaNet over a prompt's positions
  attn_step  gated attention of one token over a filled KV cache
  attn_chunk gated attention of a prompt chunk behind earlier positions
  model      a prompt, then greedy tokens, then the logits of the last one

Widths are those of the two model shapes the package names (TINY, NINE_B) and 1024 and
2048 between them. Activations are normal, weights as ``emprise_synth_write`` draws them.
"""
import math
import os
import struct
import tempfile

import numpy as np
import torch

import emprise_amd as ea

EPS = 1e-6
ROPE_BASE = 1e7
TYPES = {"q6_k": ea.Q6_K, "q4_k": ea.Q4_K}

# (heads, kv_heads, head_dim, rotary) of the named shapes
HEADS = {"9b": (16, 4, 256, 64), "tiny": (8, 2, 64, 16)}
# (key_heads, value_heads, state_dim, conv_width)
STATES = {"9b": (16, 32, 128, 4), "tiny": (4, 8, 64, 4)}
# model shapes: the smallest one whole, and four layers at the full widths
MODELS = {
    "tiny": dict(ea.TINY),
    "narrow": dict(ea.TINY, hidden=1024, ffn=3072, vocab=8192, eos=8192),
    "wide": dict(ea.NINE_B, layers=4, vocab=16384, eos=16384, context_length=4096),
}


def listed():
    return [
        # the smallest model: a short prompt and a few tokens, bound by launches
        {"name": "model_tiny", "kind": "model", "shape": "tiny", "mix": False, "prompt": 16, "count": 24},
        # the full widths: a chat turn's prompt, then decode steps
        {"name": "model_wide", "kind": "model", "shape": "wide", "mix": True, "prompt": 160, "count": 16},
        # decode: one block of each kind at the full widths
        {"name": "recurrent_step", "kind": "recurrent", "shape": "9b", "hidden": 4096, "type": "q6_k"},
        {"name": "ffn_step", "kind": "ffn", "tokens": 1, "hidden": 4096, "ffn": 12288, "type": "q6_k", "q8": False},
        # decode of a smaller model
        {"name": "ffn_step_narrow", "kind": "ffn", "tokens": 1, "hidden": 2048, "ffn": 6144, "type": "q4_k", "q8": False},
        # draft verification
        {"name": "ffn_draft", "kind": "ffn", "tokens": 5, "hidden": 4096, "ffn": 12288, "type": "q4_k", "q8": False},
        # a short prompt, a longer one on a smaller model, a full prefill chunk
        {"name": "ffn_prompt", "kind": "ffn", "tokens": 99, "hidden": 4096, "ffn": 12288, "type": "q6_k", "q8": False},
        {"name": "ffn_prompt_narrow", "kind": "ffn", "tokens": 700, "hidden": 2048, "ffn": 6144, "type": "q4_k", "q8": False},
        {"name": "ffn_chunk", "kind": "ffn", "tokens": 2048, "hidden": 4096, "ffn": 12288, "type": "q6_k", "q8": False},
        # one token late in a long conversation; the third chunk of a long prompt
        {"name": "attn_step_long", "kind": "attn_step", "shape": "9b", "position": 30000},
        {"name": "attn_chunk", "kind": "attn_chunk", "shape": "9b", "first": 4096, "count": 2048},
        # the recurrence of a prompt of ordinary length
        {"name": "delta_prompt", "kind": "delta", "shape": "9b", "count": 777},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ffn", "ffn", "ffn", "recurrent", "attn_step", "attn_chunk", "delta", "model"])
    if kind == "ffn":
        hidden = rng.choice([512, 768, 1024, 1536, 2048, 2560, 3072, 4096, 4096, 4096])
        c = {"kind": kind, "tokens": 1 if rng.random() < 0.25 else _log(rng, 2, 2047), "hidden": hidden,
             "ffn": 4096 * rng.randint(1, 3) if rng.random() < 0.3 else 256 * rng.randint(hidden // 256, hidden * 3 // 256),
             "type": rng.choice(["q6_k", "q4_k"]), "q8": False}
        c["q8"] = c["tokens"] == 1 and c["type"] == "q6_k" and rng.random() < 0.5  # --fast-q8
        return c
    if kind == "recurrent":
        return {"kind": kind, "shape": rng.choice(["9b", "tiny"]), "hidden": 256 * rng.randint(2, 15),
                "type": rng.choice(["q6_k", "q4_k"])}
    if kind == "attn_step":
        return {"kind": kind, "shape": rng.choice(["9b", "tiny"]), "position": _log(rng, 1, 32760)}
    if kind == "attn_chunk":
        first = 0 if rng.random() < 0.4 else rng.randint(1, 4095)
        return {"kind": kind, "shape": rng.choice(["9b", "tiny"]), "first": first, "count": _log(rng, 2, 2047)}
    if kind == "delta":
        return {"kind": kind, "shape": rng.choice(["9b", "tiny"]), "count": _log(rng, 2, 2047)}
    return {"kind": kind, "shape": rng.choice(["tiny", "narrow"]), "mix": rng.random() < 0.5,
            "prompt": _log(rng, 2, 400), "count": rng.randint(1, 24)}


def tolerance(case):
    # FP32 sums in another order: a layer differs by a few 1e-7 of its norm; a whole model
    # carries each layer's rounding through all that follow
    if case["kind"] == "model":
        return {"rel": 1e-4, "max": 2e-3}
    if case.get("q8"):
        return {"rel": 2e-3, "max": 0.05}  # a value that lands on the other side of a code's edge
    if case["kind"] in ("recurrent", "ffn"):
        return {"rel": 1e-5, "max": 2e-4}
    return {"rel": 6e-6, "max": 2e-4}


# ---- inputs ---------------------------------------------------------------------------


def _rng(case, seed, salt):
    return np.random.default_rng([seed, salt])


def _normal(gen, *shape, scale=1.0):
    return torch.randn(*shape, generator=gen, device="cuda") * scale


def _blocks(rng, wtype, rows, cols):
    """GGUF blocks of a rows x cols matrix, with emprise_synth_write's distributions."""
    n = rows * cols // 256
    size = 210 if wtype == ea.Q6_K else 144
    b = np.frombuffer(rng.bytes(n * size), np.uint8).reshape(n, size).copy()
    if wtype == ea.Q6_K:
        b[:, 192:208] = ((b[:, 192:208] & 63).astype(np.int8) - 32).view(np.uint8)
        b[:, 208:210] = (np.abs(rng.standard_normal(n)) * 2e-4).astype(np.float16)[:, None].view(np.uint8)
    else:
        b[:, 0:4] = (np.abs(rng.standard_normal((n, 2))) * 1e-3).astype(np.float16).view(np.uint8)
    return b


def _vector(rng, n, kind="norm"):
    z = rng.standard_normal(n)
    v = {"norm": 1 + 0.02 * z, "a": -np.exp(0.5 * z - 2), "dt": 0.5 * z - 1, "conv": 0.5 * z}[kind]
    return v.astype(np.float32)


def _ffn_weights(case, seed):
    rng, t, H, F = _rng(case, seed, 1), TYPES[case["type"]], case["hidden"], case["ffn"]
    return {"gate": _blocks(rng, t, F, H), "up": _blocks(rng, t, F, H), "down": _blocks(rng, t, H, F),
            "norm": _vector(rng, H)}


def _recurrent_weights(case, seed):
    kh, vh, sd, cw = STATES[case["shape"]]
    rng, t, H = _rng(case, seed, 2), TYPES[case["type"]], case["hidden"]
    ch, vd = (2 * kh + vh) * sd, vh * sd
    w = {"qkv": _blocks(rng, t, ch, H), "z": _blocks(rng, t, vd, H), "alpha": _blocks(rng, t, vh, H),
         "beta": _blocks(rng, t, vh, H), "out": _blocks(rng, t, H, vd), "attn_norm": _vector(rng, H)}
    w.update(_delta_weights(case, seed))
    return w


def _delta_weights(case, seed):
    kh, vh, sd, cw = STATES[case["shape"]]
    rng = _rng(case, seed, 3)
    return {"conv": _vector(rng, (2 * kh + vh) * sd * cw, "conv"), "a": _vector(rng, vh, "a"),
            "dt": _vector(rng, vh, "dt"), "norm": _vector(rng, sd)}


def _attn_weights(case, seed):
    hd = HEADS[case["shape"]][2]
    rng = _rng(case, seed, 4)
    return {"q_norm": _vector(rng, hd), "k_norm": _vector(rng, hd)}


def _inputs(case, seed):
    """The activations and states of a case, on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1))
    k = case["kind"]
    if k == "ffn":
        return {"x": _normal(g, case["tokens"], case["hidden"]), "delta": _normal(g, case["tokens"], case["hidden"])}
    if k in ("recurrent", "delta"):
        kh, vh, sd, cw = STATES[case["shape"]]
        ch, vd = (2 * kh + vh) * sd, vh * sd
        s = {"conv_state": _normal(g, ch, cw), "rec_state": _normal(g, vh, sd, sd, scale=0.1)}
        if k == "recurrent":
            s["x"], s["delta"] = _normal(g, case["hidden"]), _normal(g, case["hidden"])
        else:
            s["rows"] = _normal(g, case["count"], ch + vd + 2 * vh)
        return s
    heads, kv, hd, _ = HEADS[case["shape"]]
    past = case["position"] if k == "attn_step" else case["first"]
    n = 1 if k == "attn_step" else case["count"]
    s = {"keys": torch.zeros(past + n, kv, hd, device="cuda"), "values": torch.zeros(past + n, kv, hd, device="cuda")}
    s["keys"][:past] = _normal(g, past, kv, hd)
    s["values"][:past] = _normal(g, past, kv, hd)
    s["rows"] = _normal(g, n, heads * hd * 2 + 2 * kv * hd)
    return s


def _model_file(case, seed):
    fd, path = tempfile.mkstemp(suffix=".gguf")
    os.close(fd)
    ea.synth_write(path, seed=seed, q4_k_m_mix=case["mix"], **MODELS[case["shape"]])
    return path


def _prompt(case, seed):
    return ea.synth_prompt(seed, MODELS[case["shape"]]["vocab"], case["prompt"])


def _context(n):
    return (n + 1023) // 1024 * 1024


# ---- what a program holds, and one pass of it -------------------------------------------

_backends = {}


def _backend(q8):
    """A program opens one backend and runs all its layers on it, one after the other."""
    if q8 not in _backends:
        _backends[q8] = ea.HipBackend(quantize_activations=q8)
    return _backends[q8]


class _State(dict):
    """A layer's weights and buffers; the weights are given back with it."""

    def __init__(self, be, *a, **k):
        super().__init__(*a, **k)
        self.be, self.weights = be, []

    def upload(self, wtype, cols, rows, data):
        self.weights.append(self.be.upload_weight(wtype, cols, rows, data))
        return self.weights[-1]

    def vector(self, v):
        self.weights.append(self.be.vector(v))
        return self.weights[-1]

    def __del__(self):
        for w in self.weights:
            self.be.weight_free(w)


def prepare(case, seed):
    if case["kind"] == "model":
        path = _model_file(case, seed)
        try:
            model = ea.Model(path, context=1024)
        finally:
            os.unlink(path)
        return {"case": case, "model": model, "prompt": _prompt(case, seed)}
    s = _State(_backend(case.get("q8", False)), case=case, **_inputs(case, seed))
    up = lambda w, name, rows, cols: s.upload(TYPES[case["type"]], cols, rows, w[name])  # noqa: E731
    if case["kind"] == "ffn":
        w, H, F, M = _ffn_weights(case, seed), case["hidden"], case["ffn"], case["tokens"]
        s["w"] = (up(w, "gate", F, H), up(w, "up", F, H), up(w, "down", H, F))
        s["norm"] = s.vector(w["norm"])
        s["xn"] = torch.zeros(M, H, device="cuda")
        s["hidden"] = torch.zeros(M, F, device="cuda")
        s["y"] = torch.zeros(M, H, device="cuda")
        s["inp"] = ea.Input(s["x"].data_ptr(), s["delta"].data_ptr(), s["xn"].data_ptr(), s["norm"], EPS)
    elif case["kind"] in ("recurrent", "delta"):
        kh, vh, sd, cw = STATES[case["shape"]]
        ch, vd = (2 * kh + vh) * sd, vh * sd
        w = _delta_weights(case, seed)
        vec = (s.vector(w["conv"]), s.vector(w["a"]), s.vector(w["dt"]), s.vector(w["norm"]))
        cs, rs = s["conv_state"].data_ptr(), s["rec_state"].data_ptr()
        if case["kind"] == "recurrent":
            H = case["hidden"]
            w = _recurrent_weights(case, seed)
            mats = (up(w, "qkv", ch, H), up(w, "z", vd, H), up(w, "alpha", vh, H), up(w, "beta", vh, H), up(w, "out", H, vd))
            s["p"] = ea.RecurrentParams(*mats, *vec, kh, vh, sd, cw, EPS, cs, rs)
            s["xo"], s["y"] = torch.zeros(H, device="cuda"), torch.zeros(H, device="cuda")
            s["inp"] = ea.Input(s["x"].data_ptr(), s["delta"].data_ptr(), s["xo"].data_ptr(), s.vector(w["attn_norm"]), EPS)
        else:
            r = s["rows"].data_ptr()
            s["out"] = torch.zeros(case["count"], vd, device="cuda")
            s["p"] = ea.DeltaNetParams(kh, vh, sd, cw, EPS, r, r + 4 * ch, r + 4 * (ch + vd), r + 4 * (ch + vd + vh), *vec,
                                       cs, rs, s["out"].data_ptr())
    else:
        heads, kv, hd, rot = HEADS[case["shape"]]
        n = s["rows"].shape[0]
        w = _attn_weights(case, seed)
        total = s["keys"].shape[0]
        context = _context(total)
        for c in ("keys", "values"):
            cache = torch.zeros(context, kv, hd, device="cuda")
            cache[:total] = s[c]
            s[c] = cache
        s["position"] = torch.tensor([total - n], dtype=torch.int32, device="cuda")
        s["p"] = ea.AttentionParams(heads, kv, hd, rot, context, EPS, ROPE_BASE, s.vector(w["q_norm"]),
                                    s.vector(w["k_norm"]), s["keys"].data_ptr(), s["values"].data_ptr(),
                                    s["position"].data_ptr())
        s["out"] = torch.zeros(n, heads * hd, device="cuda")
    torch.cuda.synchronize()  # the backend works on its own stream
    return s


def run(s):
    c, k = s["case"], s["case"]["kind"]
    if k == "model":
        tokens, _ = s["model"].generate(s["prompt"], c["count"])
        return {"tokens": np.array(tokens), "logits": s["model"].evaluate(tokens[-1])}
    be = s.be
    if k == "ffn":
        gate, up, down = s["w"]
        M, H, F = c["tokens"], c["hidden"], c["ffn"]
        if M == 1:
            be.feed_forward(gate, up, down, 0, s["y"].data_ptr(), s["inp"])
            return {"y": s["y"], "x": s["xn"]}
        be.rmsnorm_rows(s["x"].data_ptr(), s["norm"], s["xn"].data_ptr(), H, M, EPS)
        be.ffn_gate_up_batch(gate, up, s["xn"].data_ptr(), H, s["hidden"].data_ptr(), F, M)
        be.linear_batch(down, s["hidden"].data_ptr(), s["y"].data_ptr(), M)
        return {"y": s["y"], "hidden": s["hidden"]}
    if k == "recurrent":
        be.recurrent(s["p"], 0, s["y"].data_ptr(), s["inp"])
        return {"y": s["y"], "rec_state": s["rec_state"], "conv_state": s["conv_state"], "x": s["xo"]}
    if k == "delta":
        be.delta_net_batch(s["p"], c["count"], s["rows"].shape[1], s["out"].shape[1])
        return {"out": s["out"], "rec_state": s["rec_state"], "conv_state": s["conv_state"]}
    rows, out = s["rows"], s["out"]
    if k == "attn_step":
        be.attention(s["p"], rows.data_ptr(), out.data_ptr())
        return {"out": out, "key": s["keys"][c["position"]], "value": s["values"][c["position"]]}
    be.attention_batch(s["p"], rows.data_ptr(), c["count"], rows.shape[1], c["first"], out.data_ptr(), out.shape[1])
    n = c["first"] + c["count"]
    return {"out": out, "keys": s["keys"][c["first"]:n], "values": s["values"][c["first"]:n]}


# ---- the bytes and operations that a pass cannot do without -----------------------------


def _encoded(wtype, n):
    return ea.encoded_bytes(wtype, n)


def _model_layers(case):
    """(matrix name, rows, cols, type) of every layer's projections, in file order."""
    m = MODELS[case["shape"]]
    H, F = m["hidden"], m["ffn"]
    low = ea.Q4_K if case["mix"] else ea.Q6_K
    layers = []
    for i in range(m["layers"]):
        if (i + 1) % m["full_attention_interval"]:
            sd, kh, vh = m["state_dim"], m["key_heads"], m["value_heads"]
            t = [("attn_qkv", (2 * kh + vh) * sd, H, low), ("attn_gate", vh * sd, H, low), ("ssm_alpha", vh, H, low),
                 ("ssm_beta", vh, H, low), ("ssm_out", H, vh * sd, low)]
        else:
            q, kv = m["heads"] * m["head_dim"], m["kv_heads"] * m["head_dim"]
            t = [("attn_q", 2 * q, H, low), ("attn_k", kv, H, low), ("attn_v", kv, H, ea.Q6_K), ("attn_output", H, q, low)]
        layers.append(t + [("ffn_gate", F, H, low), ("ffn_up", F, H, low), ("ffn_down", H, F, ea.Q6_K)])
    return layers


def work(case):
    k = case["kind"]
    if k == "model":
        m = MODELS[case["shape"]]
        mats = [t for layer in _model_layers(case) for t in layer]
        weights = sum(_encoded(t, r * c) for _, r, c, t in mats)
        head = _encoded(ea.Q4_K if case["mix"] else ea.Q6_K, m["vocab"] * m["hidden"])
        steps = case["count"] + 1
        ops = 2 * sum(r * c for _, r, c, _ in mats)
        return {"bytes": weights * (steps + (case["prompt"] > 1)) + head * steps,
                "flops": ops * (case["prompt"] - 1 + steps) + 2 * m["vocab"] * m["hidden"] * steps}
    if k == "ffn":
        M, H, F = case["tokens"], case["hidden"], case["ffn"]
        return {"bytes": 3 * _encoded(TYPES[case["type"]], H * F) + 4 * M * H * 3, "flops": 6 * M * H * F}
    if k in ("recurrent", "delta"):
        kh, vh, sd, cw = STATES[case["shape"]]
        ch, vd = (2 * kh + vh) * sd, vh * sd
        n = 1 if k == "recurrent" else case["count"]
        state = 8 * (vd * sd + ch * cw) + 4 * ch * cw
        ops = n * (2 * ch * cw + 7 * vd * sd)
        if k == "delta":
            return {"bytes": state + 4 * n * (ch + vd + 2 * vh + vd), "flops": ops}
        H = case["hidden"]
        mats = (ch + vd + 2 * vh + vd) * H
        return {"bytes": state + _encoded(TYPES[case["type"]], mats) + 16 * H, "flops": ops + 2 * mats}
    heads, kv, hd, _ = HEADS[case["shape"]]
    past, n = (case["position"], 1) if k == "attn_step" else (case["first"], case["count"])
    pairs = n * past + n * (n + 1) // 2
    row = heads * hd * 2 + 2 * kv * hd
    return {"bytes": 8 * (past + n) * kv * hd + 4 * n * (row + heads * hd), "flops": 4 * heads * hd * pairs}


# ---- the same results in 64 bits --------------------------------------------------------


def _f16(b):
    return torch.from_numpy(np.ascontiguousarray(b).view(np.float16).astype(np.float64)).cuda()


def _decode(wtype, b, rows, cols):
    """GGUF blocks as a rows x cols matrix in 64 bits."""
    b = np.ascontiguousarray(b).reshape(rows * cols // 256, -1)
    raw = torch.from_numpy(b).cuda()
    n = raw.shape[0]
    if wtype == ea.Q6_K:
        low, high = raw[:, :128].reshape(n, 2, 1, 64), raw[:, 128:192].reshape(n, 2, 1, 32)
        low = torch.cat([low & 15, low >> 4], 2).reshape(n, 2, 4, 32)
        high = torch.cat([(high >> (2 * i)) & 3 for i in range(4)], 2)
        code = (low | (high << 4)).reshape(n, 16, 16).double() - 32
        scale = raw[:, 192:208].view(torch.int8).double() * _f16(b[:, 208:210])
        return (code * scale[:, :, None]).reshape(rows, cols)
    s = raw[:, 4:16]
    scale = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
    floor = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    q = raw[:, 16:].reshape(n, 4, 1, 32)
    code = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32).double()
    d, dm = _f16(b[:, 0:2]), _f16(b[:, 2:4])
    return (code * (d * scale)[:, :, None] - (dm * floor)[:, :, None]).reshape(rows, cols)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _silu(x):
    return x * torch.sigmoid(x)


def _vec(v):
    return torch.from_numpy(np.asarray(v)).cuda().double()


def _rope(x, positions, rotary, base):
    """NEOX rotation of x[position][head][dim]; the angle is a 32-bit value by definition."""
    half = rotary // 2
    i = torch.arange(half, device="cuda", dtype=torch.float32)
    angle = positions.float()[:, None] / torch.pow(torch.tensor(base, device="cuda"), 2 * i / rotary)
    c, s = angle.double().cos()[:, None], angle.double().sin()[:, None]
    a, b = x[..., :half], x[..., half:rotary]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., rotary:]], -1)


def _attend(rows, keys, values, first, heads, rotary, base, q_norm, k_norm):
    """Gated causal attention of the positions from `first` on; keys and values hold the
    earlier rows. Returns the outputs and the new key and value rows."""
    n, (kv, hd) = rows.shape[0], keys.shape[1:]
    at = torch.arange(first, first + n, device="cuda")
    qg = rows[:, :heads * hd * 2].reshape(n, heads, 2, hd)
    q = _rope(_rms(qg[:, :, 0], q_norm), at, rotary, base)
    k = _rope(_rms(rows[:, heads * hd * 2:heads * hd * 2 + kv * hd].reshape(n, kv, hd), k_norm), at, rotary, base)
    v = rows[:, heads * hd * 2 + kv * hd:].reshape(n, kv, hd)
    ks, vs = torch.cat([keys, k]), torch.cat([values, v])
    masked = torch.arange(first + n, device="cuda")[None, :] > at[:, None]
    out = torch.empty(n, heads, hd, device="cuda", dtype=torch.float64)
    for h in range(heads):
        j = h // (heads // kv)
        p = (q[:, h] @ ks[:, j].T / math.sqrt(hd)).masked_fill(masked, -math.inf).softmax(-1)
        out[:, h] = p @ vs[:, j]
    return (out * torch.sigmoid(qg[:, :, 1])).reshape(n, -1), k, v


def _delta(rows, z, alpha, beta, w, dims, conv_state, rec_state):
    """The Gated DeltaNet over the positions of rows; returns the outputs and both states."""
    kh, vh, sd, cw = dims
    n, conv = rows.shape[0], _vec(w["conv"]).reshape(-1, cw)
    seq = torch.cat([conv_state[:, 1:].T, rows])
    mixed = _silu(sum(seq[j:j + n] * conv[:, j] for j in range(cw)))
    q, k, v = mixed.split([kh * sd, kh * sd, vh * sd], 1)
    unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + EPS)  # noqa: E731
    of = torch.arange(vh, device="cuda") % kh
    q = unit(q.reshape(n, kh, sd))[:, of] / math.sqrt(sd)
    k, v = unit(k.reshape(n, kh, sd))[:, of], v.reshape(n, vh, sd)
    decay = torch.exp(_vec(w["a"]) * torch.nn.functional.softplus(alpha + _vec(w["dt"]), threshold=1e9))
    gate = torch.sigmoid(beta)
    S, o = rec_state.clone(), torch.empty_like(v)
    for t in range(n):
        S *= decay[t, :, None, None]
        mem = (S * k[t, :, None]).sum(-1)
        S += ((v[t] - mem) * gate[t, :, None])[:, :, None] * k[t, :, None]
        o[t] = (S * q[t, :, None]).sum(-1)
    out = _rms(o, _vec(w["norm"])) * _silu(z.reshape(n, vh, sd))
    return out.reshape(n, -1), S, torch.cat([conv_state.T, rows])[-cw:].T.contiguous()


def _tensors(path):
    """The tensors of a GGUF file: name -> (type, shape, bytes)."""
    data = np.memmap(path, np.uint8, "r")
    at = 8

    def take(fmt):
        nonlocal at
        v = struct.unpack_from("<" + fmt, data, at)
        at += struct.calcsize("<" + fmt)
        return v[0]

    def text():
        nonlocal at
        n = take("Q")
        at += n
        return bytes(data[at - n:at]).decode()

    def value(t):
        if t == 8:
            return text()
        if t == 9:
            inner, n = take("I"), take("Q")
            return [value(inner) for _ in range(n)]
        return take("BbHhIif?..QqD"[t] if t < 12 else "d")

    count, keys = take("Q"), take("Q")
    meta = {}
    for _ in range(keys):
        name = text()
        meta[name] = value(take("I"))
    infos = []
    for _ in range(count):
        name, dims = text(), take("I")
        shape = [take("Q") for _ in range(dims)]
        infos.append((name, shape, take("I"), take("Q")))
    align = meta.get("general.alignment", 32)
    at = (at + align - 1) // align * align
    return {name: (t, shape, data[at + off:at + off + ea.encoded_bytes(t, math.prod(shape))])
            for name, shape, t, off in infos}


class _Exact:
    """A qwen35 model in 64 bits, from its file."""

    def __init__(self, path, m):
        self.m, self.t, self.held = m, _tensors(path), {}
        sd, kh, vh = m["state_dim"], m["key_heads"], m["value_heads"]
        self.state = [{"conv": torch.zeros((2 * kh + vh) * sd, m["conv_width"], device="cuda", dtype=torch.float64),
                       "rec": torch.zeros(vh, sd, sd, device="cuda", dtype=torch.float64),
                       "k": torch.zeros(0, m["kv_heads"], m["head_dim"], device="cuda", dtype=torch.float64),
                       "v": torch.zeros(0, m["kv_heads"], m["head_dim"], device="cuda", dtype=torch.float64)}
                      for _ in range(m["layers"])]
        self.position = 0

    def __getitem__(self, name):
        if name not in self.held:
            t, shape, raw = self.t[name]
            if t == ea.F32:
                v = torch.from_numpy(np.array(raw).view(np.float32)).cuda().double()
                self.held[name] = v if len(shape) == 1 else v.reshape(shape[::-1])
            else:
                self.held[name] = _decode(t, raw, shape[1], shape[0])
        return self.held[name]

    def step(self, tokens):
        """The logits after these further tokens."""
        m, n = self.m, len(tokens)
        x = self["token_embd.weight"][torch.tensor(tokens, device="cuda")]
        for i, s in enumerate(self.state):
            w = lambda name: self["blk.%d.%s" % (i, name)]  # noqa: B023,E731
            h = _rms(x, w("attn_norm.weight"))
            if (i + 1) % m["full_attention_interval"]:
                p = {"conv": w("ssm_conv1d.weight").cpu().numpy().reshape(-1), "a": w("ssm_a").cpu().numpy(),
                     "dt": w("ssm_dt.bias").cpu().numpy(), "norm": w("ssm_norm.weight").cpu().numpy()}
                o, s["rec"], s["conv"] = _delta(h @ w("attn_qkv.weight").T, h @ w("attn_gate.weight").T,
                                                h @ w("ssm_alpha.weight").T, h @ w("ssm_beta.weight").T, p,
                                                (m["key_heads"], m["value_heads"], m["state_dim"], m["conv_width"]),
                                                s["conv"], s["rec"])
                x = x + o @ w("ssm_out.weight").T
            else:
                rows = torch.cat([h @ w("attn_%s.weight" % c).T for c in "qkv"], 1)
                o, k, v = _attend(rows, s["k"], s["v"], self.position, m["heads"], m["rotary"], m["rope_base"],
                                  w("attn_q_norm.weight"), w("attn_k_norm.weight"))
                s["k"], s["v"] = torch.cat([s["k"], k]), torch.cat([s["v"], v])
                x = x + o @ w("attn_output.weight").T
            h = _rms(x, w("post_attention_norm.weight"))
            x = x + (_silu(h @ w("ffn_gate.weight").T) * (h @ w("ffn_up.weight").T)) @ w("ffn_down.weight").T
        self.position += n
        return self["output.weight"] @ _rms(x[-1], self["output_norm.weight"])


def exact(case, seed):
    k = case["kind"]
    if k == "model":
        path = _model_file(case, seed)
        try:
            e = _Exact(path, MODELS[case["shape"]])
            logits = e.step(_prompt(case, seed))
            for _ in range(case["count"]):
                logits = e.step([int(logits.argmax())])
        finally:
            os.unlink(path)
        return {"tokens": None, "logits": logits}
    s = _inputs(case, seed)
    d = {name: t.double() for name, t in s.items()}
    if k == "ffn":
        w, t, H, F = _ffn_weights(case, seed), TYPES[case["type"]], case["hidden"], case["ffn"]
        x = d["x"] + d["delta"] if case["tokens"] == 1 else d["x"]
        n = _rms(x, _vec(w["norm"]))
        h = _silu(n @ _decode(t, w["gate"], F, H).T) * (n @ _decode(t, w["up"], F, H).T)
        y = h @ _decode(t, w["down"], H, F).T
        return {"y": y, "x": x} if case["tokens"] == 1 else {"y": y, "hidden": h}
    if k == "recurrent":
        kh, vh, sd, cw = STATES[case["shape"]]
        w, t, H = _recurrent_weights(case, seed), TYPES[case["type"]], case["hidden"]
        x = d["x"] + d["delta"]
        n = _rms(x, _vec(w["attn_norm"]))[None]
        m = {name: n @ _decode(t, w[name], rows, H).T
             for name, rows in (("qkv", (2 * kh + vh) * sd), ("z", vh * sd), ("alpha", vh), ("beta", vh))}
        o, S, hist = _delta(m["qkv"], m["z"], m["alpha"], m["beta"], w, (kh, vh, sd, cw), d["conv_state"], d["rec_state"])
        return {"y": (o @ _decode(t, w["out"], H, vh * sd).T)[0], "rec_state": S, "conv_state": hist, "x": x}
    if k == "delta":
        kh, vh, sd, cw = STATES[case["shape"]]
        parts = d["rows"].split([(2 * kh + vh) * sd, vh * sd, vh, vh], 1)
        o, S, hist = _delta(*parts, _delta_weights(case, seed), (kh, vh, sd, cw), d["conv_state"], d["rec_state"])
        return {"out": o, "rec_state": S, "conv_state": hist}
    heads, kv, hd, rot = HEADS[case["shape"]]
    w, n = _attn_weights(case, seed), d["rows"].shape[0]
    past = d["keys"].shape[0] - n
    o, key, value = _attend(d["rows"], d["keys"][:past], d["values"][:past], past, heads, rot, ROPE_BASE,
                            _vec(w["q_norm"]), _vec(w["k_norm"]))
    if k == "attn_step":
        return {"out": o, "key": key[0], "value": value[0]}
    return {"out": o, "keys": key, "values": value}
