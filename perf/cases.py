"""Performance cases of the attention framework, through its public Python entry points.

A case is a dict of plain values; ``kind`` names the entry point it calls:

* ``laya_block``    the Laya fused split + RoPE + attention op, by its (L, L, B) keep tensor or
                    (``entry`` "structured") by validity bytes and a window
* ``jeff_op``       the Jeff full-attention op on one question row, K/V expanded to every query head
* ``jeff_rows``     batched Jeff rows with native GQA, f32 or bf16
* ``laya_layer``    a whole Laya attention layer (projections around the op)
* ``jeff_layer``    a whole Jeff attention layer over rows
* ``laya_forward``  the Laya decision model, prompts in, marker logits and action logits out

Sizes are those of the repository's configurations (12 or 16 heads of 64; 8 query and 2 key/value
heads of 256) and ragged ones around them. Row lengths of a padded batch are spread evenly from
``shortest`` to ``length``; the seed decides which row has which.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "tenferro-decision-rs_amd"))
import tenferro_ext as te  # noqa: E402
from tenferro_ext.laya_model import (ACTION_HIDDEN, AgentConfig, EncoderConfig,  # noqa: E402
                                     LayaCheckpoint, LayaModel)

DEVICE = torch.device("cuda", 0)
THETA_GLOBAL, THETA_LOCAL, THETA_JEFF, EPS_JEFF = 160000.0, 10000.0, 1.0e7, 1.0e-6
VOCAB, MARKERS, ACTIONS = 8192, 8, 4


def _laya(name, length, batch, *, heads=12, shortest=None, window=-1, entry="keep", **more):
    return dict(kind="laya_block", name=name, heads=heads, head_dim=64, length=length, batch=batch,
                shortest=shortest or length, window=window, entry=entry, **more)


def _jeff(name, kind, rows, length, *, shortest=None, dtype="f32", trim=False):
    return dict(kind=kind, name=name, rows=rows, length=length, heads=8, kv_heads=2, head_dim=256,
                rotary_dim=64, shortest=shortest or length, dtype=dtype, trim=trim)


def listed():
    return [
        # One short prompt through the drop-in op: latency and launches.
        _laya("laya_short", 64, 1, heads=16),
        # A few prompts of an odd length, padded: tile remainders in every dimension.
        _laya("laya_odd", 395, 3, shortest=57),
        # The global layers' attention over a padded batch (the headline shape).
        _laya("laya_global", 512, 8, shortest=64),
        # The local layers' attention over long documents, by validity bytes and window.
        _laya("laya_local", 2048, 4, window=64, entry="structured"),
        # One question row per call, as an engine that loops over rows calls the op.
        _jeff("jeff_row", "jeff_op", 1, 256, shortest=200),
        # All question rows of a decision in one call, left-padded.
        _jeff("jeff_rows", "jeff_rows", 16, 256, shortest=32),
        # Rows of an odd length, trimmed as the engine trims them.
        _jeff("jeff_odd", "jeff_rows", 5, 333, shortest=100, trim=True),
        # Long-context prefill in bf16.
        _jeff("jeff_bf16_long", "jeff_rows", 2, 8192, dtype="bf16"),
        # A whole encoder attention layer on the padded batch.
        dict(_laya("laya_layer", 512, 8, shortest=64), kind="laya_layer", bias=False),
        # A whole full-attention layer on the question rows.
        dict(_jeff("jeff_layer", "jeff_layer", 16, 256, shortest=32), hidden=1024),
        # One short decision prompt through the whole model, answers on the host.
        dict(kind="laya_forward", name="forward_single", hidden=768, heads=12, inter=1152,
             layers=22, length=96, batch=1, shortest=96),
        # A padded batch of prompts through the whole model, answers on the host.
        dict(kind="laya_forward", name="forward_batch", hidden=768, heads=12, inter=1152,
             layers=22, length=512, batch=8, shortest=64),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("laya_block", "laya_block", "jeff_op", "jeff_rows", "jeff_rows",
                       "laya_layer", "jeff_layer", "laya_forward"))
    if kind in ("laya_block", "laya_layer"):
        length = _log_int(rng, 8, 2048 if kind == "laya_block" else 1024)
        batch = _log_int(rng, 1, max(1, min(16, (8192 if kind == "laya_block" else 4096) // length)))
        c = _laya(None, length, batch, heads=rng.choice((12, 16)),
                  shortest=length if rng.random() < 0.3 else max(1, length // rng.randint(2, 8)),
                  window=rng.choice((-1, 64)))
        if kind == "laya_layer":
            c.update(kind=kind, bias=rng.random() < 0.5)
        elif rng.random() < 0.5:
            c["entry"] = "structured"
    elif kind == "laya_forward":
        length = _log_int(rng, 16, 512)
        c = dict(kind=kind, hidden=768, heads=12, inter=1152, layers=rng.randint(2, 12), length=length,
                 batch=_log_int(rng, 1, max(1, min(8, 4096 // length))),
                 shortest=max(12, length // rng.randint(1, 8)))
    else:
        dtype = rng.choice(("f32", "bf16")) if kind == "jeff_rows" else "f32"
        length = _log_int(rng, 16, {"jeff_op": 1024, "jeff_layer": 512}.get(
            kind, 8192 if dtype == "bf16" else 1024))
        rows = 1 if kind == "jeff_op" else _log_int(rng, 1, max(1, min(32, (
            16384 if dtype == "bf16" else 4096) // length)))
        c = _jeff(None, kind, rows, length, dtype=dtype, trim=kind == "jeff_rows" and rng.random() < 0.3,
                  shortest=length if rng.random() < 0.3 else max(1, length // rng.randint(2, 8)))
        if kind == "jeff_layer":
            c["hidden"] = 1024
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ inputs


def _lengths(case):
    """The row lengths of a batch, spread evenly from `shortest` to `length`."""
    n = case.get("batch", case.get("rows", 1))
    lo, hi = case["shortest"], case["length"]
    if n == 1:
        return [lo]
    return [lo + (hi - lo) * i // (n - 1) for i in range(n)]


def _shuffled(case, seed):
    lens = _lengths(case)
    order = np.random.default_rng(seed).permutation(len(lens))
    return [lens[i] for i in order]


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _normal(g, n, scale=1.0):
    return torch.randn(n, generator=g, device=DEVICE, dtype=torch.float32).mul_(scale)


def _keep(valid, window):
    """[b, key, query] keep bytes: a query keeps the valid keys within the window, a padded query
    every valid key."""
    B, L = valid.shape
    t = torch.arange(L, device=DEVICE)
    inside = torch.ones(L, L, dtype=torch.bool, device=DEVICE)
    if window >= 0:
        inside = (t[:, None] - t[None, :]).abs() <= window
    return valid[:, :, None] & (inside[None] | ~valid[:, None, :])


def _laya_inputs(case, seed):
    """Activations and masks of the Laya op and layer cases."""
    g = _generator(seed)
    d, L, B = case["heads"] * case["head_dim"], case["length"], case["batch"]
    lens = torch.tensor(_shuffled(case, seed), device=DEVICE)
    valid = torch.arange(L, device=DEVICE)[None, :] < lens[:, None]
    s = {"valid": valid, "keep": _keep(valid, case["window"]).to(torch.uint8).reshape(-1),
         "base": THETA_GLOBAL if case["window"] < 0 else THETA_LOCAL}
    if case["kind"] == "laya_block":
        # Projections of unit activations by N(0, 0.02^2) weights; unit ones in the local layers.
        s["qkv"] = _normal(g, 3 * d * L * B, 0.02 * math.sqrt(d) if case["window"] < 0 else 1.0)
    else:
        s["x"] = _normal(g, d * L * B)
        s["w_in"], s["w_out"] = _normal(g, 3 * d * d, 0.02), _normal(g, d * d, 0.02)
        s["b_in"] = _normal(g, 3 * d, 0.02) if case["bias"] else None
        s["b_out"] = _normal(g, d, 0.02) if case["bias"] else None
    return s


def _jeff_inputs(case, seed):
    """Activations, norms and left-padding masks of the Jeff cases."""
    g = _generator(seed)
    R, L, hd = case["rows"], case["length"], case["head_dim"]
    W, KW = case["heads"] * hd, case["kv_heads"] * hd
    lens = torch.tensor(_shuffled(case, seed), device=DEVICE)
    s = {"mask": (torch.arange(L, device=DEVICE)[None, :] >= L - lens[:, None]).float().reshape(-1),
         "q_norm": _normal(g, hd, 0.02), "k_norm": _normal(g, hd, 0.02)}
    if case["kind"] == "jeff_layer":
        n = case["hidden"]
        s["x"] = _normal(g, R * L * n)
        for name, size in (("w_q", n * W), ("w_gate", n * W), ("w_k", n * KW), ("w_v", n * KW),
                           ("w_o", W * n)):
            s[name] = _normal(g, size, 0.02)
        return s
    scale = 0.02 * math.sqrt(1024.0)  # projections of 1024 unit activations by N(0, 0.02^2) weights
    for name, size in (("q", R * L * W), ("gate", R * L * W), ("k", R * L * KW), ("v", R * L * KW)):
        s[name] = _normal(g, size, scale)
        if case["dtype"] == "bf16":
            s[name] = s[name].to(torch.bfloat16)
    if case["kind"] == "jeff_op":  # the engine's weights hold every key/value head once per query head
        for name in ("k", "v"):
            s[name] = (s[name].view(case["kv_heads"], 1, hd * L)
                       .expand(-1, case["heads"] // case["kv_heads"], -1).reshape(-1))
    return s


def _checkpoint(case, seed):
    """A decision model of the case's shape with random weights, as loaded from a checkpoint."""
    g = _generator(seed)
    d, inter = case["hidden"], case["inter"]
    enc = EncoderConfig.from_json({
        "vocab_size": VOCAB, "hidden_size": d, "intermediate_size": inter,
        "num_hidden_layers": case["layers"], "num_attention_heads": case["heads"],
        "local_attention": 128})
    agent = AgentConfig(head_layers=1, action_names=["a%d" % i for i in range(ACTIONS - 1)])

    def normal(n, scale=1.0, shift=0.0):
        return (_normal(g, n, scale) + shift).cpu().numpy()

    w = {"tok_embeddings": normal(VOCAB * d)}

    def linear(key, n_in, n_out, bias):
        w[key + ".w"] = normal(n_in * n_out, n_in ** -0.5)
        w[key + ".b"] = normal(n_out, 0.1) if bias else None

    def norm(key, bias):
        w[key + ".w"], w[key + ".b"] = normal(d, 0.1, 1.0), normal(d, 0.1) if bias else None

    norm("embed_norm", False)
    for i in range(case["layers"]):
        p = "layers.%d." % i
        if i:
            norm(p + "attn_norm", False)
        else:
            w[p + "attn_norm.w"] = w[p + "attn_norm.b"] = None
        linear(p + "wqkv", d, 3 * d, False)
        linear(p + "wo", d, d, False)
        norm(p + "mlp_norm", False)
        linear(p + "wi", d, 2 * inter, False)
        linear(p + "wo_mlp", inter, d, False)
    norm("final_norm", False)
    norm("head.0.norm1", True)
    linear("head.0.in_proj", d, 3 * d, True)
    linear("head.0.out_proj", d, d, True)
    norm("head.0.norm2", True)
    linear("head.0.linear1", d, 4 * d, True)
    linear("head.0.linear2", 4 * d, d, True)
    w["type_emb"] = normal(3 * d)
    norm("scorer_norm", True)
    linear("scorer1", d, d, True)
    linear("scorer2", d, 1, True)
    linear("act1", d + 4, ACTION_HIDDEN, True)
    linear("act2", ACTION_HIDDEN, ACTIONS, True)
    return LayaCheckpoint(enc, agent, w, max(1, d // 64))


def _prompts(case, seed):
    """(ids, mask, marker_pos, marker_mask, qtype) host arrays of a right-padded batch."""
    rng = np.random.default_rng(seed)
    L, B, lens = case["length"], case["batch"], _shuffled(case, seed)
    ids = rng.integers(0, VOCAB, L * B)
    mask = np.zeros((B, L), bool)
    pos = np.zeros((B, MARKERS), np.int64)
    for b in range(B):
        mask[b, :lens[b]] = True
        pos[b] = 1 + np.sort(rng.permutation(lens[b] - 1)[:MARKERS])
    return ids, mask.reshape(-1), pos.reshape(-1), np.ones(B * MARKERS, bool), np.arange(B) % 3


_CONTEXT = []


def _context():
    """The program's one context, on torch's current stream."""
    if not _CONTEXT:
        _CONTEXT.append(te.Context(0, stream=torch.cuda.current_stream(DEVICE).cuda_stream))
    return _CONTEXT[0]


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    if kind == "laya_forward":
        return {"case": case, "model": LayaModel(_checkpoint(case, seed), ctx=ctx),
                "prompts": _prompts(case, seed)}
    s = _laya_inputs(case, seed) if kind.startswith("laya") else _jeff_inputs(case, seed)
    if case.get("entry") == "structured":
        s["valid"] = s["valid"].to(torch.uint8).reshape(-1)
    n = (case["batch"] * case["heads"] * case["head_dim"] if kind.startswith("laya") else
         case["rows"] * case.get("hidden", case["heads"] * case["head_dim"])) * case["length"]
    s.update(case=case, ctx=ctx, out=torch.empty(n, dtype=torch.float32, device=DEVICE))
    return s


# ------------------------------------------------------------------ one pass


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "laya_forward":
        logits, action = s["model"].forward(*s["prompts"])
        return {"logits": logits, "action": action}
    L = c["length"]
    with te.asynchronous():
        if kind == "laya_block":
            d, H, B = c["heads"] * c["head_dim"], c["heads"], c["batch"]
            if c["entry"] == "structured":
                return te.laya_attention_structured(s["qkv"], s["valid"], d, H, L, B, c["window"],
                                                    s["base"], ctx=s["ctx"], out=s["out"])
            return te.laya_attention_block(s["qkv"], s["keep"], d, H, s["base"],
                                           qkv_shape=(3 * d, L, B), ctx=s["ctx"], out=s["out"])
        if kind == "laya_layer":
            return te.laya_attention_layer(s["x"], s["keep"], s["w_in"], s["b_in"], s["w_out"],
                                           s["b_out"], c["heads"] * c["head_dim"], c["heads"], L,
                                           c["batch"], s["base"], ctx=s["ctx"], out=s["out"])
        if kind == "jeff_op":
            return te.jeff_full_attention(s["q"], s["k"], s["v"], s["gate"], s["q_norm"],
                                          s["k_norm"], s["mask"], c["heads"], c["head_dim"],
                                          c["rotary_dim"], THETA_JEFF, EPS_JEFF,
                                          q_shape=(L, c["heads"] * c["head_dim"]), ctx=s["ctx"],
                                          out=s["out"], kv_heads=c["kv_heads"])
        if kind == "jeff_rows":
            return te.jeff_full_attention_rows(s["q"], s["k"], s["v"], s["gate"], s["q_norm"],
                                               s["k_norm"], s["mask"], c["rows"], L, c["heads"],
                                               c["kv_heads"], c["head_dim"], c["rotary_dim"],
                                               THETA_JEFF, EPS_JEFF, trim_leading=c["trim"],
                                               bf16=c["dtype"] == "bf16", ctx=s["ctx"], out=s["out"])
        return te.jeff_full_attention_layer_rows(s["x"], s["w_q"], s["w_gate"], s["w_k"], s["w_v"],
                                                 s["w_o"], s["q_norm"], s["k_norm"], s["mask"],
                                                 c["rows"], L, c["hidden"], c["heads"],
                                                 c["kv_heads"], c["head_dim"], c["rotary_dim"],
                                                 THETA_JEFF, EPS_JEFF, trim_leading=c["trim"],
                                                 ctx=s["ctx"], out=s["out"])


# ------------------------------------------------------------------ work and tolerance


def _pairs(case, window):
    """Kept (query, key) pairs of the batch, per head."""
    L, total = case["length"], 0
    for n in _lengths(case):
        q = np.arange(n)
        if window < 0:
            total += L * n
        else:
            total += int((np.minimum(q + window, n - 1) - np.maximum(q - window, 0) + 1).sum())
            total += (L - n) * n  # padded queries keep every valid key
    return total


def work(case):
    L, kind = case["length"], case["kind"]
    lens = _lengths(case)
    if kind == "laya_forward":
        d, inter, n = case["hidden"], case["inter"], sum(lens)
        weights = case["layers"] * (4 * d * d + 3 * d * inter) + 4 * d * d + 8 * d * d
        flops = 2.0 * n * weights
        for i in range(case["layers"] + 1):
            if i == case["layers"] or i % 3 == 0:
                flops += 4.0 * d * sum(m * m for m in lens)
            else:
                flops += 4.0 * d * sum(m * min(m, 129) for m in lens)
        return {"bytes": 4.0 * weights + 4.0 * n * d, "flops": flops}
    if kind.startswith("laya"):
        d, B = case["heads"] * case["head_dim"], case["batch"]
        mask = L * B if case["entry"] == "structured" else L * L * B
        flops = 4.0 * d * _pairs(case, case["window"])
        if kind == "laya_block":  # q and out of every token, k and v of the valid ones
            return {"bytes": 4.0 * d * (2 * L * B + 2 * sum(lens)) + mask, "flops": flops}
        return {"bytes": 4.0 * (2 * d * L * B + 4 * d * d) + mask, "flops": flops + 8.0 * d * d * L * B}
    W, KW, R = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["rows"]
    flops = 4.0 * W * sum(n * (n + 1) / 2 for n in lens)
    if kind == "jeff_layer":
        n = case["hidden"]
        weights = n * (3 * W + 2 * KW)
        return {"bytes": 4.0 * (2 * R * L * n + weights), "flops": flops + 2.0 * R * L * weights}
    size = 2 if case["dtype"] == "bf16" else 4
    return {"bytes": size * (R * L * W + sum(lens) * (W + 2 * KW)) + 4.0 * R * L * W, "flops": flops}


def tolerance(case):
    if case.get("dtype") == "bf16":
        return {"rel": 1e-2, "max": 5e-2}
    if case["kind"] == "laya_forward":
        return {"rel": 2e-5}
    return {"rel": 4e-6}


# ------------------------------------------------------------------ the same in 64 bits


def _rotary(length, dim, base):
    """cos and sin (L, dim/2) in 64 bits of the op's angles, which its definition rounds to f32."""
    i = np.arange(dim // 2, dtype=np.float32)
    expo = (np.float32(-2.0) * i / np.float32(dim)).astype(np.float64)
    freq = np.power(np.float64(np.float32(base)), expo).astype(np.float32)
    angle = np.arange(length, dtype=np.float32)[:, None] * freq[None, :]
    angle = torch.from_numpy(angle).to(DEVICE).double()
    return angle.cos(), angle.sin()


def _rotate(x, cos, sin):
    """Rotates pairs (i, i + half) of the last axis of x (..., L, dim)."""
    h = cos.shape[-1]
    a, b, rest = x[..., :h], x[..., h:2 * h], x[..., 2 * h:]
    return torch.cat((a * cos - b * sin, a * sin + b * cos, rest), -1)


def _attend(q, k, v, allowed):
    """Masked softmax attention of (n, hd) by (m, hd); no allowed key gives NaN."""
    s = (q @ k.T) / math.sqrt(q.shape[-1])
    return torch.softmax(s.masked_fill(~allowed, -math.inf), -1) @ v


def _laya_exact(qkv, keep, heads, base):
    """qkv [B, L, 3d], keep [b, key, query] -> [B, L, d]."""
    B, L, d3 = qkv.shape
    d = d3 // 3
    hd = d // heads
    out = torch.empty(B, L, d, dtype=torch.float64, device=DEVICE)
    cos, sin = _rotary(L, hd, base) if base else (None, None)
    for b in range(B):
        allowed = keep[b].T
        for h in range(heads):
            q, k, v = (qkv[b, :, j * d + h * hd:j * d + (h + 1) * hd] for j in range(3))
            if base:
                q, k = _rotate(q, cos, sin), _rotate(k, cos, sin)
            out[b, :, h * hd:(h + 1) * hd] = _attend(q, k, v, allowed)
    return out


def _jeff_exact(case, q, k, v, gate, q_norm, k_norm, mask):
    """q, gate [R, W, L], k, v [R, KW, L] -> [R, W, L]."""
    R, L, H, KV, hd = (case[n] for n in ("rows", "length", "heads", "kv_heads", "head_dim"))
    out = torch.zeros(R, H * hd, L, dtype=torch.float64, device=DEVICE)
    cos, sin = _rotary(L, case["rotary_dim"], THETA_JEFF)
    eps = float(np.float32(EPS_JEFF))
    mask = mask.view(R, L)

    def prepared(x, w, first):
        x = x.T.double()
        x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * (1.0 + w.double())
        n = x.shape[0]
        return _rotate(x, cos[first:first + n], sin[first:first + n])

    for r in range(R):
        active = mask[r] != 0
        t0 = int(active.nonzero()[0]) if case["trim"] and bool(active.any()) else 0
        t = torch.arange(t0, L, device=DEVICE)
        allowed = (t[None, :] <= t[:, None]) & active[None, t0:]
        empty = ~allowed.any(-1)
        for h in range(H):
            f, fk = slice(h * hd, (h + 1) * hd), slice(h * KV // H * hd, (h * KV // H + 1) * hd)
            o = _attend(prepared(q[r, f, t0:], q_norm, 0), prepared(k[r, fk, t0:], k_norm, 0),
                        v[r, fk, t0:].T.double(), allowed)
            o[empty] = 0.0
            out[r, f, t0:] = (o * torch.sigmoid(gate[r, f, t0:].T.double())).T
    return out


def _forward_exact(case, seed):
    ck = _checkpoint(case, seed)
    ids, mask, pos, _, qtype = _prompts(case, seed)
    L, B, d, enc = case["length"], case["batch"], case["hidden"], ck.encoder
    eps = float(np.float32(enc.norm_eps))
    up = {k: torch.from_numpy(v).to(DEVICE).double() for k, v in ck.weights.items() if v is not None}
    valid = torch.from_numpy(mask).to(DEVICE).view(B, L)

    def norm(key, x):
        return torch.nn.functional.layer_norm(x, (d,), up[key + ".w"], up.get(key + ".b"), eps)

    def linear(key, x):
        return torch.nn.functional.linear(x, up[key + ".w"].view(-1, x.shape[-1]), up.get(key + ".b"))

    def attention(p, q, o, x, heads, window, base):
        return linear(p + o, _laya_exact(linear(p + q, x), _keep(valid, window), heads, base))

    x = norm("embed_norm", up["tok_embeddings"].view(-1, d)[torch.from_numpy(ids).to(DEVICE)]).view(B, L, d)
    gelu = torch.nn.functional.gelu
    for i, kind in enumerate(enc.layer_types):
        p = "layers.%d." % i
        window = enc.local_attention // 2 if kind == "sliding_attention" else -1
        a = norm(p + "attn_norm", x) if p + "attn_norm.w" in up else x
        x = x + attention(p, "wqkv", "wo", a, case["heads"], window, enc.rope_base(kind))
        u = linear(p + "wi", norm(p + "mlp_norm", x))
        x = x + linear(p + "wo_mlp", gelu(u[..., :case["inter"]]) * u[..., case["inter"]:])
    h = norm("final_norm", x) + up["type_emb"].view(3, d)[torch.from_numpy(qtype).to(DEVICE)][:, None]
    h = h + attention("head.0.", "in_proj", "out_proj", norm("head.0.norm1", h), ck.head_heads, -1, 0.0)
    h = h + linear("head.0.linear2", torch.relu(linear("head.0.linear1", norm("head.0.norm2", h))))
    at = torch.from_numpy(pos).to(DEVICE).view(B, MARKERS)
    s = norm("scorer_norm", h[torch.arange(B, device=DEVICE)[:, None], at])
    logits = linear("scorer2", gelu(linear("scorer1", s)))[..., 0]
    prob = torch.softmax(logits, -1)
    top = prob.topk(2, -1).values
    entropy = -(prob * prob.clamp_min(1e-9).log()).sum(-1) / math.log(MARKERS)
    used = torch.full_like(entropy, MARKERS / 255.0)
    pooled = torch.cat((h[:, 0], torch.stack((top[:, 0], top[:, 0] - top[:, 1], entropy, used), -1)), -1)
    action = linear("act2", gelu(linear("act1", pooled)))
    return {"logits": logits.reshape(-1), "action": action.reshape(-1)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "laya_forward":
        return _forward_exact(case, seed)
    if kind.startswith("laya"):
        s = _laya_inputs(case, seed)
        B, L, d = case["batch"], case["length"], case["heads"] * case["head_dim"]
        keep = _keep(s["valid"], case["window"])
        if kind == "laya_block":
            return _laya_exact(s["qkv"].view(B, L, 3 * d).double(), keep, case["heads"], s["base"]).reshape(-1)
        linear = torch.nn.functional.linear
        up = {k: v.double() if v is not None else None for k, v in s.items() if k[:2] in ("x", "w_", "b_")}
        qkv = linear(up["x"].view(B, L, d), up["w_in"].view(3 * d, d), up["b_in"])
        att = _laya_exact(qkv, keep, case["heads"], s["base"])
        return linear(att, up["w_out"].view(d, d), up["b_out"]).reshape(-1)
    s = _jeff_inputs(case, seed)
    R, L, W, KW = case["rows"], case["length"], case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    if kind == "jeff_layer":
        n = case["hidden"]
        x = s["x"].view(R, n, L).double()
        q, gate, k, v = (s[w].view(-1, n).double() @ x for w in ("w_q", "w_gate", "w_k", "w_v"))
    else:
        q, gate = s["q"].view(R, W, L), s["gate"].view(R, W, L)
        k, v = s["k"].view(R, -1, L), s["v"].view(R, -1, L)
        if kind == "jeff_op":  # the first of each group's copies
            k, v = (t.view(R, case["kv_heads"], -1, case["head_dim"], L)[:, :, 0].reshape(R, KW, L) for t in (k, v))
    out = _jeff_exact(case, q, k, v, gate, s["q_norm"], s["k_norm"], s["mask"])
    if kind == "jeff_layer":
        out = s["w_o"].view(case["hidden"], W).double() @ out
    return out.reshape(-1)
