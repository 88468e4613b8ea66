"""The measured workloads: what a program that serves Qwen2.5-shaped models
through this package has the GPU do.

listed() are fixed cases, draw() gives others of the same ranges.  A case is a
dict of plain values; its "op" says which entry point runs:

    decode_step    attention.decode_step: one token of every (sequence, layer)
                   over the fp16 cache (RoPE, append, split-K attention)
    prefill_step   attention.prefill_step_vt ("keep_vt") or prefill_step: a
                   chunk of prompt tokens after `base` cached positions
    decode_layers  layers.decode_all_layers over quantized weights; with
                   "logits" the final norm and lm_head after it
    prefill_layers layers.prefill_all_layers for a chunk of rows; with
                   "logits" the last row's final norm and lm_head after it
    matvec         vecops.matvec on a GGUF tensor

Every pass writes the same cache rows from the same inputs, so it can be
repeated on its state.
"""
from __future__ import annotations

import math
import random

import torch

from tinymetalagent_amd import attention as A
from tinymetalagent_amd import layers as LY
from tinymetalagent_amd import vecops as V

DEVICE = "cuda"
THETA = 1.0e6
EPS = 1.0e-6
VOCAB = 151936

# heads, kv heads, head_dim, feed-forward width, layers
SHAPES = {
    "0.5B": (14, 2, 64, 4864, 24),
    "1.5B": (12, 2, 128, 8960, 28),
    "3B": (16, 2, 128, 11008, 36),
    "7B": (28, 4, 128, 18944, 28),
}
Q4_0, Q8_0 = V.GGML_Q4_0, V.GGML_Q8_0
TYPES = {"Q4_0": Q4_0, "Q8_0": Q8_0}
BLOCK = 32


def listed() -> list[dict]:
    return [
        # the smallest call: one layer of the smallest model at a short context,
        # as a runtime that drives the layers itself issues it
        {"name": "decode_step_0.5B_512", "op": "decode_step", "shape": "0.5B", "layers": 1, "positions": "512"},
        # one token through the attention of every layer at 8K context: the
        # benchmark's own step
        {"name": "decode_step_3B_8K", "op": "decode_step", "shape": "3B", "layers": 36, "positions": "8192"},
        # a serving batch of eight sequences of ragged lengths
        {"name": "decode_step_7B_ragged", "op": "decode_step", "shape": "7B", "layers": 28,
         "positions": "1531,15877,9040,4211,12798,2345,7007,10662"},
        # one layer's attention for a 4096-token prompt, from an empty cache
        {"name": "prefill_step_3B_4096", "op": "prefill_step", "shape": "3B", "tokens": 4096, "base": 0,
         "keep_vt": True},
        # the last 2K chunk of a 16K document
        {"name": "prefill_step_1.5B_2K_after_14K", "op": "prefill_step", "shape": "1.5B", "tokens": 2048,
         "base": 14336, "keep_vt": True},
        # a prompt of odd length after a short cached prefix, by a program that
        # keeps no transposed value cache
        {"name": "prefill_step_0.5B_777", "op": "prefill_step", "shape": "0.5B", "tokens": 777, "base": 123,
         "keep_vt": False},
        # one layer of one token of the largest model, 8-bit weights
        {"name": "decode_layer_7B_Q8_0", "op": "decode_layers", "shape": "7B", "type": "Q8_0", "layers": 1,
         "position": 3000, "logits": False},
        # one generated token: every layer, the final norm and the logits
        {"name": "decode_token_3B_Q4_0", "op": "decode_layers", "shape": "3B", "type": "Q4_0", "layers": 36,
         "position": 639, "logits": True},
        # a chat's second turn: 64 new tokens after a cached conversation, one layer
        {"name": "prefill_layer_3B_Q8_0_64", "op": "prefill_layers", "shape": "3B", "type": "Q8_0", "layers": 1,
         "tokens": 64, "base": 576, "logits": False},
        # the second chunk of a long prompt through one layer of the largest model
        {"name": "prefill_layer_7B_Q8_0_512", "op": "prefill_layers", "shape": "7B", "type": "Q8_0", "layers": 1,
         "tokens": 512, "base": 512, "logits": False},
        # a whole 512-token prompt to its first logits
        {"name": "prompt_3B_Q4_0_512", "op": "prefill_layers", "shape": "3B", "type": "Q4_0", "layers": 36,
         "tokens": 512, "base": 0, "logits": True},
        # the vocabulary projection of one token
        {"name": "lm_head_3B_Q8_0", "op": "matvec", "type": "Q8_0", "rows": VOCAB, "cols": 2048},
    ]


def _log_int(rng: random.Random, low: int, high: int) -> int:
    return round(math.exp(rng.uniform(math.log(low), math.log(high))))


def draw(rng: random.Random) -> dict:
    op = rng.choice(["decode_step", "prefill_step", "decode_layers", "prefill_layers", "prefill_layers", "matvec"])
    shape = rng.choice(sorted(SHAPES))
    kind = rng.choice(sorted(TYPES))
    if op == "decode_step":
        # up to the ragged batch's cache size, any split of it over sequences and layers
        seqs = _log_int(rng, 1, 16)
        layers = rng.choice([1, 2, SHAPES[shape][4]])
        row = 4 * SHAPES[shape][1] * SHAPES[shape][2] * layers
        longest = max(64, min(131072, int(6.0e9 / row / seqs)))
        positions = [_log_int(rng, 16, longest) for _ in range(seqs)]
        return {"op": op, "shape": shape, "layers": layers, "positions": ",".join(map(str, positions))}
    if op == "prefill_step":
        return {"op": op, "shape": shape, "tokens": _log_int(rng, 16, 4096),
                "base": rng.choice([0, _log_int(rng, 1, 14000)]), "keep_vt": rng.random() < 0.7}
    if op == "decode_layers":
        return {"op": op, "shape": shape, "type": kind, "layers": rng.choice([1, 2, 4]),
                "position": _log_int(rng, 16, 16000), "logits": False}
    if op == "prefill_layers":
        return {"op": op, "shape": shape, "type": kind, "layers": rng.choice([1, 2]), "tokens": _log_int(rng, 8, 512),
                "base": rng.choice([0, _log_int(rng, 1, 4000)]), "logits": False}
    return {"op": op, "type": kind, "rows": _log_int(rng, 500, VOCAB), "cols": BLOCK * rng.randint(16, 256)}


# ---- inputs ------------------------------------------------------------------


def _randn(g: torch.Generator, *shape: int, scale: float = 1.0) -> torch.Tensor:
    return torch.randn(shape, generator=g, device=DEVICE).mul_(scale)


def _half(g: torch.Generator, *shape: int) -> torch.Tensor:
    """fp16 cache contents, drawn one leading slice at a time."""
    out = torch.empty(shape, dtype=torch.float16, device=DEVICE)
    for part in out.view(-1, *shape[2:]):
        part.copy_(_randn(g, *shape[2:]))
    return out


def _keys(g: torch.Generator, *shape: int) -> torch.Tensor:
    """Cached keys: two channels of each head are several times the others."""
    k = _half(g, *shape)
    k[..., 3] *= 6
    k[..., shape[-1] // 2 + 5] *= 6
    return k


def _hidden(g: torch.Generator, *shape: int) -> torch.Tensor:
    """Residual-stream rows: N(0, 1) with a few large channels."""
    x = _randn(g, *shape)
    x[..., 7::shape[-1] // 4] *= 12
    return x


def _fill_tensor(g: torch.Generator, dst: torch.Tensor, kind: int, rows: int, cols: int) -> None:
    """A GGUF tensor's bytes into dst: normal codes and block scales that keep
    a projection's outputs near unit variance, of either sign as quantizers
    write them."""
    blocks = rows * cols // BLOCK
    std = 2.6 if kind == Q4_0 else 40.0
    d = _randn(g, blocks, scale=0.25).exp_().mul_(1.0 / (std * math.sqrt(cols)))
    d *= torch.where(torch.rand(blocks, generator=g, device=DEVICE) < 0.5, -1.0, 1.0)
    out = dst.view(blocks, -1)
    out[:, :2] = d.half().view(torch.uint8).view(blocks, 2)
    codes = _randn(g, blocks, BLOCK, scale=std).round_()
    if kind == Q4_0:
        n = codes.clamp_(-8, 7).add_(8).to(torch.uint8)
        out[:, 2:] = n[:, :16] | n[:, 16:] << 4
    else:
        out[:, 2:] = codes.clamp_(-127, 127).to(torch.int8).view(torch.uint8)


def _projections(shape: str) -> dict:
    heads, kv, d, ffn, _ = SHAPES[shape]
    hidden = heads * d
    return {"q": (hidden, hidden), "k": (kv * d, hidden), "v": (kv * d, hidden), "output": (hidden, hidden),
            "gate": (ffn, hidden), "up": (ffn, hidden), "down": (hidden, ffn)}


def _model(g: torch.Generator, shape: str, kind: int, layers: int, head: bool) -> dict:
    """The weights of a model file in HBM: every tensor 32-byte aligned."""
    heads, kv, d, ffn, _ = SHAPES[shape]
    hidden = heads * d
    sizes, offsets, cursor = [], {n: [] for n in _projections(shape)}, 0
    for _layer in range(layers):
        for n, (rows, cols) in _projections(shape).items():
            offsets[n].append(cursor)
            sizes.append((cursor, rows, cols))
            cursor += -(-rows * V.row_bytes(kind, cols) // 32) * 32
    head_offset = cursor
    if head:
        sizes.append((cursor, VOCAB, hidden))
        cursor += VOCAB * V.row_bytes(kind, hidden)
    mapping = torch.zeros(cursor + 64, dtype=torch.uint8, device=DEVICE)
    for off, rows, cols in sizes:
        _fill_tensor(g, mapping[off:off + rows * V.row_bytes(kind, cols)], kind, rows, cols)
    return {
        "mapping": mapping, "offsets": offsets, "head_offset": head_offset,
        "attn_norm": _randn(g, layers, hidden, scale=0.1).add_(1), "ffn_norm": _randn(g, layers, hidden, scale=0.1).add_(1),
        "out_norm": _randn(g, hidden, scale=0.1).add_(1),
        "q_bias": _randn(g, layers, hidden, scale=0.3), "k_bias": _randn(g, layers, kv * d, scale=0.3),
        "v_bias": _randn(g, layers, kv * d, scale=0.1),
    }


def _positions(case: dict) -> list[int]:
    return [int(p) for p in case["positions"].split(",")]


def prepare(case: dict, seed: int) -> dict:
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    op = case["op"]
    s = {"case": case}
    if op == "matvec":
        kind, rows, cols = TYPES[case["type"]], case["rows"], case["cols"]
        w = torch.empty(rows * V.row_bytes(kind, cols), dtype=torch.uint8, device=DEVICE)
        _fill_tensor(g, w, kind, rows, cols)
        s.update(w=w, x=_hidden(g, cols), out=torch.empty(rows, device=DEVICE))
        return s
    heads, kv, d, ffn, _ = SHAPES[case["shape"]]
    hidden = heads * d
    if op == "decode_step":
        layers, positions = case["layers"], _positions(case)
        seqs, ctx = len(positions), max(positions) + 1
        s.update(positions=positions, q=_randn(g, seqs, layers, heads, d), k=_randn(g, seqs, layers, kv, d),
                 v=_randn(g, seqs, layers, kv, d), q_bias=_randn(g, layers, hidden, scale=0.3),
                 k_bias=_randn(g, layers, kv * d, scale=0.3), v_bias=_randn(g, layers, kv * d, scale=0.1),
                 kc=_keys(g, seqs, layers, ctx, kv, d), vc=_half(g, seqs, layers, ctx, kv, d),
                 out=torch.empty(seqs, layers, heads, d, device=DEVICE),
                 ws=A.decode_workspace(seqs, layers, heads, kv, d, positions=positions, device=DEVICE))
    elif op == "prefill_step":
        tokens, base = case["tokens"], case["base"]
        ctx = base + tokens
        s.update(q=_randn(g, 1, 1, tokens, heads, d), k=_randn(g, 1, 1, tokens, kv, d),
                 v=_randn(g, 1, 1, tokens, kv, d), q_bias=_randn(g, 1, hidden, scale=0.3),
                 k_bias=_randn(g, 1, kv * d, scale=0.3), v_bias=_randn(g, 1, kv * d, scale=0.1),
                 kc=_keys(g, 1, 1, ctx, kv, d), vc=_half(g, 1, 1, ctx, kv, d),
                 out=torch.empty(1, 1, tokens, heads, d, device=DEVICE))
        if case["keep_vt"]:
            s["vt"] = A.value_t_buffer(1, 1, ctx, kv, d, device=DEVICE)
            if base:
                A.value_transpose(s["vc"], s["vt"], first_position=0, count=base)
            s["ws"] = A.prefill_vt_workspace(1, 1, tokens, heads, kv, d, base_position=base, context_tokens=ctx,
                                             device=DEVICE)
    else:
        kind, layers = TYPES[case["type"]], case["layers"]
        s.update(_model(g, case["shape"], kind, layers, case["logits"]))
        base = case["position"] if op == "decode_layers" else case["base"]
        rows = 1 if op == "decode_layers" else case["tokens"]
        ctx = base + rows
        s.update(kc=_keys(g, 1, layers, ctx, kv, d), vc=_half(g, 1, layers, ctx, kv, d))
        if op == "decode_layers":
            s.update(x=_hidden(g, hidden), ws=LY.workspace(base, hidden, kv * d, heads, kv, d, ffn, device=DEVICE))
        else:
            s.update(x=_hidden(g, rows, hidden), ws=LY.prefill_workspace(rows, hidden, kv * d, ffn, device=DEVICE))
            s["vt"] = A.value_t_buffer(1, layers, ctx, kv, d, device=DEVICE)
            if base:
                A.value_transpose(s["vc"], s["vt"], first_position=0, count=base)
        s["out"] = torch.empty_like(s["x"])
        if case["logits"]:
            s.update(norm=torch.empty(hidden, device=DEVICE), logits=torch.empty(VOCAB, device=DEVICE))
    s["cos"], s["sin"] = A.rope_table(ctx, d, THETA, device=DEVICE)
    return s


# ---- one pass ----------------------------------------------------------------


def run(s: dict):
    case = s["case"]
    op = case["op"]
    if op == "matvec":
        return V.matvec(s["w"], TYPES[case["type"]], s["x"], case["rows"], out=s["out"])
    if op == "decode_step":
        out = A.decode_step(s["q"], s["k"], s["v"], s["cos"], s["sin"], s["kc"], s["vc"], positions=s["positions"],
                            q_bias=s["q_bias"], k_bias=s["k_bias"], v_bias=s["v_bias"], out=s["out"],
                            workspace=s["ws"])
        return {"out": out, "key_cache": s["kc"], "value_cache": s["vc"]}
    if op == "prefill_step":
        biases = {"q_bias": s["q_bias"], "k_bias": s["k_bias"], "v_bias": s["v_bias"]}
        if case["keep_vt"]:
            out = A.prefill_step_vt(s["q"], s["k"], s["v"], s["cos"], s["sin"], s["kc"], s["vc"], s["vt"],
                                    base_position=case["base"], out=s["out"], workspace=s["ws"], **biases)
            return {"out": out, "key_cache": s["kc"], "value_cache": s["vc"], "value_t": s["vt"]}
        out = A.prefill_step(s["q"], s["k"], s["v"], s["cos"], s["sin"], s["kc"], s["vc"], base_position=case["base"],
                             out=s["out"], **biases)
        return {"out": out, "key_cache": s["kc"], "value_cache": s["vc"]}
    heads, kv, d, ffn, _ = SHAPES[case["shape"]]
    kind, layers = TYPES[case["type"]], case["layers"]
    ctx = s["kc"].shape[2]
    weights = (s["mapping"], s["offsets"], layers, kind, s["x"], s["attn_norm"], s["ffn_norm"], s["q_bias"],
               s["k_bias"], s["v_bias"], s["cos"], s["sin"], s["kc"], s["vc"])
    if op == "decode_layers":
        out = LY.decode_all_layers(*weights, case["position"], ctx, heads, kv, d, ffn, EPS, out=s["out"], ws=s["ws"])
        last = out
    else:
        out = LY.prefill_all_layers(*weights, s["vt"], case["base"], ctx, heads, kv, d, ffn, EPS, out=s["out"],
                                    ws=s["ws"])
        last = out[-1]
    result = {"hidden": out, "key_cache": s["kc"], "value_cache": s["vc"]}
    if op == "prefill_layers":
        result["value_t"] = s["vt"]
    if case["logits"]:
        hidden = heads * d
        V.rmsnorm(last, s["out_norm"], EPS, out=s["norm"])
        head = s["mapping"][s["head_offset"]:s["head_offset"] + VOCAB * V.row_bytes(kind, hidden)]
        result["logits"] = V.matvec(head, kind, s["norm"], VOCAB, out=s["logits"])
    return result


# ---- what a pass cannot do without -------------------------------------------


def _attention_work(shape: str, rows: int, base: int) -> tuple[float, float]:
    """Bytes and operations of one layer's attention for `rows` tokens after
    `base` cached ones: the cache up to the last row once, fp32 q / k / v in,
    fp16 k / v and fp32 rows out, the rows' rotations."""
    heads, kv, d, _, _ = SHAPES[shape]
    flops = 4.0 * heads * d * (rows * base + rows * (rows + 1) / 2)
    nbytes = 4.0 * base * kv * d + rows * (heads * d * 8 + kv * d * 12 + d * 4)
    return nbytes, flops


def work(case: dict) -> dict:
    op = case["op"]
    if op == "matvec":
        rows, cols = case["rows"], case["cols"]
        return {"bytes": rows * V.row_bytes(TYPES[case["type"]], cols) + 4.0 * (rows + cols), "flops": 2.0 * rows * cols}
    heads, _, d, _, _ = SHAPES[case["shape"]]
    if op == "decode_step":
        parts = [_attention_work(case["shape"], 1, p) for p in _positions(case)] * case["layers"]
    elif op == "prefill_step":
        parts = [_attention_work(case["shape"], case["tokens"], case["base"])]
    else:
        rows, base = (1, case["position"]) if op == "decode_layers" else (case["tokens"], case["base"])
        kind, hidden = TYPES[case["type"]], heads * d
        dims = _projections(case["shape"]).values()
        nbytes, flops = _attention_work(case["shape"], rows, base)
        nbytes += sum(n * V.row_bytes(kind, k) for n, k in dims) - rows * hidden * 8
        flops += 2.0 * rows * sum(n * k for n, k in dims)
        parts = [(nbytes, flops)] * case["layers"] + [(rows * hidden * 8.0, 0.0)]
        if case["logits"]:
            parts.append((VOCAB * (V.row_bytes(kind, hidden) + 4.0), 2.0 * VOCAB * hidden))
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case: dict) -> dict:
    """About four times the error against exact() of the outputs computed (the
    appended fp16 rows differ by one rounding at most: "max")."""
    op = case["op"]
    if op == "matvec":  # fp32 sums over inputs rounded to 22 bits: 4e-7
        return {"rel": 2.0e-6, "max": 2.0e-5}
    if op == "decode_step":  # fp32 softmax and sums over the fp16 cache: up to 1.5e-6, the cache rows 1.1e-5
        return {"rel": 2.0e-5, "max": 2.0e-3}
    if op == "prefill_step":  # fp16 queries and weights of the softmax: up to 4.1e-4
        return {"rel": 1.6e-3, "max": 2.0e-2}
    if op == "decode_layers":  # 2e-6 after 36 layers, the cache rows 9e-6
        return {"rel": 2.0e-5, "max": 2.0e-3}
    return {"rel": 2.4e-3, "max": 2.0e-2}  # fp16 attention through every layer: up to 5.8e-4


# ---- the same in 64 bits -----------------------------------------------------


def _dequantize(data: torch.Tensor, kind: int, rows: int, cols: int) -> torch.Tensor:
    b = data[:rows * V.row_bytes(kind, cols)].view(rows * cols // BLOCK, -1)
    d = b[:, :2].contiguous().view(torch.float16).double()
    if kind == Q4_0:
        n = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8
    else:
        n = b[:, 2:].contiguous().view(torch.int8).double()
    return (n * d).view(rows, cols)


def _rotate(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, first: int) -> torch.Tensor:
    """x [tokens, heads, d] at positions first, first + 1, ..."""
    half = x.shape[-1] // 2
    c = cos[first:first + x.shape[0], None].double()
    n = sin[first:first + x.shape[0], None].double()
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * n, b * c + a * n], -1)


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, base: int) -> torch.Tensor:
    """Causal attention of rows q [tokens, heads, d] at positions base.. over
    k / v [positions, kv, d], one head at a time."""
    tokens, heads, d = q.shape
    group = heads // k.shape[1]
    out = torch.empty_like(q)
    mask = None
    if tokens > 1:
        rows = torch.arange(tokens, device=q.device)[:, None] + base
        mask = torch.arange(k.shape[0], device=q.device)[None] > rows
    for h in range(heads):
        scores = q[:, h] @ k[:, h // group].T.contiguous() / math.sqrt(d)
        if mask is not None:
            scores = scores.masked_fill(mask, -math.inf)
        out[:, h] = scores.softmax(-1) @ v[:, h // group].contiguous()
    return out


def _attention_exact(s, q, k, v, kc, vc, base, exact_k, exact_v):
    """One (sequence, layer): biased q / k / v [tokens, heads, d] in, the rows
    appended to exact_k / exact_v, attention over the cache as fp16 holds it."""
    n = base + q.shape[0]
    exact_k[base:n] = _rotate(k, s["cos"], s["sin"], base)
    exact_v[base:n] = v
    keys, values = kc[:n].double(), vc[:n].double()
    keys[base:] = exact_k[base:n].half().double()
    values[base:] = exact_v[base:n].half().double()
    return _attend(_rotate(q, s["cos"], s["sin"], base), keys, values, base)


def _transposed(s, exact_v, count):
    """V^T of the first `count` positions, zeros after them."""
    vt = torch.zeros(s["vt"].shape, dtype=torch.float64, device=DEVICE)
    vt[..., :count] = exact_v[:, :, :count].permute(0, 1, 3, 4, 2)
    return vt


def exact(case: dict, seed: int):
    s = prepare(case, seed)
    op = case["op"]
    if op == "matvec":
        return _dequantize(s["w"], TYPES[case["type"]], case["rows"], case["cols"]) @ s["x"].double()
    heads, kv, d, ffn, _ = SHAPES[case["shape"]]
    exact_k, exact_v = s["kc"].double(), s["vc"].double()

    def biased(x, bias, n):
        return (x.double() + bias.double()).view(-1, n, d)

    if op in ("decode_step", "prefill_step"):
        bases = s["positions"] if op == "decode_step" else [case["base"]]
        out = torch.empty(s["out"].shape, dtype=torch.float64, device=DEVICE)
        for i, base in enumerate(bases):
            for l in range(s["kc"].shape[1]):
                rows = s["q"][i, l].reshape(-1, heads * d).shape[0]
                args = [biased(s[t][i, l].reshape(rows, -1), s[t + "_bias"][l], n)
                        for t, n in (("q", heads), ("k", kv), ("v", kv))]
                out[i, l] = _attention_exact(s, *args, s["kc"][i, l], s["vc"][i, l], base, exact_k[i, l],
                                             exact_v[i, l]).view(out[i, l].shape)
        result = {"out": out, "key_cache": exact_k, "value_cache": exact_v}
        if op == "prefill_step" and case["keep_vt"]:
            result["value_t"] = _transposed(s, exact_v, case["base"] + case["tokens"])
        return result

    kind, hidden = TYPES[case["type"]], heads * d
    base = case["position"] if op == "decode_layers" else case["base"]
    x = s["x"].double().view(-1, hidden)

    def norm(rows, weight):
        return rows / (rows.square().mean(-1, keepdim=True) + EPS).sqrt() * weight.double()

    for l in range(case["layers"]):
        def project(name, rows):
            n, k = _projections(case["shape"])[name]
            return rows @ _dequantize(s["mapping"][s["offsets"][name][l]:], kind, n, k).T

        h = norm(x, s["attn_norm"][l])
        args = [biased(project(t, h), s[t + "_bias"][l], n) for t, n in (("q", heads), ("k", kv), ("v", kv))]
        attn = _attention_exact(s, *args, s["kc"][0, l], s["vc"][0, l], base, exact_k[0, l], exact_v[0, l])
        x = x + project("output", attn.reshape(-1, hidden))
        h = norm(x, s["ffn_norm"][l])
        gate = project("gate", h)
        x = x + project("down", gate * torch.sigmoid(gate) * project("up", h))
    result = {"hidden": x.view(s["out"].shape), "key_cache": exact_k, "value_cache": exact_v}
    if op == "prefill_layers":
        result["value_t"] = _transposed(s, exact_v, base + case["tokens"])
    if case["logits"]:
        head = _dequantize(s["mapping"][s["head_offset"]:], kind, VOCAB, hidden)
        result["logits"] = head @ norm(x[-1], s["out_norm"])
    return result
