"""The work this framework is timed on, over the range its users put it to.

The shapes are the Qwen2.5-0.5B ones of ``qwenforge_amd.model.Qwen2Config``
(14 query heads over 2 kv heads of 64, hidden 896, MLP 4864, vocab 151936).
Kinds of case:

* ``decode`` / ``decode_paged`` -- the attention of one decode step, all 24
  layers captured in a hipGraph as the engines capture it, over dense or paged
  caches.
* ``prefill`` / ``prefill_ragged`` -- RoPE + append + causal attention of a
  prompt (or of packed prompts), a few layers captured in a hipGraph.
* ``attn_block`` / ``mlp_block`` -- the two halves of the fused decode step of
  1..4 rows, 24 layers of their own weights captured in a hipGraph.
* ``model_decode`` -- a whole captured decode step of the engine.
* ``model_prefill`` -- a whole prefill call of the engine.
"""

from __future__ import annotations

import math

import torch

from qwenforge_amd import ops, paged, step_ops
from qwenforge_amd.engine import DecodeEngine, cache_capacity
from qwenforge_amd.model import Qwen2Config, init_weights
from qwenforge_amd.rope import cos_sin, inv_freq

CFG = Qwen2Config()
QH, KVH, G, D = CFG.heads, CFG.kv_heads, CFG.groups, CFG.head_dim
LAYERS = CFG.layers
PREFILL_LAYERS = 4
DEV = "cuda"
F16_MIN = torch.finfo(torch.float16).min


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------

def listed():
    return [
        # One user's short chat: 512 tokens of context, latency is all.
        dict(name="decode_b1_512", kind="decode", batch=1, lo=512, hi=512, mask="none", heavy=0.0),
        # Four chats of different lengths in one padded batch, holes masked by a bias.
        dict(name="decode_b4_ragged", kind="decode", batch=4, lo=256, hi=2048, mask="bias", heavy=0.0),
        # One long document whose attention is dominated by a few keys.
        dict(name="decode_b1_32768", kind="decode", batch=1, lo=32768, hi=32768, mask="none",
             heavy=0.01),
        # An evaluation batch with long prompts; all rows share the write slot.
        dict(name="decode_b12_5760", kind="decode", batch=12, lo=5760, hi=5760, mask="slot", heavy=0.0),
        # A serving batch over a paged cache, each row at its own odd length.
        dict(name="paged_b16_ragged", kind="decode_paged", batch=16, lo=201, hi=6007, page=64),
        # A prompt of ordinary length.
        dict(name="prefill_2048", kind="prefill", batch=1, seq=2048),
        # A long prompt.
        dict(name="prefill_8192", kind="prefill", batch=1, seq=8192),
        # Four prompts admitted together, packed along the token axis.
        dict(name="prefill_ragged_4", kind="prefill_ragged", batch=4, lo=509, hi=1024),
        # The attention half of the layers of a four-row decode step.
        dict(name="attn_block_b4", kind="attn_block", batch=4, length=1024),
        # The MLP half of the layers of a one-row decode step.
        dict(name="mlp_block_b1", kind="mlp_block", batch=1),
        # A decode step of an evaluation or serving batch, whole model.
        dict(name="model_decode_b12", kind="model_decode", batch=12, length=1024),
        # The prompt of one request, whole model.
        dict(name="model_prefill_1024", kind="model_prefill", batch=1, lo=1024, hi=1024),
    ]


def _log_int(rng, lo, hi):
    """Whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode_paged", "prefill", "prefill_ragged", "attn_block",
                       "mlp_block", "model_decode", "model_prefill"])
    if kind == "decode":
        batch = _log_int(rng, 1, 32)
        hi = _log_int(rng, 128, min(32768, 69120 // batch))
        mask = rng.choice(["none", "slot", "bias", "rows"])
        lo = hi if mask in ("none", "slot") else max(1, int(hi * rng.uniform(0.1, 1.0)))
        return dict(kind=kind, batch=batch, lo=lo, hi=hi, mask=mask, heavy=rng.choice([0.0, 0.01]))
    if kind == "decode_paged":
        batch = _log_int(rng, 1, 32)
        hi = _log_int(rng, 128, min(32768, 69120 // batch))
        return dict(kind=kind, batch=batch, lo=max(1, int(hi * rng.uniform(0.03, 1.0))), hi=hi,
                    page=rng.choice([64, 64, 128, 256]))
    if kind == "prefill":
        batch = rng.choice([1, 1, 1, 2, 4, 8])
        return dict(kind=kind, batch=batch, seq=_log_int(rng, 32, 8192 // batch))
    if kind == "prefill_ragged":
        batch = rng.randint(2, 16)
        hi = _log_int(rng, 48, 8192 // batch)
        return dict(kind=kind, batch=batch, lo=max(1, int(hi * rng.uniform(0.05, 0.9))), hi=hi)
    if kind == "attn_block":
        return dict(kind=kind, batch=rng.randint(1, 4), length=_log_int(rng, 32, 4000))
    if kind == "mlp_block":
        # Four sizes there are; the salt tells draws of the same size apart.
        return dict(kind=kind, batch=rng.randint(1, 4), salt=rng.randint(1, 10**6))
    if kind == "model_decode":
        batch = _log_int(rng, 1, 32)
        return dict(kind=kind, batch=batch, length=_log_int(rng, 32, min(4000, 32768 // batch)))
    batch = rng.choice([1, 1, 2, 4, 6])
    hi = _log_int(rng, 24, 2048 // batch)
    return dict(kind="model_prefill", batch=batch,
                lo=hi if batch == 1 else max(1, int(hi * rng.uniform(0.2, 1.2))), hi=hi)


def _lengths(case):
    """The rows' lengths: evenly over [lo, hi], in an order that is not sorted."""
    b, lo, hi = case["batch"], min(case["lo"], case["hi"]), case["hi"]
    if b == 1:
        return [hi]
    row = [lo + (hi - lo) * i // (b - 1) for i in range(b)]
    return row[1::2] + row[0::2][::-1]


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------

def _gen(seed, case):
    return torch.Generator(DEV).manual_seed(int(seed) * 1000003 + int(case.get("salt", 0)))


def _randn(gen, *shape, std=1.0):
    return (torch.randn(*shape, generator=gen, device=DEV, dtype=torch.float32) * std).half()


def _capture(fn):
    """A hipGraph of ``fn`` after one warm-up on a side stream."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        fn()
    torch.cuda.synchronize()
    return graph


def _heavy(gen, k, length, frac):
    """Scale the same random ``frac`` of the first ``length`` keys of every row by 8."""
    if frac > 0:
        rows = torch.randperm(length, generator=gen, device=DEV)[:max(1, round(frac * length))]
        k[..., rows, :] *= 8


def _decode_inputs(case, seed):
    gen = _gen(seed, case)
    b, lengths = case["batch"], _lengths(case)
    cap = cache_capacity(case["hi"], 1)
    q = _randn(gen, LAYERS, b, KVH, G, D)
    k = _randn(gen, LAYERS, b, KVH, cap, D)
    v = _randn(gen, LAYERS, b, KVH, cap, D)
    _heavy(gen, k, case["hi"], case.get("heavy", 0.0))
    return q, k, v, lengths, cap


def _prepare_decode(case, seed):
    b = case["batch"]
    q, k, v, lengths, cap = _decode_inputs(case, seed)
    bias = kv_last = None
    if case["mask"] == "none":
        k, v = k[:, :, :, :case["hi"]], v[:, :, :, :case["hi"]]
        cap = case["hi"]
    elif case["mask"] == "slot":
        kv_last = torch.tensor([case["hi"] - 1], device=DEV)
    elif case["mask"] == "rows":
        kv_last = torch.tensor(lengths, device=DEV) - 1
    else:
        bias = torch.full((b, cap), F16_MIN, device=DEV, dtype=torch.float16)
        for i, n in enumerate(lengths):
            bias[i, :n] = 0.0
    flash = ops.make_flash_scratch(b, KVH, G, cap, DEV)
    outs = torch.zeros(LAYERS, b, KVH, G, D, device=DEV, dtype=torch.float16)

    def step():
        for i in range(LAYERS):
            ops.flash_decode_attention(q[i], k[i], v[i], bias,
                                       (*flash[:3], outs[i], *flash[4:]), kv_last=kv_last)

    return {"graph": _capture(step), "out": outs, "keep": (q, k, v, bias, kv_last, flash)}


def _paged_inputs(case, seed):
    gen = _gen(seed, case)
    b, lengths, page = case["batch"], _lengths(case), case["page"]
    need = [-(-n // page) for n in lengths]
    ids = torch.randperm(sum(need), generator=gen, device=DEV).to(torch.int32)
    table = torch.full((b, max(need)), -1, device=DEV, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = ids[at:at + n]
        at += n
    q = _randn(gen, LAYERS, b, KVH, G, D)
    k = _randn(gen, LAYERS, sum(need), KVH, page, D)
    v = _randn(gen, LAYERS, sum(need), KVH, page, D)
    return q, k, v, table, lengths


def _prepare_decode_paged(case, seed):
    b = case["batch"]
    q, k, v, table, lengths = _paged_inputs(case, seed)
    kv_last = torch.tensor(lengths, device=DEV) - 1
    flash = ops.make_flash_scratch(b, KVH, G, table.shape[1] * case["page"], DEV)
    outs = torch.zeros(LAYERS, b, KVH, G, D, device=DEV, dtype=torch.float16)

    def step():
        for i in range(LAYERS):
            paged.flash_decode_attention_paged(q[i], k[i], v[i], table, None,
                                               (*flash[:3], outs[i], *flash[4:]), kv_last=kv_last)

    return {"graph": _capture(step), "out": outs, "keep": (q, k, v, table, kv_last, flash)}


def _proj_inputs(case, seed, rows, tokens):
    """Fused QKV projections of ``PREFILL_LAYERS`` layers, as a linear layer leaves them."""
    return _randn(_gen(seed, case), PREFILL_LAYERS, rows, tokens, (QH + 2 * KVH) * D)


def _split_heads(proj):
    q, k, v = proj.split((QH * D, KVH * D, KVH * D), dim=-1)
    return (q.unflatten(-1, (QH, D)), k.unflatten(-1, (KVH, D)), v.unflatten(-1, (KVH, D)))


def _prepare_prefill(case, seed):
    b, s = case["batch"], case["seq"]
    proj = _proj_inputs(case, seed, b, s)
    cos, sin = cos_sin(torch.arange(s, device=DEV), inv_freq(D, CFG.rope_theta, DEV))
    caches = torch.zeros(PREFILL_LAYERS, 2, b, KVH, cache_capacity(s, 1), D, device=DEV,
                         dtype=torch.float16)
    outs = []

    def step():
        outs.clear()
        for i in range(PREFILL_LAYERS):
            q, k, v = (t.transpose(1, 2) for t in _split_heads(proj[i]))
            outs.append(torch.ops.student_qwen.gqa_flash_prefill_rope_append(
                q, k, v, cos, sin, caches[i, 0], caches[i, 1], 0))

    graph = _capture(step)
    return {"graph": graph, "out": {"out": outs, "caches": caches}, "keep": (proj, cos, sin)}


def _prepare_prefill_ragged(case, seed):
    lengths = _lengths(case)
    total = sum(lengths)
    proj = _proj_inputs(case, seed, 1, total)[:, 0]
    pos = torch.cat([torch.arange(n, device=DEV) for n in lengths])
    cos, sin = cos_sin(pos, inv_freq(D, CFG.rope_theta, DEV))
    cu = torch.tensor([sum(lengths[:i]) for i in range(len(lengths) + 1)], device=DEV,
                      dtype=torch.int32)
    caches = torch.zeros(PREFILL_LAYERS, 2, len(lengths), KVH, cache_capacity(max(lengths), 1), D,
                         device=DEV, dtype=torch.float16)
    outs = []

    def step():
        outs.clear()
        for i in range(PREFILL_LAYERS):
            q, k, v = _split_heads(proj[i])
            outs.append(ops.prefill_varlen(q, k, v, cu, max(lengths), cos, sin, caches[i, 0],
                                           caches[i, 1], 0, lengths=lengths))

    graph = _capture(step)
    return {"graph": graph, "out": {"out": outs, "caches": caches}, "keep": (proj, cos, sin, cu)}


def _block_weights(case, seed):
    """The layers of the model alone: neither block reads the embedding."""
    cfg = Qwen2Config(vocab=64)
    return cfg, init_weights(cfg, DEV, int(_gen(seed, case).initial_seed()))


def _block_hidden(case, seed):
    return _randn(_gen(int(seed) + 1, case), case["batch"], CFG.hidden)


def _block_caches(case, seed):
    return _randn(_gen(int(seed) + 2, case), LAYERS, 2, case["batch"], KVH,
                  cache_capacity(case["length"], 128), D)


def _prepare_attn_block(case, seed):
    b, n = case["batch"], case["length"]
    cfg, weights = _block_weights(case, seed)
    engine = DecodeEngine(cfg, weights, DEV)
    first, caches = _block_hidden(case, seed), _block_caches(case, seed)
    hidden = first.clone()
    write = torch.tensor([n], device=DEV)
    rope = (torch.full((b,), n, device=DEV, dtype=torch.long), engine.inv_freq)
    cap = caches.shape[4]
    flash = ops.make_flash_scratch(b, KVH, G, cap, DEV, fused=False,
                                   splits=min(ops.choose_splits(b, KVH, cap),
                                              engine.fused_max_splits(b)))
    q_rot = torch.zeros(b, QH, D, device=DEV, dtype=torch.float16)

    def step():
        for i, layer in enumerate(weights["layers"]):
            kc, vc = caches[i, 0], caches[i, 1]
            step_ops.rms_qkv_rope_append(hidden, layer["input_norm"], cfg.rms_eps,
                                         engine.projection_weights(i, b)[0], layer["qkv_bias"],
                                         None, None, kc, vc, write, q_rot, positions=rope)
            ops.flash_decode_split(q_rot.view(b, KVH, G, D), kc, vc, None, flash, kv_last=write,
                                   split_capacity=True)
            step_ops.attn_merge_o_proj(flash, engine.o_proj_weight(i, b), hidden)

    graph = _capture(step)
    out = {"hidden": hidden, "rows": caches[:, :, :, :, n], "caches": caches}
    return {"graph": graph, "out": out, "reset": [(hidden, first)],
            "keep": (engine, write, rope, flash, q_rot)}


def _prepare_mlp_block(case, seed):
    b = case["batch"]
    cfg, weights = _block_weights(case, seed)
    engine = DecodeEngine(cfg, weights, DEV)
    first = _block_hidden(case, seed)
    hidden = first.clone()
    h = torch.zeros(LAYERS, b, cfg.intermediate, device=DEV, dtype=torch.float16)

    def step():
        for i, layer in enumerate(weights["layers"]):
            step_ops.rms_gate_up_swiglu(hidden, layer["post_norm"], cfg.rms_eps,
                                        engine.projection_weights(i, b)[1], h[i])
            step_ops.gemv_residual(h[i], layer["down_weight"], hidden)

    graph = _capture(step)
    return {"graph": graph, "out": {"hidden": hidden, "h": h}, "reset": [(hidden, first)],
            "keep": (engine,)}


def _model_weights(case, seed):
    return init_weights(CFG, DEV, int(_gen(seed, case).initial_seed()))


def _tokens(case, seed, n):
    return torch.randint(CFG.vocab, (n,), generator=_gen(int(seed) + 1, case), device=DEV)


def _prepare_model_decode(case, seed):
    b, n = case["batch"], case["length"]
    engine = DecodeEngine(CFG, _model_weights(case, seed), DEV)
    caches = _block_caches(case, seed)
    ctx = engine.make_context([(caches[i, 0], caches[i, 1]) for i in range(LAYERS)], b, 128)
    first = _tokens(case, seed, b)
    start = {"token": first, "pos": torch.full_like(first, n),
             "write": torch.full((1,), n, device=DEV), "step": torch.ones(1, device=DEV).long()}
    parked = caches[:, :, :, :, -1].clone()
    graph = engine.capture(ctx)
    caches[:, :, :, :, -1] = parked     # the warm-ups of the capture append there
    out = {"logits": ctx["logits"], "rows": caches[:, :, :, :, n], "caches": caches}
    return {"graph": graph, "out": out, "reset": [(ctx[key], t) for key, t in start.items()],
            "keep": (engine, ctx)}


def _prepare_model_prefill(case, seed):
    lengths = _lengths(case)
    engine = DecodeEngine(CFG, _model_weights(case, seed), DEV)
    ids = _tokens(case, seed, sum(lengths)).split(lengths)
    caches = torch.zeros(LAYERS, 2, len(lengths), KVH, cache_capacity(max(lengths), 128), D,
                         device=DEV, dtype=torch.float16)
    pairs = [(caches[i, 0], caches[i, 1]) for i in range(LAYERS)]
    if min(lengths) == max(lengths):
        prompts = torch.stack(ids)
        call = lambda: engine.prefill(prompts, pairs)  # noqa: E731
    else:
        call = lambda: engine.prefill_ragged(list(ids), pairs)  # noqa: E731
    return {"call": call, "caches": caches}


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------

def run(state):
    if "call" in state:
        return {"logits": state["call"](), "caches": state["caches"]}
    for to, start in state.get("reset", ()):
        to.copy_(start)
    state["graph"].replay()
    return state["out"]


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------

def _causal_pairs(lengths):
    return sum(n * (n + 1) // 2 for n in lengths)


def _linear_params():
    return CFG.hidden * (CFG.qkv_width + CFG.heads * D + 3 * CFG.intermediate)


def work(case):
    kind, b = case["kind"], case["batch"]
    row = 2 * KVH * D * 2                      # bytes of one token's K and V in one layer
    if kind in ("decode", "decode_paged"):
        n = sum(_lengths(case))
        return {"bytes": LAYERS * (row * n + 2 * 2 * b * QH * D), "flops": LAYERS * 4 * n * QH * D}
    if kind in ("prefill", "prefill_ragged"):
        lengths = [case["seq"]] * b if kind == "prefill" else _lengths(case)
        t = sum(lengths)
        # q, k and v in, the output and the appended rows out, the tables once.
        return {"bytes": PREFILL_LAYERS * (t * 2 * QH * D * 2 + 2 * t * row) + 2 * 2 * D * max(lengths),
                "flops": PREFILL_LAYERS * 4 * _causal_pairs(lengths) * QH * D}
    if kind == "attn_block":
        params = CFG.hidden * (CFG.qkv_width + QH * D)
        return {"bytes": LAYERS * (2 * params + b * row * (case["length"] + 1)) + 4 * b * CFG.hidden,
                "flops": LAYERS * b * (2 * params + 4 * (case["length"] + 1) * QH * D)}
    if kind == "mlp_block":
        params = 3 * CFG.hidden * CFG.intermediate
        return {"bytes": LAYERS * 2 * params + 4 * b * CFG.hidden + LAYERS * 2 * b * CFG.intermediate,
                "flops": LAYERS * b * 2 * params}
    lengths = _lengths(case) if kind == "model_prefill" else [1] * b
    t = sum(lengths)
    seen = _causal_pairs(lengths) if kind == "model_prefill" else b * (case["length"] + 1)
    cached = t if kind == "model_prefill" else seen
    head = CFG.vocab * CFG.hidden
    return {"bytes": 2 * (LAYERS * _linear_params() + head) + LAYERS * row * cached
            + 2 * b * CFG.vocab,
            "flops": LAYERS * (2 * t * _linear_params() + 4 * seen * QH * D) + 2 * b * head}


def tolerance(case):
    # fp16 operands and results, sums in fp32: about four times the distance
    # from the 64-bit result (2.5e-4, 4.4e-4, 1.5e-3 and 4.5e-3).
    kind = case["kind"]
    if kind in ("decode", "decode_paged"):
        return {"rel": 1.2e-3}
    if kind in ("prefill", "prefill_ragged"):
        return {"rel": 2e-3}
    if kind in ("attn_block", "mlp_block"):
        return {"rel": 6e-3}
    # The roundings of one layer travel through all that follow.
    return {"rel": 2e-2}


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------

def _attend64(q, k, v, causal=False):
    """q (..., n, D), k and v (..., m, D) in fp64; with ``causal`` n == m."""
    s = q @ k.transpose(-1, -2) * D ** -0.5
    if causal:
        n = s.shape[-1]
        s.masked_fill_(torch.ones(n, n, device=DEV, dtype=torch.bool).triu_(1), -math.inf)
    return torch.softmax(s, -1) @ v


def _causal64(q, k, v):
    """q (QH, n, D), k and v (KVH, n, D) in fp64, a head at a time."""
    return torch.stack([_attend64(q[h], k[h // G], v[h // G], causal=True) for h in range(QH)])


def _rotate64(x, cos, sin):
    half = torch.cat((-x[..., D // 2:], x[..., :D // 2]), -1)
    return x * cos + half * sin


def _tables64(pos):
    freq = CFG.rope_theta ** (-torch.arange(0, D, 2, device=DEV, dtype=torch.float64) / D)
    angle = pos.double().unsqueeze(-1) * freq
    angle = torch.cat((angle, angle), -1)
    return angle.cos(), angle.sin()


def _rms64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + CFG.rms_eps) * w.double()


def _mlp64(x, layer):
    gate, up = (_rms64(x, layer["post_norm"]) @ layer["gate_up_weight"].double().T).chunk(2, -1)
    h = gate * torch.sigmoid(gate) * up
    return h, x + h @ layer["down_weight"].double().T


def _qkv64(x, layer):
    proj = _rms64(x, layer["input_norm"]) @ layer["qkv_weight"].double().T + layer["qkv_bias"].double()
    return _split_heads(proj)


def _decode_attn64(x, layer, cache, n):
    """x (b, hidden); cache (2, b, KVH, cap, D) holds n rows -> (x, the new K and V rows)."""
    b = x.shape[0]
    q, k, v = _qkv64(x, layer)
    cos, sin = _tables64(torch.tensor([n], device=DEV))
    q, k = _rotate64(q, cos, sin), _rotate64(k, cos, sin)
    keys = torch.cat((cache[0, :, :, :n].double(), k.unsqueeze(2)), 2)
    values = torch.cat((cache[1, :, :, :n].double(), v.unsqueeze(2)), 2)
    att = _attend64(q.view(b, KVH, G, D), keys, values)
    return x + att.reshape(b, QH * D) @ layer["o_weight"].double().T, torch.stack((k, v))


def _exact_decode(case, seed):
    q, k, v, lengths, _ = _decode_inputs(case, seed)
    return torch.stack([torch.stack([_attend64(q[i, r].double(), k[i, r, :, :n].double(),
                                               v[i, r, :, :n].double())
                                     for r, n in enumerate(lengths)]) for i in range(LAYERS)])


def _exact_decode_paged(case, seed):
    q, k, v, table, lengths = _paged_inputs(case, seed)
    page = case["page"]

    def rows(pool, r, n):
        pages = table[r, :-(-n // page)].long()
        return pool[pages].transpose(0, 1).reshape(KVH, -1, D)[:, :n].double()

    return torch.stack([torch.stack([_attend64(q[i, r].double(), rows(k[i], r, n), rows(v[i], r, n))
                                     for r, n in enumerate(lengths)]) for i in range(LAYERS)])


def _exact_rows(proj, lengths, cap):
    """Packed (layers, T, width) projections -> (outputs per layer (T, QH, D), caches)."""
    outs, caches = [], torch.zeros(PREFILL_LAYERS, 2, len(lengths), KVH, cap, D, device=DEV,
                                   dtype=torch.float64)
    for i in range(PREFILL_LAYERS):
        at, out = 0, []
        for r, n in enumerate(lengths):
            q, k, v = (t.double().transpose(0, 1) for t in _split_heads(proj[i, at:at + n]))
            # The fp16 tables are inputs of the call.
            cos, sin = (t.double() for t in cos_sin(torch.arange(n, device=DEV),
                                                    inv_freq(D, CFG.rope_theta, DEV)))
            q, k = _rotate64(q, cos, sin), _rotate64(k, cos, sin)
            caches[i, 0, r, :, :n], caches[i, 1, r, :, :n] = k, v
            out.append(_causal64(q, k, v).transpose(0, 1))
            at += n
        outs.append(torch.cat(out))
    return outs, caches


def _exact_prefill(case, seed):
    b, s = case["batch"], case["seq"]
    proj = _proj_inputs(case, seed, b, s).reshape(PREFILL_LAYERS, b * s, -1)
    outs, caches = _exact_rows(proj, [s] * b, cache_capacity(s, 1))
    return {"out": [o.view(b, s, QH, D).transpose(1, 2) for o in outs], "caches": caches}


def _exact_prefill_ragged(case, seed):
    lengths = _lengths(case)
    proj = _proj_inputs(case, seed, 1, sum(lengths))[:, 0]
    outs, caches = _exact_rows(proj, lengths, cache_capacity(max(lengths), 1))
    return {"out": outs, "caches": caches}


def _exact_attn_block(case, seed):
    _, weights = _block_weights(case, seed)
    x, caches, n = _block_hidden(case, seed).double(), _block_caches(case, seed), case["length"]
    after, rows = caches.double(), []
    for i, layer in enumerate(weights["layers"]):
        x, new = _decode_attn64(x, layer, caches[i], n)
        rows.append(new)
        after[i, :, :, :, n] = new
    return {"hidden": x, "rows": torch.stack(rows), "caches": after}


def _exact_mlp_block(case, seed):
    _, weights = _block_weights(case, seed)
    x, hs = _block_hidden(case, seed).double(), []
    for layer in weights["layers"]:
        h, x = _mlp64(x, layer)
        hs.append(h)
    return {"hidden": x, "h": torch.stack(hs)}


def _head64(x, weights):
    x = _rms64(x, weights["final_norm"])
    return torch.cat([x @ part.double().T for part in weights["lm_head"].split(16384)], -1)


def _exact_model_decode(case, seed):
    weights, caches, n = _model_weights(case, seed), _block_caches(case, seed), case["length"]
    x = weights["embed"][_tokens(case, seed, case["batch"])].double()
    after, rows = caches.double(), []
    for i, layer in enumerate(weights["layers"]):
        x, new = _decode_attn64(x, layer, caches[i], n)
        _, x = _mlp64(x, layer)
        rows.append(new)
        after[i, :, :, :, n] = new
    return {"logits": _head64(x, weights), "rows": torch.stack(rows), "caches": after}


def _exact_model_prefill(case, seed):
    lengths, weights = _lengths(case), _model_weights(case, seed)
    ids = _tokens(case, seed, sum(lengths)).split(lengths)
    cap = cache_capacity(max(lengths), 128)
    caches = torch.zeros(LAYERS, 2, len(lengths), KVH, cap, D, device=DEV, dtype=torch.float64)
    logits = []
    for r, n in enumerate(lengths):
        x = weights["embed"][ids[r]].double()
        cos, sin = _tables64(torch.arange(n, device=DEV))
        for i, layer in enumerate(weights["layers"]):
            q, k, v = (t.transpose(0, 1) for t in _qkv64(x, layer))
            q, k = _rotate64(q, cos, sin), _rotate64(k, cos, sin)
            caches[i, 0, r, :, :n], caches[i, 1, r, :, :n] = k, v
            att = _causal64(q, k, v).transpose(0, 1).reshape(n, QH * D)
            _, x = _mlp64(x + att @ layer["o_weight"].double().T, layer)
        logits.append(_head64(x[-1], weights))
    return {"logits": torch.stack(logits), "caches": caches}


def exact(case, seed):
    with torch.no_grad():
        return globals()["_exact_" + case["kind"]](case, seed)
