"""The native prompt pass (include/qf_prefill.h) against the torch projections
around the same attention (``DecodeEngine`` with the native call switched off,
itself pinned to the CPU oracle by the engine tests).

Token counts sit at the edges of the kernels' tiles (64 and 128 tokens) and on
both sides of the split of the down projection's k; one row, equal rows, packed
rows (an empty one among them) and paged caches.  Single layers of other
shapes, on integers, match bit for bit.  Tolerance: both passes are
within 2e-2 of the fp32 caches and 3e-2 of the fp32 logits in the engine
tests, so they are within the sum of the two of each other; the shallow model
here stays far inside (fp16 roundings of two layers).
"""

import numpy as np
import pytest
import torch

import oracle
from qwenforge_amd import prefill_ops
from qwenforge_amd.engine import DecodeEngine
from qwenforge_amd.model import Qwen2Config, init_weights
from qwenforge_amd.paged_engine import PagedDecodeEngine
from qwenforge_amd.rope import cos_sin

pytestmark = pytest.mark.gpu

TOL = 2e-2
CFG = Qwen2Config(layers=2, vocab=4096)


@pytest.fixture(scope="module")
def weights(dev):
    w = init_weights(CFG, dev, seed=4)
    gen = torch.Generator(dev).manual_seed(1)
    for layer in w["layers"]:
        layer["qkv_bias"] = torch.randn(CFG.qkv_width, generator=gen, device=dev).half() * 0.1
        layer["input_norm"] = (torch.rand(CFG.hidden, generator=gen, device=dev) + 0.5).half()
    return w


def _torch_only(engine):
    engine._native_layers = lambda *a, **k: False
    return engine


def _native_only(engine):
    inner = engine._native_layers

    def run(*a, **k):
        assert inner(*a, **k)
        return True

    engine._native_layers = run
    return engine


@pytest.mark.parametrize("lengths", [
    (1,), (63,), (64,), (65,), (127,), (128,), (129,), (300,), (1025,), (2048,), (2113,),
    (512,), (513,), (577,), (1281,), (2305,), (3585,), (4608,), (4609,),
    (5, 5, 5), (128, 128), (700, 700, 700),
    (3, 70, 1, 64), (257, 31, 900), (0, 40, 0, 65, 0),
])
def test_prefill_matches_torch_projections(dev, weights, lengths):
    gen = torch.Generator().manual_seed(sum(lengths))
    prompts = [torch.randint(0, CFG.vocab, (n,), generator=gen).to(dev) for n in lengths]
    print(f"[prefill layers] {lengths}", flush=True)
    out = []
    for make in (_native_only, _torch_only):
        eng = make(DecodeEngine(CFG, weights, dev))
        caches = eng.new_caches(len(lengths), max(lengths) + 7)
        if len(set(lengths)) == 1:
            logits = eng.prefill(torch.stack(prompts), caches)
        else:
            logits = eng.prefill_ragged(prompts, caches)
        out.append((logits.float(), [t.float() for kv in caches for t in kv]))
    (ln, cn), (lt, ct) = out
    rows = [i for i, n in enumerate(lengths) if n]  # an empty row has no last token
    assert (ln - lt)[rows].abs().max().item() <= TOL
    for a, b in zip(cn, ct):
        assert (a - b).abs().max().item() <= TOL
        for r, n in enumerate(lengths):
            assert not bool(a[r, :, n:].any())


@pytest.mark.parametrize("lengths,page", [((65,), 64), ((130, 1, 257), 128)])
def test_prefill_paged_matches_torch_projections(dev, weights, lengths, page):
    gen = torch.Generator().manual_seed(sum(lengths))
    prompts = [torch.randint(0, CFG.vocab, (n,), generator=gen).to(dev) for n in lengths]
    out = []
    for make in (_native_only, _torch_only):
        eng = make(PagedDecodeEngine(CFG, weights, dev))
        kv = eng.new_paged_cache(len(lengths) + 1, 16, page, 5)
        written = torch.zeros(16, page, device=dev, dtype=torch.bool)
        for r, n in enumerate(lengths):
            for j, p in enumerate(kv.map_row(len(lengths) - r, n)):
                written[p, :n - j * page] = True
        logits = eng.prefill_paged(prompts, kv, [len(lengths) - r for r in range(len(lengths))])
        out.append((logits.float(), [t.float() for pair in kv.pools for t in pair]))
    (ln, cn), (lt, ct) = out
    assert (ln - lt).abs().max().item() <= TOL
    for a, b in zip(cn, ct):
        assert (a - b).abs().max().item() <= TOL
        assert torch.equal((a != 0).any(-1), written[:, None].expand(-1, CFG.kv_heads, -1))


def test_graph_replays_equal_eager(dev, weights):
    """Captured with the split down projection, replayed on changed inputs:
    the result is the eager one's bits."""
    eng = DecodeEngine(CFG, weights, dev)
    caches = eng.new_caches(1, 64)
    embed = weights["embed"]
    first, other = embed[:40].clone(), embed[100:140].clone()
    hidden = first.clone()
    table = prefill_ops.layer_table(CFG, weights["layers"], caches, dev, (1, 2, 40, 64))

    def run():
        prefill_ops.prefill_layers(CFG, table, hidden, 1, 40, eng.inv_freq)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        run()
    for source in (first, other, first, other):
        hidden.copy_(source)
        graph.replay()
        got = hidden.clone()
        hidden.copy_(source)
        run()
        assert torch.equal(got, hidden)
        torch.cuda.synchronize()


def test_layouts_it_does_not_take(dev, weights):
    """Other layouts name no table (the engine then runs the torch projections)."""
    eng = DecodeEngine(CFG, weights, dev)
    caches = eng.new_caches(2, 64)
    shape = (2, 2, 64, 64)
    assert prefill_ops.layer_table(CFG, weights["layers"], caches, dev, shape) is not None
    assert prefill_ops.layer_table(CFG, weights["layers"], caches, dev, (2, 2, 65, 64)) is None
    layers = [dict(l) for l in weights["layers"]]
    layers[1]["o_weight"] = layers[1]["o_weight"].t().contiguous().t()
    assert prefill_ops.layer_table(CFG, layers, caches, dev, shape) is None
    layers[1]["o_weight"] = weights["layers"][1]["o_weight"].float()
    assert prefill_ops.layer_table(CFG, layers, caches, dev, shape) is None
    assert prefill_ops.workspace_bytes(Qwen2Config(hidden=960, heads=15, kv_heads=3), 8) < 0


def test_swiglu_rounds_every_gate_correctly(dev):
    """A layer whose h is silu(v) of chosen fp16 values: token t holds one
    number, 2^10 at place t, which the norm turns into 32 exactly; gate weights
    v / 32 and up weights 1 / 32 in that column, the down projection picks h
    out.  Every fp16 v from 2^-8 to the largest, both signs, against silu in
    fp64 rounded once (which F.silu gives for all of them)."""
    cfg = Qwen2Config(hidden=1024, heads=16, kv_heads=2, intermediate=1024, layers=1, vocab=64)
    tokens, n = 64, 1024
    bits = torch.arange(0x1C00, 0x7C00, dtype=torch.int32).to(torch.int16).view(torch.float16)
    v = torch.cat([bits, -bits])
    v = torch.cat([v, v[:tokens * (n - tokens) - v.numel()]]).view(tokens, n - tokens).to(dev)
    gate_up = torch.zeros(2 * n, n, device=dev, dtype=torch.float16)
    gate_up[tokens:n, :tokens] = (v / 32).t()
    assert torch.equal(gate_up[tokens:n, :tokens].t() * 32, v)
    gate_up[n:, :tokens] = 1 / 32
    zeros = lambda *s: torch.zeros(*s, device=dev, dtype=torch.float16)  # noqa: E731
    layer = {"input_norm": zeros(n) + 1, "post_norm": zeros(n) + 1, "qkv_bias": None,
             "qkv_weight": zeros(cfg.qkv_width, n), "o_weight": zeros(n, n),
             "gate_up_weight": gate_up, "down_weight": torch.eye(n, device=dev).half()}
    caches = [(zeros(1, 2, 64, 64), zeros(1, 2, 64, 64))]
    hidden = zeros(tokens, n)
    hidden[:, :tokens].fill_diagonal_(1024.0)
    table = prefill_ops.layer_table(cfg, [layer], caches, dev, (1, 2, tokens, 64))
    inv = torch.zeros(32, device=dev)
    prefill_ops.prefill_layers(cfg, table, hidden, 1, tokens, inv)
    # numpy rounds fp64 to fp16 once (torch by way of fp32).
    exact = v.double().cpu().numpy()
    with np.errstate(over="ignore"):  # exp(65504): silu is -0 there
        want = torch.from_numpy((exact / (1 + np.exp(-exact))).astype(np.float16)).to(dev)
    got = hidden[:, tokens:]
    print(f"[prefill silu] {int((got != want).sum())} of {want.numel()} differ", flush=True)
    assert torch.equal(torch.nn.functional.silu(v), want)
    assert torch.equal(got, want)


def _ints(gen, *shape, low=-1, high=2):
    return torch.randint(low, high, shape, generator=gen, device=gen.device).float()


def _run_layer(cfg, layer, x, rows, caches):
    table = prefill_ops.layer_table(cfg, [layer], caches, x.device, (rows, cfg.kv_heads, 1, 64))
    hidden = x.half()
    tokens = x.shape[0] // rows
    inv = oracle.inv_freq(64, cfg.rope_theta).to(x.device)
    prefill_ops.prefill_layers(cfg, table, hidden, rows, tokens, inv)
    return hidden


# hidden, heads, kv heads, intermediate, tokens: RMSNorm rows of one to four chunks a
# lane; feature counts that leave tails in the 64-, 128- and 160-wide tiles; token counts
# at tile edges and on both sides of each tile form's and k split's line at that shape.
LAYER_SHAPES = (
    [(128, 2, 1, 128, t) for t in (1, 63, 65, 129, 4100)]
    + [(128, 2, 2, 384, t) for t in (64, 200)]
    + [(640, 10, 1, 256, t) for t in (5, 128, 1000, 3000)]
    + [(1024, 16, 4, 1152, t) for t in (1, 300, 513, 1300, 2700, 3700)]
    + [(2048, 32, 2, 2176, t) for t in (2, 65, 250, 260, 700, 1500, 1700)]
    + [(896, 14, 2, 4864, t) for t in (1, 64, 129, 577, 900, 2305, 4609)])


@pytest.mark.parametrize("hidden,heads,kv,inter,tokens", LAYER_SHAPES)
def test_layer_exact_on_integers(dev, hidden, heads, kv, inter, tokens):
    """Every projection bit for bit: integer operands make the fp32 sums exact
    in any order, so one wrong tile edge or lost k share shows.  One row of all
    tokens: QKV (with RoPE and append), gate/up and down (w_o = 0, so the
    normalised rows stay +-1); a row per token: its attention is its own V, so
    o_proj is exact too (no MLP)."""
    cfg = Qwen2Config(hidden=hidden, heads=heads, kv_heads=kv, intermediate=inter, layers=1, vocab=64)
    gen = torch.Generator(dev).manual_seed(hidden + tokens)
    print(f"[prefill layer] {hidden} {heads}/{kv} {inter} T={tokens}", flush=True)
    x = _ints(gen, tokens, hidden, high=1) * 2 + 1           # +-1
    x[:, 0] = 1
    norms = [_ints(gen, hidden, low=1, high=3) for _ in range(2)]
    norms[1][0] = 1
    w_qkv, b_qkv = _ints(gen, cfg.qkv_width, hidden), _ints(gen, cfg.qkv_width, low=-3, high=4)
    w_o = _ints(gen, hidden, hidden)
    gate_up = torch.zeros(2 * inter, hidden, device=dev)
    places = torch.randint(1, hidden, (2 * inter, 8), generator=gen, device=dev)
    gate_up.scatter_(1, places, _ints(gen, 2 * inter, 8))
    gate_up[:inter, 0] = 64                                  # gates of 48..80: silu(g) = g
    w_down = _ints(gen, hidden, inter)
    half = {"input_norm": norms[0], "post_norm": norms[1], "qkv_weight": w_qkv, "qkv_bias": b_qkv,
            "o_weight": w_o, "gate_up_weight": gate_up, "down_weight": w_down}
    layer = {k: t.half().contiguous() for k, t in half.items()}
    zeros = lambda *s: torch.zeros(*s, device=dev, dtype=torch.float16)  # noqa: E731

    kc, vc = zeros(1, kv, tokens + 3, 64), zeros(1, kv, tokens + 3, 64)
    got = _run_layer(cfg, layer | {"o_weight": zeros(hidden, hidden)}, x, 1, [(kc, vc)])
    qkv = ((x * norms[0]) @ w_qkv.T + b_qkv).half()
    _, k, v = qkv.split((hidden, kv * 64, kv * 64), -1)
    # The table as torch gives it on this device (the host's cosf rounds ten of half a
    # million values otherwise).
    cos, sin = (t.cpu() for t in cos_sin(torch.arange(tokens, device=dev),
                                         oracle.inv_freq(64, cfg.rope_theta).to(dev)))
    k = oracle.apply_rope_fp16(k.view(tokens, kv, 64).cpu(), cos[:, None], sin[:, None]).to(dev)
    assert torch.equal(kc[0, :, :tokens].transpose(0, 1), k)
    assert torch.equal(vc[0, :, :tokens].transpose(0, 1), v.view(tokens, kv, 64))
    assert not bool(kc[:, :, tokens:].any()) and not bool(vc[:, :, tokens:].any())
    gate, up = ((x * norms[1]) @ gate_up.T).chunk(2, -1)
    down = ((gate * up) @ w_down.T).half()
    assert torch.equal(got, (x + down.float()).half())

    # No bias, no MLP, a row per token.
    kc, vc = zeros(tokens, kv, 1, 64), zeros(tokens, kv, 1, 64)
    plain = layer | {"qkv_bias": None, "gate_up_weight": zeros(2 * inter, hidden)}
    got = _run_layer(cfg, plain, x, tokens, [(kc, vc)])
    v = ((x * norms[0]) @ w_qkv[hidden + kv * 64:].T).half()
    assert torch.equal(vc.view(tokens, -1), v)
    att = v.view(tokens, kv, 1, 64).expand(-1, -1, cfg.groups, -1).reshape(tokens, hidden)
    assert torch.equal(got, (x + (att.float() @ w_o.T).half().float()).half())


def test_appends_stay_within_the_rows(dev, weights):
    """A cache that holds fewer rows, slots or pages than the call fills is
    refused before any launch; a packed row longer than the longest announced
    appends no further than that (slots past it exist here)."""
    eng = DecodeEngine(CFG, weights, dev)
    caches, pools = eng.new_caches(2, 40), [(torch.zeros(4, 2, 64, 64, device=dev).half(),) * 2] * 2
    hidden = weights["embed"][:40].clone()
    table = prefill_ops.layer_table(CFG, weights["layers"], caches, dev, (2, 2, 1, 64))
    paged = prefill_ops.layer_table(CFG, weights["layers"], pools, dev, (4, 2, 64, 64))
    block_table = torch.zeros(1, 1, device=dev, dtype=torch.int32)
    for args, kw in (((table, hidden, 1, 40), {}),                       # two rows, not one
                     ((table, hidden.repeat(3, 1), 2, 60), {}),          # 40 slots
                     ((paged, hidden.repeat(2, 1), 1, 80),               # one page of 64
                      dict(block_table=block_table, n_pages=4, page_size=64)),
                     ((paged, hidden, 1, 40),                            # five pages
                      dict(block_table=block_table, n_pages=5, page_size=64))):
        with pytest.raises(ValueError):
            prefill_ops.prefill_layers(CFG, *args, eng.inv_freq, **kw)
    cu = torch.tensor([0, 10, 40], device=dev, dtype=torch.int32)
    print("[prefill layers] rows of 10 and 30 announced as 20", flush=True)
    prefill_ops.prefill_layers(CFG, table, hidden, 2, 20, eng.inv_freq, cu=cu)
    for t in (t for pair in caches for t in pair):
        used = (t != 0).any(-1).any(1)
        assert used.sum(1).tolist() == [10, 20] and not bool(used[1, 20:].any())
