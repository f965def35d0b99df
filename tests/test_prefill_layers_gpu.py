"""The native prompt pass (include/qf_prefill.h) against the torch projections
around the same attention (``DecodeEngine`` with the native call switched off,
itself pinned to the CPU oracle by the engine tests).

Token counts sit at the edges of the kernels' tiles (64 and 128 tokens) and on
both sides of the split of the down projection's k; one row, equal rows, packed
rows (an empty one among them) and paged caches.  Tolerance: both passes are
within 2e-2 of the fp32 caches and 3e-2 of the fp32 logits in the engine
tests, so they are within the sum of the two of each other; the shallow model
here stays far inside (fp16 roundings of two layers).
"""

import numpy as np
import pytest
import torch

from qwenforge_amd import prefill_ops
from qwenforge_amd.engine import DecodeEngine
from qwenforge_amd.model import Qwen2Config, init_weights
from qwenforge_amd.paged_engine import PagedDecodeEngine

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
        for r, n in enumerate(lengths):
            kv.map_row(len(lengths) - r, n)
        logits = eng.prefill_paged(prompts, kv, [len(lengths) - r for r in range(len(lengths))])
        out.append((logits.float(), [t.float() for pair in kv.pools for t in pair]))
    (ln, cn), (lt, ct) = out
    assert (ln - lt).abs().max().item() <= TOL
    for a, b in zip(cn, ct):
        assert (a - b).abs().max().item() <= TOL
        assert torch.equal(a == 0, b == 0) or ((a == 0) != (b == 0)).float().mean().item() < 1e-3


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
    want = torch.from_numpy((exact / (1 + np.exp(-exact))).astype(np.float16)).to(dev)
    got = hidden[:, tokens:]
    print(f"[prefill silu] {int((got != want).sum())} of {want.numel()} differ", flush=True)
    assert torch.equal(torch.nn.functional.silu(v), want)
    assert torch.equal(got, want)
