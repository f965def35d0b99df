"""Decode-step kernels for 5..32 rows (include/qf_wide.h) against ``oracle.step``.

Batches sit at the edges of the kernels' tiles: the fewest rows, whole and
ragged blocks of four rows (rows per wave) and of 16 (matrix-core columns),
the most rows.  Integer operands make every sum exact in any order, so those
outputs match bit for bit; random ones agree to a few fp16 ulps (the bound of
the 1..4-row kernels' tests).
"""

import types

import pytest
import torch

import oracle.step as ost
from oracle.rope import inv_freq, rope_cos_sin
from qwenforge_amd import _lib, step_ops, wide_ops
from qwenforge_amd.engine import DecodeEngine
from qwenforge_amd.model import Qwen2Config, init_weights
from qwenforge_amd.paged_engine import PagedDecodeEngine

pytestmark = pytest.mark.gpu

HIDDEN, QH, KVH, D, INTER = 896, 14, 2, 64, 4864
EPS = 1e-6
STEP_TOL = 4e-3   # |got - ref| <= STEP_TOL * max(1, |ref|)
LOGIT_TOL = 3e-2  # the engine tests' bound
BATCHES = [5, 8, 13, 16, 17, 32]


def _close(got, ref):
    return (((got.float().cpu() - ref.float()).abs()) / ref.float().abs().clamp_min(1.0)).max().item()


def _int_rows(b, n, gen):
    return (torch.randint(0, 2, (b, n), generator=gen) * 2 - 1).half()


def _int_w(n, k, gen):
    return torch.randint(-1, 2, (n, k), generator=gen).half()


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("hidden", [HIDDEN, 96, 1024])
def test_qkv_rope_append_exact(dev, batch, hidden, paged):
    gen = torch.Generator().manual_seed(batch + hidden)
    x, nw = _int_rows(batch, hidden, gen), torch.ones(hidden, dtype=torch.float16)
    width = (QH + 2 * KVH) * D
    w, bias = _int_w(width, hidden, gen), torch.randint(-3, 4, (width,), generator=gen).half()
    pos = torch.randint(0, 40000, (batch,), generator=gen)
    cos, sin = rope_cos_sin(pos, inv_freq(D, 1e6))
    q, k, v = ost.qkv_rope16(x, nw, EPS, w, bias, cos, sin, QH, KVH, D)
    tiles = step_ops.pack_weight(w.to(dev), step_ops.PACK_ROPE)
    q_out = torch.zeros(batch, QH, D, device=dev, dtype=torch.float16)
    positions = (pos.to(dev), inv_freq(D, 1e6).to(dev))
    print(f"[wide qkv] B={batch} hidden={hidden} paged={paged}", flush=True)
    if paged:
        # One row's slot is past its pages and one page is unmapped: nothing is written there.
        kc = torch.zeros(2 * batch, KVH, 64, D, device=dev, dtype=torch.float16)
        vc = torch.zeros_like(kc)
        table = torch.randperm(2 * batch, generator=gen).to(torch.int32).view(batch, 2)
        slots = torch.randint(0, 128, (batch,), generator=gen)
        slots[0], slots[1] = 128, 5
        table[1, 0] = -1
        wide_ops.rms_qkv_rope_append_paged(x.to(dev), nw.to(dev), EPS, tiles, bias.to(dev), positions,
                                           kc, vc, table.to(dev), slots.to(dev), q_out)
        kr, vr = torch.zeros_like(kc, device="cpu"), torch.zeros_like(kc, device="cpu")
        for b in range(2, batch):
            page = int(table[b, int(slots[b]) // 64])
            kr[page, :, int(slots[b]) % 64], vr[page, :, int(slots[b]) % 64] = k[b], v[b]
    else:
        kc = torch.zeros(batch, KVH, 64, D, device=dev, dtype=torch.float16)
        vc = torch.zeros_like(kc)
        wide_ops.rms_qkv_rope_append(x.to(dev), nw.to(dev), EPS, tiles, bias.to(dev), positions,
                                     kc, vc, torch.tensor([37], device=dev), q_out)
        kr, vr = torch.zeros_like(kc, device="cpu"), torch.zeros_like(kc, device="cpu")
        kr[:, :, 37], vr[:, :, 37] = k, v
    assert torch.equal(q_out.cpu(), q)
    assert torch.equal(kc.cpu(), kr) and torch.equal(vc.cpu(), vr)


@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("k_dim,n", [(HIDDEN, HIDDEN), (INTER, HIDDEN), (32, 16), (1024, 48),
                                     (1056, 32), (8192, 64)])
def test_gemv_residual_exact_on_repeated_calls(dev, batch, k_dim, n):
    gen = torch.Generator().manual_seed(batch + k_dim)
    w = _int_w(n, k_dim, gen)
    tiles = step_ops.pack_weight(w.to(dev), step_ops.PACK_PLAIN)
    scratch = wide_ops.make_wide_scratch(batch, n, k_dim, dev)
    print(f"[wide gemv] B={batch} K={k_dim} N={n}", flush=True)
    for _ in range(3):  # the ticket re-arms
        inp = _int_rows(batch, k_dim, gen)
        res = torch.randint(-8, 9, (batch, n), generator=gen).half()
        hidden = res.to(dev)
        wide_ops.gemv_residual(inp.to(dev), tiles, hidden, scratch)
        assert torch.equal(hidden.cpu(), ost.residual16(res, inp, w))
    assert not bool(scratch[1].any())


@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("hidden,inter", [(HIDDEN, INTER), (64, 40)])
def test_gate_up_swiglu(dev, batch, hidden, inter):
    gen = torch.Generator().manual_seed(batch)
    x = torch.randn(batch, hidden, generator=gen).half()
    nw = (torch.rand(hidden, generator=gen) + 0.5).half()
    w = (torch.randn(2 * inter, hidden, generator=gen) * 0.02).half()
    h = torch.zeros(batch, inter, device=dev, dtype=torch.float16)
    print(f"[wide gate_up] B={batch} {hidden}x{inter}", flush=True)
    wide_ops.rms_gate_up_swiglu(x.to(dev), nw.to(dev), EPS,
                                step_ops.pack_weight(w.to(dev), step_ops.PACK_SWIGLU), h)
    assert _close(h, ost.swiglu16(x, nw, EPS, w)) <= STEP_TOL


@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("blocks", [1, 96, 512])
def test_lm_head_and_argmax_step_exact(dev, batch, blocks):
    """Integer logits, a planted tie (first index wins) and a row of NaNs
    (torch.argmax names the first)."""
    gen = torch.Generator().manual_seed(batch)
    vocab = 5008
    x, nw = _int_rows(batch, HIDDEN, gen), torch.ones(HIDDEN, dtype=torch.float16)
    w = _int_w(vocab, HIDDEN, gen)
    w[1234] = torch.sign(x[0].float()).half()
    w[4000] = w[1234]
    x[1, 5] = float("nan")
    logits = torch.zeros(batch, vocab, device=dev, dtype=torch.float16)
    keys = torch.zeros(batch, blocks, device=dev, dtype=torch.long)
    print(f"[wide lm_head] B={batch} blocks={blocks}", flush=True)
    wide_ops.rms_lm_head(x.to(dev), nw.to(dev), EPS, step_ops.pack_weight(w.to(dev)), logits, keys)
    token, rows = torch.full((batch,), -1, device=dev), torch.zeros(batch, 5, device=dev).long()
    step, write = torch.tensor([2], device=dev), torch.tensor([40], device=dev)
    pos = torch.arange(batch, device=dev) + 10
    wide_ops.argmax_step(keys, token, rows, step, write, pos)
    ref, first = ost.lm_head_argmax(x, nw, EPS, w)
    keep = [b for b in range(batch) if b != 1]
    assert torch.equal(logits.cpu()[keep], ref[keep]) and bool(logits[1].isnan().all())
    first[1] = 0
    assert int(first[0]) == 1234 and torch.equal(token.cpu(), first)
    assert torch.equal(rows.cpu()[:, 2], first) and not bool(rows[:, [0, 1, 3, 4]].any())
    assert int(step) == 3 and int(write) == 41 and torch.equal(pos.cpu(), torch.arange(batch) + 11)


@pytest.mark.parametrize("batch,paged", [(5, False), (16, True), (17, False), (32, True)])
def test_wide_step_matches_torch_step(dev, batch, paged):
    """Teacher-forced logits, appended rows and bookkeeping of the captured
    wide step equal the torch-projection step's within the engine's bound."""
    cfg = Qwen2Config(layers=3)
    w = init_weights(cfg, dev, seed=3)
    s, steps = 70, 3
    gen = torch.Generator().manual_seed(5)
    ids = torch.randint(0, cfg.vocab, (batch, s), generator=gen).to(dev)
    teacher = torch.randint(0, cfg.vocab, (steps, batch), generator=gen).to(dev)
    out = {}
    for wide in (True, False):
        eng = (PagedDecodeEngine if paged else DecodeEngine)(cfg, w, dev, tile_weights=wide)
        if paged:
            kv = eng.new_paged_cache(batch, 2 * batch, 64, 2)
            for r in range(batch):
                kv.map_row(r, 128)
            eng.prefill_paged(list(ids), kv, range(batch))
            ctx = eng.make_paged_context(kv, batch, steps + 1)
            eng.capture_paged(ctx)
        else:
            caches = eng.new_caches(batch, 128)
            eng.prefill(ids, caches)
            ctx = eng.make_context(caches, batch, steps + 1)
            eng.capture(ctx)
            ctx["write"].fill_(s)
        assert ctx["wide"] == wide
        ctx["pos"].fill_(s)
        ctx["step"].fill_(1)
        logits = []
        for t in range(steps):
            ctx["token"].copy_(teacher[t])
            ctx["graph"].replay()
            logits.append(ctx["logits"].float().cpu())
        rows = ([kv.gather(i, r, s + steps)[0] for i in range(3) for r in range(batch)] if paged
                else [k[:, :, s:s + steps] for k, _ in caches])
        out[wide] = (torch.stack(logits), ctx["pos"].cpu(), int(ctx["step"]),
                     torch.stack([r.float().cpu() for r in rows]))
    (lw, pw, sw, cw), (lt, pt, st, ct) = out[True], out[False]
    print(f"[wide vs torch step B={batch}] max|dlogit| {(lw - lt).abs().max():.3e}", flush=True)
    assert (lw - lt).abs().max().item() <= LOGIT_TOL
    assert torch.equal(pw, pt) and sw == st and (cw - ct).abs().max().item() <= 2e-2


@pytest.mark.parametrize("batch", [3, 5, 16])
def test_decode_follows_weights_changed_in_place(dev, batch):
    """Other weights copied over an engine's: generate gives a fresh engine's
    tokens on a reused graph (dense) and a new one (paged), as the torch
    projections did at 5..32 rows; 3 rows, and a context of the caller's own
    between replays, after ``repack_weights``."""
    cfg = Qwen2Config(layers=2, vocab=4096)
    gen = torch.Generator().manual_seed(batch)
    ids = torch.randint(0, cfg.vocab, (batch, 20), generator=gen).to(dev)
    other = init_weights(cfg, dev, seed=22)

    def overwrite(w, source):
        for to, frm in zip([w] + w["layers"], [source] + source["layers"]):
            for name, t in to.items():
                if isinstance(t, torch.Tensor):
                    t.data.copy_(frm[name])

    print(f"[repack] B={batch}", flush=True)
    for paged in (False, True):
        def run(engine):
            return engine.generate_paged(list(ids), 12) if paged else engine.generate(ids, 12)

        kind = PagedDecodeEngine if paged else DecodeEngine
        eng = kind(cfg, init_weights(cfg, dev, seed=21), dev)
        first, want = run(eng), run(kind(cfg, other, dev))
        assert not torch.equal(first, want)
        overwrite(eng.w, other)
        if batch < wide_ops.MIN_BATCH:
            eng.repack_weights()
        assert torch.equal(run(eng), want)
        assert paged or eng.captures == 1
    ctx = eng._ctx
    logits = []
    for change in (False, True):
        if change:  # the layers alone: the embedding is read where it lies
            back = init_weights(cfg, dev, seed=21)
            for to, frm in zip(eng.w["layers"], back["layers"]):
                for name in ("qkv_weight", "o_weight", "gate_up_weight", "down_weight"):
                    to[name].copy_(frm[name])
            eng.repack_weights()
        ctx["pos"].fill_(20)
        ctx["step"].fill_(1)
        ctx["token"].fill_(7)
        ctx["graph"].replay()
        logits.append(ctx["logits"].clone())
    assert not torch.equal(*logits)


def test_every_launch_runs_with_its_operands_device_current(dev, monkeypatch):
    """An engine on another device than the current one: each call of the wide
    step and of the packing enters its operands' device first (the null stream
    a launch names is the current device's)."""
    inside, calls = [], []

    class Guard(torch.cuda.device):
        def __enter__(self):
            inside.append(self.idx)
            return super().__enter__()

        def __exit__(self, *exc):
            inside.pop()
            return super().__exit__(*exc)

    class Lib(types.SimpleNamespace):
        def __getattr__(self, name):
            def call(*args):
                if name != "qf_wide_splits":
                    calls.append((name, list(inside)))
                return int(name == "qf_wide_splits")
            return call

    f16 = dict(device=dev, dtype=torch.float16)
    x, nw, q = torch.zeros(5, 64, **f16), torch.zeros(64, **f16), torch.zeros(5, 1, 64, **f16)
    pos, inv = torch.zeros(5, device=dev).long(), torch.zeros(32, device=dev)
    cache, pool = torch.zeros(5, 1, 8, 64, **f16), torch.zeros(5, 1, 64, 64, **f16)
    table = torch.zeros(5, 1, device=dev, dtype=torch.int32)
    keys, rows = torch.zeros(5, 2, device=dev).long(), torch.zeros(5, 2, device=dev).long()
    scratch = wide_ops.make_wide_scratch(5, 64, 64, dev)
    monkeypatch.setattr(_lib, "load", Lib)
    monkeypatch.setattr(torch.cuda, "device", Guard)
    w_qkv, w, w_gu = (step_ops.pack_weight(torch.zeros(n, 64, **f16), layout) for n, layout in (
        (192, step_ops.PACK_ROPE), (64, step_ops.PACK_PLAIN), (128, step_ops.PACK_SWIGLU)))
    wide_ops.rms_qkv_rope_append(x, nw, EPS, w_qkv, None, (pos, inv), cache, cache, pos[:1], q)
    wide_ops.rms_qkv_rope_append_paged(x, nw, EPS, w_qkv, None, (pos, inv), pool, pool, table, pos, q)
    wide_ops.gemv_residual(x, w, x, scratch)
    wide_ops.rms_gate_up_swiglu(x, nw, EPS, w_gu, x)
    wide_ops.rms_lm_head(x, nw, EPS, w, x, keys)
    wide_ops.argmax_step(keys, pos, rows, pos[:1], None, pos)
    assert len(calls) == 9 and all(where == [x.device.index] for _, where in calls), calls


@pytest.mark.parametrize("hidden", [64, 96, 160, HIDDEN])
@pytest.mark.parametrize("batch", [3, 5, 20])
def test_infinite_weights_stay_infinities(dev, batch, hidden):
    """One infinite weight in every k block in turn (k blocks past a wave's
    share re-read such a tile): its output row is an infinity of the row's
    sign, as in torch, and the others are untouched."""
    x = torch.ones(batch, hidden, dtype=torch.float16)
    x[1] = -1
    x, nw = x.to(dev), torch.ones(hidden, **dict(device=dev, dtype=torch.float16))
    pos, inv = torch.zeros(batch, device=dev).long(), inv_freq(D, 1e6).to(dev)
    print(f"[wide inf] B={batch} hidden={hidden}", flush=True)
    want = torch.full((batch,), float("inf"), device=dev, dtype=torch.float16)
    want[1] = -want[1]
    for kb in range(hidden // 32):
        w = torch.zeros(256, hidden, device=dev, dtype=torch.float16)
        w[128 + 32 * (kb % 2), 32 * kb + 5] = float("inf")  # a V row (kv head 0: rows 128..191)
        if batch >= wide_ops.MIN_BATCH:
            logits = torch.zeros(batch, 256, device=dev, dtype=torch.float16)
            wide_ops.rms_lm_head(x, nw, EPS, step_ops.pack_weight(w), logits,
                                 torch.zeros(batch, 3, device=dev).long())
            assert torch.equal(logits[:, 128 + 32 * (kb % 2)], want), kb
            assert int((logits != 0).sum()) == batch
        qkv = w[:192].contiguous()
        kc, vc = (torch.zeros(batch, 1, 4, D, device=dev, dtype=torch.float16) for _ in range(2))
        q = torch.zeros(batch, 1, D, device=dev, dtype=torch.float16)
        tiles = step_ops.pack_weight(qkv, step_ops.PACK_ROPE)
        if batch >= wide_ops.MIN_BATCH:
            wide_ops.rms_qkv_rope_append(x, nw, EPS, tiles, None, (pos, inv), kc, vc, pos[:1], q)
        else:
            step_ops.rms_qkv_rope_append(x, nw, EPS, tiles, None, None, None, kc, vc, pos[:1], q,
                                         positions=(pos, inv))
        assert torch.equal(vc[:, 0, 0, 32 * (kb % 2)], want), kb
        assert int((vc != 0).sum()) == batch and not bool(q.any()) and not bool(kc.any())
        # Gate rows 1 and 0 infinite against up rows of ones: silu(inf) * 1.
        gu = torch.zeros(32, hidden, device=dev, dtype=torch.float16)
        gu[3, 32 * kb + 5], gu[16 + 3] = float("inf"), 1 / hidden
        h = torch.zeros(batch, 16, device=dev, dtype=torch.float16)
        packed = step_ops.pack_weight(gu, step_ops.PACK_SWIGLU)
        (wide_ops if batch >= wide_ops.MIN_BATCH else step_ops).rms_gate_up_swiglu(x, nw, EPS, packed, h)
        assert bool(torch.isposinf(h[[0, 2], 3]).all()) and not bool(h[:, :3].any()), kb
