"""The single-launch merge with its workgroups shared out by the rows' lengths.

Rows with bounds of their own (``kv_last`` per row, no bias) at 2..64 rows, up
to 8 splits and at least 192 slots of capacity per split: equal rows, one long
row among empty ones (its share capped), rows of one slot, shares that leave
workgroups over, and both sides of each condition.  Against fp64 attention on
the valid slots (2e-3, the bound of the other decode tests), with NaN in every
slot past a row's end; repeated calls re-arm the tickets and replays of a graph
follow bounds that move.  Paged caches give the dense call's bits.
"""

import pytest
import torch

from qwenforge_amd import ops, paged

pytestmark = pytest.mark.gpu
TOL = 2e-3
KVH, D = 2, 64


def _case(dev, lengths, cap, g, seed):
    gen = torch.Generator(dev).manual_seed(seed)
    b = len(lengths)
    q, k, v = (torch.randn(*s, generator=gen, device=dev).half()
               for s in ((b, KVH, g, D), (b, KVH, cap, D), (b, KVH, cap, D)))
    for r, n in enumerate(lengths):
        k[r, :, n:] = float("nan")
        v[r, :, n:] = float("nan")
    return q, k, v, torch.tensor(lengths, device=dev) - 1


def _check(out, q, k, v, lengths):
    for r, n in enumerate(lengths):
        if n == 0:
            continue  # no key: the output is unspecified
        s = q[r].double() @ k[r, :, :n].double().transpose(-1, -2) * D ** -0.5
        ref = torch.softmax(s, -1) @ v[r, :, :n].double()
        assert (out[r].double() - ref).abs().max().item() <= TOL, r


@pytest.mark.parametrize("lengths,cap,splits,g", [
    ((2000, 2000), 2000, 8, 7),                # equal rows: S each
    ((1, 1999), 2048, 8, 7),
    ((0, 0, 1536, 0), 1536, 8, 7),             # one row: the cap on its share
    ((0, 0, 0), 1536, 8, 7),                   # nothing at all
    ((31, 32, 33, 1536, 700), 1536, 8, 16),
    ((640, 5, 77), 640, 3, 1),
    ((400, 384), 400, 2, 4),
    (tuple(range(1, 1537, 24)), 1536, 8, 7),   # 64 rows
    (tuple(range(1, 1537, 24))[:63] + (9, 9), 1536, 8, 7),  # 65: even splits
    ((1535, 3), 1535, 8, 7),                   # under six tiles per split: even splits
    ((2000, 100), 2000, 9, 7),                 # nine splits: even splits
])
def test_rows_share_workgroups(dev, lengths, cap, splits, g):
    q, k, v, last = _case(dev, lengths, cap, g, len(lengths) + cap)
    flash = ops.make_flash_scratch(len(lengths), KVH, g, cap, dev, splits=splits, fused=True)
    print(f"[decode rows] {len(lengths)} rows cap={cap} splits={splits} G={g}", flush=True)
    first = ops.flash_decode_attention(q, k, v, None, flash, kv_last=last).clone()
    _check(first, q, k, v, lengths)
    again = ops.flash_decode_attention(q, k, v, None, flash, kv_last=last)
    valid = [r for r, n in enumerate(lengths) if n]
    assert torch.equal(first[valid], again[valid])
    assert not bool(flash[4].any())
    if cap % 64 == 0:
        pages = cap // 64
        order = torch.randperm(len(lengths) * pages, device=dev).view(len(lengths), pages)
        pool_k, pool_v = (torch.empty(order.numel(), KVH, 64, D, device=dev, dtype=torch.float16)
                          for _ in range(2))
        for t, pool in ((k, pool_k), (v, pool_v)):
            pool[order] = t.view(len(lengths), KVH, pages, 64, D).transpose(1, 2)
        out = paged.flash_decode_attention_paged(q, pool_k, pool_v, order.to(torch.int32), None,
                                                 flash, kv_last=last)
        assert torch.equal(out[valid], first[valid])


def test_graph_replays_follow_moving_bounds(dev):
    lengths = [1, 900, 1600, 40, 1599]
    q, k, v, last = _case(dev, [1600] * 5, 1600, 7, 3)
    flash = ops.make_flash_scratch(5, KVH, 7, 1600, dev, splits=8, fused=True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ops.flash_decode_attention(q, k, v, None, flash, kv_last=last)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        ops.flash_decode_attention(q, k, v, None, flash, kv_last=last)
    for shift in range(4):
        rows = lengths[shift:] + lengths[:shift]
        last.copy_(torch.tensor(rows, device=dev) - 1)
        graph.replay()
        _check(flash[3], q, k, v, rows)
        torch.cuda.synchronize()


def test_even_splits_on_request(dev):
    """``share_rows=False``: the reference's partials per row (the combine
    launch merges them to the same output) and no trace of the other rows."""
    lengths, cap = [1, 900, 1600, 40, 1599], 1600
    q, k, v, last = _case(dev, lengths, cap, 7, 3)
    flash = ops.make_flash_scratch(5, KVH, 7, cap, dev, splits=8, fused=True)
    print("[decode rows] even", flush=True)
    first = ops.flash_decode_attention(q, k, v, None, flash, kv_last=last, share_rows=False).clone()
    _check(first, q, k, v, lengths)
    merged = ops.flash_decode_combine(flash[:4])
    assert (merged.float() - first.float()).abs().max().item() <= TOL
    for others in (0, 300, 1599):
        moved = torch.full_like(last, others)
        moved[1] = last[1]
        out = ops.flash_decode_attention(q, k, v, None, flash, kv_last=moved, share_rows=False)
        assert torch.equal(out[1], first[1])
