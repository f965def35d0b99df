"""The streaming prefill with one wave group per query tile.

The launch takes one group instead of two once the query tiles fill the CUs
twice and either no chain stands out (24 tiles for each step of the longest)
or there are five tiles per CU.  Shapes on both sides of each line, dense,
packed and paged, against fp32 attention on the rotated rows (2e-3, the bound
of the other prefill tests); packed and paged agree bit for bit.
"""

import pytest
import torch

import oracle
from qwenforge_amd import ops, paged

pytestmark = pytest.mark.gpu
TOL = 2e-3


def _rows(lengths, heads, seed):
    gen = torch.Generator().manual_seed(seed)
    return torch.randn(sum(lengths), heads, 64, generator=gen).half()


def _reference(q, k, v, groups):
    """fp32 causal attention of one row: (n, QH, 64), (n, KVH, 64) on the device."""
    out = torch.empty(q.shape, device=q.device, dtype=torch.float32)
    mask = torch.ones(q.shape[0], q.shape[0], device=q.device, dtype=torch.bool).triu_(1)
    for h in range(q.shape[1]):
        s = q[:, h].float() @ k[:, h // groups].float().T * 0.125
        out[:, h] = torch.softmax(s.masked_fill_(mask, float("-inf")), -1) @ v[:, h // groups].float()
    return out


@pytest.mark.parametrize("lengths,qh,kvh", [
    ((640,) * 2, 26, 2),      # 520 tiles, 52 a step: one group
    ((577,) * 2, 26, 2),      # the same tiles, ragged
    ((576,) * 2, 26, 2),      # 468 tiles: two groups
    ((2900,), 12, 2),         # 552 tiles, 12 a step: two groups
    ((5100,), 16, 2),         # 1280 tiles, five per CU: one group
    ((5050,), 16, 2),         # 1264: two groups
    ((130, 1, 700, 64, 333, 500, 9, 640, 700), 14, 2),  # packed: 700 tiles by tokens
])
def test_group_count_edges(dev, lengths, qh, kvh):
    b, total = len(lengths), sum(lengths)
    q, k, v = _rows(lengths, qh, 1), _rows(lengths, kvh, 2), _rows(lengths, kvh, 3)
    pos = torch.cat([torch.arange(n) for n in lengths])
    cos, sin = oracle.rope_cos_sin(pos, oracle.inv_freq(64, 1e6))
    q_rot = oracle.apply_rope_fp16(q, cos[:, None], sin[:, None]).to(dev)
    k_rot = oracle.apply_rope_fp16(k, cos[:, None], sin[:, None]).to(dev)
    starts = [sum(lengths[:i]) for i in range(b + 1)]
    cu = torch.tensor(starts, dtype=torch.int32, device=dev)
    args = [t.to(dev) for t in (q, k, v)]
    tables = (cos.to(dev), sin.to(dev))
    kc = torch.zeros(b, kvh, max(lengths), 64, device=dev, dtype=torch.float16)
    vc = torch.zeros_like(kc)
    print(f"[prefill groups] {lengths} {qh}/{kvh}", flush=True)
    out = ops.prefill_varlen(*args, cu, max(lengths), *tables, kc, vc, 0, lengths=list(lengths))
    pages = [-(-n // 64) for n in lengths]
    pool_k = torch.zeros(sum(pages), kvh, 64, 64, device=dev, dtype=torch.float16)
    pool_v = torch.zeros_like(pool_k)
    table = torch.full((b, max(pages)), -1, dtype=torch.int32)
    order = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(4)).to(torch.int32)
    for r, n in enumerate(pages):
        table[r, :n] = order[sum(pages[:r]):sum(pages[:r]) + n]
    out_paged = paged.prefill_varlen_paged(*args, cu, max(lengths), *tables, pool_k, pool_v,
                                           table.to(dev), 0, lengths=list(lengths))
    assert torch.equal(out, out_paged)
    if len(set(lengths)) == 1:
        n = lengths[0]
        dense = [t.view(b, n, -1, 64).transpose(1, 2) for t in args]
        kd, vd = torch.zeros_like(kc), torch.zeros_like(vc)
        d = ops.gqa_flash_prefill_rope_append(*dense, tables[0][:n], tables[1][:n], kd, vd, 0)
        assert torch.equal(d.transpose(1, 2).reshape(total, qh, 64), out)
    for r, n in enumerate(lengths):
        at = slice(starts[r], starts[r + 1])
        ref = _reference(q_rot[at], k_rot[at], args[2][at], qh // kvh)
        assert (out[at].float() - ref).abs().max().item() <= TOL
        assert torch.equal(kc[r, :, :n].transpose(0, 1), k_rot[at])
        assert torch.equal(vc[r, :, :n].transpose(0, 1), args[2][at])
