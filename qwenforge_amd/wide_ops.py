"""Torch-facing wrappers of the decode-step projections for 5..32 rows
(``include/qf_wide.h``).

The step of ``step_ops`` (SE:896-982) for wider batches: every weight is
``step_ops.Tiles``, o_proj takes the attention's merged output
(``ops.flash_decode_attention``), and the long down projection is split over
workgroups through the caller's ``make_wide_scratch``.  Like there, every
function launches on the current HIP stream (of its operands' device, whichever
is current); nothing computes on the host.
"""

from __future__ import annotations

import torch

from . import _lib
from .ops import HEAD_DIM, _ptr, _stream
from .paged import _pool_args, _slot_args
from .step_ops import PACK_PLAIN, PACK_ROPE, PACK_SWIGLU, Tiles, _check, _rows, _weight

MIN_BATCH, MAX_BATCH = 5, 32


def _batch(b: int) -> None:
    if not MIN_BATCH <= b <= MAX_BATCH:
        raise ValueError(f"wide decode-step kernels take {MIN_BATCH}..{MAX_BATCH} rows (got {b})")


def _tiles(name: str, w, out_f: int, in_f: int, pack: int) -> int:
    if not isinstance(w, Tiles):
        raise TypeError(f"{name} must be packed (step_ops.pack_weight)")
    return _weight(name, w, out_f, in_f, pack)[0]


def make_wide_scratch(batch: int, n: int, k: int, device):
    """(part, ticket) of ``gemv_residual`` for a (n, k) weight; the ticket is
    zeroed here and left zeroed by every call."""
    splits = _lib.load().qf_wide_splits(k)
    _lib.check(min(splits, 0), "qf_wide_splits")
    part = torch.empty(n // 16 * splits * -(-batch // 16) * 256, device=device, dtype=torch.float32)
    return part, torch.zeros(n // 16, device=device, dtype=torch.int32)


def _rms_qkv(x, norm_w, eps, w_qkv, bias, positions, caches, slots, q_out, kvh, cap):
    _check("q_out", q_out)
    if q_out.dim() != 3 or q_out.shape[2] != HEAD_DIM or q_out.stride(2) != 1:
        raise ValueError(f"q_out must be (B, QH, 64) (got {tuple(q_out.shape)})")
    b, qh, d = q_out.shape
    _batch(b)
    hidden = norm_w.shape[0]
    _check("norm_w", norm_w)
    x_sb = _rows("x", x, b, hidden)
    rows = (qh + 2 * kvh) * d
    w_ptr = _tiles("w_qkv", w_qkv, rows, hidden, PACK_ROPE)
    if bias is not None:
        _check("bias", bias)
        if tuple(bias.shape) != (rows,) or not bias.is_contiguous():
            raise ValueError("bias must be contiguous ((QH + 2 KVH) * 64,)")
    pos, inv = positions
    _check("pos", pos, torch.int64)
    _check("inv_freq", inv, torch.float32)
    if pos.shape != (b,) or not pos.is_contiguous():
        raise ValueError("pos must be contiguous (B,)")
    if inv.shape != (d // 2,) or not inv.is_contiguous():
        raise ValueError(f"inv_freq must be contiguous ({d // 2},)")
    with torch.cuda.device(x.device):
        rc = _lib.load().qf_wide_qkv(
            x.data_ptr(), x_sb, norm_w.data_ptr(), float(eps), w_ptr, _ptr(bias), pos.data_ptr(),
            inv.data_ptr(), *caches, *slots, q_out.data_ptr(), q_out.stride(0), q_out.stride(1),
            b, hidden, qh, kvh, d, cap, _stream(x.device))
    _lib.check(rc, "qf_wide_qkv")


def rms_qkv_rope_append(x: torch.Tensor, norm_w: torch.Tensor, eps: float, w_qkv: Tiles,
                        bias: torch.Tensor | None, positions, key_cache: torch.Tensor,
                        value_cache: torch.Tensor, write_index: torch.Tensor,
                        q_out: torch.Tensor) -> None:
    """q_out <- RoPE(q); caches[:, :, write_index] <- RoPE(k), v, with RoPE from
    ``positions = (pos, inv_freq)`` as in ``step_ops.rms_qkv_rope_append``."""
    _check("key_cache", key_cache)
    _check("value_cache", value_cache)
    b, kvh, cap, d = key_cache.shape
    if d != HEAD_DIM or value_cache.shape != key_cache.shape or b != q_out.shape[0]:
        raise ValueError("caches must be (B, KVH, cap, 64) and alike")
    if key_cache.stride(-1) != 1 or value_cache.stride(-1) != 1:
        raise ValueError("caches need unit stride on the head dimension")
    _check("write_index", write_index, torch.int64)
    caches = (key_cache.data_ptr(), *key_cache.stride()[:3],
              value_cache.data_ptr(), *value_cache.stride()[:3], None, 0, 0, 0, 0)
    _rms_qkv(x, norm_w, eps, w_qkv, bias, positions, caches, (write_index.data_ptr(), 0), q_out,
             kvh, cap)


def rms_qkv_rope_append_paged(x: torch.Tensor, norm_w: torch.Tensor, eps: float, w_qkv: Tiles,
                              bias: torch.Tensor | None, positions, k_pool: torch.Tensor,
                              v_pool: torch.Tensor, block_table: torch.Tensor,
                              slots: torch.Tensor, q_out: torch.Tensor) -> None:
    """The same into paged caches at per-row ``slots`` (B,) int64."""
    b = q_out.shape[0]
    pool, cap = _pool_args(k_pool, v_pool, block_table, b)
    _rms_qkv(x, norm_w, eps, w_qkv, bias, positions, pool, _slot_args(slots, b, q_out.device),
             q_out, k_pool.shape[1], cap)


def gemv_residual(inp: torch.Tensor, w: Tiles, hidden: torch.Tensor, scratch) -> None:
    """hidden <- fp16(hidden + fp16(inp @ w^T)), in place; ``scratch`` from
    ``make_wide_scratch`` for this weight's shape and batch (or a larger one)."""
    b, k = inp.shape
    _batch(b)
    n = w.shape[0]
    in_sb = _rows("inp", inp, b, k)
    w_ptr = _tiles("w", w, n, k, PACK_PLAIN)
    h_sb = _rows("hidden", hidden, b, n)
    part, ticket = scratch
    lib = _lib.load()
    _check("part", part, torch.float32)
    _check("ticket", ticket, torch.int32)
    if part.numel() < n // 16 * lib.qf_wide_splits(k) * -(-b // 16) * 256 or ticket.numel() < n // 16:
        raise ValueError("scratch too small for this weight and batch (make_wide_scratch)")
    with torch.cuda.device(inp.device):
        rc = lib.qf_wide_gemv_residual(inp.data_ptr(), in_sb, w_ptr, hidden.data_ptr(), h_sb,
                                       part.data_ptr(), ticket.data_ptr(), b, k, n,
                                       _stream(inp.device))
    _lib.check(rc, "qf_wide_gemv_residual")


def rms_gate_up_swiglu(x: torch.Tensor, norm_w: torch.Tensor, eps: float, w_gate_up: Tiles,
                       h_out: torch.Tensor) -> None:
    """h_out <- fp16(fp16(silu(g)) * u), [g | u] = rms_norm(x) @ w_gate_up^T."""
    b, hidden = x.shape
    _batch(b)
    inter = w_gate_up.shape[0] // 2
    x_sb = _rows("x", x, b, hidden)
    _check("norm_w", norm_w)
    w_ptr = _tiles("w_gate_up", w_gate_up, 2 * inter, hidden, PACK_SWIGLU)
    ho_sb = _rows("h_out", h_out, b, inter)
    with torch.cuda.device(x.device):
        rc = _lib.load().qf_wide_gate_up(x.data_ptr(), x_sb, norm_w.data_ptr(), float(eps), w_ptr,
                                         h_out.data_ptr(), ho_sb, b, hidden, inter, _stream(x.device))
    _lib.check(rc, "qf_wide_gate_up")


def rms_lm_head(x: torch.Tensor, norm_w: torch.Tensor, eps: float, w_lm: Tiles,
                logits: torch.Tensor, keys: torch.Tensor) -> None:
    """logits <- fp16(rms_norm(x) @ w_lm^T); keys (B, n_blocks) <- per-block argmax keys."""
    b, hidden = x.shape
    _batch(b)
    vocab = w_lm.shape[0]
    x_sb = _rows("x", x, b, hidden)
    _check("norm_w", norm_w)
    w_ptr = _tiles("w_lm", w_lm, vocab, hidden, PACK_PLAIN)
    lg_sb = _rows("logits", logits, b, vocab)
    _check("keys", keys, torch.int64)
    if keys.dim() != 2 or keys.shape[0] != b or not keys.is_contiguous():
        raise ValueError("keys must be contiguous (B, n_blocks) int64")
    with torch.cuda.device(x.device):
        rc = _lib.load().qf_wide_lm_head(x.data_ptr(), x_sb, norm_w.data_ptr(), float(eps), w_ptr,
                                         logits.data_ptr(), lg_sb, keys.data_ptr(), keys.shape[1], b,
                                         hidden, vocab, _stream(x.device))
    _lib.check(rc, "qf_wide_lm_head")


def argmax_step(keys: torch.Tensor, token: torch.Tensor, rows: torch.Tensor, step: torch.Tensor,
                write_index: torch.Tensor | None, pos: torch.Tensor) -> None:
    """token <- argmax from the lm_head keys; rows[:, step] <- token; step,
    write_index (if any) and pos advance by one (a parked row's stays)."""
    b, n_blocks = keys.shape
    _batch(b)
    for name, t in (("keys", keys), ("token", token), ("rows", rows), ("step", step), ("pos", pos)):
        _check(name, t, torch.int64)
    if token.shape != (b,) or not token.is_contiguous() or pos.shape != (b,) or not pos.is_contiguous():
        raise ValueError("token and pos must be contiguous (B,)")
    if rows.dim() != 2 or rows.shape[0] != b or rows.stride(1) != 1 or not keys.is_contiguous():
        raise ValueError("rows must be (B, T) with unit inner stride, keys contiguous")
    if write_index is not None:
        _check("write_index", write_index, torch.int64)
    with torch.cuda.device(keys.device):
        rc = _lib.load().qf_wide_argmax_step(keys.data_ptr(), n_blocks, b, token.data_ptr(),
                                             rows.data_ptr(), rows.stride(0), rows.shape[1],
                                             step.data_ptr(), _ptr(write_index), pos.data_ptr(),
                                             _stream(keys.device))
    _lib.check(rc, "qf_wide_argmax_step")
