"""The prompt pass over every layer in one native call (``include/qf_prefill.h``).

``prefill_layers`` enqueues rms_norm, QKV + RoPE + append, causal attention,
o_proj + residual, rms_norm, gate/up + SwiGLU and down_proj + residual of all
layers (SE:679-737, SE:1162-1204).  ``layer_table`` says whether a model and its
caches have the layouts it takes; the engine keeps the torch projections
otherwise.
"""

from __future__ import annotations

import ctypes as C

import torch

from . import _lib
from .ops import _ptr, _stream


class Layer(C.Structure):
    """``QfPrefillLayer``."""

    _fields_ = ([(n, C.c_void_p) for n in ("norm1", "w_qkv", "b_qkv", "w_o", "norm2", "w_gate_up",
                                           "w_down", "k_cache", "v_cache")]
                + [(n, C.c_int64) for n in ("kc_sb", "kc_sh", "kc_sn", "vc_sb", "vc_sh", "vc_sn")])


def layer_table(cfg, layers, caches, device, shape):
    """The ``Layer`` array of a model's weights and (K, V) caches, or None if
    any of them has another type, device, layout or size.  ``shape`` is the
    caches' (rows or pages, kv heads, least slots, 64).  Built for each call:
    no pointer outlives it.  ``rows`` and ``slots`` of the result are what every
    cache holds."""
    h, width = cfg.hidden, cfg.qkv_width
    want = (("input_norm", (h,)), ("qkv_weight", (width, h)), ("qkv_bias", (width,)),
            ("o_weight", (h, cfg.heads * cfg.head_dim)), ("post_norm", (h,)),
            ("gate_up_weight", (2 * cfg.intermediate, h)), ("down_weight", (h, cfg.intermediate)))
    if cfg.heads * cfg.head_dim != h or len(layers) != len(caches):
        return None
    table = (Layer * len(layers))()
    rows, heads, slots, dim = shape
    table.rows, table.slots = rows, min((t.shape[2] for pair in caches for t in pair), default=0)
    for entry, layer, pair in zip(table, layers, caches):
        ptrs = []
        for name, size in want:
            t = layer[name]
            if t is None and name == "qkv_bias":
                ptrs.append(None)
                continue
            ptr = t.data_ptr()
            if (t.dtype != torch.float16 or t.device != device or t.shape != size or ptr % 16
                    or not t.is_contiguous()):
                return None
            ptrs.append(ptr)
        strides = []
        for t in pair:
            ptr, n, stride = t.data_ptr(), t.shape, t.stride()
            if (t.dtype != torch.float16 or t.device != device or len(n) != 4 or n[0] != rows
                    or n[1] != heads or n[2] < slots or n[3] != dim or stride[3] != 1 or ptr % 16
                    or (stride[0] | stride[1] | stride[2]) % 8):
                return None
            ptrs.append(ptr)
            strides += stride[:3]
        (entry.norm1, entry.w_qkv, entry.b_qkv, entry.w_o, entry.norm2, entry.w_gate_up,
         entry.w_down, entry.k_cache, entry.v_cache) = ptrs
        (entry.kc_sb, entry.kc_sh, entry.kc_sn, entry.vc_sb, entry.vc_sh, entry.vc_sn) = strides
    return table


def workspace_bytes(cfg, tokens: int) -> int:
    """Bytes ``prefill_layers`` needs for ``tokens`` tokens; negative for shapes
    its kernels do not cover."""
    return _lib.load().qf_prefill_layers_workspace(tokens, cfg.hidden, cfg.heads, cfg.kv_heads,
                                                   cfg.head_dim, cfg.intermediate)


def prefill_layers(cfg, table, hidden: torch.Tensor, rows: int, longest: int,
                   inv_freq: torch.Tensor, cu: torch.Tensor | None = None,
                   block_table: torch.Tensor | None = None, n_pages: int = 0,
                   page_size: int = 0) -> None:
    """Runs the layers of ``table`` over ``hidden`` (tokens, cfg.hidden) in place:
    ``rows`` rows of ``longest`` tokens, or packed rows of at most that many
    with their offsets ``cu`` (rows + 1) int32 on the device."""
    tokens = hidden.numel() // cfg.hidden
    if block_table is None and (table.rows != rows or longest > table.slots):
        raise ValueError(f"caches of {table.rows} rows and {table.slots} slots do not hold "
                         f"{rows} rows of {longest} tokens")
    if block_table is not None and (
            (n_pages, page_size) != (table.rows, table.slots) or block_table.dim() != 2
            or longest > block_table.shape[1] * page_size):
        raise ValueError("n_pages and page_size must be the pools' and the table's rows hold "
                         f"{longest} slots")
    if hidden.dtype != torch.float16 or hidden.device.type != "cuda" or not hidden.is_contiguous():
        raise ValueError("hidden must be a contiguous fp16 device tensor")
    if cu is not None and (cu.dtype != torch.int32 or cu.shape != (rows + 1,)
                           or cu.device != hidden.device or not cu.is_contiguous()):
        raise ValueError("cu must be (rows + 1,) int32 on hidden's device")
    if inv_freq.dtype != torch.float32 or inv_freq.shape != (cfg.head_dim // 2,) \
            or inv_freq.device != hidden.device or not inv_freq.is_contiguous():
        raise ValueError("inv_freq must be (head_dim / 2,) fp32 on hidden's device")
    bt_sb = ppr = 0
    if block_table is not None:
        if (block_table.dtype != torch.int32 or block_table.device != hidden.device
                or block_table.dim() != 2 or block_table.shape[0] != rows
                or block_table.stride(1) != 1):
            raise ValueError("block_table must be (rows, pages) int32 with unit inner stride")
        bt_sb, ppr = block_table.stride(0), block_table.shape[1]
    need = workspace_bytes(cfg, tokens)
    _lib.check(min(need, 0), "qf_prefill_layers_workspace")
    with torch.cuda.device(hidden.device):
        ws = torch.empty(need, device=hidden.device, dtype=torch.uint8)
        rc = _lib.load().qf_prefill_layers(
            table, len(table), hidden.data_ptr(), tokens, rows, longest, _ptr(cu),
            inv_freq.data_ptr(), _ptr(block_table), bt_sb, ppr, n_pages, page_size, ws.data_ptr(),
            need, float(cfg.rms_eps), cfg.hidden, cfg.heads, cfg.kv_heads, cfg.head_dim,
            cfg.intermediate, _stream(hidden.device))
    _lib.check(rc, "qf_prefill_layers")
