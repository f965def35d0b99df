/* C ABI of the prompt pass over every layer (gfx950 / MI355X).
 *
 * Replaces the per-layer torch op sequence of the reference's cached prefill
 * (_prefill student_engine.py:679-737, _prefill_ragged :1162-1204): rms_norm,
 * QKV projection, RoPE, KV append, causal attention, o_proj + residual,
 * rms_norm, gate/up, SwiGLU, down_proj + residual.  Conventions as in
 * qf_attn.h: fp16 storage, plain pointers and element strides, the stream as
 * void*, a QF_* / hipError_t return code, no allocation and no
 * synchronisation inside the call (capture-safe).
 */
#ifndef QF_PREFILL_H
#define QF_PREFILL_H

#include <stdint.h>

#include "qf_attn.h"

#ifdef __cplusplus
extern "C" {
#endif

/* One layer: torch Linear weights (out, in), row-major and contiguous; b_qkv
 * may be null.  Caches (B, KVH, cap, 64) with row strides kc_sb / vc_sb, or
 * page pools (qf_paged.h) with page strides.  16-byte aligned throughout. */
typedef struct {
  const void* norm1;
  const void* w_qkv;
  const void* b_qkv;
  const void* w_o;
  const void* norm2;
  const void* w_gate_up;
  const void* w_down;
  void* k_cache;
  void* v_cache;
  int64_t kc_sb, kc_sh, kc_sn;
  int64_t vc_sb, vc_sh, vc_sn;
} QfPrefillLayer;

/* Bytes of the workspace for T tokens, or a negative QF_* code for shapes that
 * the kernels do not cover (hidden, QH * 64 and I multiples of 128, hidden <=
 * 2048, head dim 64). */
int64_t qf_prefill_layers_workspace(int T, int hidden, int QH, int KVH, int D, int I);

/* hidden (T, hidden_size) fp16 contiguous, in place: the embedded prompts in,
 * the residual stream after the last layer out; each token's rotated K and raw
 * V go to its cache slot.  cu null: B rows of S tokens each.  Otherwise packed
 * rows, cu (B + 1) int32 on the device as in qf_prefill_varlen with S the
 * longest row (a token past it in its row is not appended).  Token i of row b
 * goes to slot i of row b: every cache holds S slots at least, which the caller
 * checks; with block_table through it, a page outside the pool writing
 * nothing.  ws: 16-byte aligned, of at least the bytes above (else
 * QF_ERR_SCRATCH_LIMIT), free again when the call's work is done. */
int qf_prefill_layers(const QfPrefillLayer* layers, int n_layers, void* hidden, int T, int B, int S,
                      const int32_t* cu, const float* inv_freq, const int32_t* block_table,
                      int64_t bt_sb, int pages_per_row, int n_pages, int page_size, void* ws,
                      int64_t ws_bytes, float eps, int hidden_size, int QH, int KVH, int D, int I,
                      void* stream);

#ifdef __cplusplus
}
#endif

#endif /* QF_PREFILL_H */
