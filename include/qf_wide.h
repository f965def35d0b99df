/* C ABI of the decode-step projections for 5..32 batch rows (gfx950 / MI355X).
 *
 * qf_step.h covers 1..4 rows; these entry points are the same step for wider
 * batches (the torch op sequence of student_engine.py:896-982).  Conventions
 * and layouts as in qf_step.h; every weight is in matrix-core tiles
 * (qf_pack_weight) and every width it names a multiple of 32.  The attention
 * between them is qf_decode_attn / qf_decode_attn_paged, whose merged fp16
 * output the o_proj call takes.
 */
#ifndef QF_WIDE_H
#define QF_WIDE_H

#include <stdint.h>

#include "qf_step.h"

#ifdef __cplusplus
extern "C" {
#endif

#define QF_WIDE_MAX_B 32

/* qf_rms_qkv_rope_append with positions (pos, inv_freq) for 5..32 rows:
 * rms_norm + QKV (+ bias) + rotate-half RoPE + KV append.  w_qkv packed with
 * QF_PACK_ROPE.  Dense caches: block_table null, every row appends at
 * slots[0] (slot_sb 0) and kc_sb / vc_sb are row strides.  Paged caches
 * (qf_paged.h): kc_sb / vc_sb are page strides, row b appends at logical slot
 * slots[b * slot_sb] through block_table; cap = pages_per_row * page_size. */
int qf_wide_qkv(const void* x, int64_t x_sb, const void* norm_w, float eps, const void* w_qkv,
                const void* bias, const int64_t* pos, const float* inv_freq, void* k_cache,
                int64_t kc_sb, int64_t kc_sh, int64_t kc_sn, void* v_cache, int64_t vc_sb,
                int64_t vc_sh, int64_t vc_sn, const int32_t* block_table, int64_t bt_sb,
                int pages_per_row, int n_pages, int page_size, const int64_t* slots,
                int64_t slot_sb, void* q_out, int64_t qo_sb, int64_t qo_sh, int B, int hidden,
                int QH, int KVH, int D, int cap, void* stream);

/* Workgroups that share one row block's k range in qf_wide_gemv_residual;
 * QF_ERR_UNSUPPORTED for a K that it does not take (a multiple of 32, up to
 * 3.3 million). */
int qf_wide_splits(int K);

/* hidden <- fp16(hidden + fp16(inp @ w^T)), in place (o_proj SE:973-974,
 * down_proj SE:978).  inp (B, K); w packed with QF_PACK_PLAIN.  With
 * qf_wide_splits(K) > 1: part holds N/16 * splits * ceil(B/16) * 256 fp32 and
 * ticket N/16 zeroed int32 that the call leaves zeroed; calls that overlap
 * need their own. */
int qf_wide_gemv_residual(const void* inp, int64_t in_sb, const void* w, void* hidden,
                          int64_t h_sb, float* part, int32_t* ticket, int B, int K, int N,
                          void* stream);

/* qf_rms_gate_up_swiglu for 5..32 rows; w packed with QF_PACK_SWIGLU. */
int qf_wide_gate_up(const void* x, int64_t x_sb, const void* norm_w, float eps,
                    const void* w_gate_up, void* h_out, int64_t ho_sb, int B, int hidden, int I,
                    void* stream);

/* qf_rms_lm_head for 5..32 rows; w packed with QF_PACK_PLAIN. */
int qf_wide_lm_head(const void* x, int64_t x_sb, const void* norm_w, float eps, const void* w_lm,
                    void* logits, int64_t lg_sb, uint64_t* keys, int n_blocks, int B, int hidden,
                    int V, void* stream);

/* qf_argmax_step for 5..32 rows. */
int qf_wide_argmax_step(const uint64_t* keys, int n_blocks, int B, int64_t* token, int64_t* rows,
                        int64_t rows_sb, int n_rows, int64_t* step, int64_t* write_index,
                        int64_t* pos, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* QF_WIDE_H */
