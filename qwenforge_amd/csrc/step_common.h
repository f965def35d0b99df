// Helpers shared by the decode-step projection kernels (decode_step.hip for
// 1..4 batch rows, decode_wide.hip for 5..32).
#pragma once

#include "qf_common.h"

namespace qf {
namespace step {

constexpr int kNW = 4;          // waves per workgroup
constexpr int kNT = kNW * 64;   // threads per workgroup
constexpr int kMaxNormK = 1024; // widest normalised (hidden) row: one chunk per thread
constexpr int kHeadDim = 64;

// Sum over the 64 lanes with DPP moves (no LDS traffic): butterflies inside
// each 16-lane row, then row broadcasts leave the total in lane 63, which is
// read back as a wave-uniform value.
template <int kCtrl, int kRowMask>
__device__ __forceinline__ float dpp_add(float v) {
  const int moved = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), kCtrl, kRowMask, 0xF,
                                                false);
  return v + __builtin_bit_cast(float, moved);
}

__device__ __forceinline__ float wave_sum(float v) {
  v = dpp_add<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
  v = dpp_add<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]: quad sums
  v = dpp_add<0x141, 0xF>(v);  // row_half_mirror: 8-lane sums
  v = dpp_add<0x140, 0xF>(v);  // row_mirror: 16-lane row sums
  v = dpp_add<0x142, 0xA>(v);  // row_bcast:15 into rows 1, 3
  v = dpp_add<0x143, 0xC>(v);  // row_bcast:31 into rows 2, 3: lane 63 holds the total
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

__device__ __forceinline__ f16x8 zero8() {
  f16x8 z;
#pragma unroll
  for (int e = 0; e < 8; ++e) z[e] = (f16)0.f;
  return z;
}

// Eager rotate-half RoPE of one (d, d+32) pair with the reference's fp16
// rounding (student_engine.py:927-928): lo' = fp16(fp16(lo*cos_lo) -
// fp16(hi*sin_lo)), hi' = fp16(fp16(hi*cos_hi) + fp16(lo*sin_hi)).
__device__ __forceinline__ void rope1(float lo, float hi, float cl, float sl, float ch, float sh,
                                      f16& out_lo, f16& out_hi) {
#pragma clang fp contract(off)
  const float a = round16(lo * cl);
  const float b = round16(hi * sl);
  const float c = round16(hi * ch);
  const float d = round16(lo * sh);
  out_lo = (f16)(a - b);
  out_hi = (f16)(c + d);
}

// Packed weight tiles (qf_pack_weight): the 1 KB A operand of row block rb, k
// block kb in lane order, read once per step, so non-temporally.
__device__ __forceinline__ f16x8 tile_load(const f16* __restrict__ w, int nkb, int rb, int kb,
                                           int lane) {
  return load16_nt(w + (((int64_t)rb * nkb + kb) * 64 + lane) * 8);
}

// Orderable key of an fp16 logit at `index`: larger logit first, then the
// smaller index (torch.argmax returns the first maximum).
__device__ __forceinline__ uint64_t argmax_key(f16 v, int index) {
  const unsigned short bits = __builtin_bit_cast(unsigned short, v);
  const unsigned ord = (bits & 0x8000u) ? (~bits & 0xFFFFu) : (bits | 0x8000u);
  return ((uint64_t)ord << 32) | (uint64_t)(0xFFFFFFFFu - (unsigned)index);
}

// Arguments of the QKV kernels (row-major and tiles).
struct QkvArgs {
  const f16* x;
  int64_t x_sb;
  const int64_t* token;
  f16* hidden_out;
  int64_t ho_sb;
  const f16* norm_w;
  float eps;
  const f16* w;
  const f16* bias;
  const f16* cos;
  const f16* sin;
  int64_t cs_sb;
  // Positions mode (cos == nullptr): row b's angle for frequency i is
  // float(pos[b]) * inv_freq[i], and cos/sin are evaluated here in fp32 and
  // rounded to fp16 -- bit-identical to the torch table (SE:910-915) that
  // table mode reads.
  const int64_t* pos;
  const float* inv_freq;
  f16* kc;
  int64_t kc_sb, kc_sh, kc_sn;
  f16* vc;
  int64_t vc_sb, vc_sh, vc_sn;
  const int64_t* write_index;
  f16* q_out;
  int64_t qo_sb, qo_sh;
  int K, QH, KVH, cap, n_pairs, B;
  // Paged caches: kc/vc are page pools (page strides kc_sb/vc_sb); row b
  // appends at logical slot slots[b * slot_sb], in page
  // table[b * t_sb + (slot >> log2p)].  cap = pages per row << log2p.
  const int32_t* table;
  int64_t t_sb;
  int log2p, n_pages;
  const int64_t* slots;  // the tile kernels' dense form too: write_index, stride 0
  int64_t slot_sb;
};
static_assert(covers_lines(sizeof(QkvArgs), {offsetof(QkvArgs, x), offsetof(QkvArgs, bias),
                                             offsetof(QkvArgs, write_index), offsetof(QkvArgs, K),
                                             offsetof(QkvArgs, slots)}),
              "touch_arg_lines fields cover every line");

// Arguments of the gate/up kernels.
struct GateUpArgs {
  const f16* x;
  int64_t x_sb;
  const f16* norm_w;
  float eps;
  const f16* w;
  f16* h;
  int64_t h_sb;
  int K, I, B;
};

// The matrix-core forms of decode_wide.hip (QKV 1..32 rows, gate/up 3..32);
// a.B holds the rows.
void launch_qkv_tiles(const QkvArgs& a, bool paged, bool positions, hipStream_t st);
void launch_gate_up_tiles(const GateUpArgs& a, hipStream_t st);

}  // namespace step
}  // namespace qf
