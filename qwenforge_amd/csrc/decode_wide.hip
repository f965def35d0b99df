// Decode-step projections on packed weight tiles for up to 32 batch rows
// (gfx950 / MI355X): QKV from one row on, gate/up from three, the others from five.
//
// Below 16 rows an MFMA column is still mostly idle work, so the cost of a
// projection stays streaming its weight once, as at 1..4 rows
// (decode_step.hip).  The kernels keep that shape -- packed 16 x 32 weight
// tiles as the A operand, batch rows as MFMA columns, a row block's k range
// split over the four waves of a workgroup -- and change what more rows cost:
//
//   * rows are normalised a row per wave (no barrier for the sum of squares)
//     and staged with 16 bytes of padding per row, so the 16 columns of an
//     operand read hit distinct LDS banks (hidden * 2 bytes is a multiple of
//     all 64 banks: unpadded reads conflict 16 ways);
//   * past 16 rows a second block of 16 columns reuses the weight tile in
//     registers;
//   * o_proj takes the attention's merged output instead of merging partials
//     in every workgroup (that prologue grows with splits x rows);
//   * the long down projection splits k over workgroups too: 56 row blocks
//     alone cannot stream 8.7 MB from 56 CUs.
//
// Measured on MI355X (kernel trace, 896/4864 widths, 1024 tokens of context),
// us at B=12 / 32, with the torch projections' kernels at B=12 beside them:
// QKV + RoPE + append 4.4 / 6.6 (norm 3.6 + GEMM 7.3 + append 4.0), o_proj
// 4.1 / 5.2 (7.3 + add 4.0), gate/up 6.4 / 8.9 (norm 3.6 + GEMM 10 + silu and
// product 8), down 6.9 / 8.1 (13.4 + add 4.0), lm_head 46 / 53 (54 + argmax 49).
// The first four are bound by launch latency and the round trip of their
// loads (at B=12 1.6-17 MB of weights at 0.4-2.7 TB/s), the lm_head by HBM
// (5.9 TB/s).
//
// Replaces the torch op sequence of _decode_step_static
// (student_engine.py:896-982); same rounding points as decode_step.hip.
#include "step_common.h"
#include "../../include/qf_wide.h"

namespace qf {
namespace step {

constexpr int kPad = 8;            // halves of padding per staged row
constexpr int kNt = 2;             // non-temporal bit of a buffer access
constexpr int kNormBlk = kMaxNormK / 32 / kNW;  // k blocks per wave of a normalised row (max)

// Columns of 16 for kRows staged rows per wave (4 * kRows rows in all).
constexpr int col_blocks(int rows_per_wave) { return rows_per_wave > 4 ? 2 : 1; }

// RMSNorm staging, fp32 math and one rounding: wave w owns rows w, w + 4, ...
// Rows past B re-read row B - 1 (their columns are never stored); `token`
// gathers the rows of an embedding table.  Split so
// that the caller's weight loads go out in between.
template <int kRows>
struct WideStage {
  f16x8 x[kRows][2];
  f16x8 g[2];
};

template <int kRows>
__device__ __forceinline__ void wide_load(WideStage<kRows>& st, const f16* __restrict__ x,
                                          int64_t x_sb, int B, int C, const f16* __restrict__ nw,
                                          const int64_t* token = nullptr) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c0 = min(lane, C - 1), c1 = min(lane + 64, C - 1);
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const int r = min(w + kNW * i, B - 1);
    const f16* row = x + (token != nullptr ? token[r] : (int64_t)r) * x_sb;
    st.x[i][0] = load16(row + 8 * c0);
    st.x[i][1] = load16(row + 8 * c1);
  }
  st.g[0] = load16(nw + 8 * c0);
  st.g[1] = load16(nw + 8 * c1);
}

template <int kRows>
__device__ __forceinline__ void wide_finish(const WideStage<kRows>& st, int K, float eps, f16* xs) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, C = K / 8;
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    float s[2] = {0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 8; ++e) s[h] += (float)st.x[i][h][e] * (float)st.x[i][h][e];
    const float tot = wave_sum((lane < C ? s[0] : 0.f) + (lane + 64 < C ? s[1] : 0.f));
    const float rstd = rsqrtf(tot / (float)K + eps);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f16x8 y;
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = (f16)(((float)st.x[i][h][e] * rstd) * (float)st.g[h][e]);
      if (lane + 64 * h < C) store16(xs + (w + kNW * i) * (K + kPad) + 8 * (lane + 64 * h), y);
    }
  }
  __syncthreads();
}

// B operand of k block kb and column block cb from the staged rows.
template <int kRows>
__device__ __forceinline__ f16x8 wide_operand(const f16* xs, int K, int kb, int cb, int lane) {
  const int row = min(16 * cb + (lane & 15), kNW * kRows - 1);
  return *reinterpret_cast<const f16x8*>(xs + row * (K + kPad) + 32 * kb + 8 * (lane >> 4));
}

// The weight tiles of k blocks [kb0, kb0 + n) of row block rb, zeros past n: a
// real tile re-read there could hold infinities, which zero columns turn into
// NaN.  The buffer ends after this wave's share (all of it wave-uniform), so a
// surplus block costs neither traffic nor selects (non-temporal like
// tile_load).  rb past nrb: zeros.  MI355X, us for 24 layers, tiles re-read /
// an out-of-range offset a surplus block (in the lanes) / this: the MLP half at
// 4 rows 267 / 271 / 259, the attention half 322 / 319 / 316, a step of 12 rows
// 750 / 752 / 741, of 32 951 / - / 946.
template <int kBlk>
__device__ __forceinline__ void share_tiles(f16x8 (&wa)[kBlk], const f16* w, int nkb, int nrb,
                                            int rb, int kb0, int n, int lane) {
  const __amdgpu_buffer_rsrc_t r = buffer_rsrc(w + ((int64_t)rb * nkb + kb0) * 512,
                                               rb < nrb && n > 0 ? n * 1024 : 0);
#pragma unroll
  for (int t = 0; t < kBlk; ++t)
    wa[t] = __builtin_bit_cast(
        f16x8, __builtin_amdgcn_raw_buffer_load_b128(r, t * 1024 + lane * 16, 0, kNt));
}

// This wave's k blocks [kb0, kb0 + n) of one row block against every column
// block; the operands of all blocks are read before the first MFMA.  A block
// past n multiplies zeros on both sides (share_tiles, and here).
template <int kRows, int kBlk>
__device__ __forceinline__ void wide_mfma(const f16x8 (&wa)[kBlk], const f16* xs, int K, int kb0,
                                          int n, int lane, f32x4 (&acc)[col_blocks(kRows)]) {
  constexpr int NC = col_blocks(kRows);
  f16x8 xb[kBlk][NC];
#pragma unroll
  for (int t = 0; t < kBlk; ++t)
#pragma unroll
    for (int c = 0; c < NC; ++c)
      xb[t][c] = t < n ? wide_operand<kRows>(xs, K, kb0 + t, c, lane) : zero8();
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < kBlk; ++t)
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = mfma16x16x32(wa[t], xb[t][c], acc[c]);
}

// ---------------------------------------------------------------------------
// One 16-row block (QF_PACK_ROPE: rotate-half pairs in C registers t and
// t + 2 of a lane) per workgroup; wave c < NC finishes column block c.
template <int kRows, bool kPaged, bool kPos>
__global__ __launch_bounds__(kNT) void wide_qkv_kernel(QkvArgs a) {
  constexpr int NC = col_blocks(kRows);
  __shared__ __attribute__((aligned(16))) f16 xs[kNW * kRows * (kMaxNormK + kPad)];
  __shared__ f32x4 part[kNW][NC][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = touch_arg_lines(a.K, a.x, a.bias, a.write_index, a.slots), nkb = K / 32;
  const int per = (nkb + kNW - 1) / kNW, kb0 = w * per, n = min(per, nkb - kb0);
  const int rb = blockIdx.x;
  WideStage<kRows> st;
  // Gathered rows: the 1..4-row entry points only.
  wide_load<kRows>(st, a.x, a.x_sb, a.B, K / 8, a.norm_w, kRows == 1 ? a.token : nullptr);
  // Epilogue operands of this wave's column block, loaded ahead of the weights.
  const int q = lane >> 4, col = 16 * min(w, NC - 1) + (lane & 15), be = min(col, a.B - 1);
  const int head = rb >> 2, d0 = 8 * (rb & 3) + 2 * q;
  const int64_t slot = a.slots[be * a.slot_sb];
  const bool has_bias = a.bias != nullptr;
  const f16* bsrc = (has_bias ? a.bias : a.w) + 64 * head + d0;
  float bias[2][2], ang[2];
  float cs[2][4];  // per dim: cos_lo, sin_lo, cos_hi, sin_hi
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const float lo = (float)bsrc[t], hi = (float)bsrc[t + 32];
    bias[t][0] = has_bias ? lo : 0.f;
    bias[t][1] = has_bias ? hi : 0.f;
    if (kPos) {
      ang[t] = (float)a.pos[be] * a.inv_freq[d0 + t];
    } else {
      const f16* cp = a.cos + be * a.cs_sb + d0 + t;
      const f16* sp = a.sin + be * a.cs_sb + d0 + t;
      cs[t][0] = (float)cp[0];
      cs[t][1] = (float)sp[0];
      cs[t][2] = (float)cp[32];
      cs[t][3] = (float)sp[32];
    }
  }
  f16x8 wa[kNormBlk];
  share_tiles(wa, a.w, nkb, (int)gridDim.x, rb, kb0, n, lane);
  bool in_range = slot >= 0 && slot < a.cap;
  int64_t kro, vro;
  if (kPaged) {
    const int64_t sl = in_range ? slot : 0;
    const int page = a.table[be * a.t_sb + (sl >> a.log2p)];
    in_range = in_range && page >= 0 && page < a.n_pages;
    const int64_t prow = sl & ((1 << a.log2p) - 1);
    kro = (int64_t)page * a.kc_sb + prow * a.kc_sn;
    vro = (int64_t)page * a.vc_sb + prow * a.vc_sn;
  } else {
    kro = be * a.kc_sb + slot * a.kc_sn;
    vro = be * a.vc_sb + slot * a.vc_sn;
  }
  if (kPos) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      cs[t][0] = cs[t][2] = (float)(f16)cosf(ang[t]);
      cs[t][1] = cs[t][3] = (float)(f16)sinf(ang[t]);
    }
  }
  if (kRows == 1 && a.token != nullptr && a.hidden_out != nullptr && blockIdx.x == 0) {
    // The gathered embedding rows, as the residual stream.
#pragma unroll
    for (int i = 0; i < kRows; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (w + kNW * i < a.B && lane + 64 * h < K / 8)
          store16(a.hidden_out + (w + kNW * i) * a.ho_sb + 8 * (lane + 64 * h), st.x[i][h]);
  }
  wide_finish<kRows>(st, K, a.eps, xs);
  f32x4 acc[NC];
  wide_mfma<kRows, kNormBlk>(wa, xs, K, kb0, n, lane, acc);
#pragma unroll
  for (int c = 0; c < NC; ++c) part[w][c][lane] = acc[c];
  __syncthreads();
  if (w >= NC || col >= a.B) return;
  f32x4 sum = part[0][w][lane];
#pragma unroll
  for (int s = 1; s < kNW; ++s) sum += part[s][w][lane];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int d = d0 + t;
    const float lo = (float)(f16)(sum[t] + bias[t][0]);
    const float hi = (float)(f16)(sum[t + 2] + bias[t][1]);
    if (head < a.QH + a.KVH) {
      f16 olo, ohi;
      rope1(lo, hi, cs[t][0], cs[t][1], cs[t][2], cs[t][3], olo, ohi);
      if (head < a.QH) {
        f16* qo = a.q_out + col * a.qo_sb + head * a.qo_sh;
        qo[d] = olo;
        qo[d + 32] = ohi;
      } else if (in_range) {
        f16* kd = a.kc + kro + (head - a.QH) * a.kc_sh;
        kd[d] = olo;
        kd[d + 32] = ohi;
      }
    } else if (in_range) {
      f16* vd = a.vc + vro + (head - a.QH - a.KVH) * a.vc_sh;
      vd[d] = (f16)lo;
      vd[d + 32] = (f16)hi;
    }
  }
}

// ---------------------------------------------------------------------------
struct WideGemvArgs {
  const f16* inp;
  int64_t in_sb;
  const f16* w;
  f16* hidden;
  int64_t h_sb;
  float* part;
  int32_t* ticket;
  int B, K, N, splits;
};
static_assert(covers_lines(sizeof(WideGemvArgs),
                           {offsetof(WideGemvArgs, K), offsetof(WideGemvArgs, splits)}),
              "touch_arg_lines fields cover every line");

// hidden += inp @ w^T.  Grid (row blocks, splits): a workgroup takes one
// split of a row block's k range, a quarter of it per wave.  Each wave loads
// its B operands straight from global memory (16 rows of 64 bytes per k
// block): no wave reads another's k range, so nothing is staged and no
// barrier stands before the MFMAs.  kBlk: k blocks per wave (max).
//
// With more than one split the workgroups store their fp32 tiles with
// write-through (sc1) stores, wait for the acknowledgements and draw the row
// block's ticket; the last one sums all of them in split order (the same sum
// whichever workgroup is last), adds the residual and re-arms the ticket.
// The publication order is the decode kernel's single-launch merge's.
template <int NC, int kBlk, bool kSplit>
__global__ __launch_bounds__(kNT) void wide_gemv_kernel(WideGemvArgs a) {
  __shared__ f32x4 red[kNW][NC][64];
  __shared__ int sh_last;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int K = touch_arg_lines(a.K, a.splits), nkb = K / 32;
  const int rb = blockIdx.x, sp = blockIdx.y;
  const int parts = kNW * (kSplit ? a.splits : 1), mine = kNW * sp + w;
  // Even shares of the k blocks: [mine * nkb / parts, (mine + 1) * nkb / parts).
  const int kb0 = mine * nkb / parts, n = (mine + 1) * nkb / parts - kb0;
  const int q = lane >> 4, col = lane & 15;
  f16x8 wa[kBlk], xb[kBlk][NC];
#pragma unroll
  for (int t = 0; t < kBlk; ++t) wa[t] = tile_load(a.w, nkb, rb, min(kb0 + t, nkb - 1), lane);
#pragma unroll
  for (int t = 0; t < kBlk; ++t)
#pragma unroll
    for (int c = 0; c < NC; ++c)
      xb[t][c] = load16(a.inp + (int64_t)min(16 * c + col, a.B - 1) * a.in_sb +
                        32 * min(kb0 + t, nkb - 1) + 8 * q);
  // Wave c < NC finishes column block c: lane l rows 16 rb + 4 (l / 16) .. +3.
  const int oc = 16 * min(w, NC - 1) + col;
  f16* hp = a.hidden + (int64_t)min(oc, a.B - 1) * a.h_sb + 16 * rb + 4 * q;
  const f16x4 res = *reinterpret_cast<const f16x4*>(hp);
  f32x4 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < kBlk; ++t) {
    const f16x8 wt = t < n ? wa[t] : zero8();
#pragma unroll
    for (int c = 0; c < NC; ++c)
      // A block past this wave's share multiplies zeros on both sides (its
      // loads re-read real data, which may hold infinities).
      acc[c] = mfma16x16x32(wt, t < n ? xb[t][c] : zero8(), acc[c]);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) red[w][c][lane] = acc[c];
  __syncthreads();
  f32x4 sum;
  if (w < NC) {
    sum = red[0][w][lane];
#pragma unroll
    for (int s = 1; s < kNW; ++s) sum += red[s][w][lane];
  }
  if (kSplit) {
    const int S = a.splits;
    const int64_t row_floats = (int64_t)S * NC * 256;
    const __amdgpu_buffer_rsrc_t rp = buffer_rsrc(a.part + rb * row_floats, row_floats * 4);
    if (w < NC)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum), rp,
                                             ((sp * NC + w) * 64 + lane) * 16, 0, kSc1);
    s_waitcnt_vm(0);
    __syncthreads();
    if (threadIdx.x == 0) sh_last = atomicAdd(a.ticket + rb, 1) == S - 1;
    __syncthreads();
    if (!sh_last) return;
    if (w < NC) {
      sum = f32x4{0.f, 0.f, 0.f, 0.f};
      constexpr int kFold = 8;  // splits past S read zeros (the buffer ends there)
      for (int s0 = 0; s0 < S; s0 += kFold) {
        f32x4 v[kFold];
#pragma unroll
        for (int u = 0; u < kFold; ++u)
          v[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                               rp, (((s0 + u) * NC + w) * 64 + lane) * 16, 0, kSc1));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kFold; ++u) sum += v[u];
      }
    }
    if (threadIdx.x == 0) atomicExch(a.ticket + rb, 0);
  }
  if (w >= NC || oc >= a.B) return;
  f16x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = (f16)((float)res[i] + (float)(f16)sum[i]);
  *reinterpret_cast<f16x4*>(hp) = o;
}

// ---------------------------------------------------------------------------
// Gate/up + SwiGLU (QF_PACK_SWIGLU: gate and up of a pair in C registers t
// and t + 2 of a lane), kRB row blocks per workgroup.
template <int kRows, int kRB>
__global__ __launch_bounds__(kNT) void wide_gate_up_kernel(GateUpArgs a) {
  constexpr int NC = col_blocks(kRows);
  __shared__ __attribute__((aligned(16))) f16 xs[kNW * kRows * (kMaxNormK + kPad)];
  __shared__ f32x4 part[kNW][kRB * NC][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = a.K, nkb = K / 32, nrb = a.I / 8;
  const int per = (nkb + kNW - 1) / kNW, kb0 = w * per, n = min(per, nkb - kb0);
  const int rb0 = blockIdx.x * kRB;
  WideStage<kRows> st;
  wide_load<kRows>(st, a.x, a.x_sb, a.B, K / 8, a.norm_w);
  f16x8 wa[kRB][kNormBlk];
#pragma unroll
  for (int r = 0; r < kRB; ++r) share_tiles(wa[r], a.w, nkb, nrb, rb0 + r, kb0, n, lane);
  wide_finish<kRows>(st, K, a.eps, xs);
#pragma unroll
  for (int r = 0; r < kRB; ++r) {
    f32x4 acc[NC];
    wide_mfma<kRows, kNormBlk>(wa[r], xs, K, kb0, n, lane, acc);
#pragma unroll
    for (int c = 0; c < NC; ++c) part[w][r * NC + c][lane] = acc[c];
  }
  __syncthreads();
  for (int j = w; j < kRB * NC; j += kNW) {
    const int r = j / NC, col = 16 * (j % NC) + (lane & 15);
    f32x4 sum = part[0][j][lane];
#pragma unroll
    for (int s = 1; s < kNW; ++s) sum += part[s][j][lane];
    if (col >= a.B || rb0 + r >= nrb) continue;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      // F.silu on the fp16 gate (fp32 math, one rounding), then the fp16 product.
      const float g16 = (float)(f16)sum[t], u16 = (float)(f16)sum[t + 2];
      const float s16 = (float)(f16)(g16 / (1.f + expf(-g16)));
      a.h[col * a.h_sb + 8 * (rb0 + r) + 2 * (lane >> 4) + t] = (f16)(s16 * u16);
    }
  }
}

// ---------------------------------------------------------------------------
struct WideLmArgs {
  const f16* x;
  int64_t x_sb;
  const f16* norm_w;
  float eps;
  const f16* w;
  f16* logits;
  int64_t lg_sb;
  uint64_t* keys;
  int B, K, V;
};

// torch.argmax's order: a NaN beats every number and the two zeros are equal.
__device__ __forceinline__ uint64_t wide_key(f16 v, int index) {
  const float f = (float)v;
  const f16 canon = f != f ? __builtin_bit_cast(f16, (unsigned short)0x7FFF) : (f == 0.f ? (f16)0.f : v);
  return argmax_key(canon, index);
}

// lm_head: each wave takes whole row blocks (grid-stride) in stages of kLmKC
// tiles, the next stage's loads in flight under the current one's MFMAs.
constexpr int kWideLmKC = 7;

template <int kRows>
__global__ __launch_bounds__(kNT) void wide_lm_head_kernel(WideLmArgs a) {
  constexpr int NC = col_blocks(kRows), KC = kWideLmKC;
  __shared__ __attribute__((aligned(16))) f16 xs[kNW * kRows * (kMaxNormK + kPad)];
  __shared__ uint64_t wkeys[kNW][16 * NC];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int K = a.K, nkb = K / 32, nch = (nkb + KC - 1) / KC;
  const int nrb = a.V / 16, stride = gridDim.x * kNW, rb0 = blockIdx.x * kNW + w;
  const int items = (rb0 < nrb ? (nrb - 1 - rb0) / stride + 1 : 0) * nch;
  auto load_stage = [&](int i, f16x8 (&buf)[KC]) {
    const int ii = min(i, max(items - 1, 0));
    const int rb = min(rb0 + (ii / nch) * stride, nrb - 1), ch = ii % nch;
#pragma unroll
    for (int t = 0; t < KC; ++t) buf[t] = tile_load(a.w, nkb, rb, min(ch * KC + t, nkb - 1), lane);
  };
  WideStage<kRows> st;
  wide_load<kRows>(st, a.x, a.x_sb, a.B, K / 8, a.norm_w);
  f16x8 cur[KC], nxt[KC];
  load_stage(0, cur);
  wide_finish<kRows>(st, K, a.eps, xs);

  const int q = lane >> 4;
  uint64_t best[NC];
  f32x4 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    best[c] = 0;
    acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (int i = 0; i < items; ++i) {
    load_stage(i + 1, nxt);
    const int ch = i % nch, n = __builtin_amdgcn_readfirstlane(min(KC, nkb - ch * KC));
    if (n < KC)  // the tiles past a short stage re-read real ones, which may hold infinities
#pragma unroll
      for (int t = 1; t < KC; ++t)
        if (t >= n) cur[t] = zero8();
#pragma unroll
    for (int t = 0; t < KC; ++t)
#pragma unroll
      for (int c = 0; c < NC; ++c)
        acc[c] = mfma16x16x32(
            cur[t], t < n ? wide_operand<kRows>(xs, K, ch * KC + t, c, lane) : zero8(), acc[c]);
    if (ch == nch - 1) {
      const int n0 = 16 * (rb0 + (i / nch) * stride) + 4 * q;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int col = 16 * c + (lane & 15);
        if (col < a.B) {
          f16x4 lg;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            lg[e] = (f16)acc[c][e];
            const uint64_t key = wide_key(lg[e], n0 + e);
            best[c] = key > best[c] ? key : best[c];
          }
          *reinterpret_cast<f16x4*>(a.logits + col * a.lg_sb + n0) = lg;
        }
        acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int t = 0; t < KC; ++t) cur[t] = nxt[t];
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
#pragma unroll
    for (int off = 16; off < 64; off <<= 1) {
      const unsigned lo = __shfl_xor((unsigned)best[c], off);
      const unsigned hi = __shfl_xor((unsigned)(best[c] >> 32), off);
      const uint64_t o = ((uint64_t)hi << 32) | lo;
      best[c] = o > best[c] ? o : best[c];
    }
    if (lane < 16) wkeys[w][16 * c + lane] = best[c];
  }
  __syncthreads();
  const int b = threadIdx.x;
  if (b < a.B && b < 16 * NC) {
    uint64_t k = wkeys[0][b];
#pragma unroll
    for (int ww = 1; ww < kNW; ++ww) k = wkeys[ww][b] > k ? wkeys[ww][b] : k;
    a.keys[(int64_t)b * gridDim.x + blockIdx.x] = k;
  }
}

// ---------------------------------------------------------------------------
struct WideFinArgs {
  const uint64_t* keys;
  int n_blocks, B;
  int64_t* token;
  int64_t* rows;
  int64_t rows_sb;
  int n_rows;
  int64_t* step;
  int64_t* write_index;
  int64_t* pos;
};

// One workgroup of 16 waves, a batch row per wave: the counters it advances
// are read by every wave before any lane writes them (the barrier).
__global__ __launch_bounds__(1024) void wide_argmax_step_kernel(WideFinArgs a) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t s = a.step != nullptr ? a.step[0] : 0;
  __syncthreads();
  for (int b = w; b < a.B; b += 16) {
    const uint64_t* keys = a.keys + (int64_t)b * a.n_blocks;
    uint64_t k = 0;
    for (int j0 = lane; j0 < a.n_blocks; j0 += 8 * 64) {
      uint64_t v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = keys[min(j0 + 64 * u, a.n_blocks - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u) k = v[u] > k ? v[u] : k;
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const unsigned lo = __shfl_xor((unsigned)k, off), hi = __shfl_xor((unsigned)(k >> 32), off);
      const uint64_t o = ((uint64_t)hi << 32) | lo;
      k = o > k ? o : k;
    }
    if (lane == 0) {
      const int64_t tok = (int64_t)(0xFFFFFFFFu - (unsigned)(k & 0xFFFFFFFFu));
      a.token[b] = tok;
      if (a.rows != nullptr && s >= 0 && s < a.n_rows) a.rows[b * a.rows_sb + s] = tok;
      if (a.pos != nullptr && a.pos[b] >= 0) a.pos[b] += 1;  // a parked row stays parked
    }
  }
  if (threadIdx.x == 0) {
    if (a.write_index != nullptr) a.write_index[0] += 1;
    if (a.step != nullptr) a.step[0] = s + 1;
  }
}

}  // namespace step
}  // namespace qf

using namespace qf;
using namespace qf::step;

static bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
static bool al8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }
static bool wide_rows(int B) { return B >= 5 && B <= QF_WIDE_MAX_B; }

// Launches KERNEL<rows per wave, ...> for B rows (grid, block, st, a in scope).
#define QF_WIDE_DISPATCH(B, KERNEL, ...)                                                         \
  switch (((B) + kNW - 1) / kNW) {                                                               \
    case 2: hipLaunchKernelGGL((KERNEL<2, ##__VA_ARGS__>), grid, block, 0, st, a); break;        \
    case 3: hipLaunchKernelGGL((KERNEL<3, ##__VA_ARGS__>), grid, block, 0, st, a); break;        \
    case 4: hipLaunchKernelGGL((KERNEL<4, ##__VA_ARGS__>), grid, block, 0, st, a); break;        \
    case 5: hipLaunchKernelGGL((KERNEL<5, ##__VA_ARGS__>), grid, block, 0, st, a); break;        \
    case 6: hipLaunchKernelGGL((KERNEL<6, ##__VA_ARGS__>), grid, block, 0, st, a); break;        \
    case 7: hipLaunchKernelGGL((KERNEL<7, ##__VA_ARGS__>), grid, block, 0, st, a); break;        \
    default: hipLaunchKernelGGL((KERNEL<8, ##__VA_ARGS__>), grid, block, 0, st, a); break;       \
  }

// One row per wave up to 4 rows.  Measured on MI355X (weights past the MALL):
// at B=4 3.14 us against 4.04 for the 1..4-row form this replaced, whose
// workgroup reduced every row together and read its operands with LDS bank
// conflicts; B=2 3.13 (3.32 at both before share_tiles).
void qf::step::launch_qkv_tiles(const QkvArgs& a, bool paged, bool positions, hipStream_t st) {
  const dim3 grid((a.QH + 2 * a.KVH) * 4), block(kNT);
  if (a.B > 4) {  // positions only: the 5..32-row entry point takes no tables
    if (paged) { QF_WIDE_DISPATCH(a.B, wide_qkv_kernel, true, true) }
    else { QF_WIDE_DISPATCH(a.B, wide_qkv_kernel, false, true) }
  } else if (positions) {
    if (paged) hipLaunchKernelGGL((wide_qkv_kernel<1, true, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((wide_qkv_kernel<1, false, true>), grid, block, 0, st, a);
  } else {
    if (paged) hipLaunchKernelGGL((wide_qkv_kernel<1, true, false>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((wide_qkv_kernel<1, false, false>), grid, block, 0, st, a);
  }
}

// From 3 rows (below, re-reading the last row in the spare ones costs more than
// it saves: B=2 5.75 us against 5.46 for rms_gate_up_swiglu_mfma_kernel).
// Three row blocks per workgroup: the 608 of Qwen2.5-0.5B then take 203
// workgroups, one round of the CUs, and the rows are staged a third as often
// (MI355X, weights past the MALL, us for 1 / 2 / 3 / 4 blocks: B=12 6.50 /
// 6.64 / 5.70 / 6.30, B=32 10.5 / 11.5 / 8.4 / 9.1; with share_tiles three take
// 5.49 and 8.14).  Up to 8 rows the two-row instance: at B=4 5.21, before
// share_tiles 5.51 against 6.28 with one row per wave and 6.03 for
// rms_gate_up_swiglu_mfma_kernel (B=3 5.20, 5.51 against 5.78).
void qf::step::launch_gate_up_tiles(const GateUpArgs& a, hipStream_t st) {
  constexpr int kRB = 3;
  const dim3 grid((a.I / 8 + kRB - 1) / kRB), block(kNT);
  QF_WIDE_DISPATCH(a.B < 5 ? 5 : a.B, wide_gate_up_kernel, kRB)
}

extern "C" int qf_wide_qkv(const void* x, int64_t x_sb, const void* norm_w, float eps,
                           const void* w_qkv, const void* bias, const int64_t* pos,
                           const float* inv_freq, void* k_cache, int64_t kc_sb, int64_t kc_sh,
                           int64_t kc_sn, void* v_cache, int64_t vc_sb, int64_t vc_sh,
                           int64_t vc_sn, const int32_t* block_table, int64_t bt_sb,
                           int pages_per_row, int n_pages, int page_size, const int64_t* slots,
                           int64_t slot_sb, void* q_out, int64_t qo_sb, int64_t qo_sh, int B,
                           int hidden, int QH, int KVH, int D, int cap, void* stream) {
  if (D != kHeadDim || !wide_rows(B) || hidden < 32 || hidden > kMaxNormK || hidden % 32)
    return QF_ERR_UNSUPPORTED;
  if (!x || !norm_w || !w_qkv || !pos || !inv_freq || !k_cache || !v_cache || !slots || !q_out)
    return QF_ERR_INVALID_ARG;
  if (QH < 1 || KVH < 1 || cap < 1) return QF_ERR_INVALID_ARG;
  if (!al16(x) || !al16(norm_w) || !al16(w_qkv) || (x_sb & 7)) return QF_ERR_INVALID_ARG;
  QkvArgs a = {};
  a.x = static_cast<const f16*>(x); a.x_sb = x_sb;
  a.norm_w = static_cast<const f16*>(norm_w); a.eps = eps;
  a.w = static_cast<const f16*>(w_qkv); a.bias = static_cast<const f16*>(bias);
  a.pos = pos; a.inv_freq = inv_freq;
  a.kc = static_cast<f16*>(k_cache); a.kc_sb = kc_sb; a.kc_sh = kc_sh; a.kc_sn = kc_sn;
  a.vc = static_cast<f16*>(v_cache); a.vc_sb = vc_sb; a.vc_sh = vc_sh; a.vc_sn = vc_sn;
  a.slots = slots; a.slot_sb = slot_sb;
  a.q_out = static_cast<f16*>(q_out); a.qo_sb = qo_sb; a.qo_sh = qo_sh;
  a.B = B; a.K = hidden; a.QH = QH; a.KVH = KVH; a.cap = cap;
  a.table = block_table; a.t_sb = bt_sb; a.n_pages = n_pages;
  if (block_table != nullptr) {
    a.log2p = page_log2(page_size, pages_per_row, n_pages);
    if (a.log2p < 0) return QF_ERR_UNSUPPORTED;
    if (bt_sb < pages_per_row || cap != pages_per_row * page_size) return QF_ERR_INVALID_ARG;
  }
  launch_qkv_tiles(a, block_table != nullptr, true, static_cast<hipStream_t>(stream));
  return (int)hipGetLastError();
}

// k blocks per wave: up to 8 in one workgroup per row block; longer rows are
// split between workgroups at 5 per wave, so that 56 row blocks x 8 splits
// stream the 4864-wide down projection (MI355X, weights past the MALL, us at
// B=12 / 32: 5 blocks, 8 splits 6.73 / 7.88; 8 blocks, 5 splits 7.06 / 9.26; 4
// blocks, 10 splits 7.39 / 8.98; 13 blocks, 3 splits 7.24 / 8.94).
constexpr int kGemvBlk = 8, kSplitBlk = 5;

extern "C" int qf_wide_splits(int K) {
  if (K < 32 || K % 32) return QF_ERR_UNSUPPORTED;
  const int nkb = K / 32, per = nkb <= kNW * kGemvBlk ? kGemvBlk : kSplitBlk;
  const int splits = (nkb - 1) / (kNW * per) + 1;
  // The kernel cuts its shares at (share * nkb) / shares in 32 bits.
  if ((int64_t)kNW * splits * nkb > 0x7fffffff) return QF_ERR_UNSUPPORTED;
  return splits;
}

template <int kBlk, bool kSplit>
static void launch_gemv(const WideGemvArgs& a, hipStream_t st) {
  const dim3 grid(a.N / 16, a.splits), block(kNT);
  if (a.B <= 16) hipLaunchKernelGGL((wide_gemv_kernel<1, kBlk, kSplit>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((wide_gemv_kernel<2, kBlk, kSplit>), grid, block, 0, st, a);
}

extern "C" int qf_wide_gemv_residual(const void* inp, int64_t in_sb, const void* w, void* hidden,
                                     int64_t h_sb, float* part, int32_t* ticket, int B, int K,
                                     int N, void* stream) {
  if (!wide_rows(B) || K < 32 || K % 32 || N < 16 || N % 16) return QF_ERR_UNSUPPORTED;
  if (!inp || !w || !hidden) return QF_ERR_INVALID_ARG;
  if (!al16(inp) || !al16(w) || (in_sb & 7) || !al8(hidden) || (h_sb & 3)) return QF_ERR_INVALID_ARG;
  const int splits = qf_wide_splits(K);
  if (splits < 0) return splits;
  if (splits > 1 && (!part || !ticket || !al16(part))) return QF_ERR_INVALID_ARG;
  WideGemvArgs a;
  a.inp = static_cast<const f16*>(inp); a.in_sb = in_sb;
  a.w = static_cast<const f16*>(w);
  a.hidden = static_cast<f16*>(hidden); a.h_sb = h_sb;
  a.part = part; a.ticket = ticket;
  a.B = B; a.K = K; a.N = N; a.splits = splits;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // A wave loads kBlk blocks whatever its share is, so o_proj's 28 take the
  // 7-block form (3.82 us at B=12 against 4.05 with 8).
  const int per = (K / 32 + kNW * splits - 1) / (kNW * splits);
  if (splits > 1) launch_gemv<kSplitBlk, true>(a, st);
  else if (per <= 7) launch_gemv<7, false>(a, st);
  else launch_gemv<kGemvBlk, false>(a, st);
  return (int)hipGetLastError();
}

extern "C" int qf_wide_gate_up(const void* x, int64_t x_sb, const void* norm_w, float eps,
                               const void* w_gate_up, void* h_out, int64_t ho_sb, int B, int hidden,
                               int I, void* stream) {
  if (!wide_rows(B) || hidden < 32 || hidden > kMaxNormK || hidden % 32 || I < 8 || I % 8)
    return QF_ERR_UNSUPPORTED;
  if (!x || !norm_w || !w_gate_up || !h_out) return QF_ERR_INVALID_ARG;
  if (!al16(x) || !al16(norm_w) || !al16(w_gate_up) || (x_sb & 7)) return QF_ERR_INVALID_ARG;
  GateUpArgs a;
  a.x = static_cast<const f16*>(x); a.x_sb = x_sb;
  a.norm_w = static_cast<const f16*>(norm_w); a.eps = eps;
  a.w = static_cast<const f16*>(w_gate_up);
  a.h = static_cast<f16*>(h_out); a.h_sb = ho_sb;
  a.B = B; a.K = hidden; a.I = I;
  launch_gate_up_tiles(a, static_cast<hipStream_t>(stream));
  return (int)hipGetLastError();
}

extern "C" int qf_wide_lm_head(const void* x, int64_t x_sb, const void* norm_w, float eps,
                               const void* w_lm, void* logits, int64_t lg_sb, uint64_t* keys,
                               int n_blocks, int B, int hidden, int V, void* stream) {
  if (!wide_rows(B) || hidden < 32 || hidden > kMaxNormK || hidden % 32 || V < 16 || V % 16)
    return QF_ERR_UNSUPPORTED;
  if (!x || !norm_w || !w_lm || !logits || !keys) return QF_ERR_INVALID_ARG;
  if (n_blocks < 1 || n_blocks > 65535) return QF_ERR_INVALID_ARG;
  if (!al16(x) || !al16(norm_w) || !al16(w_lm) || (x_sb & 7)) return QF_ERR_INVALID_ARG;
  if (!al8(logits) || (lg_sb & 3)) return QF_ERR_INVALID_ARG;
  WideLmArgs a;
  a.x = static_cast<const f16*>(x); a.x_sb = x_sb;
  a.norm_w = static_cast<const f16*>(norm_w); a.eps = eps;
  a.w = static_cast<const f16*>(w_lm);
  a.logits = static_cast<f16*>(logits); a.lg_sb = lg_sb;
  a.keys = keys;
  a.B = B; a.K = hidden; a.V = V;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid(n_blocks), block(kNT);
  QF_WIDE_DISPATCH(B, wide_lm_head_kernel)
  return (int)hipGetLastError();
}

extern "C" int qf_wide_argmax_step(const uint64_t* keys, int n_blocks, int B, int64_t* token,
                                   int64_t* rows, int64_t rows_sb, int n_rows, int64_t* step,
                                   int64_t* write_index, int64_t* pos, void* stream) {
  if (!wide_rows(B)) return QF_ERR_UNSUPPORTED;
  if (!keys || !token || n_blocks < 1) return QF_ERR_INVALID_ARG;
  if (rows != nullptr && step == nullptr) return QF_ERR_INVALID_ARG;
  WideFinArgs a;
  a.keys = keys; a.n_blocks = n_blocks; a.B = B;
  a.token = token; a.rows = rows; a.rows_sb = rows_sb; a.n_rows = n_rows;
  a.step = step; a.write_index = write_index; a.pos = pos;
  hipLaunchKernelGGL(wide_argmax_step_kernel, dim3(1), dim3(1024), 0,
                     static_cast<hipStream_t>(stream), a);
  return (int)hipGetLastError();
}
