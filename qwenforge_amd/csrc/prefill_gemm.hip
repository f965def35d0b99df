// Prompt projections of the cached prefill (student_engine.py:679-737) on
// gfx950: hand-written MFMA GEMMs with the step around each projection in
// their epilogues, and one native call that enqueues every layer.
//
// Y (tokens x features) = X (tokens x K) . W (features x K)^T, fp16 in, fp32
// sums.  The weight rows are the A operand and the tokens the columns of
// v_mfma_f32_16x16x32_f16, so a lane ends with four consecutive features of
// one token per tile, and a rotate-half pair (d, d + 32) or a gate/up pair
// sits in one lane: bias + RoPE + cache append (QKV), residual add (o_proj,
// down) and SwiGLU (gate/up) need no pass of their own.
//
// Both operands go HBM/L2 -> LDS by direct-to-LDS loads (16 bytes a lane),
// kStages deep: a stage's loads are issued kStages - 1 stages ahead and
// waited for with a counted vmcnt, one barrier per stage.  LDS rows hold kBK
// halves; chunk c of row r lives at c ^ f(r) (applied to the global address of
// the load, since the DMA writes LDS in lane order), which puts the 16 rows of
// an operand read on 16 distinct 16-byte bank groups.
#include <algorithm>
#include <type_traits>

#include "step_common.h"
#include "../../include/qf_prefill.h"

namespace qf {
namespace pgemm {

using step::rope1;
using step::wave_sum;

typedef __attribute__((address_space(3))) void lds_void;

// kEpiPartial: fp32 sums of one k share of a residual product, for
// prefill_rms_kernel to add up.
enum Epilogue { kEpiQkv = 0, kEpiResidual = 1, kEpiSwiglu = 2, kEpiPartial = 3 };

struct GemmArgs {
  const f16* x;     // (T, K), row stride x_sn
  int64_t x_sn;
  const f16* w;     // (N, K) row-major, contiguous
  f16* y;           // qkv (T, N) / hidden (T, N) in place / h (T, N / 2)
  int64_t y_sn;
  int T, N, K;
  int n_ft, n_tt;   // feature and token tiles
  int xt;           // XCD rectangles along the tokens: 1, 2, 4 or 8
  // QKV epilogue
  const f16* bias;
  const f16* cs;    // (T, 64): cos of the 32 frequencies, then sin
  const int2* info; // per token: cache row or page (-1: append nothing), slot within it
  f16* kc;
  int64_t kc_sb, kc_sh, kc_sn;
  f16* vc;
  int64_t vc_sb, vc_sh, vc_sn;
  int QH, KVH;
  // split k (partial epilogue): (splits, T, N) sums
  int splits;
  float* part;
};

// 16 bytes per lane from byte `off` of the resource to LDS byte `dst` + 16 *
// lane, as inline asm: the compiler would wait for every such load in flight
// (vmcnt(0)) before any LDS read it can see, since it cannot tell one stage
// from another.  The load writes no register; the counted waits at the
// barriers (stage_barrier) order it before the reads of its stage.
__device__ __forceinline__ void load_lds(u32x4 rsrc, unsigned dst, int off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :
               : "s"(dst), "v"(off), "s"(rsrc)
               : "memory", "m0");
}

// Buffer resource words over `bytes` bytes at `base` (wave-uniform).
__device__ __forceinline__ u32x4 rsrc_words(const void* base, int64_t bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  return u32x4{(unsigned)p, (unsigned)(p >> 32) & 0xFFFFu,
               (unsigned)(bytes < 0x7fffffff ? bytes : 0x7fffffff), 0x00020000u};
}

// This wave's LDS reads are done and all but its newest kLoads loads have
// landed; after the barrier that holds for every wave.
template <int kLoads>
__device__ __forceinline__ void stage_barrier() {
  static_assert(kLoads >= 0 && kLoads < 64, "vmcnt is six bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "i"(kLoads) : "memory");
}

// 16-row blocks that a lane needs together: QKV a whole head (rotate-half
// pairs), SwiGLU a gate block and its up block.
constexpr int group_blocks(int epi) { return epi == kEpiQkv ? 4 : (epi == kEpiSwiglu ? 2 : 1); }

// exp(-g) of an fp16 g as 2^k 2^a: hi holds 11 bits of log2(e), so hi * g is
// exact, and the reduced argument a carries the rest.  With it and the hardware
// reciprocal (1 ulp) silu rounds all 65536 fp16 gates as F.silu's expf and
// division do; exp2 of the once-rounded -g log2(e) was off on one more gate.
// expf itself costs the prefill of 1024 tokens 24 us of 2201, this 7.
__device__ __forceinline__ float exp_neg16(float g) {
  constexpr float hi = 1.4423828125f, lo = (float)(1.4426950408889634074 - 1.4423828125);
  const float p = __builtin_amdgcn_fmed3f(-hi * g, -150.f, 126.f), k = rintf(p);
  return __builtin_amdgcn_ldexpf(fast_exp2(__builtin_fmaf(-lo, g, p - k)), (int)k);
}

// Outputs of token t in the group whose first weight row (SwiGLU: of the
// interleaved gate and up rows) is f0: acc[f][i] is row f0 + 16 f + 4 q + i.
template <int kEpi>
__device__ __forceinline__ void finish(const GemmArgs& a, int f0, int t, int q,
                                       const f32x4 (&acc)[group_blocks(kEpi)]) {
  if (f0 >= a.N) return;
  if constexpr (kEpi == kEpiPartial) {
    *reinterpret_cast<f32x4*>(a.part + ((int64_t)blockIdx.y * a.T + t) * a.N + f0 + 4 * q) = acc[0];
  } else if constexpr (kEpi == kEpiResidual) {
    f16* y = a.y + t * a.y_sn + f0 + 4 * q;
    const f16x4 res = *reinterpret_cast<const f16x4*>(y);
    f16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (f16)((float)res[i] + (float)(f16)acc[0][i]);
    *reinterpret_cast<f16x4*>(y) = o;
  } else if constexpr (kEpi == kEpiSwiglu) {
    f16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // F.silu on the fp16 gate (fp32 math, one rounding), then the fp16
      // product; equal to F.silu's bits for every fp16 gate.
      const float g16 = (float)(f16)acc[0][i], u16 = (float)(f16)acc[1][i];
      const float s16 = (float)(f16)(g16 * __builtin_amdgcn_rcpf(1.f + exp_neg16(g16)));
      o[i] = (f16)(s16 * u16);
    }
    *reinterpret_cast<f16x4*>(a.y + t * a.y_sn + f0 / 2 + 4 * q) = o;
  } else {
    const int head = f0 >> 6;
    f16x4 o[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      f16x4 bias = {(f16)0.f, (f16)0.f, (f16)0.f, (f16)0.f};
      if (a.bias != nullptr) bias = *reinterpret_cast<const f16x4*>(a.bias + f0 + 16 * f + 4 * q);
#pragma unroll
      for (int i = 0; i < 4; ++i) o[f][i] = (f16)(acc[f][i] + (float)bias[i]);
    }
    if (head < a.QH + a.KVH) {
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const f16x4 c = *reinterpret_cast<const f16x4*>(a.cs + 64 * t + 16 * f + 4 * q);
        const f16x4 s = *reinterpret_cast<const f16x4*>(a.cs + 64 * t + 32 + 16 * f + 4 * q);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f16 lo, hi;
          rope1((float)o[f][i], (float)o[f + 2][i], (float)c[i], (float)s[i], (float)c[i],
                (float)s[i], lo, hi);
          o[f][i] = lo;
          o[f + 2][i] = hi;
        }
      }
    }
    f16* y = a.y + t * a.y_sn + f0 + 4 * q;
#pragma unroll
    for (int f = 0; f < 4; ++f) *reinterpret_cast<f16x4*>(y + 16 * f) = o[f];
    if (head >= a.QH) {
      const int2 at = a.info[t];
      if (at.x >= 0) {
        f16* dst = head < a.QH + a.KVH
                       ? a.kc + at.x * a.kc_sb + at.y * a.kc_sn + (head - a.QH) * a.kc_sh
                       : a.vc + at.x * a.vc_sb + at.y * a.vc_sn + (head - a.QH - a.KVH) * a.vc_sh;
#pragma unroll
        for (int f = 0; f < 4; ++f)
          *reinterpret_cast<f16x4*>(dst + 16 * f + 4 * q) = o[f];
      }
    }
  }
}

// kWN x kWM waves, each kFW x kTW blocks of 16 features x 16 tokens, times kWK
// waves that split the k of a stage; kBK of k per stage.
template <int kFW, int kTW, int kWN, int kWM, int kWK, int kBK, int kStages, int kEpi>
__global__ __launch_bounds__(kWN* kWM* kWK * 64, 1) void prefill_gemm_kernel(GemmArgs a) {
  constexpr int kBN = 16 * kFW * kWN, kBM = 16 * kTW * kWM;
  constexpr int M = kFW * kTW;                       // MFMAs per k block
  constexpr int NW = kWN * kWM * kWK;
  constexpr int CPR = kBK / 8;                       // 16-byte chunks per LDS row
  constexpr int kStageBytes = (kBN + kBM) * kBK * 2;
  constexpr int LPW = kStageBytes / 1024 / NW;       // loads per wave and stage
  constexpr int LW = kBN * kBK * 2 / 1024 / NW;      // of them, weight rows
  constexpr int KB = kBK / 32 / kWK;                 // k blocks per wave and stage
  static_assert(LPW <= M && kFW % group_blocks(kEpi) == 0, "a load per MFMA at most; whole groups");
  static_assert(LPW * NW * 1024 == kStageBytes && LW * NW * 1024 == kBN * kBK * 2, "even loads");
  constexpr int kRedBytes = kWK > 1 ? NW * M * 1024 : 0;
  constexpr int kLds = kStages * kStageBytes > kRedBytes ? kStages * kStageBytes : kRedBytes;
  __shared__ __attribute__((aligned(16))) unsigned char lds[kLds];

  // Workgroup i runs on XCD i % 8: each XCD takes one of a.xt x (8 / a.xt)
  // rectangles of tiles, tokens fastest (see launch_as).
  const int xcd = (int)(blockIdx.x & 7), idx = (int)(blockIdx.x >> 3), xf = 8 / a.xt;
  const int xi = xcd % a.xt, xj = xcd / a.xt;
  const int t0 = a.n_tt * xi / a.xt, tn = a.n_tt * (xi + 1) / a.xt - t0;
  const int g0 = a.n_ft * xj / xf, gn = a.n_ft * (xj + 1) / xf - g0;
  if (idx >= tn * gn) return;
  const int tt = t0 + idx % tn, ft = g0 + idx / tn, lin = ft * a.n_tt + tt;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = lane >> 4, r16 = lane & 15;
  const int K = a.K;
  const int tok0 = tt * kBM;

  // Stages of this workgroup's k range.
  int s_lo = 0, s_n = K / kBK;
  if (kEpi == kEpiPartial) {
    const int all = K / kBK;
    s_lo = (int)blockIdx.y * all / a.splits;
    s_n = ((int)blockIdx.y + 1) * all / a.splits - s_lo;
  }

  // Byte offsets of this lane's loads from the stage's first k (0x7ffffff0:
  // past the operand, reads as zero).
  int off[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const bool is_w = i < LW;
    const int c = ((is_w ? i : i - LW) * NW + wv) * 64 + lane;
    const int row = c / CPR, chunk = (c % CPR) ^ (((row & 15) * CPR / 16) & (CPR - 1));
    if (is_w) {
      int wr;
      bool ok;
      if (kEpi == kEpiSwiglu) {
        const int blk = row >> 4, j = ft * (kBN / 2) + 16 * (blk >> 1) + (row & 15);
        ok = j < a.N / 2;
        wr = (blk & 1) ? a.N / 2 + j : j;
      } else {
        wr = ft * kBN + row;
        ok = wr < a.N;
      }
      off[i] = ok ? (wr * K + 8 * chunk) * 2 : 0x7ffffff0;
    } else {
      off[i] = tok0 + row < a.T ? (int)(row * a.x_sn + 8 * chunk) * 2 : 0x7ffffff0;
    }
  }
  const f16* xt = a.x + (int64_t)tok0 * a.x_sn;
  const int64_t x_bytes = ((int64_t)(min(kBM, a.T - tok0) - 1) * a.x_sn + K) * 2;
  const int64_t w_bytes = (int64_t)a.N * K * 2;
  const unsigned lds0 = (unsigned)(uintptr_t)(const lds_void*)lds;
  // Loads of stage s (relative); a stage past the range reads nothing (an
  // empty resource), so every stage issues the same number of loads.
  u32x4 rw, rx;
  unsigned st = 0;
  const auto aim = [&](int s, unsigned slot) {
    const bool in = s < s_n;
    const int64_t k0 = (int64_t)(s_lo + (in ? s : 0)) * kBK * 2;
    rw = rsrc_words(reinterpret_cast<const unsigned char*>(a.w) + k0, in ? w_bytes - k0 : 0);
    rx = rsrc_words(reinterpret_cast<const unsigned char*>(xt) + k0, in ? x_bytes - k0 : 0);
    st = lds0 + slot + wv * 1024;
  };
  const auto load = [&](int i) {
    if (i < LW) load_lds(rw, st + i * NW * 1024, off[i]);
    else load_lds(rx, st + kBN * kBK * 2 + (i - LW) * NW * 1024, off[i]);
  };
#pragma unroll
  for (int s = 0; s < kStages; ++s) {
    aim(s, s * kStageBytes);
#pragma unroll
    for (int i = 0; i < LPW; ++i) load(i);
  }

  const int wk = wv % kWK, wm = (wv / kWK) % kWM, wn = wv / (kWK * kWM);
  // Operand reads of k block kb (of this wave's KB): rows 16 f + r16.
  int ra[KB], rb[KB];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int chunk = (4 * (wk * KB + kb) + q) ^ ((r16 * CPR / 16) & (CPR - 1));
    ra[kb] = (16 * kFW * wn + r16) * kBK * 2 + 16 * chunk;
    rb[kb] = kBN * kBK * 2 + (16 * kTW * wm + r16) * kBK * 2 + 16 * chunk;
  }
  const auto read = [&](unsigned slot, int kb, f16x8 (&av)[kFW], f16x8 (&bv)[kTW]) {
#pragma unroll
    for (int f = 0; f < kFW; ++f)
      av[f] = *reinterpret_cast<const f16x8*>(lds + slot + ra[kb] + f * 16 * kBK * 2);
#pragma unroll
    for (int t = 0; t < kTW; ++t)
      bv[t] = *reinterpret_cast<const f16x8*>(lds + slot + rb[kb] + t * 16 * kBK * 2);
  };
  f32x4 acc[kFW][kTW];
#pragma unroll
  for (int f = 0; f < kFW; ++f)
#pragma unroll
    for (int t = 0; t < kTW; ++t) acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // The operands of the next k block are read while the current one's MFMAs
  // run.  Before the first read of stage s + 1: that stage has landed, and
  // every wave has read all of stage s, whose slot takes stage s + kStages.
  f16x8 av[2][kFW], bv[2][kTW];
  stage_barrier<LPW*(kStages - 1)>();
  read(0, 0, av[0], bv[0]);
  unsigned slot = 0;
  const auto stage = [&](int s, auto parity) {  // parity: the set its first operands are in
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      constexpr int P = decltype(parity)::value;
      const int cur = (P + kb) & 1, nxt = cur ^ 1;
      if (kb + 1 < KB) {
        read(slot, kb + 1, av[nxt], bv[nxt]);
      } else {
        stage_barrier<LPW*(kStages - 2)>();
        aim(s + kStages, slot);
        slot = slot + kStageBytes == kStages * kStageBytes ? 0 : slot + kStageBytes;
        read(slot, 0, av[nxt], bv[nxt]);  // past the last stage: stale LDS, never used
      }
      // The loads go out between the MFMAs: issuing one holds its wave until
      // the address path has taken it, so a burst of them behind the barrier
      // kept the matrix core idle for the whole burst.
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const int li = (m * LPW + M - 1) / M;
        if (kb + 1 == KB && li < LPW && li * M / LPW == m) {
          load(li);
          __builtin_amdgcn_sched_barrier(0);
        }
        const int f = m / kTW, t = m % kTW;
        acc[f][t] = mfma16x16x32(av[cur][f], bv[cur][t], acc[f][t]);
        if (kb + 1 == KB) __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  int s = 0;
  for (; s + 2 <= s_n; s += 2) {
    stage(s, std::integral_constant<int, 0>{});
    stage(s + 1, std::integral_constant<int, KB & 1>{});
  }
  if (s < s_n) stage(s, std::integral_constant<int, 0>{});
  stage_barrier<0>();

  const int f0 = ft * kBN + 16 * kFW * wn;
  constexpr int GB = group_blocks(kEpi);
  if constexpr (kWK == 1) {
#pragma unroll
    for (int t = 0; t < kTW; ++t) {
      const int tok = tok0 + 16 * (kTW * wm + t) + r16;
#pragma unroll
      for (int f = 0; f < kFW; f += GB) {
        f32x4 g[GB];
#pragma unroll
        for (int u = 0; u < GB; ++u) g[u] = acc[f + u][t];
        if (tok < a.T) finish<kEpi>(a, f0 + 16 * f, tok, q, g);
      }
    }
  } else {
    // The k shares of a tile meet in LDS (free once every load and read of the
    // loop is done); wave wk finishes the tokens of its column block.
    static_assert(kWN == 1 && kWM == 1 && kWK == kTW, "one column block per k share");
    f32x4* red = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int f = 0; f < kFW; ++f)
#pragma unroll
      for (int t = 0; t < kTW; ++t) red[((wv * kTW + t) * kFW + f) * 64 + lane] = acc[f][t];
    __syncthreads();
    f32x4 g[kFW];
#pragma unroll
    for (int f = 0; f < kFW; ++f) {
      g[f] = red[(wk * kFW + f) * 64 + lane];
#pragma unroll
      for (int s = 1; s < kWK; ++s) g[f] += red[((s * kTW + wk) * kFW + f) * 64 + lane];
    }
    const int tok = tok0 + 16 * wk + r16;
#pragma unroll
    for (int f = 0; f < kFW; f += GB) {
      f32x4 o[GB];
#pragma unroll
      for (int u = 0; u < GB; ++u) o[u] = g[f + u];
      if (tok < a.T) finish<kEpi>(a, f0 + 16 * f, tok, q, o);
    }
  }
}

// rms_norm of T rows, a row per wave: fp16((x * rsqrt(mean(x^2) + eps)) * w).
// kParts: first x <- fp16(x + fp16(sum of the row's `splits` partials)), in
// place and in split order, so a repeat gives the same bits; w == nullptr then
// ends there.  The whole chip adds the partials up while it would have waited
// for this row's load anyway; the last workgroup of a tile reading them back
// (write-through stores, a ticket) was alone with them.
constexpr int kMaxChunks = 4;  // 16-byte chunks per lane: hidden <= 2048

template <bool kParts>
__global__ __launch_bounds__(256) void prefill_rms_kernel(f16* x, const f16* __restrict__ w, f16* y,
                                                          const float* __restrict__ part, int splits,
                                                          int T, int K, float eps) {
  const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  const int C = K / 8;
  f16x8 v[kMaxChunks], g[kMaxChunks];
#pragma unroll
  for (int i = 0; i < kMaxChunks; ++i)
    if (64 * i < C) {
      const int c = min(64 * i + lane, C - 1);
      v[i] = load16(x + (int64_t)t * K + 8 * c);
      if (!kParts || w != nullptr) g[i] = load16(w + 8 * c);
    }
  if constexpr (kParts) {
    f32x4 sum[kMaxChunks][2];
#pragma unroll
    for (int i = 0; i < kMaxChunks; ++i) sum[i][0] = sum[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < splits; s += 4) {
      f32x4 p[4][kMaxChunks][2];  // a batch of loads in flight together
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float* row = part + ((int64_t)(s + u) * T + t) * K;
#pragma unroll
        for (int i = 0; i < kMaxChunks; ++i) {
          p[u][i][0] = p[u][i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (64 * i < C && s + u < splits) {
            const float* src = row + 8 * min(64 * i + lane, C - 1);
            p[u][i][0] = *reinterpret_cast<const f32x4*>(src);
            p[u][i][1] = *reinterpret_cast<const f32x4*>(src + 4);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < kMaxChunks; ++i) {
          sum[i][0] += p[u][i][0];
          sum[i][1] += p[u][i][1];
        }
    }
#pragma unroll
    for (int i = 0; i < kMaxChunks; ++i)
      if (64 * i + lane < C) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = (f16)((float)v[i][e] + (float)(f16)sum[i][e >> 2][e & 3]);
        store16(x + (int64_t)t * K + 8 * (64 * i + lane), v[i]);
      }
    if (w == nullptr) return;
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < kMaxChunks; ++i)
    if (64 * i + lane < C) {
      float p = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) p += (float)v[i][e] * (float)v[i][e];
      s += p;
    }
  const float rstd = rsqrtf(wave_sum(s) / (float)K + eps);
#pragma unroll
  for (int i = 0; i < kMaxChunks; ++i)
    if (64 * i + lane < C) {
      f16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = (f16)(((float)v[i][e] * rstd) * (float)g[i][e]);
      store16(y + (int64_t)t * K + 8 * (64 * i + lane), o);
    }
}

// Per token of the packed rows: the fp16 RoPE table of its position (the same
// values as the torch table, student_engine.py:910-915) and where it is
// appended.  cu == nullptr: rows of S tokens; else rows of at most S, a token
// past them appending nothing.  One wave per two tokens.
__global__ __launch_bounds__(256) void prefill_tokens_kernel(const int* cu, int B, int S, int T,
                                                             const float* inv_freq,
                                                             const int32_t* table, int64_t t_sb,
                                                             int log2p, int ppr, int n_pages,
                                                             f16* cs, int2* info) {
  const int t = blockIdx.x * 8 + (threadIdx.x >> 5), i = threadIdx.x & 31;
  if (t >= T) return;
  int b, pos;
  if (cu != nullptr) {
    int lo = 0, hi = B;  // the last row that starts at or before t
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (cu[mid] <= t) lo = mid;
      else hi = mid;
    }
    b = lo;
    pos = t - cu[b];
  } else {
    b = t / S;
    pos = t - b * S;
  }
  const float ang = (float)pos * inv_freq[i];
  cs[64 * t + i] = (f16)cosf(ang);
  cs[64 * t + 32 + i] = (f16)sinf(ang);
  if (i == 0) {
    int2 at = make_int2(pos < S ? b : -1, pos);
    if (table != nullptr) {
      const int lp = pos >> log2p;
      const int page = pos < S && lp < ppr ? table[b * t_sb + lp] : -1;
      at = make_int2(page >= 0 && page < n_pages ? page : -1, pos & ((1 << log2p) - 1));
    }
    info[t] = at;
  }
}

// ---------------------------------------------------------------------------
static bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Every XCD fetches the tokens and the weight rows of its rectangle of tiles
// into its own L2, X / xt + W / (8 / xt) bytes: of the splits that leave no XCD
// more than an even share of the tiles (rounded up), the one with the fewest.
// (One strip of features per XCD made all eight read every token: 90 MB for
// down_proj at 1024 tokens, where 4 x 2 rectangles read 55.)
static int xcd_split(int n_ft, int n_tt, int64_t x_bytes, int64_t w_bytes, int& largest) {
  int best = 0;
  int64_t best_bytes = 0;
  for (int pass = 0; pass < 2 && best == 0; ++pass)
    for (int xt = 1; xt <= 8; xt *= 2) {
      const int xf = 8 / xt;
      const int most = ((n_tt + xt - 1) / xt) * ((n_ft + xf - 1) / xf);
      const int64_t bytes = x_bytes / xt + w_bytes / xf;
      // No split may be even (few tiles): then the one with the least to do.
      const int64_t rank = pass == 0 ? bytes : most;
      if (pass == 0 && most > (n_ft * n_tt + 7) / 8) continue;
      if (best == 0 || rank < best_bytes) {
        best = xt;
        best_bytes = rank;
        largest = most;
      }
    }
  return best;
}

template <int kFW, int kTW, int kWN, int kWM, int kWK, int kBK, int kStages, int kEpi>
static int launch_as(GemmArgs a, hipStream_t st) {
  constexpr int kBN = 16 * kFW * kWN, kBM = 16 * kTW * kWM;
  a.n_ft = (a.N + kBN - 1) / kBN;
  a.n_tt = (a.T + kBM - 1) / kBM;
  int largest = 0;
  a.xt = xcd_split(a.n_ft, a.n_tt, (int64_t)a.T * a.K * 2, (int64_t)a.N * a.K * 2, largest);
  const dim3 grid((unsigned)largest * 8u, (unsigned)a.splits);
  hipLaunchKernelGGL((prefill_gemm_kernel<kFW, kTW, kWN, kWM, kWK, kBK, kStages, kEpi>), grid,
                     dim3(kWN * kWM * kWK * 64), 0, st, a);
  return (int)hipGetLastError();
}

// Tile sizes, by how many tiles the product has on `cus` compute units
// (MI355X, weights past the MALL, us):
//   - 128 x 128, half the operand bytes per product of 64 x 64, from nine
//     tiles per 16 CUs on for gate/up (152 tiles at 256 tokens: 13.8 against
//     16.1; 608 at 1024: 28.7 against 40.1) and from thirteen for the others
//     (kernel trace, 128 / 64: QKV at 2560 tokens, 180 tiles, 22.2 / 21.8, 3072,
//     216, 22.1 / 23.4, 4096, 288, 26.2 / 32.5; o_proj at 2048, 112, 18.6 /
//     12.9, 2560, 140, 19.4 / 17.3, 4096, 224, 19.0 / 22.0 -- and ahead by 2 at
//     3072 and 3584 already, 168 and 196 tiles, where QKV is not);
//   - gate/up 160 features wide from two tiles per CU on: its 9728 rows then
//     fill whole rounds of workgroups (two per CU) at 1024 x n tokens (28.2
//     against 28.7, at 4096 81.7 against 88.4, at 8192 160 against 199);
//   - below that 64 x 64, each stage's k split over the four waves (o_proj at
//     1024 tokens, 224 tiles: 7.9 against 15.5), three stages deep with one
//     workgroup per CU, two stages and two workgroups once there are more
//     tiles than CUs (QKV at 1024 tokens, 288 tiles: 10.9 against 13.5).
// hipBLASLt beside them (without the epilogues' work): gate/up 30 / 85 / 154
// at 1024 / 4096 / 8192 tokens, down 21 / 44 / 78, o_proj 8.7 at 1024.
template <int kEpi>
static int launch(const GemmArgs& a, int cus, hipStream_t st) {
  const int64_t t128 = (int64_t)((a.N + 127) / 128) * ((a.T + 127) / 128);
  const int64_t t64 = (int64_t)((a.N + 63) / 64) * ((a.T + 63) / 64);
  if (t128 * 16 >= (kEpi == kEpiSwiglu ? 9 : 13) * (int64_t)cus) {
    if constexpr (kEpi == kEpiSwiglu)
      if (t128 >= 2 * (int64_t)cus) return launch_as<10, 2, 1, 4, 1, 64, 2, kEpi>(a, st);
    return launch_as<4, 4, 2, 2, 1, 64, 2, kEpi>(a, st);
  }
  if (t64 <= cus) return launch_as<4, 4, 1, 1, 4, 128, 3, kEpi>(a, st);
  return launch_as<4, 4, 1, 1, 4, 128, 2, kEpi>(a, st);
}

// The down projection's k split over workgroups whose partial sums the next
// rms_norm adds up.
struct KSplit {
  int splits;  // 1: not split
  int form;    // 0: 64 x 64 tiles, 1: 128 x 128 and one workgroup per CU, 2: 128 x 128 and two
};

// 64 x 64 tiles: as many shares as the CUs hold at one workgroup each, at most
// eight and none under four stages of 128.
static int shares64(int T, int N, int K, int cus) {
  const int tiles = (N + 63) / 64 * ((T + 63) / 64);
  return std::max(1, std::min({cus / tiles, 8, K / 128 / 4}));
}

// 128 x 128 tiles: as many shares as the fullest XCD's tiles leave room for in
// one round of workgroups (of more, the last ones wait for a whole share: 42
// tiles in 6 shares are 36 workgroups on an XCD's 32 CUs, 2027 us against 1815
// in 5), none under eight stages of 64.
static int shares128(int T, int N, int K, int slots) {
  int most = 0;
  xcd_split((N + 127) / 128, (T + 127) / 128, (int64_t)T * K * 2, (int64_t)N * K * 2, most);
  return std::max(1, std::min({slots / 8 / most, 8, K / 64 / 8}));
}

// Up to one 64 x 64 tile per two CUs the small tiles; then 128 x 128, four
// stages deep with a CU to itself while that allows two shares, two stages and
// two workgroups per CU past that.  Measured on MI355X for the whole prefill of
// 24 layers, us, unsplit or in 64 x 64 shares merged behind a ticket / this
// rule: 64 tokens 1242 / 1206, 300 1522 / 1496, 512 1771 / 1755; 600 1832 /
// 1749, 1024 2312 / 2224, 1280 2947 / 2720, 2048 3744 / 3404; 2400 4653 / 4176,
// 3000 5243 / 4500, 4096 6325 / 6005.  Across the first line: seven 128 x 128
// shares at 512 tokens 1785, three 64 x 64 ones at 600 1771.
static KSplit k_split(int T, int N, int K, int cus) {
  const int64_t t64 = (int64_t)((N + 63) / 64) * ((T + 63) / 64);
  if (t64 * 2 <= cus) return {shares64(T, N, K, cus), 0};
  const int one = shares128(T, N, K, cus);
  if (one > 1) return {one, 1};
  return {shares128(T, N, K, 2 * cus), 2};
}

static int launch_split(const GemmArgs& a, int form, hipStream_t st) {
  if (form == 0) return launch_as<4, 4, 1, 1, 4, 128, 3, kEpiPartial>(a, st);
  if (form == 1) return launch_as<4, 4, 2, 2, 1, 64, 4, kEpiPartial>(a, st);
  return launch_as<4, 4, 2, 2, 1, 64, 2, kEpiPartial>(a, st);
}

}  // namespace pgemm
}  // namespace qf

using namespace qf;
using namespace qf::pgemm;

namespace {

constexpr int kMaxCus = 256;

struct Workspace {
  int64_t x, qkv, att, h, cs, info, part, bytes;
};

// For a whole part's CUs: each form's shares only grow with the CU count, but
// fewer CUs may take another form, so the partials hold the most of them.
Workspace workspace(int T, int H, int QH, int KVH, int I) {
  Workspace w;
  int64_t at = 0;
  const auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  };
  w.x = take((int64_t)T * H * 2);
  w.qkv = take((int64_t)T * (QH + 2 * KVH) * 64 * 2);
  w.att = take((int64_t)T * QH * 64 * 2);
  w.h = take((int64_t)T * I * 2);
  w.cs = take((int64_t)T * 64 * 2);
  w.info = take((int64_t)T * 8);
  const int most = std::max(shares64(T, H, I, kMaxCus), shares128(T, H, I, 2 * kMaxCus));
  w.part = take(most > 1 ? (int64_t)most * T * H * 4 : 0);
  w.bytes = at;
  return w;
}

bool shapes_ok(int T, int H, int QH, int KVH, int D, int I) {
  const int64_t lim = 0x7ffffff0;
  return T >= 1 && D == 64 && QH >= 1 && KVH >= 1 && QH % KVH == 0 && H >= 128 && H % 128 == 0 &&
         H <= 64 * 8 * kMaxChunks && (QH * 64) % 128 == 0 && I >= 128 && I % 128 == 0 &&
         (int64_t)2 * I * H * 2 < lim && (int64_t)(QH + 2 * KVH) * 64 * H * 2 < lim &&
         (int64_t)T * (I > 2 * H ? I : 2 * H) < lim;
}

}  // namespace

extern "C" int64_t qf_prefill_layers_workspace(int T, int hidden, int QH, int KVH, int D, int I) {
  if (!shapes_ok(T, hidden, QH, KVH, D, I)) return QF_ERR_UNSUPPORTED;
  return workspace(T, hidden, QH, KVH, I).bytes;
}

extern "C" int qf_prefill_layers(const QfPrefillLayer* layers, int n_layers, void* hidden_p, int T,
                                 int B, int S, const int32_t* cu, const float* inv_freq,
                                 const int32_t* block_table, int64_t bt_sb, int pages_per_row,
                                 int n_pages, int page_size, void* ws, int64_t ws_bytes, float eps,
                                 int H, int QH, int KVH, int D, int I, void* stream) {
  if (!shapes_ok(T, H, QH, KVH, D, I)) return QF_ERR_UNSUPPORTED;
  if (!layers || n_layers < 1 || !hidden_p || !inv_freq || !ws || B < 1 || S < 1)
    return QF_ERR_INVALID_ARG;
  if (cu == nullptr && (int64_t)B * S != T) return QF_ERR_INVALID_ARG;
  if (!al16(hidden_p) || !al16(ws)) return QF_ERR_INVALID_ARG;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int found = stream_cus(st), cus = found > 0 && found < kMaxCus ? found : kMaxCus;
  const Workspace w = workspace(T, H, QH, KVH, I);
  if (ws_bytes < w.bytes) return QF_ERR_SCRATCH_LIMIT;
  int l2 = 0;
  if (block_table != nullptr) {
    l2 = page_log2(page_size, pages_per_row, n_pages);
    if (l2 < 0) return QF_ERR_UNSUPPORTED;
    if (bt_sb < pages_per_row) return QF_ERR_INVALID_ARG;
  }
  for (int i = 0; i < n_layers; ++i) {
    const QfPrefillLayer& y = layers[i];
    if (!y.norm1 || !y.w_qkv || !y.w_o || !y.norm2 || !y.w_gate_up || !y.w_down || !y.k_cache ||
        !y.v_cache)
      return QF_ERR_INVALID_ARG;
    if (!al16(y.norm1) || !al16(y.w_qkv) || !al16(y.w_o) || !al16(y.norm2) || !al16(y.w_gate_up) ||
        !al16(y.w_down) || !al16(y.k_cache) || !al16(y.v_cache) || !al16(y.b_qkv))
      return QF_ERR_INVALID_ARG;
    if (((y.kc_sb | y.kc_sh | y.kc_sn | y.vc_sb | y.vc_sh | y.vc_sn) & 7) != 0)
      return QF_ERR_INVALID_ARG;
  }
  unsigned char* base = static_cast<unsigned char*>(ws);
  f16* hidden = static_cast<f16*>(hidden_p);
  f16* x = reinterpret_cast<f16*>(base + w.x);
  f16* qkv = reinterpret_cast<f16*>(base + w.qkv);
  f16* att = reinterpret_cast<f16*>(base + w.att);
  f16* h = reinterpret_cast<f16*>(base + w.h);
  f16* cs = reinterpret_cast<f16*>(base + w.cs);
  int2* info = reinterpret_cast<int2*>(base + w.info);
  const int W = (QH + 2 * KVH) * 64, A = QH * 64;
  float* part = reinterpret_cast<float*>(base + w.part);
  const KSplit down = k_split(T, H, I, cus);
  const auto norm = [&](const f16* weight, bool parts) {
    const dim3 grid((T + 3) / 4), block(256);
    if (parts)
      hipLaunchKernelGGL(prefill_rms_kernel<true>, grid, block, 0, st, hidden, weight, x, part,
                         down.splits, T, H, eps);
    else
      hipLaunchKernelGGL(prefill_rms_kernel<false>, grid, block, 0, st, hidden, weight, x, nullptr,
                         0, T, H, eps);
  };
  hipLaunchKernelGGL(prefill_tokens_kernel, dim3((T + 7) / 8), dim3(256), 0, st, cu, B, S, T,
                     inv_freq, block_table, bt_sb, l2, pages_per_row, n_pages, cs, info);
  int rc = (int)hipGetLastError();
  for (int i = 0; i < n_layers && rc == 0; ++i) {
    const QfPrefillLayer& y = layers[i];
    GemmArgs g = {};
    g.T = T;
    g.splits = 1;
    g.cs = cs;
    g.info = info;
    g.QH = QH;
    g.KVH = KVH;
    g.kc = static_cast<f16*>(y.k_cache);
    g.kc_sb = y.kc_sb; g.kc_sh = y.kc_sh; g.kc_sn = y.kc_sn;
    g.vc = static_cast<f16*>(y.v_cache);
    g.vc_sb = y.vc_sb; g.vc_sh = y.vc_sh; g.vc_sn = y.vc_sn;
    g.bias = static_cast<const f16*>(y.b_qkv);
    g.part = part;

    // Split: the layer before left its down_proj as partials.
    norm(static_cast<const f16*>(y.norm1), i > 0 && down.splits > 1);
    GemmArgs gq = g;
    gq.x = x; gq.x_sn = H; gq.w = static_cast<const f16*>(y.w_qkv); gq.y = qkv; gq.y_sn = W;
    gq.N = W; gq.K = H;
    rc = launch<kEpiQkv>(gq, cus, st);
    if (rc) break;
    if (cu == nullptr)
      rc = qf_prefill_attn(qkv, (int64_t)S * W, 64, W, qkv + A, (int64_t)S * W, 64, W,
                           qkv + A + KVH * 64, (int64_t)S * W, 64, W, nullptr, nullptr, 0, 0,
                           nullptr, 0, 0, 0, nullptr, 0, 0, 0, 0, 0, att, (int64_t)S * A, 64, A, B,
                           QH, KVH, S, D, 0.125f, stream);
    else
      rc = qf_prefill_varlen(qkv, 64, W, qkv + A, 64, W, qkv + A + KVH * 64, 64, W, cu, T, S,
                             nullptr, nullptr, 0, nullptr, 0, 0, 0, nullptr, 0, 0, 0, 0, 0, att, 64,
                             A, B, QH, KVH, D, 0.125f, stream);
    if (rc) break;
    GemmArgs go = g;
    go.x = att; go.x_sn = A; go.w = static_cast<const f16*>(y.w_o); go.y = hidden; go.y_sn = H;
    go.N = H; go.K = A;
    rc = launch<kEpiResidual>(go, cus, st);
    if (rc) break;
    norm(static_cast<const f16*>(y.norm2), false);
    GemmArgs gu = g;
    gu.x = x; gu.x_sn = H; gu.w = static_cast<const f16*>(y.w_gate_up); gu.y = h; gu.y_sn = I;
    gu.N = 2 * I; gu.K = H;
    rc = launch<kEpiSwiglu>(gu, cus, st);
    if (rc) break;
    GemmArgs gd = g;
    gd.x = h; gd.x_sn = I; gd.w = static_cast<const f16*>(y.w_down); gd.y = hidden; gd.y_sn = H;
    gd.N = H; gd.K = I;
    gd.splits = down.splits;
    rc = down.splits > 1 ? launch_split(gd, down.form, st) : launch<kEpiResidual>(gd, cus, st);
  }
  if (rc == 0 && down.splits > 1) {
    norm(nullptr, true);
    rc = (int)hipGetLastError();
  }
  return rc;
}
