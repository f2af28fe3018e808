// A prompt's tokens through the decoder layers in one pass: sh_llm_generate's
// prompt, all but its last token. Every linear is a GEMM over the tokens,
// attention is causal over the KV cache, which the pass fills as decode steps
// would. The reference has no LLM path.
//
// Token row m = b * T + i of a chunk is token i of the chunk in sequence b,
// at position lens[b] + i0 + i.
//
// The pass computes what steps over the same tokens compute, bit for bit:
// every sum, norm, softmax and rounding is taken in the order of the kernels
// that the model's steps run on (kStepOps: llm_kernels.hip, kStepGpt2Layers:
// gpt2_layers.hip, kStepQwenLayers: decode_layers.hip). A cache therefore does
// not depend on how its tokens came in, on the batch or on the chunk, and a
// model in 16 bits gives the same tokens either way. This file has the parts
// for the first two, which are compiled with the compiler's own contraction of
// multiply-adds, as their step kernels are; prefill_layers.hip has the third's.
#include <hip/hip_runtime.h>

#include "common.h"
#include "llm.h"
#include "llm_device.h"
#include "prefill_gemm.h"

namespace sh {
namespace {

using prompt::f16x4;
using prompt::kT;
using prompt::lds_barrier;

// ---- embedding -----------------------------------------------------------------

// grid (B * T): the fp32 residual row of each token, its position and history
// entry and, for Qwen3, its RoPE factors (cos | sin, [d] per token).
__global__ __launch_bounds__(kT) void prefill_embed_kernel(const PrefillArgs a) {
  const int m = blockIdx.x, t = threadIdx.x;
  const int b = m / a.T, i = m - b * a.T;
  const int pos = max(a.lens[b], 0) + a.i0 + i;
  const int tok = a.tokens[(size_t)b * a.prompt_len + a.i0 + i];
  if (t == 0) {
    a.pos[m] = pos;
    if (pos < a.hist_len) a.hist[(size_t)b * a.hist_len + pos] = tok;
  }
  if (a.rope && t < a.d / 2) {
    float sn, cs;
    sincosf((float)pos * a.inv_freq[t], &sn, &cs);
    a.rope[(size_t)m * a.d + t] = cs;
    a.rope[(size_t)m * a.d + a.d / 2 + t] = sn;
  }
  float *x = a.x + (size_t)m * a.H;
  // 8 consecutive k of a row are contiguous in both tiled layouts
  for (int k = 8 * t; k < a.H; k += 8 * kT) {
    f16x8 h;
    float sc = 1.0f;
    if (a.head8) {
      const u32x2 q = *reinterpret_cast<const u32x2 *>(a.head8 + fp8_tiled_offset(tok, k, a.H));
      h = e4m3x8_to_f16(q.x, q.y);
      sc = a.head_scale[tok];
    } else {
      h = *reinterpret_cast<const f16x8 *>(a.head16 + f16_tiled_offset(tok, k, a.H));
    }
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = (float)h[e] * sc;
    if (a.wpe) {
      const f16x8 w = *reinterpret_cast<const f16x8 *>(
          a.wpe + (size_t)min(pos, a.max_pos - 1) * a.H + k);
#pragma unroll
      for (int e = 0; e < 8; e++) v[e] += (float)w[e];
    }
    *reinterpret_cast<f32x4 *>(x + k) = f32x4{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4 *>(x + k + 4) = f32x4{v[4], v[5], v[6], v[7]};
  }
}

// lens[b] += n for the B sequences.
__global__ void prefill_finish_kernel(int *lens, int B, int n) {
  if ((int)threadIdx.x < B) lens[threadIdx.x] += n;
}

// ---- norms -----------------------------------------------------------------------

// The per-op GEMV's prologue (its Stager), one wave per row: the order of its
// sums and its expressions.
template <int kPro>
__global__ __launch_bounds__(kT) void prefill_norm_ops_kernel(const float *x, const float *gamma,
                                                              const float *beta, uint16_t *out16,
                                                              int M, int K, float eps) {
  const int m = blockIdx.x * (kT / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (m >= M) return;
  const float *row = x + (size_t)m * K;
  float mean = 0.0f;
  if (kPro == kProLayer) {
    float sm = 0.0f;
    for (int k = lane; k < K; k += 64) sm += row[k];
    mean = wave_sum(sm) / (float)K;
  }
  float ss = 0.0f;
  for (int k = lane; k < K; k += 64) {
    const float d = row[k] - mean;
    ss += d * d;
  }
  ss = wave_sum(ss);
  const float inv = 1.0f / sqrtf(ss / (float)K + eps);
  for (int k = lane; k < K; k += 64) {
    float y = (row[k] - mean) * inv * gamma[k];
    if (kPro == kProLayer) y += beta[k];
    out16[f16_tiled_offset(m, k, K)] = f32_to_f16_bits(y);
  }
}

// The GPT-2 layers kernel's LayerNorm (its stage_ln), one workgroup per row:
// a wave holds a quarter of the row as 2-value pairs, and the quarters' means
// and squared deviations are merged. kP: pairs per thread.
template <int kP>
__global__ __launch_bounds__(kT) void prefill_norm_gpt2_kernel(const float *x, const float *gamma,
                                                               const float *beta, uint16_t *out16,
                                                               int K, float eps) {
  __shared__ float part[2][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c2 = K >> 1;
  const float *row = x + (size_t)blockIdx.x * K;
  auto pair = [&](int i) { return wave * (K >> 3) + lane + 64 * i; };
  auto pair_ok = [&](int i) { return lane + 64 * i < (K >> 3); };
  f32x2 gv[kP], bv[kP], v[kP];
#pragma unroll
  for (int i = 0; i < kP; i++) {
    const int c = min(pair(i), c2 - 1);
    gv[i] = *reinterpret_cast<const f32x2 *>(gamma + c * 2);
    bv[i] = *reinterpret_cast<const f32x2 *>(beta + c * 2);
    v[i] = *reinterpret_cast<const f32x2 *>(row + c * 2);
  }
  const float nw = (float)(K >> 2);
  float sm = 0.0f;
#pragma unroll
  for (int i = 0; i < kP; i += 2) {
    const float s0 = pair_ok(i) ? v[i][0] + v[i][1] : 0.0f;
    const float s1 = pair_ok(i + 1) ? v[i + 1][0] + v[i + 1][1] : 0.0f;
    sm += s0 + s1;
  }
  const float mw = wave_sum_rows(sm) / nw;
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < kP; i += 2) {
    const f32x2 d0 = v[i] - mw, d1 = v[i + 1] - mw;
    const float s0 = pair_ok(i) ? d0[0] * d0[0] + d0[1] * d0[1] : 0.0f;
    const float s1 = pair_ok(i + 1) ? d1[0] * d1[0] + d1[1] * d1[1] : 0.0f;
    ss += s0 + s1;
  }
  ss = wave_sum_rows(ss);
  if (lane == 0) {
    part[0][wave] = mw;
    part[1][wave] = ss;
  }
  lds_barrier();
  const float mean = ((part[0][0] + part[0][1]) + (part[0][2] + part[0][3])) * 0.25f;
  const float e0 = part[0][0] - mean, e1 = part[0][1] - mean, e2 = part[0][2] - mean, e3 = part[0][3] - mean;
  const float m2 = ((part[1][0] + part[1][1]) + (part[1][2] + part[1][3])) +
                   nw * ((e0 * e0 + e1 * e1) + (e2 * e2 + e3 * e3));
  const float inv = 1.0f / sqrtf(m2 / (float)K + eps);
#pragma unroll
  for (int i = 0; i < kP; i++) {
    if (pair_ok(i)) {
      const f32x2 y = (v[i] - mean) * inv * gv[i] + bv[i];
      *reinterpret_cast<f16x2 *>(out16 + f16_tiled_offset(blockIdx.x, pair(i) * 2, K)) =
          f16x2{(_Float16)y[0], (_Float16)y[1]};
    }
  }
}

// ---- GPT-2: k and v to the caches -------------------------------------------------

// grid (B * T): k and v of a token, rounded to fp16, 4 values per thread.
__global__ __launch_bounds__(kT) void prefill_append_kernel(const PrefillArgs a) {
  const int m = blockIdx.x, b = m / a.T, pos = a.pos[m], n = a.kv_heads * a.d;
  if (pos >= a.max_pos) return;
  const float *qkv = a.qkv + (size_t)m * a.qkv_n + a.heads * a.d;
  for (int e = 4 * threadIdx.x; e < 2 * n; e += 4 * kT) {
    const bool is_k = e < n;
    const int c = is_k ? e : e - n, kvh = c / a.d, dd = c % a.d;
    const f32x4 x = *reinterpret_cast<const f32x4 *>(qkv + e);
    uint16_t *o = (is_k ? a.kcache : a.vcache) + (((size_t)b * a.kv_heads + kvh) * a.max_pos + pos) * a.d + dd;
    *reinterpret_cast<f16x4 *>(o) = f16x4{(_Float16)x[0], (_Float16)x[1], (_Float16)x[2], (_Float16)x[3]};
  }
}

// ---- GPT-2: attention as the layers kernel's -----------------------------------------

constexpr int kHd = 64;             // head dim
constexpr int kMaxChunk = 256;      // positions per split, one per thread
constexpr int kVJ = kMaxChunk / 32;  // V rows per thread
constexpr int kTok = 4;             // tokens per workgroup
constexpr int kPStride = kHd + 2;   // a partial: V sums, maximum, sum

// x + x of lane l ^ kX (16 or 32) in every lane (see add_lane_swap in
// gpt2_layers.hip; an fp32 sum of two values does not depend on their order).
template <int kX>
__device__ __forceinline__ float add_lane_xor(float x) {
  return x + __shfl_xor(x, kX, 64);
}

// grid (heads, ceil(T / kTok)), one sequence: kTok tokens of one head over the
// splits of the positions up to each token's own. A split's K and V rows are
// held in registers for all of the tokens as the layers kernel's attention
// item holds them for its one, and each token's arithmetic is that item's:
// thread t = 4 g + q sums dims 16 q .. of positions g + 64 m, the quad adds its
// quarters, the softmax runs over the split, thread (d8, pg) sums V over
// positions pg + 32 j. At the end the splits are merged as its O items merge
// them (stage_attn_n).
__global__ __launch_bounds__(kT) void prefill_attn_gpt2_kernel(const PrefillArgs a) {
  __shared__ __attribute__((aligned(16))) float qs[kTok][kHd];
  __shared__ float p[kMaxChunk], wmax[4], wl[4];
  __shared__ float pv[4][kHd], part[kTok][kGpt2Splits][kPStride];
  const int h = blockIdx.x, i0 = blockIdx.y * kTok;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int n = min(kTok, a.T - i0);
  const int base = max(a.lens[0], 0) + a.i0 + i0;  // the first token's position
  auto context = [&](int i) { return min(base + i + 1, a.max_pos); };
  const int end = context(n - 1);
  const uint16_t *kb = a.kcache + (size_t)h * a.max_pos * kHd;
  const uint16_t *vb = a.vcache + (size_t)h * a.max_pos * kHd;
  const int kq = t & 3, kg = t >> 2, d8 = t & 7, pg = t >> 3;
  static_assert(kT == kTok * kHd, "a thread per token and dim");
  qs[t / kHd][t % kHd] = a.qkv[(size_t)(i0 + min(t / kHd, n - 1)) * a.qkv_n + h * kHd + t % kHd] * a.scale;
  lds_barrier();
#pragma unroll 1
  for (int s = 0; s * a.chunk < end; s++) {
    const int p0 = s * a.chunk, last = min(end, p0 + a.chunk) - 1;
    f16x8 k[8], v[kVJ];
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
      for (int hh = 0; hh < 2; hh++)
        k[2 * m + hh] = *reinterpret_cast<const f16x8 *>(kb + (size_t)min(p0 + kg + 64 * m, last) * kHd + 16 * kq + 8 * hh);
#pragma unroll
    for (int j = 0; j < kVJ; j++)
      v[j] = *reinterpret_cast<const f16x8 *>(vb + (size_t)min(p0 + pg + 32 * j, last) * kHd + 8 * d8);
#pragma unroll 1
    for (int i = 0; i < n; i++) {
      const int L = context(i);
      if (p0 >= L) continue;  // uniform
      const int np = min(a.chunk, L - p0);
      f32x4 qr[4];
#pragma unroll
      for (int e = 0; e < 4; e++) qr[e] = *reinterpret_cast<const f32x4 *>(&qs[i][16 * kq + 4 * e]);
      float s4[4];
#pragma unroll
      for (int m = 0; m < 4; m++) {
        float acc = 0.0f;
#pragma unroll
        for (int hh = 0; hh < 2; hh++)
#pragma unroll
          for (int e = 0; e < 8; e++) acc += qr[2 * hh + e / 4][e % 4] * (float)k[2 * m + hh][e];
        s4[m] = acc;
      }
#pragma unroll
      for (int m = 0; m < 4; m++) {
        s4[m] += dpp_f32<0xB1>(s4[m]);
        s4[m] += dpp_f32<0x4E>(s4[m]);
      }
      const int pi_own = kg + 64 * kq;  // this thread's position in the split
      float sc = kq == 0 ? s4[0] : kq == 1 ? s4[1] : kq == 2 ? s4[2] : s4[3];
      sc = pi_own < np ? sc : -INFINITY;
      float mx = wave_max_rows(sc);
      if (lane == 0) wmax[wave] = mx;
      lds_barrier();
      mx = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
      const float ex = pi_own < np ? expf(sc - mx) : 0.0f;
      p[pi_own] = ex;
      const float ls = wave_sum_rows(ex);
      if (lane == 0) wl[wave] = ls;
      lds_barrier();
      const float lsum = (wl[0] + wl[1]) + (wl[2] + wl[3]);
      float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < kVJ; j++) {
        const int pi = pg + 32 * j;
        const float pw = p[pi];
        // (later tokens' V are not this one's: 0 times an infinity is not 0)
        const f16x8 vr = pi < np ? v[j] : f16x8{};
#pragma unroll
        for (int q = 0; q < 8; q++) o[q] += pw * (float)vr[q];
      }
#pragma unroll
      for (int q = 0; q < 8; q++) {
        o[q] += dpp_f32<0x128>(o[q]);
        o[q] = add_lane_xor<16>(o[q]);
        o[q] = add_lane_xor<32>(o[q]);
      }
      if (lane < 8) {
#pragma unroll
        for (int q = 0; q < 8; q++) pv[wave][8 * lane + q] = o[q];
      }
      lds_barrier();
      // (pv is written again two barriers on)
      if (wave == 0) {
        part[i][s][lane] = (pv[0][lane] + pv[1][lane]) + (pv[2][lane] + pv[3][lane]);
        if (lane == 0) {
          part[i][s][kHd] = mx;
          part[i][s][kHd + 1] = lsum;
        }
      }
    }
  }
  lds_barrier();
  const int i = t / kHd, dd = t % kHd;
  if (i >= n) return;
  const int ns = (context(i) + a.chunk - 1) / a.chunk;
  float M = -INFINITY;
  for (int s = 0; s < ns; s++) M = fmaxf(M, part[i][s][kHd]);
  float num = 0.0f, den = 0.0f;
  for (int s = 0; s < ns; s++) {
    const float f = expf(part[i][s][kHd] - M);
    num += f * part[i][s][dd];
    den += f * part[i][s][kHd + 1];
  }
  a.attn[f16_tiled_offset(i0 + i, h * kHd + dd, a.heads * kHd)] = f32_to_f16_bits(num / den);
}

}  // namespace

hipError_t launch_prefill_embed(hipStream_t s, const PrefillArgs &a) {
  prefill_embed_kernel<<<a.B * a.T, kT, 0, s>>>(a);
  return hipGetLastError();
}

hipError_t launch_prefill_finish(hipStream_t s, int *lens, int B, int n) {
  prefill_finish_kernel<<<1, 64, 0, s>>>(lens, B, n);
  return hipGetLastError();
}

hipError_t launch_prefill_norm(hipStream_t s, const PrefillArgs &a, const float *gamma,
                               const float *beta, int form) {
  const int M = a.B * a.T;
  if (form == kStepGpt2Layers) {
    if (a.H > 1024) return hipErrorInvalidValue;
    prefill_norm_gpt2_kernel<2><<<M, kT, 0, s>>>(a.x, gamma, beta, a.h16, a.H, a.eps);
  } else if (beta) {
    prefill_norm_ops_kernel<kProLayer><<<(M + 3) / 4, kT, 0, s>>>(a.x, gamma, beta, a.h16, M, a.H, a.eps);
  } else {
    prefill_norm_ops_kernel<kProRms><<<(M + 3) / 4, kT, 0, s>>>(a.x, gamma, beta, a.h16, M, a.H, a.eps);
  }
  return hipGetLastError();
}

hipError_t launch_prefill_gemm(hipStream_t s, const PrefillGemmArgs &g, int weight_type, int epi,
                               int form) {
  const bool fp8 = weight_type == kWeightFp8;
  if (g.M < 1 || g.N % 64 != 0 || g.K % (fp8 ? 256 : 128) != 0 || g.K < 128) return hipErrorInvalidValue;
  if (fp8 ? !g.scale || g.bias : g.scale || !g.bias) return hipErrorInvalidValue;
#define SH_GEMM(W, E, F) \
  if (weight_type == W && epi == E && form == F) return prompt::launch_gemm<W, E, F>(s, g);
  SH_GEMM(kWeightFp8, kEpiStore, kStepOps)
  SH_GEMM(kWeightFp8, kEpiResidual, kStepOps)
  SH_GEMM(kWeightFp8, kEpiSwiGLU, kStepOps)
  SH_GEMM(kWeightFp16, kEpiStore, kStepOps)
  SH_GEMM(kWeightFp16, kEpiResidual, kStepOps)
  SH_GEMM(kWeightFp16, kEpiGelu, kStepOps)
  SH_GEMM(kWeightFp16, kEpiStore, kStepGpt2Layers)
  SH_GEMM(kWeightFp16, kEpiResidual, kStepGpt2Layers)
  SH_GEMM(kWeightFp16, kEpiGelu, kStepGpt2Layers)
#undef SH_GEMM
  return hipErrorInvalidValue;
}

hipError_t launch_prefill_append(hipStream_t s, const PrefillArgs &a) {
  prefill_append_kernel<<<a.B * a.T, kT, 0, s>>>(a);
  return hipGetLastError();
}

hipError_t launch_prefill_attention_gpt2(hipStream_t s, const PrefillArgs &a) {
  if (a.B != 1 || a.d != kHd || a.chunk > kMaxChunk || a.max_pos > kGpt2Splits * a.chunk)
    return hipErrorInvalidValue;
  prefill_attn_gpt2_kernel<<<dim3(a.heads, (a.T + kTok - 1) / kTok), kT, 0, s>>>(a);
  return hipGetLastError();
}

}  // namespace sh
