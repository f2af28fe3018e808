// A prompt's tokens through the decoder layers in one pass: sh_llm_generate's
// prompt, all but its last token. Every linear is a GEMM over the tokens
// (fp16 activations, the model's own tiled FP8 / fp16 weights, fp32 sums on
// MFMA), attention is causal flash attention over the KV cache, which the
// pass fills as decode steps would. The reference has no LLM path.
//
// Token row m = b * T + i of a chunk is token i of the chunk in sequence b,
// at position lens[b] + i0 + i. Rounding points are the decode steps' own:
// fp32 residual stream, norm outputs, attention and MLP activations rounded
// to fp16, K and V cached as fp16.
//
// Every output element's sum runs in one fixed order whatever the batch, the
// chunk or the tile size, so a sequence's caches do not depend on what else
// is in the batch.
#include <hip/hip_runtime.h>

#include "common.h"
#include "llm.h"
#include "llm_device.h"

namespace sh {
namespace {

constexpr int kT = 256;
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

// Workgroup barrier for LDS traffic only: __syncthreads() would also wait for
// the outstanding global loads of the next stage.
__device__ __forceinline__ void lds_barrier() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// ---- embedding -----------------------------------------------------------------

// grid (B * T): the fp32 residual row of each token, its history entry and,
// for Qwen3, its RoPE factors (cos | sin, [d] per token).
__global__ __launch_bounds__(kT) void prefill_embed_kernel(const PrefillArgs a) {
  const int m = blockIdx.x, t = threadIdx.x;
  const int b = m / a.T, i = m - b * a.T;
  const int pos = max(a.lens[b], 0) + a.i0 + i;
  const int tok = a.tokens[(size_t)b * a.prompt_len + a.i0 + i];
  if (t == 0 && pos < a.hist_len) a.hist[(size_t)b * a.hist_len + pos] = tok;
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

// ---- linears -------------------------------------------------------------------

// C[m][n] = sum_k A[m][k] W[n][k], then the epilogue. A: fp16 rows; W: tiled
// weights (N a multiple of 64, K of 128). A workgroup owns 32 kMI tokens x
// 32 kMI outputs as 2 x 2 waves of kMI x kMI MFMA tiles. K advances in 64-wide
// stages: the tokens' stage goes through LDS (double buffered, 16-byte chunks
// XOR-swizzled by the row so that 8 rows of a read hit 8 bank groups); a
// weight tile is already in MFMA operand order, so each wave loads its own
// straight into registers. Both are requested two stages ahead. The MFMA is
// issued as W x A, which leaves a lane with 4 consecutive outputs of one
// token (16-byte fp32, 8-byte fp16 stores).
template <int kW, int kEpi, int kMI>
__global__ __launch_bounds__(kT, kMI == 4 ? 2 : 4) void prefill_gemm_kernel(const PrefillGemmArgs g, int tiles_m,
                                                          int ntiles, int per_xcd) {
  constexpr int kBM = 32 * kMI;
  constexpr int kChunks = kBM * 8 / kT;            // 16-byte chunks per thread and stage
  constexpr int kWL = kW == kWeightFp8 ? 1 : 2;    // 16-byte weight loads per tile and stage
  __shared__ __attribute__((aligned(16))) uint8_t lds[2][kBM * 128];
  // each XCD takes a run of tiles, tokens fastest: its L2 then reads few
  // weight rows, once
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= ntiles) return;
  const int tm = tile % tiles_m, tn = tile / tiles_m;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = tm * kBM, nt0 = tn * 2 * kMI + wn * kMI;  // first 16-row weight tile of the wave
  const int K = g.K, nk = K / 64;

  const uint16_t *arow[kChunks];
  int aoff[kChunks];
#pragma unroll
  for (int u = 0; u < kChunks; u++) {
    const int c = t + kT * u, r = c >> 3, ch = c & 7;
    arow[u] = g.a + (size_t)min(m0 + r, g.M - 1) * g.lda + ch * 8;
    aoff[u] = r * 128 + ((ch ^ (r & 7)) * 16);
  }
  u32x4 ra[2][kChunks], wv[2][kMI][kWL];
  auto load_a = [&](int s, int kt) {
#pragma unroll
    for (int u = 0; u < kChunks; u++)
      ra[s][u] = *reinterpret_cast<const u32x4 *>(arow[u] + (size_t)kt * 64);
  };
  auto load_w = [&](int s, int kt) {
#pragma unroll
    for (int j = 0; j < kMI; j++)
#pragma unroll
      for (int h = 0; h < kWL; h++)
        wv[s][j][h] = *reinterpret_cast<const u32x4 *>(
            g.w + ((size_t)(nt0 + j) * (nk * kWL) + (size_t)kt * kWL + h) * 1024 + lane * 16);
  };
  auto store_a = [&](int s, int buf) {
#pragma unroll
    for (int u = 0; u < kChunks; u++) *reinterpret_cast<u32x4 *>(&lds[buf][aoff[u]]) = ra[s][u];
  };

  f32x4 acc[kMI][kMI];
#pragma unroll
  for (int i = 0; i < kMI; i++)
#pragma unroll
    for (int j = 0; j < kMI; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int frow = wm * 16 * kMI + (lane & 15);
  auto compute = [&](int s, int buf) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      f16x8 fa[kMI], fw[kMI];
#pragma unroll
      for (int i = 0; i < kMI; i++) {
        const int r = frow + 16 * i, ch = 4 * h + (lane >> 4);
        fa[i] = *reinterpret_cast<const f16x8 *>(&lds[buf][r * 128 + ((ch ^ (r & 7)) * 16)]);
      }
#pragma unroll
      for (int j = 0; j < kMI; j++) {
        if (kW == kWeightFp8)
          fw[j] = e4m3x8_to_f16(wv[s][j][0][2 * h], wv[s][j][0][2 * h + 1]);
        else
          fw[j] = __builtin_bit_cast(f16x8, wv[s][j][h % kWL]);
      }
#pragma unroll
      for (int i = 0; i < kMI; i++)
#pragma unroll
        for (int j = 0; j < kMI; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[j], fa[i], acc[i][j], 0, 0, 0);
    }
  };

  load_a(0, 0);
  load_w(0, 0);
  load_a(1, 1);  // nk >= 2
  load_w(1, 1);
  store_a(0, 0);
  lds_barrier();
  // stage kt (even part: set / buffer 0, odd part: 1); the next stage's rows
  // go to the other buffer, which every wave has finished reading (the
  // barrier that ended the previous stage)
  for (int kt = 0; kt < nk; kt += 2) {
    const int k2 = min(kt + 2, nk - 1), k3 = min(kt + 3, nk - 1);  // past the end: re-read, unused
    // (the order is kept: a store moved up ahead of the loads would wait for
    // the stage requested last, not the one before it)
    load_a(0, k2);
    __builtin_amdgcn_sched_barrier(0);
    compute(0, 0);
    load_w(0, k2);
    __builtin_amdgcn_sched_barrier(0);
    store_a(1, 1);
    lds_barrier();
    load_a(1, k3);
    __builtin_amdgcn_sched_barrier(0);
    compute(1, 1);
    load_w(1, k3);
    __builtin_amdgcn_sched_barrier(0);
    store_a(0, 0);
    lds_barrier();
  }

  const int nl = 4 * (lane >> 4);  // this lane's 4 outputs within a 16-row tile
#pragma unroll
  for (int i = 0; i < kMI; i++) {
    const int m = m0 + frow + 16 * i;
    if (m >= g.M) continue;
#pragma unroll
    for (int j = 0; j < kMI; j++) {
      if (kEpi == kEpiSwiGLU && (j & 1)) continue;
      const int n = (nt0 + j) * 16 + nl;
      f32x4 v = acc[i][j];
      if (g.scale) {
        const f32x4 sc = *reinterpret_cast<const f32x4 *>(g.scale + n);
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] *= sc[r];
      }
      if (g.bias) {
        const f32x4 bi = *reinterpret_cast<const f32x4 *>(g.bias + n);
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] += bi[r];
      }
      if (kEpi == kEpiStore) {
        *reinterpret_cast<f32x4 *>(g.out + (size_t)m * g.out_ld + n) = v;
      } else if (kEpi == kEpiResidual) {
        f32x4 *o = reinterpret_cast<f32x4 *>(g.out + (size_t)m * g.out_ld + n);
        const f32x4 x = *o;
        *o = f32x4{x[0] + v[0], x[1] + v[1], x[2] + v[2], x[3] + v[3]};
      } else if (kEpi == kEpiGelu) {
        *reinterpret_cast<f16x4 *>(g.out16 + (size_t)m * g.out_ld + n) =
            f16x4{(_Float16)gelu_tanh(v[0]), (_Float16)gelu_tanh(v[1]), (_Float16)gelu_tanh(v[2]),
                  (_Float16)gelu_tanh(v[3])};
      } else {  // SwiGLU: tile j is a gate tile, j + 1 its up tile
        const f32x4 us = *reinterpret_cast<const f32x4 *>(g.scale + n + 16);
        f16x4 o;
#pragma unroll
        for (int r = 0; r < 4; r++)
          o[r] = (_Float16)(silu(v[r]) * (acc[i][(j + 1) % kMI][r] * us[r]));
        const int no = (nt0 + j) / 2 * 16 + nl;
        *reinterpret_cast<f16x4 *>(g.out16 + (size_t)m * g.out_ld + no) = o;
      }
    }
  }
}

// ---- q, k, v of the chunk ---------------------------------------------------------

constexpr int kPostTokens = 16;

// grid (ceil(T / 16), heads + 2 kv_heads, B): one head of 16 tokens. Query
// heads: RMSNorm and RoPE (Qwen3), times the softmax scale, as fp16 (and, for
// kSplit, the rounding's remainder as a second fp16); key heads: the same
// without the scale, appended to the K cache; value heads: appended to the V
// cache (kVT: transposed, [d][vt_stride]).
template <int kD, bool kQwen, bool kVT, bool kSplit>
__global__ __launch_bounds__(kT) void prefill_qkv_kernel(const PrefillArgs a, int first_head) {
  constexpr int kE = kD / 64;  // values per lane: dims lane, lane + 64
  __shared__ _Float16 vt[kPostTokens][kD + 2];
  const int hh = blockIdx.y + first_head, b = blockIdx.z;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int i_first = blockIdx.x * kPostTokens;
  const int p_first = max(a.lens[b], 0) + a.i0 + i_first;
  const bool is_q = hh < a.heads, is_k = !is_q && hh < a.heads + a.kv_heads;
  const int kvh = is_q ? 0 : (hh - a.heads) % a.kv_heads;
  const size_t cache = (size_t)b * a.kv_heads + kvh;
#pragma unroll
  for (int u = 0; u < kPostTokens / 4; u++) {
    const int r = wave * (kPostTokens / 4) + u, i = i_first + r, pos = p_first + r;
    if (i >= a.T) break;  // wave-uniform
    const size_t m = (size_t)b * a.T + i;
    float v[kE];
#pragma unroll
    for (int e = 0; e < kE; e++) v[e] = a.qkv[m * a.qkv_n + (size_t)hh * kD + lane + 64 * e];
    if (kQwen && (is_q || is_k)) {  // kD is 128: this lane holds a rotated pair
      float ss = 0.0f;
#pragma unroll
      for (int e = 0; e < kE; e++) ss += v[e] * v[e];
      ss = wave_sum(ss);
      const float inv = 1.0f / sqrtf(ss / kD + a.eps);
      const float *gain = is_q ? a.q_norm : a.k_norm;
#pragma unroll
      for (int e = 0; e < kE; e++) v[e] = v[e] * inv * gain[lane + 64 * e];
      const float cs = a.rope[m * kD + lane], sn = a.rope[m * kD + kD / 2 + lane];
      const float x1 = v[0], x2 = v[kE - 1];
      v[0] = x1 * cs - x2 * sn;
      v[kE - 1] = x2 * cs + x1 * sn;
    }
#pragma unroll
    for (int e = 0; e < kE; e++) {
      const int dd = lane + 64 * e;
      if (is_q) {
        const float q = v[e] * a.scale;
        const _Float16 hi = (_Float16)q;
        const size_t at = (m * a.heads + hh) * kD + dd;
        a.q[at] = __builtin_bit_cast(uint16_t, hi);
        if (kSplit) a.q_lo[at] = f32_to_f16_bits(q - (float)hi);
      } else if (is_k || !kVT) {
        uint16_t *c = is_k ? a.kcache : a.vcache;
        if (pos < a.max_pos) c[(cache * a.max_pos + pos) * kD + dd] = f32_to_f16_bits(v[e]);
      } else {
        vt[r][dd] = (_Float16)v[e];
      }
    }
  }
  if (!kVT || is_q || is_k) return;  // workgroup-uniform
  __syncthreads();
  // 16 positions of each dim's row: in two 16-byte stores where they are
  // all there and aligned
  const int n = min(min(kPostTokens, a.T - i_first), a.max_pos - p_first);
  for (int c = t; c < kD * 2; c += kT) {
    const int dd = c >> 1, r0 = (c & 1) * 8;
    uint16_t *o = a.vcache + (cache * kD + dd) * a.vt_stride + p_first + r0;
    f16x8 v;
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = r0 + e < n ? vt[r0 + e][dd] : (_Float16)0.0f;
    if (n == kPostTokens && (p_first & 7) == 0) {
      *reinterpret_cast<f16x8 *>(o) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const _Float16 x = v[e];
        if (r0 + e < n) o[e] = __builtin_bit_cast(uint16_t, x);
      }
    }
  }
}

// ---- causal attention ---------------------------------------------------------------

constexpr int kKeys = 64;  // positions per K / V tile

// grid (ceil(T / (64 kQT)), heads, B): 64 kQT tokens of one head against the
// cache, 16 kQT per wave; tiles of 64 positions from position 0, so that a
// token's running softmax passes over the same tiles whatever chunk it is in.
//  - scores as K x q: a lane holds one token (lane % 16) and 4 consecutive
//    positions of each 16-position tile, so the softmax's row maximum needs
//    two lane moves and the exponentials are the P operand in place;
//  - V sums as V^T x P with the MFMA's k slots numbered as P has them (slot
//    (g, e): position 4 g + e of the first 16-position tile for e < 4, of the
//    second for e >= 4), V^T read to match as two 8-byte LDS reads;
//  - K and V^T tiles go through registers to LDS one tile ahead.
// kSplit: q and P as two fp16 each (22 bits), for the models whose decode
// steps keep both in fp32; otherwise one fp16 each, the softmax sum taken
// over the rounded P, as the decode-layers kernel does.
template <int kD, bool kVT, bool kSplit, int kQT>
__global__ __launch_bounds__(kT) void prefill_attn_kernel(const PrefillArgs a) {
  constexpr int kKRow = kD + 8, kVRow = kKeys + 4;  // padded LDS rows (fp16)
  constexpr int kKK = kD / 32, kDT = kD / 16;
  constexpr int kLoads = kKeys * kD / 8 / kT;  // 16-byte loads per thread, tile and operand
  constexpr int kParts = kSplit ? 2 : 1;
  __shared__ __attribute__((aligned(16))) _Float16 ks[kKeys * kKRow];
  __shared__ __attribute__((aligned(16))) _Float16 vs[kD * kVRow];

  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int r = lane & 15, grp = lane >> 4;
  const int h = blockIdx.y, b = blockIdx.z, kvh = h / (a.heads / a.kv_heads);
  const int q0 = (gridDim.x - 1 - blockIdx.x) * 64 * kQT;  // the longest first
  const int base = max(a.lens[b], 0) + a.i0;
  const int kend = min(base + min(q0 + 64 * kQT, a.T), a.max_pos);  // positions any token sees

  int qpos[kQT];
  size_t qrow[kQT];
  f16x8 qf[kQT][kParts][kKK];
#pragma unroll
  for (int u = 0; u < kQT; u++) {
    const int i = min(q0 + (wave * kQT + u) * 16 + r, a.T - 1);
    qpos[u] = min(base + i, a.max_pos - 1);
    qrow[u] = (((size_t)b * a.T + i) * a.heads + h) * kD;
#pragma unroll
    for (int kk = 0; kk < kKK; kk++) {
      qf[u][0][kk] = *reinterpret_cast<const f16x8 *>(a.q + qrow[u] + 32 * kk + 8 * grp);
      if (kSplit)
        qf[u][kParts - 1][kk] =
            *reinterpret_cast<const f16x8 *>(a.q_lo + qrow[u] + 32 * kk + 8 * grp);
    }
  }

  const size_t cache = (size_t)b * a.kv_heads + kvh;
  const uint16_t *kb = a.kcache + cache * a.max_pos * kD;
  const uint16_t *vb = a.vcache + (kVT ? cache * kD * a.vt_stride : cache * a.max_pos * kD);
  u32x4 kr[kLoads], vr[kLoads];
  // tile pt of K and V into registers, clamped to cached positions
  auto load = [&](int pt) {
#pragma unroll
    for (int u = 0; u < kLoads; u++) {
      const int c = t + kT * u;
      const int p = min(pt + c / (kD / 8), kend - 1);
      kr[u] = *reinterpret_cast<const u32x4 *>(kb + (size_t)p * kD + (c % (kD / 8)) * 8);
      if (kVT) {  // 8 positions of one dim
        const int dd = c >> 3, p8 = min(pt + (c & 7) * 8, (kend - 1) & ~7);
        vr[u] = *reinterpret_cast<const u32x4 *>(vb + (size_t)dd * a.vt_stride + p8);
      } else {  // 8 dims of one position
        vr[u] = *reinterpret_cast<const u32x4 *>(vb + (size_t)p * kD + (c % (kD / 8)) * 8);
      }
    }
  };
  auto store = [&](int pt) {
#pragma unroll
    for (int u = 0; u < kLoads; u++) {
      const int c = t + kT * u;
      const int row = c / (kD / 8), c8 = (c % (kD / 8)) * 8;
      *reinterpret_cast<u32x4 *>(&ks[row * kKRow + c8]) = kr[u];
      const f16x8 v = __builtin_bit_cast(f16x8, vr[u]);
      if (kVT) {
        // positions past the cached ones may hold anything: zeros instead
        // (their P is 0, but 0 x NaN is not)
        const int dd = c >> 3, pl = (c & 7) * 8;
        f16x4 w[2];
#pragma unroll
        for (int e = 0; e < 8; e++) w[e >> 2][e & 3] = pt + pl + e < kend ? v[e] : (_Float16)0.0f;
        *reinterpret_cast<f16x4 *>(&vs[dd * kVRow + pl]) = w[0];
        *reinterpret_cast<f16x4 *>(&vs[dd * kVRow + pl + 4]) = w[1];
      } else {
#pragma unroll
        for (int e = 0; e < 8; e++) vs[(c8 + e) * kVRow + row] = v[e];
      }
    }
  };

  float m_run[kQT], l_run[kQT];
  f32x4 acc[kQT][kDT];
#pragma unroll
  for (int u = 0; u < kQT; u++) {
    m_run[u] = -INFINITY;
    l_run[u] = 0.0f;
#pragma unroll
    for (int dt = 0; dt < kDT; dt++) acc[u][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  load(0);
  for (int pt = 0; pt < kend; pt += kKeys) {
    lds_barrier();  // the previous tile's reads are done
    store(pt);
    lds_barrier();
    if (pt + kKeys < kend) load(pt + kKeys);

    f32x4 s[kQT][4];
#pragma unroll
    for (int u = 0; u < kQT; u++)
#pragma unroll
      for (int tt = 0; tt < 4; tt++) s[u][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int tt = 0; tt < 4; tt++)
#pragma unroll
      for (int kk = 0; kk < kKK; kk++) {
        const f16x8 kf =
            *reinterpret_cast<const f16x8 *>(&ks[(16 * tt + r) * kKRow + 32 * kk + 8 * grp]);
#pragma unroll
        for (int u = 0; u < kQT; u++)
#pragma unroll
          for (int part = 0; part < kParts; part++)
            s[u][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[u][part][kk], s[u][tt], 0, 0, 0);
      }

    f16x8 p[kQT][kParts][2];
#pragma unroll
    for (int u = 0; u < kQT; u++) {
      float mx = -INFINITY;
#pragma unroll
      for (int tt = 0; tt < 4; tt++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if (pt + 16 * tt + 4 * grp + e > qpos[u]) s[u][tt][e] = -INFINITY;
          mx = fmaxf(mx, s[u][tt][e]);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m_run[u], mx);  // finite: position 0 is always visible
      const float corr = expf(m_run[u] - m_new);
      m_run[u] = m_new;
      float ls = 0.0f;
#pragma unroll
      for (int tt = 0; tt < 4; tt++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float pr = expf(s[u][tt][e] - m_new);
          const _Float16 hi = (_Float16)pr;
          p[u][0][tt >> 1][(tt & 1) * 4 + e] = hi;
          if (kSplit) {
            p[u][kParts - 1][tt >> 1][(tt & 1) * 4 + e] = (_Float16)(pr - (float)hi);
            ls += pr;
          } else {
            ls += (float)hi;
          }
        }
      l_run[u] = l_run[u] * corr + ls;  // this lane's positions; the groups are summed at the end
#pragma unroll
      for (int dt = 0; dt < kDT; dt++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[u][dt][e] *= corr;
    }
#pragma unroll
    for (int dt = 0; dt < kDT; dt++)
#pragma unroll
      for (int sl = 0; sl < 2; sl++) {
        const _Float16 *vrow = &vs[(16 * dt + r) * kVRow + 32 * sl + 4 * grp];
        const f16x4 v0 = *reinterpret_cast<const f16x4 *>(vrow);
        const f16x4 v1 = *reinterpret_cast<const f16x4 *>(vrow + 16);
        const f16x8 vf = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int u = 0; u < kQT; u++)
#pragma unroll
          for (int part = 0; part < kParts; part++)
            acc[u][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, p[u][part][sl], acc[u][dt], 0, 0, 0);
      }
  }

#pragma unroll
  for (int u = 0; u < kQT; u++) {
    float l = l_run[u];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (q0 + (wave * kQT + u) * 16 + r < a.T) {
#pragma unroll
      for (int dt = 0; dt < kDT; dt++)
        *reinterpret_cast<f16x4 *>(a.attn + qrow[u] + 16 * dt + 4 * grp) =
            f16x4{(_Float16)(acc[u][dt][0] / l), (_Float16)(acc[u][dt][1] / l),
                  (_Float16)(acc[u][dt][2] / l), (_Float16)(acc[u][dt][3] / l)};
    }
  }
}

template <int kW, int kEpi, int kMI>
hipError_t launch_gemm_tile(hipStream_t s, const PrefillGemmArgs &g) {
  const int tiles_m = (g.M + 32 * kMI - 1) / (32 * kMI);
  const int ntiles = tiles_m * (g.N / (32 * kMI)), per_xcd = (ntiles + 7) / 8;
  prefill_gemm_kernel<kW, kEpi, kMI><<<per_xcd * 8, kT, 0, s>>>(g, tiles_m, ntiles, per_xcd);
  return hipGetLastError();
}

template <int kW, int kEpi>
hipError_t launch_gemm_epi(hipStream_t s, const PrefillGemmArgs &g) {
  // 128 x 128 tiles where they give every CU one, else 64 x 64
  if (g.N % 128 == 0 && (long long)((g.M + 127) / 128) * (g.N / 128) >= 256)
    return launch_gemm_tile<kW, kEpi, 4>(s, g);
  return launch_gemm_tile<kW, kEpi, 2>(s, g);
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

hipError_t launch_prefill_gemm(hipStream_t s, const PrefillGemmArgs &g, int weight_type, int epi) {
  if (g.M < 1 || g.N % 64 != 0 || g.K % 128 != 0 || g.K < 128) return hipErrorInvalidValue;
  if (weight_type == kWeightFp8) {
    if (epi == kEpiStore) return launch_gemm_epi<kWeightFp8, kEpiStore>(s, g);
    if (epi == kEpiResidual) return launch_gemm_epi<kWeightFp8, kEpiResidual>(s, g);
    if (epi == kEpiSwiGLU) return launch_gemm_epi<kWeightFp8, kEpiSwiGLU>(s, g);
  } else {
    if (epi == kEpiStore) return launch_gemm_epi<kWeightFp16, kEpiStore>(s, g);
    if (epi == kEpiResidual) return launch_gemm_epi<kWeightFp16, kEpiResidual>(s, g);
    if (epi == kEpiGelu) return launch_gemm_epi<kWeightFp16, kEpiGelu>(s, g);
  }
  return hipErrorInvalidValue;
}

// The forms the runners have: Qwen3 with the decode-layers kernel's caches
// (V transposed) or the per-op ones, GPT-2 with head_dim 64 or 128.
hipError_t launch_prefill_qkv(hipStream_t s, const PrefillArgs &a, bool qwen, bool kv_only) {
  const int first = kv_only ? a.heads : 0;
  const dim3 grid((a.T + kPostTokens - 1) / kPostTokens, a.heads + 2 * a.kv_heads - first, a.B);
  if (qwen && a.d == 128 && a.vt_stride)
    prefill_qkv_kernel<128, true, true, false><<<grid, kT, 0, s>>>(a, first);
  else if (qwen && a.d == 128)
    prefill_qkv_kernel<128, true, false, true><<<grid, kT, 0, s>>>(a, first);
  else if (!qwen && a.d == 128)
    prefill_qkv_kernel<128, false, false, true><<<grid, kT, 0, s>>>(a, first);
  else if (!qwen && a.d == 64)
    prefill_qkv_kernel<64, false, false, true><<<grid, kT, 0, s>>>(a, first);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_prefill_attention(hipStream_t s, const PrefillArgs &a) {
  // 128 tokens per workgroup where that leaves two workgroups per CU, else 64
  const bool wide = (long long)((a.T + 127) / 128) * a.heads * a.B >= 512;
  const int per = wide ? 128 : 64;
  const dim3 grid((a.T + per - 1) / per, a.heads, a.B);
#define SH_ATTN(D, VT, SPLIT)                                        \
  do {                                                               \
    if (wide)                                                        \
      prefill_attn_kernel<D, VT, SPLIT, 2><<<grid, kT, 0, s>>>(a);   \
    else                                                             \
      prefill_attn_kernel<D, VT, SPLIT, 1><<<grid, kT, 0, s>>>(a);   \
  } while (0)
  if (a.d == 128 && a.vt_stride)
    SH_ATTN(128, true, false);
  else if (a.d == 128)
    SH_ATTN(128, false, true);
  else if (a.d == 64 && !a.vt_stride)
    SH_ATTN(64, false, true);
  else
    return hipErrorInvalidValue;
#undef SH_ATTN
  return hipGetLastError();
}

}  // namespace sh
