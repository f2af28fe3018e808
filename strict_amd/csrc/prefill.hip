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

#include <type_traits>

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

// Groups of 4 waves that share a tile's K stages (every kGroups-th each); fixed
// per epilogue, so that a sum's order is. Two where the outputs are few (the
// residual linears, N = hidden): their stages are a serial chain on a chip that
// is not full. O and down, 1,023 tokens of 1024 x 2048 and 1024 x 3072: 15.0 and
// 21.4 us with one group, 11.2 and 15.2 with two; 128 tokens of 768 x 3072 23.7
// and 18.6; 4,090 tokens 35 and 48, 29 and 39; 8,000 tokens of 768 x 768 17.6
// and 19.0. The wide linears lose by it once the chip is full: QKV at 4,090
// tokens 56 and 71 us, gate / up at 1,023 23.9 and 27.5.
constexpr int groups_of(int epi) { return epi == kEpiResidual ? 2 : 1; }

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
__global__ __launch_bounds__(kT * groups_of(kEpi), kMI == 4 ? 2 : 4) void prefill_gemm_kernel(
    const PrefillGemmArgs g, int tiles_m, int ntiles, int per_xcd) {
  constexpr int kBM = 32 * kMI, kGroups = groups_of(kEpi);
  constexpr int kChunks = kBM * 8 / kT;            // 16-byte chunks per thread and stage
  constexpr int kWL = kW == kWeightFp8 ? 1 : 2;    // 16-byte weight loads per tile and stage
  __shared__ __attribute__((aligned(16))) uint8_t lds_all[kGroups][2][kBM * 128];
  // each XCD takes a run of tiles, tokens fastest: its L2 then reads few
  // weight rows, once
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= ntiles) return;
  const int tm = tile % tiles_m, tn = tile / tiles_m;
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / kT);
  const int t = threadIdx.x % kT, lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = tm * kBM, nt0 = tn * 2 * kMI + wn * kMI;  // first 16-row weight tile of the wave
  const int K = g.K, nk = K / 64;
  uint8_t (*lds)[kBM * 128] = lds_all[group];

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

  // this group's stages: group, group + kGroups, ..; nk is a multiple of
  // kGroups. Iteration it uses set / buffer it % 2; the next stage's rows go to
  // the other buffer, which every wave has finished reading (the barrier that
  // ended the previous iteration). (The order is kept: a store moved up ahead of
  // the loads would wait for the stage requested last, not the one before it.)
  const int nit = nk / kGroups;
  auto stage = [&](int it) { return min(it, nit - 1) * kGroups + group; };  // past the end: unused
  auto step = [&](int it, auto par_c) __attribute__((always_inline)) {
    constexpr int kPar = decltype(par_c)::value;
    load_a(kPar, stage(it + 2));
    __builtin_amdgcn_sched_barrier(0);
    compute(kPar, kPar);
    load_w(kPar, stage(it + 2));
    __builtin_amdgcn_sched_barrier(0);
    store_a(kPar ^ 1, kPar ^ 1);
    lds_barrier();
  };
  load_a(0, stage(0));
  load_w(0, stage(0));
  load_a(1, stage(1));
  load_w(1, stage(1));
  store_a(0, 0);
  lds_barrier();
  int it = 0;
  for (; it + 1 < nit; it += 2) {
    step(it, std::integral_constant<int, 0>{});
    step(it + 1, std::integral_constant<int, 1>{});
  }
  if (it < nit) step(it, std::integral_constant<int, 0>{});

  // the groups' sums: group q finishes the q-th part of the wave's token tiles
  constexpr int kOwn = kMI / kGroups;
  if constexpr (kGroups == 2) {
    f32x4 *red = reinterpret_cast<f32x4 *>(&lds_all[0][0][0]);  // [from group][i][j][thread]
#pragma unroll
    for (int i = 0; i < kOwn; i++)
#pragma unroll
      for (int j = 0; j < kMI; j++) {
        const f32x4 give = group == 0 ? acc[kOwn + i][j] : acc[i][j];
        red[((group * kOwn + i) * kMI + j) * kT + t] = give;
      }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < kOwn; i++)
#pragma unroll
      for (int j = 0; j < kMI; j++) {
        const f32x4 x = red[(((group ^ 1) * kOwn + i) * kMI + j) * kT + t];
        const f32x4 own = group == 0 ? acc[i][j] : acc[kOwn + i][j];
        acc[i][j] = f32x4{own[0] + x[0], own[1] + x[1], own[2] + x[2], own[3] + x[3]};
      }
  }

  const int nl = 4 * (lane >> 4);  // this lane's 4 outputs within a 16-row tile
#pragma unroll
  for (int i = 0; i < kOwn; i++) {
    const int m = m0 + frow + 16 * (group * kOwn + i);
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

constexpr int kAttnT = 512;

// Key parts of an attention tile, fixed per head size: 32 positions each.
constexpr int attn_parts(int d) { return d == 128 ? 4 : 2; }
// Tokens per workgroup: the 8 waves are parts x groups of 16 tokens.
constexpr int attn_tokens(int d) { return 128 / attn_parts(d); }

// grid (heads, ceil(T / attn_tokens), B): a block of tokens of one head against
// the cache. Tiles of 32 kKP positions start at position 0 and a part is a
// fixed 32 of each, so a token's kKP running softmaxes pass over the same
// positions whatever chunk of the prompt it is in; they are merged in one order
// at the end.
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
//
// What bounds it is a tile's way from the L2 through LDS to the MFMAs, step
// after step behind barriers: of 22.3 us at 1,023 tokens of 16 heads of 128 the
// loads and LDS stores alone take 14.5, all but the loads 18.5. So the keys of
// a tile are split over waves (4 waves of 16 tokens on a 64-position tile:
// 37.5 us, 400 at 4,090 tokens; now 23 and 222) and two workgroups share a CU,
// one's loads beside the other's MFMAs. 64 tokens per workgroup with half the
// K and V traffic but one workgroup per CU: 26 us, 266 at 4,090 tokens.
// Fragments straight from the cache, no LDS and no barrier: 32 us.
template <int kD, bool kVT, bool kSplit>
__global__ __launch_bounds__(kAttnT, kSplit && kD == 128 ? 2 : 4) void prefill_attn_kernel(
    const PrefillArgs a) {
  constexpr int kKP = attn_parts(kD), kKeys = 32 * kKP, kGroupsT = 8 / kKP;
  // padded LDS rows (fp16): 16 rows on 16 different bank groups
  constexpr int kKRow = kD + 8, kVRow = kKeys + 8;
  constexpr int kKK = kD / 32, kDT = kD / 16;
  constexpr int kLoads = kKeys * kD / 8 / kAttnT;  // 16-byte loads per thread, tile and operand
  constexpr int kParts = kSplit ? 2 : 1;
  __shared__ __attribute__((aligned(16))) union {
    struct {
      _Float16 k[kKeys * kKRow], v[kD * kVRow];
    } tile;
    f32x4 acc[kKP][kGroupsT][kDT][64];
  } lds;
  __shared__ float stat[kKP][kGroupsT][2][64];  // maximum, sum
  _Float16 *ks = lds.tile.k, *vs = lds.tile.v;

  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane((t >> 6) % kGroupsT);  // token group
  const int kh = __builtin_amdgcn_readfirstlane((t >> 6) / kGroupsT);    // key part
  const int r = lane & 15, grp = lane >> 4;
  // workgroups x, x + kv_heads, .. share a KV head: with 8 of those an XCD's L2
  // holds the one it works on
  const int kvh = blockIdx.x % a.kv_heads, b = blockIdx.z;
  const int h = kvh * (a.heads / a.kv_heads) + blockIdx.x / a.kv_heads;
  // the longest half of the blocks first, longest first; then the others,
  // shortest first: a CU's second workgroup evens out its first
  const int blocks = gridDim.y, by = blockIdx.y, half = (blocks + 1) / 2;
  const int q0 = attn_tokens(kD) * (by < half ? blocks - 1 - by : by - half);
  const int base = max(a.lens[b], 0) + a.i0;
  const int kend = min(base + min(q0 + attn_tokens(kD), a.T), a.max_pos);  // positions any token sees

  // this lane's token, and the first and the last position of the wave's tokens
  const int w0 = q0 + 16 * wave, i = min(w0 + r, a.T - 1);
  const int qpos = min(base + i, a.max_pos - 1);
  const int qlo = min(base + min(w0, a.T - 1), a.max_pos - 1);
  const int qhi = min(base + min(w0 + 15, a.T - 1), a.max_pos - 1);
  const size_t qrow = (((size_t)b * a.T + i) * a.heads + h) * kD;
  f16x8 qf[kParts][kKK];
#pragma unroll
  for (int kk = 0; kk < kKK; kk++) {
    qf[0][kk] = *reinterpret_cast<const f16x8 *>(a.q + qrow + 32 * kk + 8 * grp);
    if (kSplit)
      qf[kParts - 1][kk] = *reinterpret_cast<const f16x8 *>(a.q_lo + qrow + 32 * kk + 8 * grp);
  }

  const size_t cache = (size_t)b * a.kv_heads + kvh;
  const uint16_t *kb = a.kcache + cache * a.max_pos * kD;
  const uint16_t *vb = a.vcache + (kVT ? cache * kD * a.vt_stride : cache * a.max_pos * kD);
  u32x4 kr[kLoads], vr[kLoads];
  // tile pt of K and V into registers, clamped to cached positions
  auto load = [&](int pt) {
    const uint16_t *kt = kb + (size_t)pt * kD, *vt = vb + (kVT ? (size_t)pt : (size_t)pt * kD);
    const int last = kend - 1 - pt;
#pragma unroll
    for (int u = 0; u < kLoads; u++) {
      const int c = t + kAttnT * u;
      kr[u] = *reinterpret_cast<const u32x4 *>(kt + min(c / (kD / 8), last) * kD + c % (kD / 8) * 8);
      if (kVT)  // 8 positions of one dim
        vr[u] = *reinterpret_cast<const u32x4 *>(
            vt + (size_t)(c / (kKeys / 8)) * a.vt_stride + min(c % (kKeys / 8) * 8, last & ~7));
      else  // 8 dims of one position, positions along the lanes for the transposing store
        vr[u] = *reinterpret_cast<const u32x4 *>(vt + min(c % kKeys, last) * kD + c / kKeys * 8);
    }
  };
  auto store = [&](int pt) {
#pragma unroll
    for (int u = 0; u < kLoads; u++) {
      const int c = t + kAttnT * u;
      const int row = c / (kD / 8), c8 = (c % (kD / 8)) * 8;
      *reinterpret_cast<u32x4 *>(&ks[row * kKRow + c8]) = kr[u];
      const f16x8 v = __builtin_bit_cast(f16x8, vr[u]);
      if (kVT) {
        // positions past the cached ones may hold anything: zeros instead
        // (their P is 0, but 0 x NaN is not)
        const int dd = c / (kKeys / 8), pl = c % (kKeys / 8) * 8;
        f16x8 w = v;
        if (pt + kKeys > kend) {
#pragma unroll
          for (int e = 0; e < 8; e++) w[e] = pt + pl + e < kend ? v[e] : (_Float16)0.0f;
        }
        *reinterpret_cast<f16x8 *>(&vs[dd * kVRow + pl]) = w;
      } else {
        const int pv = c % kKeys, d8 = c / kKeys * 8;
#pragma unroll
        for (int e = 0; e < 8; e++) vs[(d8 + e) * kVRow + pv] = v[e];
      }
    }
  };

  float m_run = -INFINITY, l_run = 0.0f;
  f32x4 acc[kDT];
#pragma unroll
  for (int dt = 0; dt < kDT; dt++) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // this wave's part of the tile in LDS, positions p0 ..
  auto attend = [&](int p0) __attribute__((always_inline)) {
    f32x4 s[2];
#pragma unroll
    for (int tt = 0; tt < 2; tt++) s[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < kKK; kk++)
#pragma unroll
      for (int tt = 0; tt < 2; tt++) {
        const f16x8 kf = *reinterpret_cast<const f16x8 *>(
            &ks[(32 * kh + 16 * tt + r) * kKRow + 32 * kk + 8 * grp]);
#pragma unroll
        for (int part = 0; part < kParts; part++)
          s[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[part][kk], s[tt], 0, 0, 0);
      }
    if (p0 + 31 > qlo) {
      const int seen = qpos - p0 - 4 * grp;  // positions up to this one
#pragma unroll
      for (int tt = 0; tt < 2; tt++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (16 * tt + e > seen) s[tt][e] = -INFINITY;
    }
    float mx = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                     fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (__any(mx > m_run)) {
      const float m_new = fmaxf(m_run, mx);
      const float corr = m_run == m_new ? 1.0f : exp_neg(m_run - m_new);
      m_run = m_new;
      l_run *= corr;
#pragma unroll
      for (int dt = 0; dt < kDT; dt++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[dt][e] *= corr;
    }
    // (-inf while this part has shown the token nothing)
    const float m = m_run == -INFINITY ? 0.0f : m_run;
    f16x8 p[kParts];
    float ls = 0.0f;
#pragma unroll
    for (int tt = 0; tt < 2; tt++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        // (one fp16 holds 11 bits of P: the plain exp2 is far below that)
        const float x = s[tt][e] - m;
        const float pr = kSplit ? exp_neg(x) : __builtin_amdgcn_exp2f(x * 1.44269504f);
        const _Float16 hi = (_Float16)pr;
        p[0][tt * 4 + e] = hi;
        if (kSplit) {
          p[kParts - 1][tt * 4 + e] = (_Float16)(pr - (float)hi);
          ls += pr;
        } else {
          ls += (float)hi;
        }
      }
    l_run += ls;  // this lane's positions; the groups are summed at the end
#pragma unroll
    for (int dt = 0; dt < kDT; dt++) {
      const _Float16 *vrow = &vs[(16 * dt + r) * kVRow + 32 * kh + 4 * grp];
      const f16x4 v0 = *reinterpret_cast<const f16x4 *>(vrow);
      const f16x4 v1 = *reinterpret_cast<const f16x4 *>(vrow + 16);
      const f16x8 vf = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
      for (int part = 0; part < kParts; part++)
        acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, p[part], acc[dt], 0, 0, 0);
    }
  };
  load(0);
  for (int pt = 0; pt < kend; pt += kKeys) {
    lds_barrier();  // the previous tile's reads are done
    store(pt);
    lds_barrier();
    if (pt + kKeys < kend) load(pt + kKeys);
    if (pt + 32 * kh <= qhi) attend(pt + 32 * kh);
  }

  float l = l_run;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  lds_barrier();  // the last tile's reads are done
#pragma unroll
  for (int dt = 0; dt < kDT; dt++) lds.acc[kh][wave][dt][lane] = acc[dt];
  stat[kh][wave][0][lane] = m_run;
  stat[kh][wave][1][lane] = l;
  lds_barrier();
  // part kh's wave finishes the kh-th of the dims; position 0 is in part 0, so
  // the maximum is finite
  float f[kKP], m = -INFINITY, sum = 0.0f;
#pragma unroll
  for (int k = 0; k < kKP; k++) m = fmaxf(m, f[k] = stat[k][wave][0][lane]);
#pragma unroll
  for (int k = 0; k < kKP; k++) {
    f[k] = exp_neg(f[k] - m);
    sum += stat[k][wave][1][lane] * f[k];
  }
  if (w0 + r >= a.T) return;
#pragma unroll
  for (int dj = 0; dj < kDT / kKP; dj++) {
    const int dt = kh * (kDT / kKP) + dj;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kKP; k++) {
      const f32x4 x = lds.acc[k][wave][dt][lane];
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] += x[e] * f[k];
    }
    f16x4 y;
#pragma unroll
    for (int e = 0; e < 4; e++) y[e] = (_Float16)(o[e] / sum);
    *reinterpret_cast<f16x4 *>(a.attn + qrow + 16 * dt + 4 * grp) = y;
  }
}

template <int kW, int kEpi, int kMI>
hipError_t launch_gemm_tile(hipStream_t s, const PrefillGemmArgs &g) {
  const int tiles_m = (g.M + 32 * kMI - 1) / (32 * kMI);
  const int ntiles = tiles_m * (g.N / (32 * kMI)), per_xcd = (ntiles + 7) / 8;
  prefill_gemm_kernel<kW, kEpi, kMI><<<per_xcd * 8, kT * groups_of(kEpi), 0, s>>>(g, tiles_m, ntiles, per_xcd);
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
  const int per = attn_tokens(a.d);
  const dim3 grid(a.heads, (a.T + per - 1) / per, a.B);
  if (a.d == 128 && a.vt_stride)
    prefill_attn_kernel<128, true, false><<<grid, kAttnT, 0, s>>>(a);
  else if (a.d == 128)
    prefill_attn_kernel<128, false, true><<<grid, kAttnT, 0, s>>>(a);
  else if (a.d == 64 && !a.vt_stride)
    prefill_attn_kernel<64, false, true><<<grid, kAttnT, 0, s>>>(a);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace sh
