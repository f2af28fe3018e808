// The parts of a prompt's pass (prefill.hip) for models whose steps run on the
// decode-layers kernel: its RMSNorm, q / k norms, RoPE, attention and merge,
// operation by operation, over many tokens at once. Compiled without
// floating-point contraction, as decode_layers.hip is; what that kernel fuses
// it writes as fmaf, and so does this file.
#include <hip/hip_runtime.h>

#include "common.h"
#include "llm.h"
#include "llm_device.h"
#include "prefill_gemm.h"

namespace sh {
namespace {

using prompt::kT;
using prompt::lds_barrier;

constexpr int kD = 128;  // head dim
constexpr int kG = 2;    // query heads per KV head

// ---- norm ------------------------------------------------------------------------

// One workgroup per row (stage_rms with kPost): fp16 x * g, and the scale 1 /
// rms, which the linear's epilogue applies. kP: 2-value pairs per thread.
template <int kP>
__global__ __launch_bounds__(kT) void prefill_norm_layers_kernel(const float *x, const float *gamma,
                                                                 uint16_t *out16, float *inv, int K,
                                                                 float eps) {
  __shared__ float part[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c2 = K >> 1;
  const float *row = x + (size_t)blockIdx.x * K;
  auto pair = [&](int i) { return wave * (K >> 3) + lane + 64 * i; };
  auto pair_ok = [&](int i) { return lane + 64 * i < (K >> 3); };
  f32x2 gv[kP], v[kP];
#pragma unroll
  for (int i = 0; i < kP; i++) {
    const int c = min(pair(i), c2 - 1);
    gv[i] = *reinterpret_cast<const f32x2 *>(gamma + c * 2);
    v[i] = *reinterpret_cast<const f32x2 *>(row + c * 2);
  }
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < kP; i += 2) {
    const float s0 = pair_ok(i) ? fmaf(v[i][0], v[i][0], v[i][1] * v[i][1]) : 0.0f;
    const float s1 = pair_ok(i + 1) ? fmaf(v[i + 1][0], v[i + 1][0], v[i + 1][1] * v[i + 1][1]) : 0.0f;
    ss += s0 + s1;
  }
  ss = wave_sum_rows(ss);
  if (lane == 0) part[wave] = ss;
#pragma unroll
  for (int i = 0; i < kP; i++) {
    if (pair_ok(i)) {
      const f32x2 y = v[i] * gv[i];
      *reinterpret_cast<f16x2 *>(out16 + f16_tiled_offset(blockIdx.x, pair(i) * 2, K)) =
          f16x2{(_Float16)y[0], (_Float16)y[1]};
    }
  }
  lds_barrier();
  if (threadIdx.x == 0) {
    const float sum = (part[0] + part[1]) + (part[2] + part[3]);
    inv[blockIdx.x] = 1.0f / sqrtf(sum / (float)K + eps);
  }
}

// ---- q, k, v of the chunk ---------------------------------------------------------

constexpr int kPostTokens = 16;

// grid (ceil(T / 16), heads + 2 kv_heads, B): one head of 16 tokens, as
// attn_item prepares them: lane j holds values 2 j and 2 j + 1, RMSNorm over
// the head, RoPE with the partner in lane j +- 32. Query heads: times the
// softmax scale, as fp16; key heads: appended to the K cache; value heads:
// appended to the V cache (transposed, [d][vt_stride]).
__global__ __launch_bounds__(kT) void prefill_qkv_layers_kernel(const PrefillArgs a, int first_head) {
  __shared__ _Float16 vt[kPostTokens][kD + 2];
  const int hh = blockIdx.y + first_head, b = blockIdx.z;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int i_first = blockIdx.x * kPostTokens;
  const int p_first = max(a.lens[b], 0) + a.i0 + i_first;
  const bool is_q = hh < a.heads, is_k = !is_q && hh < a.heads + a.kv_heads;
  const int kvh = is_q ? 0 : (hh - a.heads) % a.kv_heads;
  const size_t cache = (size_t)b * a.kv_heads + kvh;
  const int e0 = 2 * lane, fe = e0 & (kD / 2 - 1);
  const f32x2 g = *reinterpret_cast<const f32x2 *>((is_q ? a.q_norm : a.k_norm) + e0);
#pragma unroll
  for (int u = 0; u < kPostTokens / 4; u++) {
    const int r = wave * (kPostTokens / 4) + u, i = i_first + r, pos = p_first + r;
    if (i >= a.T) break;  // wave-uniform
    const size_t m = (size_t)b * a.T + i;
    const f32x2 v = *reinterpret_cast<const f32x2 *>(a.qkv + m * a.qkv_n + (size_t)hh * kD + e0);
    float v0 = v.x, v1 = v.y;
    if (is_q || is_k) {
      const f32x2 cs = *reinterpret_cast<const f32x2 *>(a.rope + m * kD + fe);
      const f32x2 sn = *reinterpret_cast<const f32x2 *>(a.rope + m * kD + kD / 2 + fe);
      const float ss = wave_sum_rows(fmaf(v0, v0, v1 * v1));
      const float inv = 1.0f / sqrtf(ss / kD + a.eps);
      v0 = v0 * inv * g.x;
      v1 = v1 * inv * g.y;
      const float o0 = __shfl_xor(v0, 32, 64), o1 = __shfl_xor(v1, 32, 64);
      if (lane < 32) {
        v0 = fmaf(v0, cs.x, -(o0 * sn.x));
        v1 = fmaf(v1, cs.y, -(o1 * sn.y));
      } else {
        v0 = fmaf(v0, cs.x, o0 * sn.x);
        v1 = fmaf(v1, cs.y, o1 * sn.y);
      }
    }
    if (is_q) {
      *reinterpret_cast<f16x2 *>(a.q + (m * a.heads + hh) * kD + e0) =
          f16x2{f16_of_f32(v0 * a.scale), f16_of_f32(v1 * a.scale)};
    } else if (is_k) {
      if (pos < a.max_pos)
        *reinterpret_cast<f16x2 *>(a.kcache + (cache * a.max_pos + pos) * kD + e0) =
            f16x2{f16_of_f32(v0), f16_of_f32(v1)};
    } else {
      vt[r][e0] = (_Float16)v0;
      vt[r][e0 + 1] = (_Float16)v1;
    }
  }
  if (is_q || is_k) return;  // workgroup-uniform
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

constexpr int kMaxSplits = 64;
constexpr int kGroups = 16;    // split groups of a merge (merge_item)
constexpr int kSumTiles = 16;  // 16-position partial sums of the softmax

__device__ __forceinline__ bool finite_f16(_Float16 v) {
  return (__builtin_bit_cast(uint16_t, v) & 0x7c00u) != 0x7c00u;
}

// A workgroup's part of the attention: kU 16-row MFMA operands, rows (token,
// query head of the KV head), against the cache of KV head kvh in sequence b.
// Token k sees positions 0 .. base + k; rows past the last token repeat it.
template <int kU>
struct AttnBlock {
  static constexpr int kRows = 16 * kU, kTokens = kRows / kG;
  int kvh, b, i0, n, base, end, active;
  const uint16_t *kb;
  __device__ __forceinline__ explicit AttnBlock(const PrefillArgs &a) {
    // workgroups x, x + kv_heads, .. share a KV head: with 8 of those an XCD's L2
    // holds the one it works on. The longest half of the blocks first, longest
    // first; then the others, shortest first: a CU's second workgroup evens out
    // its first
    kvh = blockIdx.x;
    b = blockIdx.z;
    const int blocks = gridDim.y, by = blockIdx.y, half = (blocks + 1) / 2;
    i0 = kTokens * (by < half ? blocks - 1 - by : by - half);
    n = min(kTokens, a.T - i0);
    base = max(a.lens[b], 0) + a.i0 + i0;
    end = min(base + n, a.max_pos);
    active = (end + a.chunk - 1) / a.chunk;
    kb = a.kcache + ((size_t)b * a.kv_heads + kvh) * a.max_pos * kD;
  }
  __device__ __forceinline__ int token(int row) const { return i0 + min(row / kG, n - 1); }
  __device__ __forceinline__ int seen(const PrefillArgs &a, int row) const {
    return min(base + min(row / kG, n - 1) + 1, a.max_pos);
  }
  // (token, query head) of a row as an index
  __device__ __forceinline__ size_t head_row(const PrefillArgs &a, int row) const {
    return ((size_t)b * a.T + token(row)) * a.heads + kvh * kG + row % kG;
  }
  __device__ __forceinline__ void load_q(const PrefillArgs &a, f16x8 (&qa)[kU][4]) const {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const uint16_t *q = a.q + head_row(a, 16 * u + (lane & 15)) * kD + 8 * (lane >> 4);
#pragma unroll
      for (int kk = 0; kk < 4; kk++) qa[u][kk] = *reinterpret_cast<const f16x8 *>(q + 32 * kk);
    }
  }
  // K of tile x (this wave's: 16 positions from pb + 16 (wave + 4 x)), dims 32 kk
  // .., as load_rows takes them (positions past the last seen one re-read it:
  // never counted)
  __device__ __forceinline__ void load_k(int pb, int x, f16x8 (&raw)[4]) const {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p = min(pb + 16 * (wave + 4 * x) + (lane >> 2), end - 1);
#pragma unroll
    for (int kk = 0; kk < 4; kk++)
      raw[kk] = *reinterpret_cast<const f16x8 *>(kb + (size_t)p * kD + 8 * (lane & 3) + 32 * kk);
  }
};

// Sixteen rows of 32 values as an MFMA operand has them: lane % 16 the row,
// 8 (lane / 16) .. the values. Loaded like that, every lane would be a request
// of its own to the cache (64 a load); so four neighbouring lanes load 64 bytes
// of a row (raw), and the wave turns them round in LDS of its own. The 16-byte
// slots are swizzled by the row, which keeps both ways free of bank conflicts.
__device__ __forceinline__ void turn_rows(_Float16 *area, const f16x8 (&raw)[4], f16x8 (&frag)[4]) {
  const int lane = threadIdx.x & 63, wr = lane >> 2, rd = lane & 15;
  _Float16 *w = area + wr * 32 + (((lane & 3) ^ ((wr >> 2) & 3)) * 8);
  const _Float16 *r = area + rd * 32 + (((lane >> 4) ^ ((rd >> 2) & 3)) * 8);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);  // (a wave's LDS accesses run in order)
#pragma unroll
  for (int i = 0; i < 4; i++) *reinterpret_cast<f16x8 *>(w + 512 * i) = raw[i];
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
#pragma unroll
  for (int i = 0; i < 4; i++) frag[i] = *reinterpret_cast<const f16x8 *>(r + 512 * i);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// A step splits the context into fixed chunks, takes each chunk's softmax
// against its own maximum (P rounded to fp16, its sum over the rounded values)
// and merges the chunks. The pass does the same in two kernels. The first,
// grid (kv_heads, ceil(T / 16), B): the maximum of each chunk's scores for
// every row of 16 tokens (a maximum does not depend on an order). (32 tokens:
// 18 us for 14 at 1,023 tokens of 16 heads, 97 for 106 at 4,090.)
constexpr int kMaxU = 2;
__global__ __launch_bounds__(kT, 2) void prefill_attn_max_kernel(const PrefillArgs a) {
  constexpr int kX = 3, kRows = 16 * kMaxU;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  _Float16 *turn = reinterpret_cast<_Float16 *>(smem) + (threadIdx.x >> 6) * 2048;  // 4 KiB a wave
  float (*mx)[4][kRows] = reinterpret_cast<float (*)[4][kRows]>(smem + 4 * 4096);  // [splits]
  const AttnBlock<kMaxU> B(a);
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r16 = lane & 15, grp = lane >> 4;
  f16x8 qa[kMaxU][4], raw[kX][4];
  B.load_q(a, qa);
  auto load_k = [&](int pb) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < kX; x++) B.load_k(pb, x, raw[x]);
  };
  load_k(0);
  for (int j = 0; j < B.active; j++) {
    f32x4 top[kMaxU];
#pragma unroll
    for (int u = 0; u < kMaxU; u++) top[u] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    const int p0 = j * a.chunk, pe = min(p0 + a.chunk, B.end);
    for (int pb = p0; pb < pe; pb += 64 * kX) {
      f32x4 sc[kX][kMaxU];
#pragma unroll
      for (int x = 0; x < kX; x++) {
        f16x8 kf[4];
        turn_rows(turn, raw[x], kf);
#pragma unroll
        for (int u = 0; u < kMaxU; u++) sc[x][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
          for (int u = 0; u < kMaxU; u++)
            sc[x][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(qa[u][kk], kf[kk], sc[x][u], 0, 0, 0);
      }
      load_k(pb + 64 * kX < pe ? pb + 64 * kX : p0 + a.chunk);
#pragma unroll
      for (int x = 0; x < kX; x++) {
        const int pt = pb + 16 * (wave + 4 * x), p = pt + r16;
        if (pt >= pe) continue;  // wave-uniform
        if (pe <= B.base + 1) {  // uniform: every row sees the whole chunk
#pragma unroll
          for (int u = 0; u < kMaxU; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) top[u][r] = fmaxf(top[u][r], sc[x][u][r]);
        } else {
#pragma unroll
          for (int u = 0; u < kMaxU; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const bool is = p < min(B.seen(a, 16 * u + 4 * grp + r), pe);
              top[u][r] = fmaxf(top[u][r], is ? sc[x][u][r] : -INFINITY);
            }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kMaxU; u++) {
#pragma unroll
      for (int r = 0; r < 4; r++) top[u][r] = row16_max(top[u][r]);
      if (r16 == 0) *reinterpret_cast<f32x4 *>(&mx[j][wave][16 * u + 4 * grp]) = top[u];
    }
  }
  lds_barrier();
  for (int e = t; e < kRows * B.active; e += kT) {
    const int row = e / B.active, j = e % B.active;
    if (row / kG >= B.n) break;  // (rows of later e are larger)
    a.smax[B.head_row(a, row) * a.splits + j] =
        fmaxf(fmaxf(mx[j][0][row], mx[j][1][row]), fmaxf(mx[j][2][row], mx[j][3][row]));
  }
}

// LDS, then (dynamic), per split and row: the chunk's maximum (-inf where the row
// has no such split), its weight exp(m - M_group) and its softmax sum.
template <int kX, int kU>
struct AttnLds {
  static constexpr int kRows = 16 * kU;
  typedef float PerSplit[kRows];
  static size_t bytes(int splits) { return sizeof(AttnLds) + (size_t)splits * 3 * sizeof(PerSplit); }
  alignas(16) _Float16 q[kRows][kD + 8];            // rows padded
  alignas(16) _Float16 turn[4][2048];               // turn_rows, 4 KiB a wave
  alignas(16) _Float16 p[2][kRows][64 * kX + 8];    // P of a block, rows padded
  alignas(16) float tile_sum[2][kSumTiles][kRows];  // softmax sums per 16-position tile
  alignas(16) float mg[kGroups][kRows];             // maximum of a group's chunks; at the end its l
  alignas(16) float wg[kGroups][kRows];             // exp(M_group - M) of a row, 0 without active splits
  alignas(16) float inv[kRows];
};

// The second kernel, grid (kv_heads, ceil(T / (8 kU)), B): chunk after chunk in
// the merge's order, the scores again, P, the sums of P by 16-position tiles as
// the step's lanes and waves add them, V sums in 32-position MFMA steps from
// the chunk's start, weighted into the sums of the chunk's group, the groups
// added as the merge's lanes and waves add them. Scores and V sums are the
// step's MFMAs with 16 kU rows in place of its two. A wave scores every fourth
// tile of 16 positions, kX of them per block of 64 kX positions, and owns 32
// output dims. kX: 3 where a block holds a chunk (192 positions or fewer), else
// 2, of which two blocks fill the 16 tiles that the softmax sums are kept by.
//
// What bounds it is the vector work of the softmax as the step does it (an
// expf, two conversions and a lane sum per score: some 900 instructions per
// wave and chunk of 144 positions) with two waves per SIMD. 1,023 tokens of 16
// heads 44 us, 4,090 tokens 360; one 16-row operand per workgroup 63 and 650.
template <int kX, int kU>
__global__ __launch_bounds__(kT, 2) void prefill_attn_layers_kernel(const PrefillArgs a) {
  constexpr bool kOne = kX == 3;            // one block per chunk
  constexpr int kBlock = 64 * kX, kRows = 16 * kU;
  typedef AttnLds<kX, kU> Lds;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  Lds &S = *reinterpret_cast<Lds *>(smem);
  typename Lds::PerSplit *sm = reinterpret_cast<typename Lds::PerSplit *>(smem + sizeof(Lds));
  typename Lds::PerSplit *sw = sm + a.splits, *sl = sw + a.splits;
  const AttnBlock<kU> B(a);
  const int base = B.base, end = B.end, active = B.active, chunk = a.chunk;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r16 = lane & 15, grp = lane >> 4;
  for (int e = t; e < kRows * kD / 8; e += kT) {
    const int row = e / (kD / 8), c = e % (kD / 8) * 8;
    *reinterpret_cast<f16x8 *>(&S.q[row][c]) = *reinterpret_cast<const f16x8 *>(a.q + B.head_row(a, row) * kD + c);
  }
  // V^T rows of this wave's dims: by output column, and as the loads take them
  const uint16_t *vb = a.vcache + (((size_t)B.b * a.kv_heads + B.kvh) * kD + 32 * wave + r16) * a.vt_stride;
  const uint16_t *vl = vb + (ptrdiff_t)((lane >> 2) - r16) * a.vt_stride;
  int lim[kU][4];  // positions that this lane's accumulator rows, 16 u + 4 grp + r, see
#pragma unroll
  for (int u = 0; u < kU; u++)
#pragma unroll
    for (int r = 0; r < 4; r++) lim[u][r] = B.seen(a, 16 * u + 4 * grp + r);
  // blocks of chunk j that any token sees
  auto blocks = [&](int j) { return kOne ? 1 : (min(chunk, end - j * chunk) + kBlock - 1) / kBlock; };

  for (int e = t; e < active * kRows; e += kT) {
    const int row = e / active, j = e % active;
    sm[j][row] = j * chunk < B.seen(a, row) ? a.smax[B.head_row(a, row) * a.splits + j] : -INFINITY;
  }
  for (int e = t; e < 2 * kSumTiles * kRows; e += kT) (&S.tile_sum[0][0][0])[e] = 0.0f;
  lds_barrier();
  // group g: chunks g, g + 16, ..
  for (int e = t; e < kGroups * kRows; e += kT) {
    const int g = e / kRows, row = e % kRows;
    float mg = -INFINITY;
    for (int j = g; j < active; j += kGroups) mg = fmaxf(mg, sm[j][row]);
    S.mg[g][row] = mg;
  }
  lds_barrier();
  for (int e = t; e < kGroups * kRows; e += kT) {
    const int g = e / kRows, row = e % kRows;
    float M = -INFINITY;
#pragma unroll
    for (int k = 0; k < kGroups; k++) M = fmaxf(M, S.mg[k][row]);
    const float mg = S.mg[g][row];
    S.wg[g][row] = mg == -INFINITY ? 0.0f : expf(mg - M);
    for (int j = g; j < active; j += kGroups) sw[j][row] = expf(sm[j][row] - mg);  // (used where the row has the split)
  }
  lds_barrier();

  // out: the merge's waves added so far; pair: its lanes 0 + 1, and 2, of a
  // wave; gs: a group
  f32x4 out[kU][2], pair[2][kU][2];
#pragma unroll
  for (int u = 0; u < kU; u++)
#pragma unroll
    for (int nt = 0; nt < 2; nt++) out[u][nt] = pair[0][u][nt] = pair[1][u][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  int buf = 0;
  for (int g = 0; g < kGroups; g++) {
    f32x4 gs[kU][2];
#pragma unroll
    for (int u = 0; u < kU; u++)
#pragma unroll
      for (int nt = 0; nt < 2; nt++) gs[u][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int j = g; j < active; j += kGroups) {
      const int p0 = j * chunk, pe = p0 + chunk, nb = blocks(j);
      f32x4 oacc[kU][2];
      f32x4 es[4][kU];  // (kX = 2) P by tile % 16 = wave + 4 x, this lane's position of the tile
#pragma unroll
      for (int u = 0; u < kU; u++) {
#pragma unroll
        for (int nt = 0; nt < 2; nt++) oacc[u][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int x = 0; x < 4; x++) es[x][u] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      auto block = [&](int h, auto odd_c) __attribute__((always_inline)) {
        constexpr int kX0 = decltype(odd_c)::value * 2;
        const int pb = p0 + h * kBlock;
        // K of the block, and V^T: two 16-dim operands per 32-position step
        // (positions past the chunk re-read its last ones, which P is 0 for)
        f16x8 kr[kX][4], vr[kX][4];
#pragma unroll
        for (int x = 0; x < kX; x++) B.load_k(pb, x, kr[x]);
#pragma unroll
        for (int x = 0; x < kX; x++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const int p = min(pb + 64 * x + 32 * (i >> 1) + 8 * (lane & 3), min(pe, a.vt_stride) - 8);
            vr[x][i] = *reinterpret_cast<const f16x8 *>(vl + (size_t)(16 * (i & 1)) * a.vt_stride + p);
          }
        f32x4 sc[kX][kU];
#pragma unroll
        for (int x = 0; x < kX; x++) {
          f16x8 kf[4];
          turn_rows(S.turn[wave], kr[x], kf);
#pragma unroll
          for (int u = 0; u < kU; u++) sc[x][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int u = 0; u < kU; u++) {
              const f16x8 qa = *reinterpret_cast<const f16x8 *>(&S.q[16 * u + r16][32 * kk + 8 * grp]);
              sc[x][u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(qa, kf[kk], sc[x][u], 0, 0, 0);
            }
        }
#pragma unroll
        for (int x = 0; x < kX; x++) {
          const int pt = pb + 16 * (wave + 4 * x), p = pt + r16;
          const bool any = pt < min(pe, end);  // wave-uniform: the tile has positions of the chunk
#pragma unroll
          for (int u = 0; u < kU; u++) {
            const f32x4 mrow = *reinterpret_cast<const f32x4 *>(&sm[j][16 * u + 4 * grp]);
            f32x4 e4 = {0.f, 0.f, 0.f, 0.f};
            if (any) {
#pragma unroll
              for (int r = 0; r < 4; r++) e4[r] = (float)(_Float16)expf(sc[x][u][r] - mrow[r]);
              if (pe > base + 1) {  // uniform: not every row sees the whole chunk
#pragma unroll
                for (int r = 0; r < 4; r++) e4[r] = p < lim[u][r] ? e4[r] : 0.0f;
              }
            }
#pragma unroll
            for (int r = 0; r < 4; r++) S.p[buf][16 * u + 4 * grp + r][16 * (wave + 4 * x) + r16] = (_Float16)e4[r];
            if constexpr (kOne) {
#pragma unroll
              for (int r = 0; r < 4; r++) e4[r] = row16_sum(e4[r]);
              if (r16 == 0) *reinterpret_cast<f32x4 *>(&S.tile_sum[buf][wave + 4 * x][16 * u + 4 * grp]) = e4;
            } else {
#pragma unroll
              for (int r = 0; r < 4; r++) es[(kX0 + x) & 3][u][r] += e4[r];
            }
          }
        }
        lds_barrier();
        const int pv_end = min(pe, end);  // positions from here on have no weight
        bool odd = false;
#pragma unroll
        for (int x = 0; x < kX; x++) {
          if (pb + 64 * x >= pv_end) break;  // uniform
          f16x8 vf[4];
          turn_rows(S.turn[wave], vr[x], vf);
          if (pb + 64 * x + 64 > base + 1) {  // uniform: some of the positions are not every token's
            // 0 times an infinity or NaN is not 0: such values of the last tokens'
            // positions are taken out, and added to the tokens that see them below
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
              for (int e = 0; e < 8; e++) {
                const int p = pb + 64 * x + 32 * (i >> 1) + 8 * grp + e;
                const bool bad = p > base && !finite_f16(vf[i][e]);
                odd |= bad && p < pv_end;
                vf[i][e] = p < pv_end && !bad ? vf[i][e] : (_Float16)0.0f;
              }
          }
#pragma unroll
          for (int h2 = 0; h2 < 2; h2++) {
            const int ks = 2 * x + h2;
            if (pb + 32 * ks >= pv_end) break;  // uniform
#pragma unroll
            for (int u = 0; u < kU; u++) {
              const f16x8 pa = *reinterpret_cast<const f16x8 *>(&S.p[buf][16 * u + r16][32 * ks + 8 * grp]);
#pragma unroll
              for (int nt = 0; nt < 2; nt++)
                oacc[u][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa, vf[2 * h2 + nt], oacc[u][nt], 0, 0, 0);
            }
          }
        }
        if (__any(odd)) {
#pragma unroll 1
          for (int p = max(pb, base + 1); p < min(pb + kBlock, pv_end); p++)
#pragma unroll
            for (int nt = 0; nt < 2; nt++) {
              const uint16_t bits = vb[(size_t)(16 * nt) * a.vt_stride + p];
              const _Float16 v = __builtin_bit_cast(_Float16, bits);
#pragma unroll
              for (int u = 0; u < kU; u++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                  const float x = (float)S.p[buf][16 * u + 4 * grp + r][p - pb] * (float)v;
                  if (!finite_f16(v) && p < lim[u][r]) oacc[u][nt][r] += x;
                }
            }
        }
        buf ^= 1;  // (a wave two blocks ahead has passed a barrier after this block's reads)
      };
      if constexpr (kOne) {
        block(0, std::integral_constant<int, 0>{});
      } else {
        for (int h = 0; h < nb; h += 2) {
          block(h, std::integral_constant<int, 0>{});
          if (h + 1 < nb) block(h + 1, std::integral_constant<int, 1>{});
        }
#pragma unroll
        for (int x = 0; x < 4; x++)
#pragma unroll
          for (int u = 0; u < kU; u++) {
            f32x4 v;
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = row16_sum(es[x][u][r]);
            if (r16 == 0) *reinterpret_cast<f32x4 *>(&S.tile_sum[buf ^ 1][wave + 4 * x][16 * u + 4 * grp]) = v;
          }
        lds_barrier();
      }
      if (t < kRows) {  // this chunk's softmax sum
        float w4[4];
#pragma unroll
        for (int w = 0; w < 4; w++)
          w4[w] = (S.tile_sum[buf ^ 1][4 * w][t] + S.tile_sum[buf ^ 1][4 * w + 1][t]) +
                  (S.tile_sum[buf ^ 1][4 * w + 2][t] + S.tile_sum[buf ^ 1][4 * w + 3][t]);
        sl[j][t] = (w4[0] + w4[1]) + (w4[2] + w4[3]);
      }
      // the chunk into its group, against the group's maximum
#pragma unroll
      for (int u = 0; u < kU; u++) {
        const f32x4 wj = *reinterpret_cast<const f32x4 *>(&sw[j][16 * u + 4 * grp]);
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
          for (int nt = 0; nt < 2; nt++)
            gs[u][nt][r] = p0 < lim[u][r] ? fmaf(wj[r], oacc[u][nt][r], gs[u][nt][r]) : gs[u][nt][r];
      }
    }
    // the groups' tree: lanes (4 w + 0) + (4 w + 1), (4 w + 2) + (4 w + 3), their sum, then
    // the waves w one after another
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const f32x4 w = *reinterpret_cast<const f32x4 *>(&S.wg[g][16 * u + 4 * grp]);
#pragma unroll
      for (int nt = 0; nt < 2; nt++) {
        const f32x4 v = gs[u][nt] * w;
        switch (g & 3) {
          case 0: pair[0][u][nt] = v; break;
          case 1: pair[0][u][nt] = pair[0][u][nt] + v; break;
          case 2: pair[1][u][nt] = v; break;
          default: out[u][nt] = out[u][nt] + (pair[0][u][nt] + (pair[1][u][nt] + v)); break;
        }
      }
    }
    if (g + 1 >= active && (g & 3) == 3) break;  // the other groups add zeros
  }
  lds_barrier();  // the last chunk's sum
  for (int e = t; e < kGroups * kRows; e += kT) {
    const int g = e / kRows, row = e % kRows, row_seen = B.seen(a, row);
    float l = 0.0f;
    for (int j = g; j < active; j += kGroups)
      if (j * chunk < row_seen) l = fmaf(sw[j][row], sl[j][row], l);
    S.mg[g][row] = l * S.wg[g][row];
  }
  lds_barrier();
  if (t < kRows) {
    float lsum = 0.0f;
#pragma unroll
    for (int w = 0; w < kGroups / 4; w++)
      lsum += (S.mg[4 * w][t] + S.mg[4 * w + 1][t]) + (S.mg[4 * w + 2][t] + S.mg[4 * w + 3][t]);
    S.inv[t] = 1.0f / lsum;
  }
  lds_barrier();
#pragma unroll
  for (int u = 0; u < kU; u++) {
    const f32x4 inv = *reinterpret_cast<const f32x4 *>(&S.inv[16 * u + 4 * grp]);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int row = 16 * u + 4 * grp + r;
      if (row / kG >= B.n) continue;
      const int col = (B.kvh * kG + row % kG) * kD + 32 * wave + r16;
#pragma unroll
      for (int nt = 0; nt < 2; nt++)
        a.attn[f16_tiled_offset(B.b * a.T + B.i0 + row / kG, col + 16 * nt, a.heads * kD)] =
            __builtin_bit_cast(uint16_t, f16_product(out[u][nt][r], inv[r]));
    }
  }
}

template <int kX, int kU>
void launch_attn(hipStream_t s, const PrefillArgs &a) {
  const dim3 grid(a.kv_heads, (a.T + 8 * kU - 1) / (8 * kU), a.B);
  prefill_attn_layers_kernel<kX, kU><<<grid, kT, AttnLds<kX, kU>::bytes(a.splits), s>>>(a);
}

}  // namespace

hipError_t launch_prefill_norm_layers(hipStream_t s, const PrefillArgs &a, const float *gamma) {
  const int M = a.B * a.T;
  if (a.H <= 1024)
    prefill_norm_layers_kernel<2><<<M, kT, 0, s>>>(a.x, gamma, a.h16, a.inv, a.H, a.eps);
  else if (a.H <= 4096)
    prefill_norm_layers_kernel<8><<<M, kT, 0, s>>>(a.x, gamma, a.h16, a.inv, a.H, a.eps);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_prefill_gemm_layers(hipStream_t s, const PrefillGemmArgs &g, int epi) {
  if (g.M < 1 || g.N % 64 != 0 || g.K % 256 != 0 || g.K < 256 || !g.scale || g.bias) return hipErrorInvalidValue;
  if (epi == kEpiResidual) return prompt::launch_gemm<kWeightFp8, kEpiResidual, kStepQwenLayers>(s, g);
  if (!g.inv) return hipErrorInvalidValue;
  if (epi == kEpiStore) return prompt::launch_gemm<kWeightFp8, kEpiStore, kStepQwenLayers>(s, g);
  if (epi == kEpiSwiGLU) return prompt::launch_gemm<kWeightFp8, kEpiSwiGLU, kStepQwenLayers>(s, g);
  return hipErrorInvalidValue;
}

hipError_t launch_prefill_qkv_layers(hipStream_t s, const PrefillArgs &a, bool kv_only) {
  if (a.d != kD) return hipErrorInvalidValue;
  const int first = kv_only ? a.heads : 0;
  const dim3 grid((a.T + kPostTokens - 1) / kPostTokens, a.heads + 2 * a.kv_heads - first, a.B);
  prefill_qkv_layers_kernel<<<grid, kT, 0, s>>>(a, first);
  return hipGetLastError();
}

// LDS of prefill_attn_max_kernel.
static size_t attn_max_lds(int splits) { return 4 * 4096 + (size_t)splits * 4 * 16 * kMaxU * sizeof(float); }

hipError_t prepare_prefill_kernels() {
  const struct {
    const void *kernel;
    size_t lds;
  } all[] = {{reinterpret_cast<const void *>(&prefill_attn_max_kernel), attn_max_lds(kMaxSplits)},
             {reinterpret_cast<const void *>(&prefill_attn_layers_kernel<3, 2>), AttnLds<3, 2>::bytes(kMaxSplits)},
             {reinterpret_cast<const void *>(&prefill_attn_layers_kernel<2, 1>), AttnLds<2, 1>::bytes(kMaxSplits)}};
  for (const auto &k : all) {
    const hipError_t e = hipFuncSetAttribute(k.kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)k.lds);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_prefill_attention_layers(hipStream_t s, const PrefillArgs &a) {
  if (a.d != kD || a.heads != kG * a.kv_heads || a.chunk % 16 != 0 || a.splits > kMaxSplits ||
      (long long)a.splits * a.chunk < a.max_pos)
    return hipErrorInvalidValue;
  const dim3 grid(a.kv_heads, (a.T + 8 * kMaxU - 1) / (8 * kMaxU), a.B);
  prefill_attn_max_kernel<<<grid, kT, attn_max_lds(a.splits), s>>>(a);
  if (a.chunk > 64 * 3)
    launch_attn<2, 1>(s, a);
  else
    launch_attn<3, 2>(s, a);
  return hipGetLastError();
}

}  // namespace sh
