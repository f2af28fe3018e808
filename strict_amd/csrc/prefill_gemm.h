// The linears of a prompt's pass (prefill.hip, prefill_layers.hip): GEMMs over
// the token rows, fp16 activations times the model's own tiled FP8 / fp16
// weights, on MFMA. A decode step's GEMV fixes the order in which an output's
// products are summed, and this kernel keeps that order:
//  - K in four quarters (the GEMVs' four waves), a quarter's 32-wide MFMA steps
//    dealt to kCh accumulator chains in turn, the chains added in order;
//  - the quarters added as (0 + 1) + (2 + 3) (the layers kernels) or one after
//    another (the per-op GEMV), then the step's epilogue.
// So an output does not depend on which of the two computed it, on the batch
// or on the tile it is in.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.h"
#include "llm.h"
#include "llm_device.h"

namespace sh {
namespace prompt {

constexpr int kT = 256;
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

// Workgroup barrier for LDS traffic only: __syncthreads() would also wait for
// outstanding global loads.
__device__ __forceinline__ void lds_barrier() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Accumulator chains of a K quarter in the step kernels (decode_layers.hip
// and gpt2_layers.hip mfma_weights; the per-op GEMV has one).
constexpr int chains_of(int form, int epi) {
  return form == kStepOps ? 1 : form == kStepQwenLayers && epi == kEpiSwiGLU ? 2 : 4;
}

// Token rows whose tiles are taken together, so that they stay in an XCD's L2
// while the weights pass: gate / up of 4,090 tokens (8 MB of rows) 116 us in one
// panel, 93 in panels of 2 MiB, down 53 and 38.
constexpr int kPanelBytes = 2 << 20;

// A workgroup owns 16 kI tokens x 16 kJ outputs, each of its waves a quarter of
// K for all of them. Weight tiles are in MFMA operand order, and so are the
// token rows (f16_tiled_offset). Row-major rows lie a power of two apart: 16
// of them at a time kept the L2's channels waiting for two of their number (gate
// / up of 1,023 tokens 41 us, 28 with tiles). Both go straight into registers,
// two 64-wide stages ahead, and the waves only meet to add their sums, through
// LDS. The MFMA is issued as W x A, which leaves a lane with 4 consecutive
// outputs of one token (16-byte fp32, 8-byte fp16 stores).
// kI x kJ: 16-row tiles of tokens and of outputs. kHalf: the quarter ends with
// half a stage.
template <int kW, int kEpi, int kForm, int kI, int kJ, bool kHalf>
__global__ __launch_bounds__(kT, 2) void gemm_kernel(const PrefillGemmArgs g, int tiles_m, int ntiles,
                                                     int per_xcd, int panel) {
  constexpr int kOwn = kI * kJ / 4;              // tiles that a wave finishes
  static_assert(kJ % kOwn == 0 && kOwn % 2 == 0, "a wave's tiles are of the same tokens, in pairs");
  constexpr int kWL = kW == kWeightFp8 ? 1 : 2;  // 16-byte weight loads per tile and stage
  constexpr int kCh = chains_of(kForm, kEpi);
  __shared__ f32x4 red[4][kI * kJ][64];
  // each XCD takes a run of tiles, tokens fastest: its L2 then reads few
  // weight rows, once
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= ntiles) return;
  int tm, tn;
  {
    // panels of token tiles, whole but for the last one
    const int width = g.N / (16 * kJ), p = tile / (panel * width);
    const int rest = tile - p * panel * width, high = min(panel, tiles_m - p * panel);
    tn = rest / high;
    tm = p * panel + rest % high;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, grp = lane >> 4;
  const int m0 = tm * 16 * kI, nt0 = tn * kJ;
  // this wave's quarter in 32-wide steps and in 64-wide stages (fp16: the
  // last stage may be half of one)
  const int steps = g.K / 128, nst = (steps + 1) / 2;

  const uint16_t *arow[kI];
  const size_t astep = g.a_tiled ? 512 : 32;  // fp16 values from one 32-wide step to the next
#pragma unroll
  for (int i = 0; i < kI; i++)
    arow[i] = g.a_tiled ? g.a + ((size_t)min(m0 / 16 + i, (g.M - 1) / 16) * (g.K / 32) + wave * steps) * 512 + lane * 8
                        : g.a + (size_t)min(m0 + 16 * i + r16, g.M - 1) * g.K + wave * (g.K / 4) + 8 * grp;
  const int row_tiles = g.K / (kW == kWeightFp8 ? 64 : 32);  // 1 KiB tiles of an output tile's K
  const uint8_t *wrow[kJ];
#pragma unroll
  for (int j = 0; j < kJ; j++)
    wrow[j] = g.w + ((size_t)(nt0 + j) * row_tiles + (size_t)wave * (row_tiles / 4)) * 1024 + lane * 16;

  f16x8 ra[2][kI][2];
  u32x4 rw[2][kJ][kWL];
  // (past the end of the quarter: its last step again, unused)
  auto load = [&](int s, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int step = min(2 * st + h, steps - 1);
#pragma unroll
      for (int i = 0; i < kI; i++)
        ra[s][i][h] = *reinterpret_cast<const f16x8 *>(arow[i] + step * astep);
      if (h < kWL) {
        const int at = kWL == 2 ? step : min(st, nst - 1);
#pragma unroll
        for (int j = 0; j < kJ; j++)
          rw[s][j][h] = *reinterpret_cast<const u32x4 *>(wrow[j] + (size_t)at * 1024);
      }
    }
  };
  // Two chains at a time: a quarter's stages 0, 2, .. first, their steps on
  // chains 0 and 1 of four, then stages 1, 3, .. on chains 2 and 3 (with fewer
  // chains, the stages as they come).
  constexpr int kLive = kCh < 2 ? kCh : 2;
  f32x4 acc[kLive][kI][kJ], sum[kI][kJ];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < kLive; c++)
#pragma unroll
      for (int i = 0; i < kI; i++)
#pragma unroll
        for (int j = 0; j < kJ; j++) acc[c][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto compute = [&](int s, int st) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      if (kHalf && h == 1 && 2 * st + 1 >= steps) break;  // wave-uniform
      f16x8 fw[kJ];
#pragma unroll
      for (int j = 0; j < kJ; j++)
        fw[j] = kW == kWeightFp8 ? e4m3x8_to_f16(rw[s][j][0][2 * h], rw[s][j][0][2 * h + 1])
                                 : __builtin_bit_cast(f16x8, rw[s][j][h % kWL]);
#pragma unroll
      for (int i = 0; i < kI; i++)
#pragma unroll
        for (int j = 0; j < kJ; j++)
          acc[h % kLive][i][j] =
              __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[j], ra[s][i][h], acc[h % kLive][i][j], 0, 0, 0);
    }
  };
  // the q-th stage taken
  const int evens = kCh == 4 ? (nst + 1) / 2 : nst;
  auto stage = [&](int q) {
    const int p = min(q, nst - 1);
    return kCh != 4 ? p : p < evens ? 2 * p : 2 * (p - evens) + 1;
  };
  load(0, stage(0));
  load(1, stage(1));
  clear();
  auto run = [&](int q, int s) __attribute__((always_inline)) {
    if (kCh == 4 && q == evens) {  // wave-uniform
#pragma unroll
      for (int i = 0; i < kI; i++)
#pragma unroll
        for (int j = 0; j < kJ; j++) sum[i][j] = acc[0][i][j] + acc[kLive - 1][i][j];
      clear();
    }
    compute(s, stage(q));
  };
  int q = 0;
  for (; q + 1 < nst; q += 2) {
    run(q, 0);
    load(0, stage(q + 2));
    run(q + 1, 1);
    load(1, stage(q + 3));
  }
  if (q < nst) run(q, 0);

#pragma unroll
  for (int i = 0; i < kI; i++)
#pragma unroll
    for (int j = 0; j < kJ; j++) {
      f32x4 y = acc[0][i][j];
      if constexpr (kCh == 4) {
        // (one stage: chains 2 and 3 have no step)
        y = nst > 1 ? (sum[i][j] + acc[0][i][j]) + acc[kLive - 1][i][j] : acc[0][i][j] + acc[kLive - 1][i][j];
      } else if constexpr (kCh == 2) {
        y += acc[kLive - 1][i][j];
      }
      red[wave][i * kJ + j][lane] = y;
    }
  lds_barrier();
  // wave w finishes tiles w kOwn ..
  const int i = wave * kOwn / kJ, j0 = wave * kOwn % kJ, m = m0 + 16 * i + r16;
  if (m >= g.M) return;
  f32x4 y[kOwn];
#pragma unroll
  for (int e = 0; e < kOwn; e++) {
    const int q = wave * kOwn + e;
    const f32x4 s0 = red[0][q][lane], s1 = red[1][q][lane], s2 = red[2][q][lane], s3 = red[3][q][lane];
    y[e] = kForm == kStepOps ? ((s0 + s1) + s2) + s3 : (s0 + s1) + (s2 + s3);
  }
  const float inv = kForm == kStepQwenLayers && kEpi != kEpiResidual ? g.inv[m] : 1.0f;
#pragma unroll
  for (int e = 0; e < kOwn; e++) {
    const int n = (nt0 + j0 + e) * 16 + 4 * grp;
    f32x4 v = y[e];
    if constexpr (kEpi == kEpiSwiGLU) {  // a gate tile and its up tile
      if (e & 1) continue;
      const f32x4 sg = *reinterpret_cast<const f32x4 *>(g.scale + n);
      const f32x4 su = *reinterpret_cast<const f32x4 *>(g.scale + n + 16);
      f16x4 o;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float u = y[(e + 1) % kOwn][r];
        o[r] = kForm == kStepQwenLayers ? f16_product(silu(v[r] * inv * sg[r]), u * inv * su[r])
                                        : f16_product(silu(v[r] * sg[r]), u * su[r]);
      }
      *reinterpret_cast<f16x4 *>(g.out16 + f16_tiled_offset(m, (nt0 + j0 + e) / 2 * 16 + 4 * grp, g.out_ld)) = o;
    } else if constexpr (kW == kWeightFp8) {
#pragma clang fp contract(off)
      f32x4 *o = reinterpret_cast<f32x4 *>(g.out + (size_t)m * g.out_ld + n);
      const f32x4 sc = *reinterpret_cast<const f32x4 *>(g.scale + n);
      if constexpr (kEpi == kEpiResidual) {
        const f32x4 x = *o;
#pragma unroll
        for (int r = 0; r < 4; r++)
          v[r] = kForm == kStepQwenLayers ? fmaf(v[r], sc[r], x[r]) : x[r] + v[r] * sc[r];
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = kForm == kStepQwenLayers ? v[r] * inv * sc[r] : v[r] * sc[r];
      }
      *o = v;
    } else {
      v += *reinterpret_cast<const f32x4 *>(g.bias + n);
      if constexpr (kEpi == kEpiGelu) {
        f16x4 h;
#pragma unroll
        for (int r = 0; r < 4; r++) h[r] = gelu_tanh_f16(v[r]);
        *reinterpret_cast<f16x4 *>(g.out16 + f16_tiled_offset(m, n, g.out_ld)) = h;
      } else {
        f32x4 *o = reinterpret_cast<f32x4 *>(g.out + (size_t)m * g.out_ld + n);
        if constexpr (kEpi == kEpiResidual) v = *o + v;
        *o = v;
      }
    }
  }
}

template <int kW, int kEpi, int kForm>
hipError_t launch_gemm(hipStream_t s, const PrefillGemmArgs &g) {
  // 32 x 64 tiles: 64 x 32 reads the tokens twice as often for the same work (gate
  // / up of 4,090 tokens 212 us against 115), 64 x 64 leaves fewer workgroups than
  // it saves reads (129)
  constexpr int kI = 2, kJ = 4;
  const int tiles_m = (g.M + 16 * kI - 1) / (16 * kI);
  const int ntiles = tiles_m * (g.N / (16 * kJ)), per_xcd = (ntiles + 7) / 8;
  const int panel = std::max(1, kPanelBytes / (g.K * 2 * 16 * kI));
  constexpr bool kHalf = kW == kWeightFp16;
  if (kHalf && g.K % 256 != 0)
    gemm_kernel<kW, kEpi, kForm, kI, kJ, kHalf><<<per_xcd * 8, kT, 0, s>>>(g, tiles_m, ntiles, per_xcd, panel);
  else
    gemm_kernel<kW, kEpi, kForm, kI, kJ, false><<<per_xcd * 8, kT, 0, s>>>(g, tiles_m, ntiles, per_xcd, panel);
  return hipGetLastError();
}

}  // namespace prompt
}  // namespace sh
