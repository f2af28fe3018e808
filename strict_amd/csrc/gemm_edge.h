// The GEMM kernel for every shape that the 256 x 256-tile kernels do not take
// (or would leave most of the chip idle on): any M, N, K, leading dimensions
// and element alignment, on MFMA. Shared by the bf16 and the FP8 GEMM:
//   kFp8 = false: C = A B,            A bf16 [M][lda], B bf16 [K][ldb]
//   kFp8 = true:  C = sa sb^T (A Bt), A e4m3 [M][lda], Bt e4m3 [N][ldb]
// fp32 accumulation, bf16 result. e4m3 values go to the MFMA as fp16, which
// holds them exactly: the fp8 MFMAs drop what lies more than ~17 bits below
// the largest product of a step, the fp16 one sums as fp32 does (an operand
// row whose large products cancel: error 2^-24 of the largest against 2^-17).
//
// What bounds such shapes is the latency of a K stage times the stages, and
// how many of the CUs have a tile at all. So:
//  - tiles of 64 x 64 (128 x 128 where there are enough of them for every CU);
//  - kGroups groups of 4 waves share a tile, each with every kGroups-th K
//    stage and a staging area of its own; their fp32 sums are added in group
//    order at the end, through LDS;
//  - a stage is 128 bytes of K (64 bf16, 128 e4m3), loaded through registers
//    two stages ahead into a double-buffered LDS.
// The element sums run in an order that depends on K and kGroups only.
// It took the place of a bounds-checked fp32 FMA kernel: bf16 1000 x 1003 x 517
// 78.3 -> 8.0 us, fp8 517 x 6144 x 1024 193 -> 15.5 us, bf16 4000 x 4001 x 3999
// 213 us (0.60 PFLOP/s).
//
// Loads are 16 bytes at any element alignment. A chunk that crosses the end
// of its row reads the next row's first elements, and only at the end of the
// matrix, where there is nothing more, its elements one by one. Of A (and Bt)
// everything past K is then zeroed, as are B's rows past K; columns past N
// and rows past M hold whatever was read and are not stored.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"
#include "llm_device.h"

namespace sh {
namespace edge {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
#define SH_EDGE_LDS __attribute__((address_space(3)))

struct Args {
  const uint8_t *a, *b;  // operands as bytes
  const float *sa, *sb;  // FP8: row / column scales
  uint16_t *c;
  int M, N, K;
  size_t lda, ldb;       // bytes
  int ldc;               // elements
  size_t span_a, span_b;  // bytes from an operand's first element to its last
  int tiles_m, ntiles, per_xcd;
};

__device__ __forceinline__ uint32_t bf16_bits(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;  // quiet NaN
  u += 0x7fffu + ((u >> 16) & 1u);                                  // round to nearest even
  return u >> 16;
}

__device__ __forceinline__ void lds_barrier() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): global loads stay in flight
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// 16 bytes at any global address (no alignment needed). The pointers are cast
// to the global address space: generic loads would count against the LDS wait
// counter too, and every LDS wait would empty the load pipeline.
#define SH_EDGE_GLOBAL __attribute__((address_space(1)))
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));
__device__ __forceinline__ u32x4 load16(const SH_EDGE_GLOBAL uint8_t *p) {
  return *reinterpret_cast<const SH_EDGE_GLOBAL u32x4_any *>(p);
}

// Stands in for an operand of fewer than 16 bytes in the 16-byte loads.
static __device__ __attribute__((aligned(16))) const uint32_t kNothing[4] = {0, 0, 0, 0};

// The bytes [off, off + 16) of a span, zeros past its end, from `raw`, the 16
// bytes at min(off, span - 16); byte by byte of a span shorter than 16.
__device__ __forceinline__ u32x4 at_edge(u32x4 raw, const uint8_t *base, size_t off, size_t span) {
  unsigned __int128 x = __builtin_bit_cast(unsigned __int128, raw);
  if (span >= 16) {
    const size_t cut = off + 16 > span ? off + 16 - span : 0;
    x = cut < 16 ? x >> (8 * (int)cut) : 0;
  } else {
    x = 0;
#pragma unroll 1
    for (size_t i = off; i < span; i++) x |= (unsigned __int128)base[i] << (8 * (int)(i - off));
  }
  return __builtin_bit_cast(u32x4, x);
}

// The first n bytes of v (n >= 16: all), zeros after them.
__device__ __forceinline__ u32x4 keep_bytes(u32x4 v, int n) {
#pragma unroll
  for (int d = 0; d < 4; d++) {
    const int nb = min(max(n - 4 * d, 0), 4);
    v[d] = nb == 4 ? v[d] : v[d] & ((1u << (8 * nb)) - 1u);
  }
  return v;
}

template <bool kFp8, int kTile, int kGroups>
__global__ __launch_bounds__(256 * kGroups, kTile == 128 ? 2 : 4) void gemm_edge_kernel(const Args g) {
  constexpr int kI = kTile / 32;       // 16-row MFMA tiles per wave and operand
  constexpr int kC = kTile * 8 / 256;  // 16-byte chunks per thread, operand and stage
  constexpr int kArea = kTile * 128;   // bytes of one operand's stage
  constexpr int kEl = kFp8 ? 1 : 2;
  constexpr int kSK = 128 / kEl;       // K elements per stage
  // B's rows of a bf16 stage: kTile columns of one k
  constexpr int kBRow = kTile * 2, kBChunks = kBRow / 16;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // [group][buffer][A | B]

  const int tile = (blockIdx.x & 7) * g.per_xcd + (blockIdx.x >> 3);
  if (tile >= g.ntiles) return;
  const int tm = tile % g.tiles_m, tn = tile / g.tiles_m;
  const int group = kGroups == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int t = threadIdx.x & 255, lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = tm * kTile, n0 = tn * kTile;
  uint8_t *area = lds + group * (4 * kArea);
  const long long kbytes = (long long)g.K * kEl;
  const int nk = (int)((kbytes + 127) / 128);

  // rows of A (and Bt): chunk t % 8 of rows t / 8 + 32 u; B's k rows: chunk
  // c % kBChunks of row c / kBChunks, c = t + 256 u
  size_t a_off[kC], b_off[kC];
  int a_lds[kC], b_lds[kC];
#pragma unroll
  for (int u = 0; u < kC; u++) {
    const int r = (t >> 3) + 32 * u, ch = t & 7;
    a_off[u] = (size_t)min(m0 + r, g.M - 1) * g.lda + ch * 16;
    a_lds[u] = r * 128 + ((ch ^ (r & 7)) * 16);
    if (kFp8) {
      b_off[u] = (size_t)min(n0 + r, g.N - 1) * g.ldb + ch * 16;
      b_lds[u] = kArea + a_lds[u];
    } else {
      const int c = t + 256 * u, kr = c / kBChunks, cc = c % kBChunks;
      // (a chunk past the last column reads the last one's)
      b_off[u] = (size_t)kr * g.ldb + (size_t)min(n0 + cc * 8, (g.N - 1) / 8 * 8) * 2;
      // the transposing reads take 4 rows x 2 chunks per 16 lanes, rows 8
      // apart in the next 16: swizzled so that 32 lanes hit 64 banks
      const int f = kTile == 64 ? ((kr >> 1) & 1) | ((kr >> 2) & 2) : (kr & 3) | ((kr >> 1) & 4);
      b_lds[u] = kArea + kr * kBRow + ((cc ^ (2 * f)) * 16);
    }
  }

  // the stages before `plain` lie whole inside both operands
  int plain = (int)(kbytes / 128);
  if (!kFp8) {
    // the furthest read of a stage: its last k row, from the last column on
    while (plain > 0 && ((size_t)plain * kSK - 1) * g.ldb + (size_t)(g.N - 1) * 2 + 16 > g.span_b) plain--;
  }
  typedef const SH_EDGE_GLOBAL uint8_t *Global;
  const Global src_a = (Global)(g.span_a < 16 ? (const uint8_t *)kNothing : g.a);
  const Global src_b = (Global)(g.span_b < 16 ? (const uint8_t *)kNothing : g.b);
  const size_t last_a = g.span_a < 16 ? 0 : g.span_a - 16, last_b = g.span_b < 16 ? 0 : g.span_b - 16;
  auto stage_off_b = [&](int kt) { return kFp8 ? (size_t)kt * 128 : (size_t)kt * kSK * g.ldb; };

  u32x4 ra[2][kC], rb[2][kC];
  // stage kt into register set s: as it is (plain stages), or any stage, from
  // clamped addresses. No load sits under a branch: the compiler would wait
  // for all loads in flight where the paths join.
  auto load_plain = [&](int s, int kt) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kC; u++) {
      ra[s][u] = load16(src_a + a_off[u] + (size_t)kt * 128);
      rb[s][u] = load16(src_b + b_off[u] + stage_off_b(kt));
    }
  };
  auto load_any = [&](int s, int kt) __attribute__((always_inline)) {
    const int kc = min(kt, nk - 1);
#pragma unroll
    for (int u = 0; u < kC; u++) {
      ra[s][u] = load16(src_a + min(a_off[u] + (size_t)kc * 128, last_a));
      rb[s][u] = load16(src_b + min(b_off[u] + stage_off_b(kc), last_b));
    }
  };
  auto store_plain = [&](int s, int buf) __attribute__((always_inline)) {
    uint8_t *p = area + buf * (2 * kArea);
#pragma unroll
    for (int u = 0; u < kC; u++) {
      *reinterpret_cast<u32x4 *>(p + a_lds[u]) = ra[s][u];
      *reinterpret_cast<u32x4 *>(p + b_lds[u]) = rb[s][u];
    }
  };
  auto store_any = [&](int s, int buf, int kt) __attribute__((always_inline)) {
    if (kt >= plain) {
      const long long left = kbytes - ((long long)kt * 128 + (t & 7) * 16);  // of this chunk's row
      const int keep = (int)max(min(left, 16LL), 0LL);
#pragma unroll
      for (int u = 0; u < kC; u++) {
        ra[s][u] = keep_bytes(at_edge(ra[s][u], g.a, a_off[u] + (size_t)kt * 128, g.span_a), keep);
        rb[s][u] = at_edge(rb[s][u], g.b, b_off[u] + stage_off_b(kt), g.span_b);
        const int kr = kt * kSK + (t + 256 * u) / kBChunks;
        rb[s][u] = keep_bytes(rb[s][u], kFp8 ? keep : kr < g.K ? 16 : 0);
      }
    }
    store_plain(s, buf);
  };

  f32x4 acc[kI][kI];
#pragma unroll
  for (int i = 0; i < kI; i++)
#pragma unroll
    for (int j = 0; j < kI; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int r16 = lane & 15, grp = lane >> 4;
  auto compute = [&](int buf) __attribute__((always_inline)) {
    const uint8_t *p = area + buf * (2 * kArea);
    auto chunk = [&](const uint8_t *rows, int r, int ch) {
      return *reinterpret_cast<const u32x4 *>(rows + r * 128 + ((ch ^ (r & 7)) * 16));
    };
    if constexpr (kFp8) {
      // 16 bytes a lane, 8 for each of two k-steps; the k order, the same for
      // both operands, does not matter
#pragma unroll
      for (int h = 0; h < 2; h++) {
        u32x4 ca[kI], cb[kI];
#pragma unroll
        for (int i = 0; i < kI; i++) {
          ca[i] = chunk(p, wm * (kTile / 2) + 16 * i + r16, 4 * h + grp);
          cb[i] = chunk(p + kArea, wn * (kTile / 2) + 16 * i + r16, 4 * h + grp);
        }
#pragma unroll
        for (int q = 0; q < 2; q++) {
          f16x8 fa[kI], fb[kI];
#pragma unroll
          for (int i = 0; i < kI; i++) {
            fa[i] = e4m3x8_to_f16(ca[i][2 * q], ca[i][2 * q + 1]);
            fb[i] = e4m3x8_to_f16(cb[i][2 * q], cb[i][2 * q + 1]);
          }
#pragma unroll
          for (int i = 0; i < kI; i++)
#pragma unroll
            for (int j = 0; j < kI; j++)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[j], fa[i], acc[i][j], 0, 0, 0);
        }
      }
    } else {
      const SH_EDGE_LDS uint8_t *pb = (const SH_EDGE_LDS uint8_t *)(p + kArea);
      const int ti = (lane >> 2) & 3, tq = lane & 3;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        bf16x8 fa[kI], fb[kI];
#pragma unroll
        for (int i = 0; i < kI; i++) {
          fa[i] = __builtin_bit_cast(bf16x8, chunk(p, wm * (kTile / 2) + 16 * i + r16, 4 * h + grp));
          s16x4 half[2];
#pragma unroll
          for (int q = 0; q < 2; q++) {
            const int kr = 32 * h + 8 * grp + 4 * q + ti;
            const int f = kTile == 64 ? ((kr >> 1) & 1) | ((kr >> 2) & 2) : (kr & 3) | ((kr >> 1) & 4);
            const int cc = wn * (kTile / 16) + 2 * i + (tq >> 1);
            half[q] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (SH_EDGE_LDS s16x4 *)(pb + kr * kBRow + ((cc ^ (2 * f)) * 16) + (tq & 1) * 8));
          }
          fb[i] = __builtin_bit_cast(
              bf16x8, __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7));
        }
#pragma unroll
        for (int i = 0; i < kI; i++)
#pragma unroll
          for (int j = 0; j < kI; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j], fa[i], acc[i][j], 0, 0, 0);
      }
    }
  };

  // iteration it: this group's stage it * kGroups + group, in LDS buffer and
  // register set it % 2; the stage two ahead is requested, the next one stored
  const int nit = (nk + kGroups - 1) / kGroups;
  auto step = [&](int it, auto par_c, auto plain_c) __attribute__((always_inline)) {
    constexpr int kPar = decltype(par_c)::value;
    const int kt = it * kGroups + group;
    if constexpr (decltype(plain_c)::value) {
      // the order is kept: a store moved up ahead of the loads would wait for
      // the stage requested last, not the one before it
      load_plain(kPar, kt + 2 * kGroups);
      __builtin_amdgcn_sched_barrier(0);
      compute(kPar);
      __builtin_amdgcn_sched_barrier(0);
      store_plain(kPar ^ 1, kPar ^ 1);
    } else {
      load_any(kPar, kt + 2 * kGroups);
      if (kt < nk) compute(kPar);
      if (kt + kGroups < nk) store_any(kPar ^ 1, kPar ^ 1, kt + kGroups);
    }
    lds_barrier();
  };
  load_any(0, group);
  load_any(1, kGroups + group);
  if (group < nk) store_any(0, 0, group);
  lds_barrier();
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  int it = 0;
  // pairs of iterations whose loads, in every group, are of plain stages
  for (; (it + 4) * kGroups <= plain; it += 2) {
    step(it, c0, std::true_type{});
    step(it + 1, c1, std::true_type{});
  }
  for (; it < nit; it += 2) {
    step(it, c0, std::false_type{});
    if (it + 1 < nit) step(it + 1, c1, std::false_type{});
  }

  // lane: row m, columns n .. n + 3
  auto store_c = [&](int i, int j, f32x4 v) __attribute__((always_inline)) {
    const int m = m0 + wm * (kTile / 2) + 16 * i + r16;
    const int n = n0 + wn * (kTile / 2) + 16 * j + 4 * grp;
    if (m >= g.M || n >= g.N) return;
    uint16_t *o = g.c + (size_t)m * g.ldc + n;
    if constexpr (kFp8) {
      const float s = g.sa[m];
#pragma unroll
      for (int r = 0; r < 4; r++) v[r] = v[r] * s * g.sb[min(n + r, g.N - 1)];
    }
    const u32x2 w = {bf16_bits(v[0]) | (bf16_bits(v[1]) << 16), bf16_bits(v[2]) | (bf16_bits(v[3]) << 16)};
    if (n + 4 <= g.N) {
      __builtin_memcpy(o, &w, 8);
    } else {
#pragma unroll
      for (int r = 0; r < 3; r++)
        if (n + r < g.N) o[r] = (uint16_t)(w[r / 2] >> (16 * (r & 1)));
    }
  };
  if constexpr (kGroups == 1) {
#pragma unroll
    for (int i = 0; i < kI; i++)
#pragma unroll
      for (int j = 0; j < kI; j++) store_c(i, j, acc[i][j]);
  } else {
    // every group's sums to LDS (the staging is no longer read: the last
    // iteration's barrier), then group q adds its share of the wave's tiles
    constexpr int kTiles = kI * kI, kShare = kTiles / kGroups;
    static_assert(kTiles % kGroups == 0, "a group adds whole tiles");
    f32x4 *red = reinterpret_cast<f32x4 *>(lds);  // [group][tile][wave][lane]
#pragma unroll
    for (int q = 0; q < kTiles; q++) red[((group * kTiles + q) * 4 + wave) * 64 + lane] = acc[q / kI][q % kI];
    lds_barrier();
#pragma unroll
    for (int sh = 0; sh < kShare; sh++) {
      const int q = group * kShare + sh;
      f32x4 v = red[(q * 4 + wave) * 64 + lane];
#pragma unroll
      for (int k = 1; k < kGroups; k++) {
        const f32x4 x = red[((k * kTiles + q) * 4 + wave) * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] += x[r];
      }
      store_c(q / kI, q % kI, v);
    }
  }
}

template <bool kFp8, int kTile, int kGroups>
hipError_t launch_tiles(hipStream_t s, Args g) {
  const size_t lds = (size_t)kGroups * 4 * kTile * 128;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(
        reinterpret_cast<const void *>(&gemm_edge_kernel<kFp8, kTile, kGroups>),
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const long long tiles_m = (g.M + (long long)kTile - 1) / kTile;
  const long long nt = tiles_m * ((g.N + (long long)kTile - 1) / kTile);
  if (nt > 0x7fffffffLL - 8) return hipErrorInvalidValue;
  g.tiles_m = (int)tiles_m;
  g.ntiles = (int)nt;
  g.per_xcd = (g.ntiles + 7) / 8;
  gemm_edge_kernel<kFp8, kTile, kGroups><<<g.per_xcd * 8, 256 * kGroups, lds, s>>>(g);
  return hipGetLastError();
}

// Tile and groups by the tiles a shape has and its K stages, where the
// variants crossed (us a pass, bf16 | fp8):
//  - 128 x 128 once nearly every CU gets one: 2000^3 (256 tiles) 31.5 against
//    44.9 with 64 x 64 | 28.8, 29.5; 517 x 6144 x 1024 (240) 20.0, 20.3 | 19.3,
//    16.4; 3000 x 400 x 1111 (96) 22.6, 16.7 | 21.9, 13.1. FP8's waves convert
//    less per MFMA with it, but have half the bytes to wait for: 2048^3 (256) |
//    29.0, 27.8; 2304 x 2816 x 2048 (396) | 39.4, 40.7; 2560^3 (400) | 45.9, 50.1.
//  - four groups where at most half of the CUs have a tile (FP8: one tile each)
//    and the K stages are many: 16 x 4096 x 4096 (64 tiles) 18.9 against 21.8 |
//    13.5, 18.3; 300 x 3000 x 3000 (235) 19.2, 19.3 | 14.9, 17.6; 1000 x 1003 x
//    517 (256) 10.9, 8.4 | 10.0, 8.3; 600^3 (100) | 6.5, 7.2.
template <bool kFp8>
hipError_t launch(hipStream_t s, const Args &g) {
  auto tiles = [&](long long t) { return ((g.M + t - 1) / t) * ((g.N + t - 1) / t); };
  const long long stages = ((long long)g.K * (kFp8 ? 1 : 2) + 127) / 128;
  if (tiles(128) >= (kFp8 ? 384 : 240)) return launch_tiles<kFp8, 128, 1>(s, g);
  if (stages >= 5 && tiles(64) <= (kFp8 && stages >= 8 ? 256 : 128)) return launch_tiles<kFp8, 64, 4>(s, g);
  return launch_tiles<kFp8, 64, 1>(s, g);
}

}  // namespace edge
}  // namespace sh
