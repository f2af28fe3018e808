// Standalone decoder building blocks behind the C ABI: RMSNorm, LayerNorm,
// RoPE, SwiGLU, GELU, argmax and decode attention on caller buffers. The
// model runners fuse the same operations into their GEMV prologues and
// epilogues and into the decode-layers kernel; these entry points let a
// caller launch each one on its own buffers (and let each one be checked on
// its own).
//
// Rounding: the norms take their statistics in fp64 and RoPE its cos / sin
// in fp64 of the fp32 angle; every fp32 product and sum after that is
// rounded on its own (no contraction into FMAs), which are the rounding
// points of the oracle (oracle/llm.py).
//
// Decode attention is split-K flash decoding: grid (split, KV head, row),
// each workgroup takes its split's positions with a running softmax (max,
// sum, unnormalised V sum) per query head, and writes those three as a
// partial; a merge kernel per (row, head) combines the partials (with one
// split the first kernel writes the output). The partials live in a work
// buffer: the context's (sh_attn_decode_f16) or a fixed device array
// (sh_attn_decode_f16_noalloc).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "llm_device.h"

namespace sh {
namespace {

constexpr int kT = 256;

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Sum over the workgroup (kT threads), the same value in every thread.
__device__ __forceinline__ double block_sum_f64(double v, double *red) {
  v = wave_sum_f64(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const double r = (red[0] + red[1]) + (red[2] + red[3]);
  __syncthreads();
  return r;
}

// ---- row norms -------------------------------------------------------------

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

// Values 4 c .. 4 c + 3 of a row of n (zeros past its end).
__device__ __forceinline__ f32x4 load_row4(const float *row, int c, int n) {
  if (4 * c + 4 <= n) return *reinterpret_cast<const f32x4_any *>(row + 4 * c);
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int e = 0; e < 3; e++)
    if (4 * c + e < n) v[e] = row[4 * c + e];
  return v;
}

__device__ __forceinline__ void store_row4(float *row, int c, int n, f32x4 v) {
  if (4 * c + 4 <= n) {
    *reinterpret_cast<f32x4_any *>(row + 4 * c) = v;
    return;
  }
#pragma unroll
  for (int e = 0; e < 3; e++)
    if (4 * c + e < n) row[4 * c + e] = v[e];
}

// One row per kWaves waves (1 or 4), its values in registers between the
// statistics and the result, as kPer vectors of 4 per lane: one read and one
// write of the row, all loads (gains and biases too) requested together. With
// one wave per row nothing waits for a barrier. Statistics in fp64.
//   kLayer false: y = (x * inv) * g, inv = fp32(1 / sqrt(mean(x^2) + eps))
//   kLayer true:  y = ((x - mean) * inv) * g + b, mean and variance in two
//                 passes over the registers, inv = fp32(1 / sqrt(var + eps))
// 512 rows of 1,024: RMSNorm 4.2 -> 3.3 us a launch (4 MB, bound by latency).
template <bool kLayer, int kWaves, int kPer>
__global__ __launch_bounds__(kT) void norm_kernel(const float *x, const float *__restrict__ g,
                                                  const float *__restrict__ bias, float *y, int rows,
                                                  int n, float eps) {
#pragma clang fp contract(off)
  __shared__ double red[4];
  const int t = threadIdx.x % (64 * kWaves);
  const int row = blockIdx.x * (kT / (64 * kWaves)) + threadIdx.x / (64 * kWaves);
  if (row >= rows) return;  // (one wave per row: no barrier follows)
  const float *xr = x + (size_t)row * n;
  float *yr = y + (size_t)row * n;
  auto sum = [&](double v) {
    return kWaves == 1 ? wave_sum_f64(v) : block_sum_f64(v, red);
  };
  f32x4 v[kPer], gv[kPer], bv[kPer];
#pragma unroll
  for (int u = 0; u < kPer; u++) v[u] = load_row4(xr, t + 64 * kWaves * u, n);
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    gv[u] = load_row4(g, t + 64 * kWaves * u, n);
    if (kLayer) bv[u] = load_row4(bias, t + 64 * kWaves * u, n);
  }
  double mean = 0.0;
  if (kLayer) {
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < kPer; u++)
#pragma unroll
      for (int e = 0; e < 4; e++) s += (double)v[u][e];
    mean = sum(s) / (double)n;
  }
  double ss = 0.0;
#pragma unroll
  for (int u = 0; u < kPer; u++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const double d = (double)v[u][e] - mean;
      if (!kLayer || 4 * (t + 64 * kWaves * u) + e < n) ss += d * d;
    }
  const float inv = (float)(1.0 / sqrt(sum(ss) / (double)n + (double)eps));
  const float mf = (float)mean;
#pragma unroll
  for (int u = 0; u < kPer; u++) {
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      if (kLayer)
        o[e] = ((v[u][e] - mf) * inv) * gv[u][e] + bv[u][e];
      else
        o[e] = (v[u][e] * inv) * gv[u][e];
    }
    store_row4(yr, t + 64 * kWaves * u, n, o);
  }
}

// Rows longer than the registers hold: grid (rows), the row read again for
// each pass (y may be x: each thread re-reads its values before it overwrites
// them, after the workgroup's sums).
template <bool kLayer>
__global__ __launch_bounds__(kT) void norm_long_kernel(const float *x, const float *__restrict__ g,
                                                       const float *__restrict__ bias, float *y,
                                                       int n, float eps) {
#pragma clang fp contract(off)
  __shared__ double red[4];
  const float *xr = x + (size_t)blockIdx.x * n;
  float *yr = y + (size_t)blockIdx.x * n;
  double mean = 0.0;
  if (kLayer) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += kT) s += (double)xr[i];
    mean = block_sum_f64(s, red) / (double)n;
  }
  double ss = 0.0;
  for (int i = threadIdx.x; i < n; i += kT) {
    const double d = (double)xr[i] - mean;
    ss += d * d;
  }
  const float inv = (float)(1.0 / sqrt(block_sum_f64(ss, red) / (double)n + (double)eps));
  const float mf = (float)mean;
  for (int i = threadIdx.x; i < n; i += kT)
    yr[i] = kLayer ? ((xr[i] - mf) * inv) * g[i] + bias[i] : (xr[i] * inv) * g[i];
}

template <bool kLayer>
hipError_t launch_norm(hipStream_t s, const float *x, const float *g, const float *bias, float *y,
                       int rows, int n, float eps) {
  // one wave per row up to 8 vectors a lane, four waves up to 8 of theirs
  const int blocks4 = (rows + 3) / 4;
  if (n <= 1024)
    norm_kernel<kLayer, 1, 4><<<blocks4, kT, 0, s>>>(x, g, bias, y, rows, n, eps);
  else if (n <= 2048)
    norm_kernel<kLayer, 1, 8><<<blocks4, kT, 0, s>>>(x, g, bias, y, rows, n, eps);
  else if (n <= 8192)
    norm_kernel<kLayer, 4, 8><<<rows, kT, 0, s>>>(x, g, bias, y, rows, n, eps);
  else
    norm_long_kernel<kLayer><<<rows, kT, 0, s>>>(x, g, bias, y, n, eps);
  return hipGetLastError();
}

// ---- RoPE ------------------------------------------------------------------

// cos and sin of an fp32 angle to fp32: reduction by pi / 2 in two parts
// (Cody and Waite) and Taylor polynomials on [-pi / 4, pi / 4], all in fp64.
// Angles of 2^40 and more, infinities and NaN go to the library's sincos.
__device__ __forceinline__ void cos_sin(float angle, float *c, float *s) {
  const double a = (double)angle;
  double sd, cd;
  if (__builtin_fabsf(angle) < 1099511627776.0f) {
    const double q = rint(a * 0.63661977236758134308);  // 2 / pi
    // pi / 2 as the nearest double and the rest
    double r = fma(-q, 1.57079632679489655800, a);
    r = fma(-q, 6.12323399573676603587e-17, r);
    const double z = r * r;
    // r - r^3/3! + .. - r^15/15!; 1 - r^2/2! + .. + r^16/16!: the next terms are
    // below 2^-53
    double ps = fma(z, -7.64716373181981647590e-13, 1.60590438368216145994e-10);
    ps = fma(z, ps, -2.50521083854417187751e-8);
    ps = fma(z, ps, 2.75573192239858906526e-6);
    ps = fma(z, ps, -1.98412698412698412698e-4);
    ps = fma(z, ps, 8.33333333333333333333e-3);
    ps = fma(z, ps, -1.66666666666666666667e-1);
    const double sr = fma(r * z, ps, r);
    double pc = fma(z, 4.77947733238738529744e-14, -1.14707455977297247139e-11);
    pc = fma(z, pc, 2.08767569878680989792e-9);
    pc = fma(z, pc, -2.75573192239858906526e-7);
    pc = fma(z, pc, 2.48015873015873015873e-5);
    pc = fma(z, pc, -1.38888888888888888889e-3);
    pc = fma(z, pc, 4.16666666666666666667e-2);
    pc = fma(z, pc, -5.0e-1);
    const double cr = fma(z, pc, 1.0);
    const int k = (int)((long long)q & 3);
    sd = (k & 1) ? cr : sr;
    cd = (k & 1) ? sr : cr;
    if (k & 2) sd = -sd;
    if (k == 1 || k == 2) cd = -cd;
  } else {
    sincos(a, &sd, &cd);
  }
  *c = (float)cd;
  *s = (float)sd;
}

// Rotate-half of x[row][head][0..d) at positions[row]: angle = fp32(pos) *
// fp32(theta^(-2i/d)), cos / sin in fp64. A unit of `width` lanes (the pairs of
// a head, in whole waves) takes kRopeHeads heads of a row: their values are
// requested first and the factors, the same for all of them, worked out
// meanwhile. log2_theta: log2 of theta in fp64.
// 512 rows of 16 heads of 128: 8.5 -> 3.9 us (a power and a library sincos in
// fp64 per pair and head before).
constexpr int kRopeHeads = 4;
__global__ __launch_bounds__(kT) void rope_kernel(float *__restrict__ x, const int *__restrict__ pos,
                                                  int rows, int heads, int d, int width,
                                                  double log2_theta) {
#pragma clang fp contract(off)
  const int half = d / 2, i = threadIdx.x % width;
  const int chunks = (heads + kRopeHeads - 1) / kRopeHeads;
  const long long unit = (long long)blockIdx.x * (kT / width) + threadIdx.x / width;
  if (threadIdx.x / width >= kT / width || unit >= (long long)rows * chunks || i >= half) return;
  const int row = (int)(unit / chunks), h0 = (int)(unit % chunks) * kRopeHeads;
  float *xp = x + ((size_t)row * heads + h0) * d + i;
  float x1[kRopeHeads], x2[kRopeHeads];
#pragma unroll
  for (int u = 0; u < kRopeHeads; u++) {
    const size_t at = (size_t)min(u, heads - 1 - h0) * d;
    x1[u] = xp[at];
    x2[u] = xp[at + half];
  }
  // (theta^0 is 1 for an infinite theta, too)
  const float inv_freq = i == 0 ? 1.0f : (float)exp2(log2_theta * (-2.0 * (double)i / (double)d));
  const float ang = (float)pos[row] * inv_freq;
  float c, s;
  cos_sin(ang, &c, &s);
#pragma unroll
  for (int u = 0; u < kRopeHeads; u++) {
    if (h0 + u >= heads) break;
    xp[(size_t)u * d] = x1[u] * c - x2[u] * s;
    xp[(size_t)u * d + half] = x2[u] * c + x1[u] * s;
  }
}

// ---- elementwise -------------------------------------------------------------

// Two vectors of 4 per thread and input, requested together (one value at a
// time left the loads of a grid-stride step behind each other): 512 x 3072
// SwiGLU 4.3 -> 4.1 us a launch (19 MB).
constexpr int kPerThread = 2;

// Vectors of 4 at any alignment, and the n % 4 values after them one each. (One
// round but for sizes past the grid's limit.)
template <class Op>
__device__ __forceinline__ void map4(size_t n, const float *a, const float *b, float *out, Op op) {
  const size_t n4 = n / 4;
  for (size_t base = (size_t)blockIdx.x * kT * kPerThread + threadIdx.x; base < n4;
       base += (size_t)gridDim.x * kT * kPerThread) {
    f32x4 va[kPerThread], vb[kPerThread];
#pragma unroll
    for (int u = 0; u < kPerThread; u++) {
      const size_t i = min(base + (size_t)u * kT, n4 - 1);
      va[u] = reinterpret_cast<const f32x4_any *>(a)[i];
      vb[u] = reinterpret_cast<const f32x4_any *>(b)[i];
    }
#pragma unroll
    for (int u = 0; u < kPerThread; u++) {
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] = op(va[u][e], vb[u][e]);
      if (base + (size_t)u * kT < n4) reinterpret_cast<f32x4_any *>(out)[base + (size_t)u * kT] = o;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < (n & 3)) {
    const size_t i = n4 * 4 + threadIdx.x;
    out[i] = op(a[i], b[i]);
  }
}

// (A launch takes fewer than 2^32 threads.)
unsigned map4_grid(size_t n) {
  return (unsigned)std::min<size_t>(std::max<size_t>(1, (n / 4 + kT * kPerThread - 1) / (kT * kPerThread)), 1u << 23);
}

__global__ __launch_bounds__(kT) void swiglu_kernel(const float *gate, const float *up, float *out,
                                                    size_t n) {
#pragma clang fp contract(off)
  map4(n, gate, up, out, [](float g, float u) { return silu(g) * u; });
}

__global__ __launch_bounds__(kT) void gelu_kernel(const float *x, float *y, size_t n) {
  map4(n, x, x, y, [](float v, float) { return gelu_tanh(v); });
}

// ---- argmax ------------------------------------------------------------------

// Order of the values: argmax_key's (its high word here), by which -0 lies
// below +0; NaN, of either sign, above everything (as numpy's argmax, which
// returns the first NaN). Equal values: the smaller index.
__device__ __forceinline__ uint32_t order_key(uint32_t u) {
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// The largest of a, b, c; -0 < +0. Of no use where one of them is NaN.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// Minimum over the workgroup of kArgT threads, in every thread.
template <int kArgT>
__device__ __forceinline__ uint32_t block_min_u32(uint32_t v, uint32_t *red) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, off, 64));
  __syncthreads();  // red's earlier readers are done
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = red[0];
#pragma unroll
  for (int w = 1; w < kArgT / 64; w++) v = min(v, red[w]);
  return v;
}

// grid (rows): index[row] = the first position of the row's maximum. One
// workgroup reads a row, 8 vectors of 4 values in flight per thread, so a row
// streams at what one CU can load. A vector's maximum is
// found as floats and only that compared (as its order key) with the thread's
// best, whose vector is remembered; the position within it is looked up at the
// end. A row that holds a NaN is scanned again for the first one. 16 rows of
// 151936: 189 us with 4 waves per row, one value and one 64-bit key comparison
// at a time; 8.5 us a pass here.
template <int kArgT>
__global__ __launch_bounds__(kArgT) void argmax_kernel(const float *__restrict__ x, int n,
                                                       int32_t *__restrict__ index) {
  constexpr int kU = 8;
  __shared__ uint32_t red[kArgT / 64];
  const float *xr = x + (size_t)blockIdx.x * n;
  const int t = threadIdx.x;
  uint32_t best = 0;  // below every value's key
  int at = 0;         // first position of the best vector
  bool nan = false;
  // vectors at 0, 4, .., the last one at n - 4 (clamped starts: a vector read
  // twice changes nothing); unsigned, as a start ahead may pass 2^31
  const uint32_t un = (uint32_t)n;
  if (n >= 4) {
    for (uint32_t v0 = 4 * t; v0 < un; v0 += 4 * kArgT * kU) {
      f32x4 v[kU];
#pragma unroll
      for (int u = 0; u < kU; u++)
        v[u] = *reinterpret_cast<const f32x4_any *>(xr + min(v0 + 4 * kArgT * u, un - 4));
#pragma unroll
      for (int u = 0; u < kU; u++) {
        nan |= __builtin_isunordered(v[u].x, v[u].y) | __builtin_isunordered(v[u].z, v[u].w);
        const float m = max3(max3(v[u].x, v[u].y, v[u].z), v[u].w, v[u].w);
        const uint32_t k = order_key(__builtin_bit_cast(uint32_t, m));
        const bool better = k > best;
        best = better ? k : best;
        at = better ? (int)min(v0 + 4 * kArgT * u, un - 4) : at;
      }
    }
  } else if (t < n) {
    const float m = xr[t];
    nan = m != m;
    best = order_key(__builtin_bit_cast(uint32_t, m));
    at = t;
  }
  if (__syncthreads_or(nan)) {
    uint32_t first = 0xffffffffu;
    for (uint32_t i = t; i < un && first == 0xffffffffu; i += kArgT)
      if (xr[i] != xr[i]) first = i;
    first = block_min_u32<kArgT>(first, red);
    if (t == 0) index[blockIdx.x] = (int32_t)first;
    return;
  }
  const uint32_t top = ~block_min_u32<kArgT>(~best, red);
  uint32_t first = 0xffffffffu;
  if (best == top) {
#pragma unroll
    for (int e = 3; e >= 0; e--) {
      const int i = (int)min((uint32_t)at + e, un - 1);
      if (order_key(__builtin_bit_cast(uint32_t, xr[i])) == top) first = (uint32_t)i;
    }
  }
  first = block_min_u32<kArgT>(first, red);
  if (t == 0) index[blockIdx.x] = (int32_t)first;
}

// The same for short rows: one wave per row, four rows per workgroup (a row's
// barriers would take longer than its values). A value's key has its order in
// the high word and ~index in the low one, so that the largest key is the
// first of the largest values.
__global__ __launch_bounds__(kT) void argmax_short_kernel(const float *__restrict__ x, int rows, int n,
                                                          int32_t *__restrict__ index) {
  constexpr int kU = 4;
  const long long row = (long long)blockIdx.x * (kT / 64) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float *xr = x + (size_t)row * n;
  const int lane = threadIdx.x & 63;
  unsigned long long best = 0;
  for (int i0 = lane; i0 < n; i0 += 64 * kU) {
    float v[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) v[u] = xr[min(i0 + 64 * u, n - 1)];
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const int i = min(i0 + 64 * u, n - 1);  // (a value read twice changes nothing)
      const uint32_t k = v[u] != v[u] ? 0xffffffffu : order_key(__builtin_bit_cast(uint32_t, v[u]));
      const unsigned long long key = ((unsigned long long)k << 32) | (uint32_t)~i;
      best = key > best ? key : best;
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const unsigned long long o = __shfl_xor(best, off, 64);
    best = o > best ? o : best;
  }
  if (lane == 0) index[row] = (int32_t)~(uint32_t)best;
}

// By the row's length, where the variants crossed: 100,000 rows of 1,000 70 us with
// a wave each, 237 with 256 threads, of 64 21 and 117 (1,024 threads: 746); 16 rows
// of 2,048 5.9 and 4.7. 20,000 rows of 8,192 106 us with 256 threads, 345 with 1,024;
// 16 rows of 32,768 5.5 with 1,024, 22.8 with 256 (one value at a time). A launch
// takes fewer than 2^32 threads.
hipError_t launch_argmax(hipStream_t s, const float *x, int rows, int n, int32_t *index) {
  if (n <= 1024)
    argmax_short_kernel<<<(unsigned)((rows + 3LL) / 4), kT, 0, s>>>(x, rows, n, index);
  else if (n <= 8192 || rows >= (1 << 22))
    argmax_kernel<256><<<rows, 256, 0, s>>>(x, n, index);
  else
    argmax_kernel<1024><<<rows, 1024, 0, s>>>(x, n, index);
  return hipGetLastError();
}

// ---- decode attention ----------------------------------------------------------

constexpr int kMaxGroup = 16;  // query heads per KV head
typedef short s16x4 __attribute__((ext_vector_type(4)));
#define SH_OPS_LDS __attribute__((address_space(3)))

struct AttnOpArgs {
  const float *q;            // [B][heads][d]
  const uint16_t *k, *v;     // [B][kv_heads][max_pos][d] fp16
  const int *lengths;        // [B] positions attended: 0 .. length - 1
  float *out;                // [B][heads][d]
  float *part;               // [B][heads][splits][d + 2]: V sum, max, sum
  int heads, kv_heads, max_pos, splits, chunk;
  float scale;
};

// Positions whose K and V a workgroup requests at once (64 KiB): 8 loads of 16
// bytes of each per thread.
template <int kD>
constexpr int kAttnTile = 8 * 256 * 8 / kD;

constexpr float kPScale = 16384.0f;  // of P, and so of a partial's V sums and sum

// The result of a split for value i (head, dim) of the G heads from h0: its
// partial or, where the split is the whole row, the output.
template <int kD>
__device__ __forceinline__ void attn_store(const AttnOpArgs &a, int b, int h0, int s, int i, float sum,
                                           float m, float l) {
  if (a.splits == 1) {
    a.out[((size_t)b * a.heads + h0) * kD + i] = sum / l;
    return;
  }
  float *pp = a.part + (((size_t)b * a.heads + h0 + i / kD) * a.splits + s) * (size_t)(kD + 2);
  pp[i % kD] = sum;
  if (i % kD == 0) {
    pp[kD] = m;
    pp[kD + 1] = l;
  }
}

// Positions [p0, p1) in fp32 throughout, 64 at a time: a wave scores a head
// (lane: position), a thread sums V for (head, dim) pairs t, t + kT, ... Slow,
// for splits whose sums in two fp16 are not finite: infinities and NaN in q, K
// or V. A score of -inf has no weight.
struct AttnFp32 {
  float p[kMaxGroup][64], corr[kMaxGroup], m[kMaxGroup], l[kMaxGroup];
};
template <int kD>
__device__ __forceinline__ void attn_fp32(const AttnOpArgs &a, int b, int kvh, int s, int p0,
                                                    int p1, AttnFp32 &lds) {
  constexpr int kAcc = kMaxGroup * kD / kT;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, G = a.heads / a.kv_heads, h0 = kvh * G;
  const size_t row0 = ((size_t)b * a.kv_heads + kvh) * (size_t)a.max_pos;
  const _Float16 *kb = reinterpret_cast<const _Float16 *>(a.k) + row0 * kD;
  const _Float16 *vb = reinterpret_cast<const _Float16 *>(a.v) + row0 * kD;
  if (t < kMaxGroup) {
    lds.m[t] = -INFINITY;
    lds.l[t] = 0.0f;
  }
  float acc[kAcc];
#pragma unroll
  for (int j = 0; j < kAcc; j++) acc[j] = 0.0f;
  for (int pt = p0; pt < p1; pt += 64) {
    const int n = min(64, p1 - pt);
    __syncthreads();  // the last tile's p and corr are read; m and l are set
    for (int g = wave; g < G; g += 4) {
      const float *q = a.q + ((size_t)b * a.heads + h0 + g) * kD;
      const _Float16 *k = kb + (size_t)min(pt + lane, p1 - 1) * kD;
      float dot = 0.0f;
#pragma unroll 1
      for (int c = 0; c < kD; c += 8) {
        const f16x8 kk = *reinterpret_cast<const f16x8 *>(k + c);
#pragma unroll
        for (int e = 0; e < 8; e++) dot = fmaf(q[c + e] * a.scale, (float)kk[e], dot);
      }
      const float sc = lane < n ? dot : -INFINITY, old = lds.m[g];
      const float m = fmaxf(old, wave_max(sc));
      const float p = sc == -INFINITY ? 0.0f : expf(sc - m), c = old == m ? 1.0f : expf(old - m);
      const float sum = wave_sum(p);
      lds.p[g][lane] = p;
      if (lane == 0) {
        lds.corr[g] = c;
        lds.m[g] = m;
        lds.l[g] = lds.l[g] * c + sum;
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kAcc; j++) {
      const int i = t + kT * j, g = i / kD;
      if (g >= G) break;
      float sum = 0.0f;
      for (int p = 0; p < n; p++) sum = fmaf(lds.p[g][p], (float)vb[(size_t)(pt + p) * kD + i % kD], sum);
      acc[j] = acc[j] * lds.corr[g] + sum;
    }
  }
#pragma unroll
  for (int j = 0; j < kAcc; j++) {
    const int i = t + kT * j, g = i / kD;
    if (g < G) attn_store<kD>(a, b, h0, s, i, acc[j] * kPScale, lds.m[g], lds.l[g] * kPScale);
  }
}

// grid (splits, kv_heads, B): positions [s * chunk, min((s + 1) * chunk, L)) of
// row b for the G = heads / kv_heads query heads of KV head kvh, in tiles of
// kAttnTile positions. The kernel is bound by the K and V bytes, so all of a
// tile's loads are issued before any is used, and no wave waits for another in
// the loop: each takes a quarter of the tile's positions and keeps a running
// softmax (maximum, sum and V sum per head) of its own; the four are combined
// at the end. The arithmetic is MFMA's, whatever G is (the unused columns cost
// nothing that is missed):
//  - scores as K x q: K fragments straight from memory (a lane: 8 dims of
//    position lane % 16), heads in the columns; a lane then holds 4 consecutive
//    positions of each 16-position block for head lane % 16;
//  - V sums as V^T x P, the k slots numbered as P has them (slot (g, e):
//    position 4 g + e of the first block for e < 4, of the second for e >= 4);
//    V goes through LDS rows as it is and comes back by transposing reads.
// q and P stay fp32 to 2^-22: q as two fp16 after an exact power-of-two scaling
// of each head to below 1, the remainder times 2^12 and on sums of its own (so
// that values far below their head's largest keep their bits, too: to 2^-37 of
// it), P times 2^14 as two fp16. (Error against 64 bits 2.3e-7; the fp32 kernel
// before it, 64-position tiles staged in LDS with one serial V sum per thread,
// 4.1e-7.)
// Infinities do not survive that (a part of the other sign, or 0, times one is
// NaN): a split whose sums are not finite is worked out again in fp32.
// Measured, both kernels of a call, the fp32 kernel and this one: 4 rows of 4,096
// positions, 16 / 8 heads of 128: 30.8 and 17.6 us (67 MB, 3.8 TB/s); 16 rows 72.4
// and 49.3 (5.4 TB/s); 16 rows of 8,192, 16 / 1 heads 74.5 and 27.4; 1 row of 384,
// 12 / 12 heads of 64 9.2 and 8.8. fp32 FMAs from registers in its place were as
// fast at one query head per KV head and slower from two on (16 / 1 heads: 65.8).
// (The low part's own sums cost 0.1 to 2.5 us of these; at head_dim 128, 7 values
// beyond the 168 registers lie in scratch, 4 without those sums.)
template <int kD>
__global__ __launch_bounds__(kT, 3) void attn_op_partials_kernel(const AttnOpArgs a) {
  constexpr int kKK = kD / 32, kDT = kD / 16;
  constexpr int kBlocks = kAttnTile<kD> / 4 / 16;  // 16-position blocks per wave and tile
  constexpr int kVLoads = kBlocks * 16 * kD / 8 / 64;
  constexpr int kRow = kD * 2, kChunks = kD / 8;   // a V row in LDS: bytes, 16-byte chunks
  constexpr float kQLow = 4096.0f;
  union Lds {
    uint8_t v[4][kBlocks * 16 * kRow];
    float acc[4][kMaxGroup][kD];
    float q[kMaxGroup][kD];
    AttnFp32 fp32;
  };
  __shared__ __attribute__((aligned(16))) Lds lds;
  __shared__ __attribute__((aligned(16))) _Float16 qh[2][kMaxGroup][kD + 8];
  __shared__ float qscale[kMaxGroup], stat[4][kMaxGroup][2];

  const int s = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int r16 = lane & 15, grp = lane >> 4;
  const int G = a.heads / a.kv_heads;
  const int L = min(a.lengths[b], a.max_pos);
  const int p0 = s * a.chunk;
  const int h0 = kvh * G;
  if (p0 >= L) {  // uniform: nothing of this row in the split
    if (a.splits == 1)
      for (int i = t; i < G * kD; i += kT) a.out[((size_t)b * a.heads + h0) * kD + i] = 0.0f;
    return;
  }
  const int p1 = min(p0 + a.chunk, L);

  const size_t row0 = ((size_t)b * a.kv_heads + kvh) * (size_t)a.max_pos;
  const uint16_t *kb = a.k + row0 * kD + grp * 8;
  const uint16_t *vb = a.v + row0 * kD + (lane % kChunks) * 8;
  f16x8 kf[kBlocks][kKK];
  u32x4 vr[kVLoads];
  // positions past the split re-read its last one (never weighted)
  auto load_k = [&](int pt) __attribute__((always_inline)) {
    const int pw = pt + wave * (16 * kBlocks);
#pragma unroll
    for (int tt = 0; tt < kBlocks; tt++)
#pragma unroll
      for (int kk = 0; kk < kKK; kk++)
        kf[tt][kk] = *reinterpret_cast<const f16x8 *>(
            kb + (size_t)min(pw + 16 * tt + r16, p1 - 1) * kD + 32 * kk);
  };
  auto load_v = [&](int pt) __attribute__((always_inline)) {
    const int pw = pt + wave * (16 * kBlocks);
#pragma unroll
    for (int u = 0; u < kVLoads; u++)
      vr[u] = *reinterpret_cast<const u32x4 *>(
          vb + (size_t)min(pw + (u * 64 + lane) / kChunks, p1 - 1) * kD);
  };
  // q is requested ahead of K and V, so that waiting for it does not wait for them
  constexpr int kQ = kMaxGroup * kD / kT;
  float q[kQ];
#pragma unroll
  for (int u = 0; u < kQ; u++)
    q[u] = a.q[((size_t)b * a.heads + h0) * kD + min(t + kT * u, G * kD - 1)];
  __builtin_amdgcn_sched_barrier(0);
  load_k(p0);
  load_v(p0);
  __builtin_amdgcn_sched_barrier(0);
  auto lds_barrier = [] {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): K and V stay in flight
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };
#pragma unroll
  for (int u = 0; u < kQ; u++)
    if (t + kT * u < G * kD) (&lds.q[0][0])[t + kT * u] = q[u] * a.scale;
  lds_barrier();
  for (int g = wave; g < G; g += 4) {
    float x[kD / 64], mx = 0.0f;
#pragma unroll
    for (int e = 0; e < kD / 64; e++) {
      x[e] = lds.q[g][lane + 64 * e];
      mx = fmaxf(mx, fabsf(x[e]));
    }
    mx = wave_max_rows(mx);
    // 2^ex > mx >= 2^(ex - 1) (0 for zero, infinity and NaN)
    const int ex = min(max(__builtin_amdgcn_frexp_expf(mx), -120), 120);
    if (lane == 0) qscale[g] = ldexpf(1.0f, ex);
#pragma unroll
    for (int e = 0; e < kD / 64; e++) {
      const float y = ldexpf(x[e], -ex);
      const _Float16 hi = (_Float16)y;
      qh[0][g][lane + 64 * e] = hi;
      qh[1][g][lane + 64 * e] = (_Float16)((y - (float)hi) * kQLow);
    }
  }
  lds_barrier();
  const float qs = qscale[min(r16, G - 1)];  // (columns past G repeat the last head, unused)

  float m_run = -INFINITY, l_run = 0.0f;
  f32x4 acc[kDT];
#pragma unroll
  for (int dt = 0; dt < kDT; dt++) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint8_t *vl = lds.v[wave];
  // chunk c of row r lies at c ^ 2 f(r): a transposing read's 32 lanes (8 rows,
  // 2 chunks each) then hit 64 banks
  auto swz = [](int r) { return kD == 128 ? 2 * (r & 7) : 2 * ((r >> 1) & 3); };
  // (more_c: another tile follows; its K is requested as soon as the scores have
  // used this one's, its V as soon as this one's is in LDS)
  auto tile = [&](int pt, auto more_c) __attribute__((always_inline)) {
    constexpr bool kMore = decltype(more_c)::value;
    f32x4 sc[kBlocks], low[kBlocks];
#pragma unroll
    for (int tt = 0; tt < kBlocks; tt++) sc[tt] = low[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < kKK; kk++)
#pragma unroll
      for (int part = 0; part < 2; part++) {
        const f16x8 qf = *reinterpret_cast<const f16x8 *>(&qh[part][min(r16, G - 1)][32 * kk + 8 * grp]);
        f32x4 (&to)[kBlocks] = part ? low : sc;
#pragma unroll
        for (int tt = 0; tt < kBlocks; tt++)
          to[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[tt][kk], qf, to[tt], 0, 0, 0);
      }
#pragma unroll
    for (int tt = 0; tt < kBlocks; tt++)
#pragma unroll
      for (int e = 0; e < 4; e++) sc[tt][e] = fmaf(low[tt][e], 1.0f / kQLow, sc[tt][e]);
    if constexpr (kMore) {
      __builtin_amdgcn_sched_barrier(0);
      load_k(pt + kAttnTile<kD>);
      __builtin_amdgcn_sched_barrier(0);
    }
    // V to this wave's LDS rows (LDS works in order: after the last tile's reads)
#pragma unroll
    for (int u = 0; u < kVLoads; u++) {
      const int r = (u * 64 + lane) / kChunks, c = lane % kChunks;
      *reinterpret_cast<u32x4 *>(vl + r * kRow + ((c ^ swz(r)) * 16)) = vr[u];
    }
    if constexpr (kMore) {
      __builtin_amdgcn_sched_barrier(0);
      load_v(pt + kAttnTile<kD>);
      __builtin_amdgcn_sched_barrier(0);
    }
    float mx = -INFINITY;
    const int pw = pt + wave * (16 * kBlocks) + 4 * grp;
#pragma unroll
    for (int tt = 0; tt < kBlocks; tt++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        sc[tt][e] = pw + 16 * tt + e < p1 ? sc[tt][e] * qs : -INFINITY;
        mx = fmaxf(mx, sc[tt][e]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m = fmaxf(m_run, mx);
    const float corr = m_run == m ? 1.0f : exp_neg(m_run - m);
    m_run = m;
    float ls = 0.0f;
    f16x8 p[kBlocks / 2][2];
#pragma unroll
    for (int tt = 0; tt < kBlocks; tt++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float w = pw + 16 * tt + e < p1 ? exp_neg(sc[tt][e] - m) * kPScale : 0.0f;
        const _Float16 hi = (_Float16)w;
        p[tt / 2][0][(tt & 1) * 4 + e] = hi;
        p[tt / 2][1][(tt & 1) * 4 + e] = (_Float16)(w - (float)hi);
        ls += w;
      }
    l_run = l_run * corr + ls;  // this lane's positions; the groups are summed at the end
#pragma unroll
    for (int dt = 0; dt < kDT; dt++)
#pragma unroll
      for (int e = 0; e < 4; e++) acc[dt][e] *= corr;
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // this wave's V rows are in LDS
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    const int ti = (lane >> 2) & 3, tq = lane & 3;
#pragma unroll
    for (int sl = 0; sl < kBlocks / 2; sl++)
#pragma unroll
      for (int dt = 0; dt < kDT; dt++) {
        s16x4 half[2];
#pragma unroll
        for (int q2 = 0; q2 < 2; q2++) {
          const int r = 32 * sl + 16 * q2 + 4 * grp + ti, c = 2 * dt + (tq >> 1);
          half[q2] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (SH_OPS_LDS s16x4 *)((SH_OPS_LDS uint8_t *)vl + r * kRow + ((c ^ swz(r)) * 16) + (tq & 1) * 8));
        }
        const f16x8 vf = __builtin_bit_cast(
            f16x8, __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
        for (int part = 0; part < 2; part++)
          acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, p[sl][part], acc[dt], 0, 0, 0);
      }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  };
  int pt = p0;
  for (; pt + kAttnTile<kD> < p1; pt += kAttnTile<kD>) tile(pt, std::true_type{});
  tile(pt, std::false_type{});

  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if (grp == 0) {
    stat[wave][r16][0] = m_run;
    stat[wave][r16][1] = l_run;
  }
  lds_barrier();  // every wave's V reads are done: lds.v becomes lds.acc
  if (r16 < G) {
#pragma unroll
    for (int dt = 0; dt < kDT; dt++)
      *reinterpret_cast<f32x4 *>(&lds.acc[wave][r16][16 * dt + 4 * grp]) = acc[dt];
  }
  lds_barrier();
  // the split's partial: the four waves' sums against their common maximum
  bool finite = true;
  for (int i = t; i < G * kD; i += kT) {
    const int g = i / kD, dd = i % kD;
    float m = stat[0][g][0];
#pragma unroll
    for (int w = 1; w < 4; w++) m = fmaxf(m, stat[w][g][0]);
    float sum = 0.0f, l = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const float f = stat[w][g][0] == m ? 1.0f : exp_neg(stat[w][g][0] - m);
      sum = fmaf(f, lds.acc[w][g][dd], sum);
      l = fmaf(f, stat[w][g][1], l);
    }
    finite = finite && __builtin_fabsf(sum) < INFINITY && l < INFINITY;
    attn_store<kD>(a, b, h0, s, i, sum, m, l);
  }
  if (__syncthreads_or(finite ? 0 : 1)) attn_fp32<kD>(a, b, kvh, s, p0, p1, lds.fp32);
}

// grid (heads, B), 4 kD threads:
//   out = sum_j exp(m_j - M) acc_j / sum_j exp(m_j - M) l_j,  M = max_j m_j
// over the row's active splits j (rows of length <= 0: zeros). Thread (part,
// dim) takes splits part, part + 4, .. against their own maximum, 8 requested
// at once; the four parts are combined at the end.
constexpr int kMergeParts = 4;
template <int kD>
__global__ __launch_bounds__(kD * kMergeParts) void attn_op_merge_kernel(const AttnOpArgs a) {
  constexpr int kStep = 8;
  __shared__ float red[kMergeParts][kD], lred[kMergeParts], mred[kMergeParts];
  const int h = blockIdx.x, b = blockIdx.y, t = threadIdx.x, i = t % kD, part = t / kD;
  const int L = min(a.lengths[b], a.max_pos);
  float *o = a.out + ((size_t)b * a.heads + h) * kD;
  if (L <= 0) {
    if (part == 0) o[i] = 0.0f;
    return;
  }
  const int active = (L + a.chunk - 1) / a.chunk;
  const size_t pstride = (size_t)kD + 2;
  const float *pp = a.part + ((size_t)b * a.heads + h) * a.splits * pstride;
  float M = -INFINITY, num = 0.0f, den = 0.0f;
  for (int j0 = part; j0 < active; j0 += kMergeParts * kStep) {
    float x[kStep], m[kStep], l[kStep], top = M;
#pragma unroll
    for (int u = 0; u < kStep; u++) {
      const float *p = pp + (size_t)min(j0 + kMergeParts * u, active - 1) * pstride;
      x[u] = p[i];
      m[u] = p[kD];
      l[u] = p[kD + 1];
    }
#pragma unroll
    for (int u = 0; u < kStep; u++)
      if (j0 + kMergeParts * u < active) top = fmaxf(top, m[u]);
    const float c = M == top ? 1.0f : exp_neg(M - top);
    M = top;
    num *= c;
    den *= c;
#pragma unroll
    for (int u = 0; u < kStep; u++) {
      const bool is = j0 + kMergeParts * u < active;
      const float w = m[u] == M ? 1.0f : exp_neg(m[u] - M);
      num = is ? fmaf(w, x[u], num) : num;  // (0 times an infinity is not 0)
      den = is ? fmaf(w, l[u], den) : den;
    }
  }
  red[part][i] = num;
  if (i == 0) {
    lred[part] = den;
    mred[part] = M;
  }
  __syncthreads();
  if (part != 0) return;
  const float top = fmaxf(fmaxf(mred[0], mred[1]), fmaxf(mred[2], mred[3]));
  num = den = 0.0f;
#pragma unroll
  for (int w = 0; w < kMergeParts; w++) {
    const float f = mred[w] == top ? 1.0f : exp_neg(mred[w] - top);
    num = fmaf(f, red[w][i], num);
    den = fmaf(f, lred[w], den);
  }
  o[i] = num / den;
}

// Split layout of a call. The lengths are on the device, so the splits cover
// max_pos; one of no active position ends at once. Splits of one tile, up to
// about 2,048 workgroups, of more tiles beyond that. Three per CU, 768, are
// resident together (registers; 42 KiB of LDS at head_dim 128), but planned for 768
// a call took longer: 4 rows of 4,096 positions, 16 / 8 heads of 128, 19.0 us
// against 17.5, 64 rows of 1,000 55.1 against 51.0, 1 row of 131,200, 4 / 1 heads,
// a half-filled cache 25.3 against 20.3 (16 rows of 8,192, 16 / 1 heads 24.0
// against 27.4); 1,536 is level. Where the partials of that layout would exceed the
// allocation-free entry's array, the coarser one of about two workgroups per CU.
void attn_split(int batch, int heads, int kv_heads, int head_dim, int max_pos, int *splits, int *chunk) {
  const long long rows = (long long)batch * kv_heads;
  const int tile = head_dim == 64 ? kAttnTile<64> : kAttnTile<128>;
  const long long tiles = (max_pos + tile - 1) / tile;
  const long long per = std::max(1LL, (tiles * rows + 2047) / 2048);
  const long long fine = (tiles + per - 1) / per;
  if (fine <= 1024 && (long long)batch * heads * fine * (head_dim + 2) * 4 <=
                          (long long)SH_ATTN_NOALLOC_MAX_BYTES) {
    *chunk = (int)(per * tile);
    *splits = (int)fine;
    return;
  }
  const int want = (int)std::max(1LL, std::min(1024LL, (512 + rows - 1) / rows));
  int c = (max_pos + want - 1) / want;
  c = (c + 63) / 64 * 64;
  *chunk = c;
  *splits = (max_pos + c - 1) / c;
}

size_t attn_part_bytes(int batch, int heads, int head_dim, int splits) {
  return (size_t)batch * heads * splits * (head_dim + 2) * sizeof(float);
}

int check_attn(sh_ctx *ctx, const float *q, const uint16_t *k, const uint16_t *v,
               const int32_t *lengths, float *out, int batch, int heads, int kv_heads,
               int head_dim, int max_positions) {
  if (batch < 1 || heads < 1 || kv_heads < 1 || max_positions < 1)
    return fail(SH_ERR_INVALID_ARGUMENT,
                "attention sizes must be positive (batch=%d heads=%d kv_heads=%d max_positions=%d)",
                batch, heads, kv_heads, max_positions);
  if (heads % kv_heads != 0 || heads / kv_heads > kMaxGroup)
    return fail(SH_ERR_INVALID_ARGUMENT, "heads %d must be kv_heads %d times 1..%d", heads, kv_heads,
                kMaxGroup);
  if (head_dim != 64 && head_dim != 128)
    return fail(SH_ERR_UNSUPPORTED, "attention head_dim %d (64 or 128 are built)", head_dim);
  if (max_positions > (1 << 24)) return fail(SH_ERR_INVALID_ARGUMENT, "max_positions > 2^24");
  if ((reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v)) & 15)
    return fail(SH_ERR_INVALID_ARGUMENT, "k and v caches must be 16-byte aligned");
  const size_t qn = (size_t)batch * heads * head_dim;
  const size_t kvn = (size_t)batch * kv_heads * max_positions * head_dim;
  int rc;
  if ((rc = check_range(ctx, q, qn * 4, "q")) || (rc = check_range(ctx, k, kvn * 2, "k")) ||
      (rc = check_range(ctx, v, kvn * 2, "v")) ||
      (rc = check_range(ctx, lengths, (size_t)batch * 4, "lengths")) ||
      (rc = check_range(ctx, out, qn * 4, "out")))
    return rc;
  return SH_OK;
}

template <int kD>
hipError_t launch_attn_d(hipStream_t st, const AttnOpArgs &a, int batch) {
  const dim3 grid_p(a.splits, a.kv_heads, batch), grid_m(a.heads, batch);
  attn_op_partials_kernel<kD><<<grid_p, kT, 0, st>>>(a);
  if (a.splits > 1) attn_op_merge_kernel<kD><<<grid_m, kD * kMergeParts, 0, st>>>(a);
  return hipGetLastError();
}

hipError_t launch_attn(hipStream_t st, const AttnOpArgs &a, int batch, int head_dim) {
  return head_dim == 64 ? launch_attn_d<64>(st, a, batch) : launch_attn_d<128>(st, a, batch);
}

int run_attn(sh_ctx *ctx, const float *q, const uint16_t *k, const uint16_t *v,
             const int32_t *lengths, float *out, int batch, int heads, int kv_heads, int head_dim,
             int max_positions, float scale, float *part, int splits, int chunk) {
  AttnOpArgs a;
  a.q = q;
  a.k = k;
  a.v = v;
  a.lengths = lengths;
  a.out = out;
  a.part = part;
  a.heads = heads;
  a.kv_heads = kv_heads;
  a.max_pos = max_positions;
  a.splits = splits;
  a.chunk = chunk;
  a.scale = scale;
  const hipError_t e = launch_attn(stream_of(ctx), a, batch, head_dim);
  return e == hipSuccess ? SH_OK : hip_fail(e, "attention decode");
}

// ---- the allocation-free attention's work buffer --------------------------------

// Partials of sh_attn_decode_f16_noalloc: one array per device, held from the
// library's load until the process ends. Host code never passes `scratch`
// itself to a kernel (in host code the name is a stand-in, not a device
// address): the device address comes from hipGetSymbolAddress, once per
// device with that device current, and is kept in g_scratch_dev.
constexpr size_t kNoAllocScratchBytes = SH_ATTN_NOALLOC_MAX_BYTES;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_dev[kMaxDevices] = {};

// The current device's address of `scratch` (ctx's device is current).
int noalloc_scratch(sh_ctx *ctx, void **ptr) {
  const int dev = device_of(ctx);
  if (dev < 0 || dev >= kMaxDevices) return fail(SH_ERR_NO_DEVICE, "device %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_dev[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!p) return fail(SH_ERR_HIP, "hipGetSymbolAddress(scratch) returned NULL");
    g_scratch_dev[dev] = p;
  }
  *ptr = g_scratch_dev[dev];
  return SH_OK;
}

}  // namespace
}  // namespace sh

using namespace sh;

extern "C" {

SH_API int sh_rmsnorm_f32(sh_ctx *ctx, const float *x, const float *gain, float *y, int rows,
                          int n, float eps) {
  int rc = enter(ctx);
  if (rc != SH_OK) return rc;
  if (rows < 0 || n < 0) return fail(SH_ERR_INVALID_ARGUMENT, "negative size rows=%d n=%d", rows, n);
  if (rows == 0 || n == 0) return SH_OK;
  if (!(eps >= 0.0f)) return fail(SH_ERR_INVALID_ARGUMENT, "eps must be >= 0");
  const size_t bytes = (size_t)rows * n * 4;
  if ((rc = check_range(ctx, x, bytes, "x")) || (rc = check_range(ctx, gain, (size_t)n * 4, "gain")) ||
      (rc = check_range(ctx, y, bytes, "y")))
    return rc;
  const hipError_t e = launch_norm<false>(stream_of(ctx), x, gain, nullptr, y, rows, n, eps);
  return e == hipSuccess ? SH_OK : hip_fail(e, "rmsnorm");
}

SH_API int sh_layernorm_f32(sh_ctx *ctx, const float *x, const float *gain, const float *bias,
                            float *y, int rows, int n, float eps) {
  int rc = enter(ctx);
  if (rc != SH_OK) return rc;
  if (rows < 0 || n < 0) return fail(SH_ERR_INVALID_ARGUMENT, "negative size rows=%d n=%d", rows, n);
  if (rows == 0 || n == 0) return SH_OK;
  if (!(eps >= 0.0f)) return fail(SH_ERR_INVALID_ARGUMENT, "eps must be >= 0");
  const size_t bytes = (size_t)rows * n * 4;
  if ((rc = check_range(ctx, x, bytes, "x")) || (rc = check_range(ctx, gain, (size_t)n * 4, "gain")) ||
      (rc = check_range(ctx, bias, (size_t)n * 4, "bias")) || (rc = check_range(ctx, y, bytes, "y")))
    return rc;
  const hipError_t e = launch_norm<true>(stream_of(ctx), x, gain, bias, y, rows, n, eps);
  return e == hipSuccess ? SH_OK : hip_fail(e, "layernorm");
}

SH_API int sh_rope_f32(sh_ctx *ctx, float *x, const int32_t *positions, int rows, int heads,
                       int head_dim, float theta) {
  int rc = enter(ctx);
  if (rc != SH_OK) return rc;
  if (rows < 0 || heads < 0) return fail(SH_ERR_INVALID_ARGUMENT, "negative size rows=%d heads=%d", rows, heads);
  if (head_dim < 2 || head_dim % 2 != 0 || head_dim > 512)
    return fail(SH_ERR_INVALID_ARGUMENT, "head_dim %d must be even and 2..512", head_dim);
  if (!(theta > 0.0f)) return fail(SH_ERR_INVALID_ARGUMENT, "theta must be positive");
  if (rows == 0 || heads == 0) return SH_OK;
  if ((long long)rows * heads > 0x7fffffffLL)
    return fail(SH_ERR_INVALID_ARGUMENT, "rows * heads exceeds 2^31 - 1");
  if ((rc = check_range(ctx, x, (size_t)rows * heads * head_dim * 4, "x")) ||
      (rc = check_range(ctx, positions, (size_t)rows * 4, "positions")))
    return rc;
  const int width = (head_dim / 2 + 63) / 64 * 64;  // 64 .. 256
  const long long units = (long long)rows * ((heads + kRopeHeads - 1) / kRopeHeads);
  const int per_block = kT / width;
  rope_kernel<<<(unsigned)((units + per_block - 1) / per_block), kT, 0, stream_of(ctx)>>>(
      x, positions, rows, heads, head_dim, width, std::log2((double)theta));
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SH_OK : hip_fail(e, "rope");
}

SH_API int sh_swiglu_f32(sh_ctx *ctx, const float *gate, const float *up, float *out, size_t n) {
  int rc = enter(ctx);
  if (rc != SH_OK) return rc;
  if (n == 0) return SH_OK;
  if ((rc = check_range(ctx, gate, n * 4, "gate")) || (rc = check_range(ctx, up, n * 4, "up")) ||
      (rc = check_range(ctx, out, n * 4, "out")))
    return rc;
  swiglu_kernel<<<map4_grid(n), kT, 0, stream_of(ctx)>>>(gate, up, out, n);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SH_OK : hip_fail(e, "swiglu");
}

SH_API int sh_gelu_f32(sh_ctx *ctx, const float *x, float *y, size_t n) {
  int rc = enter(ctx);
  if (rc != SH_OK) return rc;
  if (n == 0) return SH_OK;
  if ((rc = check_range(ctx, x, n * 4, "x")) || (rc = check_range(ctx, y, n * 4, "y"))) return rc;
  gelu_kernel<<<map4_grid(n), kT, 0, stream_of(ctx)>>>(x, y, n);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? SH_OK : hip_fail(e, "gelu");
}

SH_API int sh_argmax_f32(sh_ctx *ctx, const float *x, int rows, int n, int32_t *index) {
  int rc = enter(ctx);
  if (rc != SH_OK) return rc;
  if (rows < 0 || n < 1) return fail(SH_ERR_INVALID_ARGUMENT, "need rows >= 0 and n >= 1 (rows=%d n=%d)", rows, n);
  if (rows == 0) return SH_OK;
  if ((rc = check_range(ctx, x, (size_t)rows * n * 4, "x")) ||
      (rc = check_range(ctx, index, (size_t)rows * 4, "index")))
    return rc;
  const hipError_t e = launch_argmax(stream_of(ctx), x, rows, n, index);
  return e == hipSuccess ? SH_OK : hip_fail(e, "argmax");
}

SH_API int sh_attn_decode_f16(sh_ctx *ctx, const float *q, const uint16_t *k, const uint16_t *v,
                              const int32_t *lengths, float *out, int batch, int heads,
                              int kv_heads, int head_dim, int max_positions, float scale) {
  int rc = enter(ctx);
  if (rc != SH_OK) return rc;
  if ((rc = check_attn(ctx, q, k, v, lengths, out, batch, heads, kv_heads, head_dim, max_positions)))
    return rc;
  int splits = 0, chunk = 0;
  attn_split(batch, heads, kv_heads, head_dim, max_positions, &splits, &chunk);
  void *part = nullptr;
  // at least what the fine layout may ask for: a later call whose splits are finer
  // finds its partials there and does not allocate (its stream may be capturing)
  const size_t need = attn_part_bytes(batch, heads, head_dim, splits);
  if ((rc = context_scratch(ctx, std::max(need, SH_ATTN_NOALLOC_MAX_BYTES), &part))) return rc;
  return run_attn(ctx, q, k, v, lengths, out, batch, heads, kv_heads, head_dim, max_positions, scale,
                  static_cast<float *>(part), splits, chunk);
}

SH_API int sh_attn_decode_f16_noalloc(sh_ctx *ctx, const float *q, const uint16_t *k,
                                      const uint16_t *v, const int32_t *lengths, float *out,
                                      int batch, int heads, int kv_heads, int head_dim,
                                      int max_positions, float scale) {
  int rc = enter(ctx);
  if (rc != SH_OK) return rc;
  if ((rc = check_attn(ctx, q, k, v, lengths, out, batch, heads, kv_heads, head_dim, max_positions)))
    return rc;
  int splits = 0, chunk = 0;
  attn_split(batch, heads, kv_heads, head_dim, max_positions, &splits, &chunk);
  const size_t need = attn_part_bytes(batch, heads, head_dim, splits);
  if (need > kNoAllocScratchBytes)
    return fail(SH_ERR_INVALID_ARGUMENT,
                "attention partials need %zu bytes, more than the %zu-byte allocation-free "
                "work buffer (batch * heads * splits * (head_dim + 2) * 4, %d splits)",
                need, kNoAllocScratchBytes, splits);
  void *part = nullptr;
  if ((rc = noalloc_scratch(ctx, &part))) return rc;
  return run_attn(ctx, q, k, v, lengths, out, batch, heads, kv_heads, head_dim, max_positions, scale,
                  static_cast<float *>(part), splits, chunk);
}

}  // extern "C"
