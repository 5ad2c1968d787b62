// Per-token and block activation quantisers (memory-bound pre-passes of the W8A8 GEMMs).  16-bit activations in rows of
// whole 16-byte units take quant_rows_kernel / quant_row_blocks_kernel (one read of x, 16-byte accesses); fp32, ragged
// or unaligned rows, static scales and tiles of several rows take the element-wise kernels.
//
// INT8 (forge/kernels/ref/gemm_int8.py:17-35): s = amax / 127 with IEEE division (1 where amax > 0 is false),
//   q = clamp(round_half_even(x / s), -127, 127), x / s again IEEE-divided, so codes equal the CPU oracle's bit for
//   bit, ties included.  NaN inputs give code 0, like the oracle's float->int8 cast.
// FP8 (forge/kernels/ref/gemm_fp8.py:43-85,130-150): optional fused RMSNorm y = x * (1 / sqrt(mean(x^2) + eps)) * w in
//   fp32, s = amax(y) / 448 (IEEE; 1 where amax > 0 is false, so NaN rows get scale 1 as in the oracle), or a static
//   device scale; q = e4m3fn(clamp(y / s, -448, 448)) with gfx950's round-to-nearest-even OCP fp8 conversion.
#include <algorithm>

#include "fg_device.h"

namespace fg {

__device__ __forceinline__ float block_reduce(float v, bool is_max, float* red) {
  v = is_max ? wave_max(v) : wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float r = red[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = is_max ? fmaxf(r, red[w]) : r + red[w];
  return r;
}

__global__ void __launch_bounds__(256) quant_int8_rowwise_kernel(const void* __restrict__ x, int64_t ldx, int xdt,
                                                                 int8_t* __restrict__ q, int64_t ldq,
                                                                 float* __restrict__ s, int K) {
  __shared__ float red[8];
  __shared__ int nan_flag;
  const int64_t row = blockIdx.x;
  if (threadIdx.x == 0) nan_flag = 0;
  __syncthreads();
  float amax = 0.f;
  bool has_nan = false;
  for (int k = threadIdx.x; k < K; k += blockDim.x) {
    const float v = load_f(x, xdt, row * ldx + k);
    has_nan |= __builtin_isnan(v);
    amax = fmaxf(amax, fabsf(v));
  }
  if (has_nan) nan_flag = 1;
  amax = block_reduce(amax, true, red);
  // torch.amax propagates NaN and `NaN > 0` is false: such rows take scale 1
  const float scale = (!nan_flag && amax > 0.f) ? __fdiv_rn(amax, 127.f) : 1.f;
  if (threadIdx.x == 0) s[row] = scale;
  for (int k = threadIdx.x; k < K; k += blockDim.x) {
    const float v = __fdiv_rn(load_f(x, xdt, row * ldx + k), scale);
    const float r = __builtin_isnan(v) ? 0.f : rintf(fminf(fmaxf(v, -127.f), 127.f));
    q[row * ldq + k] = (int8_t)(int)r;
  }
}

__device__ __forceinline__ uint8_t f32_to_e4m3(float v) {
  // v_cvt_pk_fp8_f32: OCP e4m3 (gfx950), round to nearest even; inputs are pre-clamped to +-448.  A NaN becomes the
  // e4m3fn NaN code with its sign (0x7F / 0xFF), as torch's cast writes it.
  const int packed = __builtin_amdgcn_cvt_pk_fp8_f32(v, 0.f, 0, false);
  const uint8_t nan_code = (__float_as_uint(v) >> 24 & 0x80) | 0x7F;
  return __builtin_isnan(v) ? nan_code : (uint8_t)(packed & 0xff);
}

__global__ void __launch_bounds__(256) quant_fp8_rowwise_kernel(const void* __restrict__ x, int64_t ldx, int xdt,
                                                                uint8_t* __restrict__ q, int64_t ldq,
                                                                float* __restrict__ s, int K,
                                                                const float* __restrict__ static_scale,
                                                                const void* __restrict__ rms_w, int wdt, float eps,
                                                                int fuse) {
  __shared__ float red[8];
  __shared__ int nan_flag;
  const int64_t row = blockIdx.x;
  if (threadIdx.x == 0) nan_flag = 0;
  __syncthreads();
  float rs = 1.f;
  if (fuse) {
    float ss = 0.f;
    for (int k = threadIdx.x; k < K; k += blockDim.x) {
      const float v = load_f(x, xdt, row * ldx + k);
      ss = __builtin_fmaf(v, v, ss);
    }
    ss = block_reduce(ss, false, red);
    rs = __fdiv_rn(1.f, __fsqrt_rn(__fdiv_rn(ss, (float)K) + eps));
  }
  auto yval = [&](int k) {
    float v = load_f(x, xdt, row * ldx + k);
    if (fuse) {
      v = v * rs;
      if (rms_w) v = v * load_f(rms_w, wdt, k);
    }
    return v;
  };
  float scale;
  if (static_scale) {
    scale = static_scale[row];
  } else {
    float amax = 0.f;
    bool has_nan = false;
    for (int k = threadIdx.x; k < K; k += blockDim.x) {
      const float v = yval(k);
      has_nan |= __builtin_isnan(v);
      amax = fmaxf(amax, fabsf(v));
    }
    if (has_nan) nan_flag = 1;
    amax = block_reduce(amax, true, red);
    scale = (!nan_flag && amax > 0.f) ? __fdiv_rn(amax, 448.f) : 1.f;
    if (threadIdx.x == 0) s[row] = scale;
  }
  for (int k = threadIdx.x; k < K; k += blockDim.x) {
    const float v = __fdiv_rn(yval(k), scale);
    const float c = __builtin_isnan(v) ? v : fminf(fmaxf(v, -448.f), 448.f);
    q[row * ldq + k] = f32_to_e4m3(c);
  }
}

// ------------------------------------------------------------------------------------------- 16-byte quantisers
// What bounds these is the latency of one row for few rows and HBM for many.  The element-wise kernels above read x
// twice (three times with the norm) in 2-byte accesses and divide with the ~12-instruction IEEE sequence: 20.6 us for 32
// rows of 4096..14336, 79 us for 4096 x 8192 (1.3 TB/s), 24 us for 1024 x 4096 with the norm, and 45 us for 600 x 8192
// in 1 x 128 blocks (a workgroup per block).  Here a row is read once, 8 values per lane and 16-byte load, and stays in
// registers; the absolute maximum is a packed 16-bit integer maximum of the bit patterns (their order is the order of
// magnitudes, a NaN above every number); and the quotient by the row's scale is exact with five multiply-adds.  The same
// four calls: 4.8, 18.9 (5.3 TB/s), 8.3 and 7.3 us (kernel trace; the third with the norm's sum in the element-wise
// kernel's order, which costs 0.5 us of it: row_sum_sq).

// RN(a / b) from y = RN(1 / b): q0 = a y is within two units in the last place, one correction brings it within one,
// and the second correction of a quotient that close is the correctly rounded one (Markstein, "Computation of
// elementary functions on the IBM RISC System/6000 processor", 1990, theorem on division with a fused multiply-add).
// It holds while no intermediate leaves the normal range: the callers use it for 2^-60 <= b <= 2^60.  There a residual
// can only lose bits for |a| < 2^-102, where the quotient is below 2^-42 and its code is zero either way.
__device__ __forceinline__ float div_by(float a, float b, float y) {
  const float q0 = a * y;
  const float q1 = __builtin_fmaf(__builtin_fmaf(-b, q0, a), y, q0);
  return __builtin_fmaf(__builtin_fmaf(-b, q1, a), y, q1);
}
__device__ __forceinline__ bool div_by_ok(float b) { return b >= 0x1p-60f && b <= 0x1p60f; }

template <bool BF16>
__device__ __forceinline__ void unpack8(const uint4& u, float (&f)[8]) {
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (BF16) {
      f[2 * i] = __uint_as_float(w[i] << 16);
      f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    } else {
      f[2 * i] = f16_bits_to_f32((uint16_t)w[i]);
      f[2 * i + 1] = f16_bits_to_f32((uint16_t)(w[i] >> 16));
    }
  }
}

// Largest magnitude among 8 packed 16-bit floats, folded into `m` (two bit patterns, one per half).
__device__ __forceinline__ uint32_t absmax8(const uint4& u, uint32_t m) {
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  u16x2 r = __builtin_bit_cast(u16x2, m);
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) r = __builtin_elementwise_max(r, __builtin_bit_cast(u16x2, w[i] & 0x7fff7fffu));
  return __builtin_bit_cast(uint32_t, r);
}

// Codes of 8 values as they lie in memory.  `fast`: div_by applies (finite values, a scale in its range).
template <bool FP8>
__device__ __forceinline__ uint2 encode8(const float (&v)[8], float scale, float y, bool fast) {
  float c[8];
  if (fast) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float q = div_by(v[i], scale, y);
      // the corrections turn -0 into +0; an e4m3 code keeps the sign of a zero
      c[i] = FP8 ? __builtin_copysignf(fminf(fmaxf(q, -448.f), 448.f), v[i]) : fminf(fmaxf(q, -127.f), 127.f);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float q = __fdiv_rn(v[i], scale);
      if (FP8)
        c[i] = __builtin_isnan(q) ? q : fminf(fmaxf(q, -448.f), 448.f);
      else
        c[i] = __builtin_isnan(q) ? 0.f : fminf(fmaxf(q, -127.f), 127.f);
    }
  }
  uint32_t w[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float* d = c + 4 * h;
    if (FP8) {
      if (fast) {
        int p = __builtin_amdgcn_cvt_pk_fp8_f32(d[0], d[1], 0, false);
        p = __builtin_amdgcn_cvt_pk_fp8_f32(d[2], d[3], p, true);
        w[h] = (uint32_t)p;
      } else {
        w[h] = (uint32_t)f32_to_e4m3(d[0]) | (uint32_t)f32_to_e4m3(d[1]) << 8 | (uint32_t)f32_to_e4m3(d[2]) << 16 |
               (uint32_t)f32_to_e4m3(d[3]) << 24;
      }
    } else {
      // |d| <= 127: adding 1.5 * 2^23 rounds to the nearest integer, ties to even, and leaves it in the low byte
      uint32_t b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = __float_as_uint(d[i] + 12582912.f);
      w[h] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(b[3], b[2], 0x0c0c0400u),
                                   __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u), 0x05040100u);
    }
  }
  return make_uint2(w[0], w[1]);
}

__device__ __forceinline__ void load8_f(const void* p, int dt, int64_t i, float (&f)[8]) {
  if (dt == FG_F32) {
    const float4 a = *reinterpret_cast<const float4*>(static_cast<const float*>(p) + i);
    const float4 b = *reinterpret_cast<const float4*>(static_cast<const float*>(p) + i + 4);
    f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
    f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
  } else {
    const uint4 u = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p) + i);
    if (dt == FG_BF16) unpack8<true>(u, f);
    else unpack8<false>(u, f);
  }
}

template <bool BF16>
__device__ __forceinline__ float pattern_f(uint32_t b) {
  return BF16 ? bf16_bits_to_f32(b) : f16_bits_to_f32((uint16_t)b);
}
__device__ __forceinline__ bool pattern_nan(bool bf16, uint32_t b) { return b > (bf16 ? 0x7f80u : 0x7c00u); }

// Sum of squares of a row of K 16-bit values that lies in LDS as pairs, in the order of quant_fp8_rowwise_kernel's 256
// threads (thread v sums columns v, v + 256, .. in turn, then wave_sum, then the four wavefronts in turn), so that the
// normed values and their codes are the same bytes whichever kernel a row takes.  A thread of the first two wavefronts
// (with one wavefront, each thread twice) stands for two neighbours v = 2 t, 2 t + 1, whose columns are one pair.  (us,
// graph replays, element-wise kernel / this one / each thread summing the units it holds: 32 x 4096 13.3 / 3.8 / 3.3,
// 1024 x 4096 18.7 / 7.0 / 6.5, 1024 x 14336 77.4 / 17.1 / 16.4.)
template <bool BF16>
__device__ __forceinline__ float row_sum_sq(const uint32_t* pairs, int K, int T, float* red) {
  const auto lo = [](uint32_t w) { return BF16 ? __uint_as_float(w << 16) : f16_bits_to_f32((uint16_t)w); };
  const auto hi = [](uint32_t w) { return BF16 ? __uint_as_float(w & 0xffff0000u) : f16_bits_to_f32((uint16_t)(w >> 16)); };
  if (threadIdx.x < 128) {
    for (int t = threadIdx.x; t < 128; t += T) {  // T is 64 or at least 128
      float a = 0.f, b = 0.f;
#pragma unroll 4
      for (int p = t; p < K / 2; p += 128) {
        const uint32_t w = pairs[p];
        a = __builtin_fmaf(lo(w), lo(w), a);
        b = __builtin_fmaf(hi(w), hi(w), b);
      }
#pragma unroll
      for (int off = 16; off > 0; off >>= 1) {  // wave_sum's exchanges over 32, 16, .., 2 columns' threads
        a += __shfl_xor(a, off, kWave);
        b += __shfl_xor(b, off, kWave);
      }
      if ((t & 31) == 0) red[t >> 5] = a + b;  // ... and over neighbours
    }
  }
  __syncthreads();
  return ((red[0] + red[1]) + red[2]) + red[3];
}

// One workgroup per row; thread t holds the row's 16-byte units t, t + T, .. (C of them at most, T threads).  With the norm
// the row also goes through LDS (2 K bytes), for the order of the sum above.
template <int C, bool BF16, bool FP8, bool RMS>
__global__ void __launch_bounds__(1024) quant_rows_kernel(const uint16_t* __restrict__ x, int64_t ldx,
                                                          uint8_t* __restrict__ q, int64_t ldq, float* __restrict__ s,
                                                          int K, const void* __restrict__ rms_w, int wdt, float eps) {
  extern __shared__ __align__(16) uint4 row_units[];
  __shared__ uint32_t red[16];
  __shared__ float red_ss[4];
  const int64_t row = blockIdx.x;
  const int T = blockDim.x, units = K / 8, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = T >> 6;
  const uint4* xr = reinterpret_cast<const uint4*>(x + row * ldx);
  uint4 u[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int k = threadIdx.x + c * T;
    u[c] = k < units ? xr[k] : make_uint4(0, 0, 0, 0);
  }
  float rs = 1.f;
  if (RMS) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int k = threadIdx.x + c * T;
      if (k < units) row_units[k] = u[c];
    }
    __syncthreads();
    const float ss = row_sum_sq<BF16>(reinterpret_cast<const uint32_t*>(row_units), K, T, red_ss);
    rs = __fdiv_rn(1.f, __fsqrt_rn(__fdiv_rn(ss, (float)K) + eps));
  }
  auto normed = [&](int c, float (&f)[8]) {
    unpack8<BF16>(u[c], f);
    if (RMS) {
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] *= rs;
      const int k = threadIdx.x + c * T;
      if (rms_w && k < units) {
        float g[8];
        load8_f(rms_w, wdt, (int64_t)k * 8, g);
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] *= g[i];
      }
    }
  };
  uint32_t m = 0;  // bit pattern of the largest magnitude (16-bit without the norm, fp32 with it)
  if (RMS) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (threadIdx.x + c * T >= units) continue;  // zeros past the row, which an infinite rs would turn into NaN
      float f[8];
      normed(c, f);
#pragma unroll
      for (int i = 0; i < 8; ++i) m = max(m, __float_as_uint(f[i]) & 0x7fffffffu);
    }
  } else {
#pragma unroll
    for (int c = 0; c < C; ++c) m = absmax8(u[c], m);
    m = max(m & 0xffffu, m >> 16);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, kWave));
  if (waves > 1) {
    if (lane == 0) red[wave] = m;
    __syncthreads();
    for (int w = 0; w < waves; ++w) m = max(m, red[w]);
  }
  const bool nan = RMS ? m > 0x7f800000u : pattern_nan(BF16, m);
  const float amax = RMS ? __uint_as_float(m) : pattern_f<BF16>(m);
  const float top = FP8 ? 448.f : 127.f;
  // torch.amax propagates NaN and `NaN > 0` is false: such rows take scale 1
  const float scale = (!nan && amax > 0.f) ? __fdiv_rn(amax, top) : 1.f;
  if (threadIdx.x == 0) s[row] = scale;
  const bool fast = !nan && div_by_ok(scale);
  const float y = __fdiv_rn(1.f, scale);
  uint2* qr = reinterpret_cast<uint2*>(q + row * ldq);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int k = threadIdx.x + c * T;
    if (k < units) {
      float f[8];
      normed(c, f);
      qr[k] = encode8<FP8>(f, scale, y, fast);
    }
  }
}

// FP8 in 1 x bk blocks: L = bk / 8 lanes (a power of two up to 64) hold one block, so a wavefront covers 64 / L of them
// and the amax needs no LDS.
template <bool BF16>
__global__ void __launch_bounds__(256) quant_row_blocks_kernel(const uint16_t* __restrict__ x, int64_t ldx,
                                                               uint8_t* __restrict__ q, int64_t ldq,
                                                               float* __restrict__ s, int64_t lds, int64_t ldk, int M,
                                                               int K, int kb, int log_l) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const uint32_t block = (uint32_t)(t >> log_l), row = block / (uint32_t)kb, b = block - row * (uint32_t)kb;
  const int l = (int)(t & ((1 << log_l) - 1)), k = (int)((b << log_l) + l) * 8;
  const bool in = row < (uint32_t)M && k < K;
  const uint4 u = in ? *reinterpret_cast<const uint4*>(x + (int64_t)row * ldx + k) : make_uint4(0, 0, 0, 0);
  uint32_t m = absmax8(u, 0);
  m = max(m & 0xffffu, m >> 16);
  for (int off = (1 << log_l) >> 1; off > 0; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, kWave));
  const bool nan = pattern_nan(BF16, m);
  const float amax = pattern_f<BF16>(m);
  const float scale = (!nan && amax > 0.f) ? __fdiv_rn(amax, 448.f) : 1.f;
  const bool fast = !nan && div_by_ok(scale);
  if (!in) return;
  if (l == 0) s[(int64_t)row * lds + b * ldk] = scale;
  float f[8];
  unpack8<BF16>(u, f);
  *reinterpret_cast<uint2*>(q + (int64_t)row * ldq + k) = encode8<true>(f, scale, __fdiv_rn(1.f, scale), fast);
}

constexpr int kQuantNormMaxK = 32000;

// Whether x and q can be accessed in 16- and 8-byte units: 16-bit values in whole units, aligned rows.
static bool quant_vec_ok(const void* x, int64_t ldx, int xdt, const void* q, int64_t ldq, int64_t K) {
  return (xdt == FG_BF16 || xdt == FG_F16) && K % 8 == 0 && ldx % 8 == 0 && ldq % 8 == 0 &&
         reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(q) % 8 == 0;
}

// Threads per row and units per thread: one unit per thread while the rows are too few to fill the CUs (up to two
// workgroups each; a row's latency counts), else about four (rows in flight count).  Rows past 65536 columns do not
// fit: returns 0.
static int quant_rows_plan(int64_t M, int64_t K, int* C) {
  const int64_t units = K / 8, per = M <= 2 * device_cus() ? 1 : 4;
  const int64_t t = std::min<int64_t>(1024, ((units + per - 1) / per + kWave - 1) / kWave * kWave);
  const int64_t c = (units + t - 1) / t;
  *C = c <= 1 ? 1 : (c <= 2 ? 2 : (c <= 4 ? 4 : 8));
  return c > 8 ? 0 : (int)t;
}

template <bool FP8, bool RMS>
static hipError_t launch_quant_rows(const void* x, int64_t ldx, int xdt, uint8_t* q, int64_t ldq, float* s, int M,
                                    int K, int T, int C, const void* rms_w, int wdt, float eps, hipStream_t st) {
  auto go = [&](auto c_tag, auto bf_tag) {
    hipLaunchKernelGGL((quant_rows_kernel<decltype(c_tag)::value, decltype(bf_tag)::value, FP8, RMS>), dim3(M), dim3(T),
                       RMS ? (size_t)K * 2 : 0, st, static_cast<const uint16_t*>(x), ldx, q, ldq, s, K, rms_w, wdt, eps);
    return hipGetLastError();
  };
  auto pick = [&](auto bf_tag) {
    if (C == 1) return go(std::integral_constant<int, 1>{}, bf_tag);
    if (C == 2) return go(std::integral_constant<int, 2>{}, bf_tag);
    if (C == 4) return go(std::integral_constant<int, 4>{}, bf_tag);
    return go(std::integral_constant<int, 8>{}, bf_tag);
  };
  return xdt == FG_BF16 ? pick(std::true_type{}) : pick(std::false_type{});
}

// One workgroup per [block_m x block_k] tile: amax over the tile, one scale, then the codes.
__global__ void __launch_bounds__(256) quant_fp8_block_kernel(const void* __restrict__ x, int64_t ldx, int xdt,
                                                              uint8_t* __restrict__ q, int64_t ldq,
                                                              float* __restrict__ s, int64_t lds, int64_t ldk, int M,
                                                              int K, int bm, int bk,
                                                              const float* __restrict__ static_scale) {
  __shared__ float red[8];
  __shared__ int nan_flag;
  const int r0 = blockIdx.y * bm, c0 = blockIdx.x * bk;
  const int rows = min(bm, M - r0), cols = min(bk, K - c0);
  const int64_t n = (int64_t)rows * cols;
  if (threadIdx.x == 0) nan_flag = 0;
  __syncthreads();
  float scale;
  if (static_scale) {
    scale = static_scale[0];
  } else {
    float amax = 0.f;
    bool has_nan = false;
    for (int64_t t = threadIdx.x; t < n; t += blockDim.x) {
      const int r = (int)(t / cols), c = (int)(t - (int64_t)r * cols);
      const float v = load_f(x, xdt, (int64_t)(r0 + r) * ldx + c0 + c);
      has_nan |= __builtin_isnan(v);
      amax = fmaxf(amax, fabsf(v));
    }
    if (has_nan) nan_flag = 1;
    amax = block_reduce(amax, true, red);
    scale = (!nan_flag && amax > 0.f) ? __fdiv_rn(amax, 448.f) : 1.f;
    if (threadIdx.x == 0) s[(int64_t)blockIdx.y * lds + blockIdx.x * ldk] = scale;
  }
  for (int64_t t = threadIdx.x; t < n; t += blockDim.x) {
    const int r = (int)(t / cols), c = (int)(t - (int64_t)r * cols);
    const float v = __fdiv_rn(load_f(x, xdt, (int64_t)(r0 + r) * ldx + c0 + c), scale);
    const float cl = __builtin_isnan(v) ? v : fminf(fmaxf(v, -448.f), 448.f);
    q[(int64_t)(r0 + r) * ldq + c0 + c] = f32_to_e4m3(cl);
  }
}

// Few large tiles (a per-tensor scale: one tile of M x K) would leave all but a few CUs idle in the kernel above.  Then
// each tile is cut into `parts` contiguous element ranges, one workgroup each, over up to four launches: zero the
// amax words, fold each part's amax into its tile's word (atomic max on the bit pattern: amax >= 0, and a NaN's
// pattern exceeds every number's, so NaN wins like torch.amax), turn the words into scales, then encode.  The scale
// buffer holds the amax bits in between, so no workspace is needed.
__global__ void __launch_bounds__(256) quant_fp8_tile_zero_kernel(float* __restrict__ s, int64_t lds, int mb, int kb) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < mb * kb) s[(int64_t)(t / kb) * lds + t % kb] = 0.f;
}

__device__ __forceinline__ void tile_part(int M, int K, int bm, int bk, int parts, int64_t* r0, int64_t* c0,
                                          int64_t* cols, int64_t* e0, int64_t* e1) {
  *r0 = (int64_t)blockIdx.y * bm;
  *c0 = (int64_t)blockIdx.x * bk;
  const int64_t rows = min((int64_t)bm, M - *r0);
  *cols = min((int64_t)bk, K - *c0);
  const int64_t n = rows * *cols, chunk = (n + parts - 1) / parts;
  *e0 = min(n, (int64_t)blockIdx.z * chunk);
  *e1 = min(n, *e0 + chunk);
}

__global__ void __launch_bounds__(256) quant_fp8_tile_amax_kernel(const void* __restrict__ x, int64_t ldx, int xdt,
                                                                  float* __restrict__ s, int64_t lds, int M, int K,
                                                                  int bm, int bk, int parts) {
  __shared__ float red[8];
  __shared__ int nan_flag;
  int64_t r0, c0, cols, e0, e1;
  tile_part(M, K, bm, bk, parts, &r0, &c0, &cols, &e0, &e1);
  if (threadIdx.x == 0) nan_flag = 0;
  __syncthreads();
  float amax = 0.f;
  bool has_nan = false;
  for (int64_t t = e0 + threadIdx.x; t < e1; t += blockDim.x) {
    const int64_t r = t / cols, c = t - r * cols;
    const float v = load_f(x, xdt, (r0 + r) * ldx + c0 + c);
    has_nan |= __builtin_isnan(v);
    amax = fmaxf(amax, fabsf(v));
  }
  if (has_nan) nan_flag = 1;
  amax = block_reduce(amax, true, red);  // its barriers also publish nan_flag
  if (threadIdx.x == 0) {
    unsigned* word = reinterpret_cast<unsigned*>(s + (int64_t)blockIdx.y * lds + blockIdx.x);
    atomicMax(word, nan_flag ? 0x7FC00000u : __float_as_uint(amax));
  }
}

__global__ void __launch_bounds__(256) quant_fp8_tile_scale_kernel(float* __restrict__ s, int64_t lds, int mb,
                                                                   int kb) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= mb * kb) return;
  float* p = s + (int64_t)(t / kb) * lds + t % kb;
  const float amax = *p;  // the bit pattern the atomics left is the amax itself (or a NaN)
  *p = (!__builtin_isnan(amax) && amax > 0.f) ? __fdiv_rn(amax, 448.f) : 1.f;
}

__global__ void __launch_bounds__(256) quant_fp8_tile_encode_kernel(const void* __restrict__ x, int64_t ldx, int xdt,
                                                                    uint8_t* __restrict__ q, int64_t ldq,
                                                                    const float* __restrict__ s, int64_t lds,
                                                                    int64_t ldx_s, int M, int K, int bm, int bk,
                                                                    int parts) {
  int64_t r0, c0, cols, e0, e1;
  tile_part(M, K, bm, bk, parts, &r0, &c0, &cols, &e0, &e1);
  const float scale = s[(int64_t)blockIdx.y * lds + blockIdx.x * ldx_s];  // strides 0, 0: one static scale
  for (int64_t t = e0 + threadIdx.x; t < e1; t += blockDim.x) {
    const int64_t r = t / cols, c = t - r * cols;
    const float v = __fdiv_rn(load_f(x, xdt, (r0 + r) * ldx + c0 + c), scale);
    const float cl = __builtin_isnan(v) ? v : fminf(fmaxf(v, -448.f), 448.f);
    q[(r0 + r) * ldq + c0 + c] = f32_to_e4m3(cl);
  }
}

// One row per block, 16-byte accesses, several blocks per wavefront: units a power of two of lanes holds.  A launch has
// fewer than 2^32 threads, one per unit here.
static bool quant_row_blocks_ok(const void* x, int64_t ldx, int xdt, const void* q, int64_t ldq, int64_t M, int64_t K,
                                int64_t bk) {
  return bk >= 8 && bk <= 512 && (bk & (bk - 1)) == 0 && M * ((K + bk - 1) / bk) * (bk / 8) < (1LL << 32) - 256 &&
         quant_vec_ok(x, ldx, xdt, q, ldq, K);
}

// Blocks of 1 x bk, scale of (row, block) at s[row * lds + block * ldk].
hipError_t launch_quant_fp8_row_blocks(const void* x, int64_t ldx, int xdt, uint8_t* q, int64_t ldq, float* s,
                                       int64_t lds, int64_t ldk, int M, int K, int bk, hipStream_t st) {
  const int kb = (K + bk - 1) / bk;
  if (quant_row_blocks_ok(x, ldx, xdt, q, ldq, M, K, bk)) {
    const int log_l = __builtin_ctz((unsigned)bk) - 3;
    const unsigned grid = (unsigned)((((int64_t)M * kb << log_l) + 255) / 256);
    auto k = xdt == FG_BF16 ? quant_row_blocks_kernel<true> : quant_row_blocks_kernel<false>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(256), 0, st, static_cast<const uint16_t*>(x), ldx, q, ldq, s, lds, ldk, M, K,
                       kb, log_l);
  } else {
    hipLaunchKernelGGL(quant_fp8_block_kernel, dim3(kb, M), dim3(256), 0, st, x, ldx, xdt, q, ldq, s, lds, ldk, M, K, 1,
                       bk, nullptr);
  }
  return hipGetLastError();
}

hipError_t launch_quant_fp8_block(const void* x, int64_t ldx, int xdt, uint8_t* q, int64_t ldq, float* s,
                                  int64_t lds, int M, int K, int bm, int bk, const float* static_scale,
                                  hipStream_t st) {
  const int kb = (K + bk - 1) / bk, mb = (M + bm - 1) / bm;
  const int64_t tiles = (int64_t)kb * mb, per_tile = (int64_t)min(bm, M) * min(bk, K);
  const int64_t cus = device_cus();
  if (bm == 1 && !static_scale && quant_row_blocks_ok(x, ldx, xdt, q, ldq, M, K, bk))
    return launch_quant_fp8_row_blocks(x, ldx, xdt, q, ldq, s, lds, 1, M, K, bk, st);
  // one workgroup per tile while the tiles cover the CUs or are small; else parts of 64 Ki elements, up to 4 rounds
  int64_t parts = 1;
  if (tiles < cus && per_tile > 65536) parts = min((per_tile + 65535) / 65536, (4 * cus + tiles - 1) / tiles);
  if (parts == 1) {
    hipLaunchKernelGGL(quant_fp8_block_kernel, dim3(kb, mb), dim3(256), 0, st, x, ldx, xdt, q, ldq, s, lds,
                       (int64_t)1, M, K, bm, bk, static_scale);
    return hipGetLastError();
  }
  const dim3 grid(kb, mb, (unsigned)parts);
  const float* scale = static_scale;
  int64_t slds = 0, sldx = 0;
  if (!static_scale) {
    const unsigned small = (unsigned)((tiles + 255) / 256);
    hipLaunchKernelGGL(quant_fp8_tile_zero_kernel, dim3(small), dim3(256), 0, st, s, lds, mb, kb);
    hipLaunchKernelGGL(quant_fp8_tile_amax_kernel, grid, dim3(256), 0, st, x, ldx, xdt, s, lds, M, K, bm, bk,
                       (int)parts);
    hipLaunchKernelGGL(quant_fp8_tile_scale_kernel, dim3(small), dim3(256), 0, st, s, lds, mb, kb);
    scale = s;
    slds = lds;
    sldx = 1;
  }
  hipLaunchKernelGGL(quant_fp8_tile_encode_kernel, grid, dim3(256), 0, st, x, ldx, xdt, q, ldq, scale, slds, sldx, M,
                     K, bm, bk, (int)parts);
  return hipGetLastError();
}

hipError_t launch_quant_int8(const void* x, int64_t ldx, int xdt, int8_t* q, int64_t ldq, float* s, int M, int K,
                             hipStream_t st) {
  int C = 0;
  const int T = quant_vec_ok(x, ldx, xdt, q, ldq, K) ? quant_rows_plan(M, K, &C) : 0;
  if (T)
    return launch_quant_rows<false, false>(x, ldx, xdt, reinterpret_cast<uint8_t*>(q), ldq, s, M, K, T, C, nullptr, 0,
                                           0.f, st);
  hipLaunchKernelGGL(quant_int8_rowwise_kernel, dim3(M), dim3(256), 0, st, x, ldx, xdt, q, ldq, s, K);
  return hipGetLastError();
}

hipError_t launch_quant_fp8(const void* x, int64_t ldx, int xdt, uint8_t* q, int64_t ldq, float* s, int M, int K,
                            const float* static_scale, const void* rms_w, int wdt, float eps, int fuse,
                            hipStream_t st) {
  int C = 0;
  // with the norm a row lies in LDS beside the reductions' words: at most 32000 columns
  const int T = !static_scale && quant_vec_ok(x, ldx, xdt, q, ldq, K) && !(fuse && K > kQuantNormMaxK) &&
                        reinterpret_cast<uintptr_t>(rms_w) % 16 == 0
                    ? quant_rows_plan(M, K, &C)
                    : 0;
  if (T && fuse) return launch_quant_rows<true, true>(x, ldx, xdt, q, ldq, s, M, K, T, C, rms_w, wdt, eps, st);
  if (T) return launch_quant_rows<true, false>(x, ldx, xdt, q, ldq, s, M, K, T, C, nullptr, 0, 0.f, st);
  hipLaunchKernelGGL(quant_fp8_rowwise_kernel, dim3(M), dim3(256), 0, st, x, ldx, xdt, q, ldq, s, K, static_scale,
                     rms_w, wdt, eps, fuse);
  return hipGetLastError();
}

}  // namespace fg
