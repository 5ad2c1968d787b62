// Column gather of the activations for act-order W4 weights: out[m, c] = x[m, perm[c]] (16-bit elements), so that every
// kernel of the policy reads a sorted weight with contiguous x.  The kernels that take the permutation themselves gather
// 2-byte elements one by one inside their K loop and rule out direct-to-LDS loads.  Whole calls, us, permutation in the
// kernel / gather in front (the same weight without act order): K = 14336, N = 4096 at 1 / 16 / 64 / 512 rows 25.8 / 105 /
// 235 / 1779 against 11.1 / 17.1 / 27.1 / 81 (8.6 / 13.4 / 23.4 / 76); K = 4096, N = 28672 at 1 / 16 / 1024 rows 20.8 /
// 140 / 4016 against 15.1 / 20.7 / 213 (12.7 / 18.6 / 214).
//
// Two forms.  Few rows (kGatherDirectM): one output unit of 8 columns per thread and row, picked straight from x in L2;
// the launch is the latency of a permutation load and an x load, and a row spreads over many workgroups.  More rows: a
// workgroup keeps the permutation of its columns in registers (C units per thread) and walks rows m, m + grid, ..: a row
// is staged into LDS with 16-byte loads, each output unit picks its 8 elements there and is stored whole; bound by one
// read and one write of x and 8 two-byte LDS reads per unit.
#include <algorithm>

#include "fg_device.h"

namespace fg {

constexpr int kGatherThreads = 512;
constexpr int kGatherMaxK = 32768;   // columns of a row in LDS (64 KiB)
constexpr int kGatherDirectM = 64;

// The 8 permutation entries of output unit u; entries past K read as 0.
template <bool VEC>
__device__ __forceinline__ void load_perm8(const int32_t* perm, int u, int K, int (&idx)[8]) {
  if (VEC) {
    const int4 a = reinterpret_cast<const int4*>(perm)[2 * u], b = reinterpret_cast<const int4*>(perm)[2 * u + 1];
    idx[0] = a.x; idx[1] = a.y; idx[2] = a.z; idx[3] = a.w;
    idx[4] = b.x; idx[5] = b.y; idx[6] = b.z; idx[7] = b.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) idx[e] = 8 * u + e < K ? perm[8 * u + e] : 0;
  }
}

template <int C, bool VEC>
__global__ void __launch_bounds__(kGatherThreads) gather_lds_kernel(const uint16_t* __restrict__ x, int64_t ldx,
                                                                    const int32_t* __restrict__ perm,
                                                                    uint16_t* __restrict__ out, int64_t ldo, int M,
                                                                    int K) {
  extern __shared__ __align__(16) uint16_t row[];
  const int units = (K + 7) / 8;
  int idx[C][8];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int u = threadIdx.x + c * kGatherThreads;
    if (u < units) load_perm8<VEC>(perm, u, K, idx[c]);
  }
  for (int m = blockIdx.x; m < M; m += gridDim.x) {
    const uint16_t* xr = x + (int64_t)m * ldx;
    if (VEC) {
      for (int u = threadIdx.x; u < units; u += kGatherThreads)
        reinterpret_cast<uint4*>(row)[u] = reinterpret_cast<const uint4*>(xr)[u];
    } else {
      for (int k = threadIdx.x; k < K; k += kGatherThreads) row[k] = xr[k];
    }
    __syncthreads();
    uint4* orow = reinterpret_cast<uint4*>(out + (int64_t)m * ldo);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int u = threadIdx.x + c * kGatherThreads;
      if (u < units) {
        uint32_t w[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) w[p] = (uint32_t)row[idx[c][2 * p]] | (uint32_t)row[idx[c][2 * p + 1]] << 16;
        orow[u] = make_uint4(w[0], w[1], w[2], w[3]);
      }
    }
    __syncthreads();  // the row is read before the next one overwrites it
  }
}

template <bool VEC>
__global__ void __launch_bounds__(64) gather_direct_kernel(const uint16_t* __restrict__ x, int64_t ldx,
                                                           const int32_t* __restrict__ perm,
                                                           uint16_t* __restrict__ out, int64_t ldo, int M, int K) {
  const int u = blockIdx.x * 64 + threadIdx.x;
  if (u >= (K + 7) / 8) return;
  int idx[8];
  load_perm8<VEC>(perm, u, K, idx);
  for (int m = blockIdx.y; m < M; m += gridDim.y) {
    const uint16_t* xr = x + (int64_t)m * ldx;
    uint32_t h[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) h[e] = xr[idx[e]];
    reinterpret_cast<uint4*>(out + (int64_t)m * ldo)[u] =
        make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
  }
}

// `out` rows are 16-byte aligned and hold K rounded up to 8 elements (checked by the caller); the columns past K repeat
// element 0.
hipError_t launch_gather(const void* x, int64_t ldx, const int32_t* perm, void* out, int64_t ldo, int M, int K,
                         hipStream_t s) {
  const uint16_t* xi = static_cast<const uint16_t*>(x);
  uint16_t* o = static_cast<uint16_t*>(out);
  const int units = (K + 7) / 8, c = (units + kGatherThreads - 1) / kGatherThreads;
  note_kernel("gather_columns");
  const bool vec = K % 8 == 0 && reinterpret_cast<uintptr_t>(perm) % 16 == 0;  // whole units of perm ...
  if (M <= kGatherDirectM || K > kGatherMaxK) {
    auto k = vec ? gather_direct_kernel<true> : gather_direct_kernel<false>;
    hipLaunchKernelGGL(k, dim3((units + 63) / 64, std::min(M, 4096)), dim3(64), 0, s, xi, ldx, perm, o, ldo, M, K);
    return hipGetLastError();
  }
  const bool xvec = vec && ldx % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0;  // ... and of x
  // four workgroups of 512 threads per CU (two past 16384 columns, by their LDS rows)
  const dim3 grid(std::min(M, 4 * device_cus()));
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, grid, dim3(kGatherThreads), (size_t)units * 16, s, xi, ldx, perm, o, ldo, M, K);
    return hipGetLastError();
  };
  if (c <= 1) return go(xvec ? gather_lds_kernel<1, true> : gather_lds_kernel<1, false>);
  if (c <= 2) return go(xvec ? gather_lds_kernel<2, true> : gather_lds_kernel<2, false>);
  if (c <= 4) return go(xvec ? gather_lds_kernel<4, true> : gather_lds_kernel<4, false>);
  return go(xvec ? gather_lds_kernel<8, true> : gather_lds_kernel<8, false>);
}

}  // namespace fg
