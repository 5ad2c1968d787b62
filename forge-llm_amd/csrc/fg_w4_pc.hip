// W4A16 prefill with producer and consumer wavefronts: y[M,N] = x[M,K] @ dequant(W)[N,K]^T (+bias).  W8A16 (int8
// weights) takes the same kernel with tiles of 64 and 128 rows: twice the staging bytes, no zero words.  Its instances for a
// K that ends inside a slice (pc_exact) keep the weights exact: the integers are the MFMA operands and each 32-column
// product takes its fp32 scale as it joins the sum, since the kernel that reads such a K otherwise multiplies in fp32 (error
// against 64 bits, bf16 x, K=4128: 1.66e-3 in both, 2.32e-3 with the scaled weight rounded to bf16, which took 39 us at 512
// rows of N=4096, groups of 32, against 48).
//
// A workgroup owns a BM x 128 output tile (BM = 256, 128 or 64; below 256 rows) and walks K in 64-column slices through
// a three-stage LDS ring.  Its eight wavefronts split the work by role, one of each role per SIMD (wavefronts 0-3 on SIMDs 0-3, 4-7 likewise):
//   * consumers (wavefronts 0-3, a 2 x 2 grid of BM/2 x 64 tiles): read A and B fragments from LDS and run
//     v_mfma_f32_16x16x32_{bf16,f16}; they issue no global memory instruction;
//   * producers (wavefronts 4-7): every global access of the slice is a direct-to-LDS load (global_load_lds, no
//     registers): the BM x 64 tile of x (BM / 32 1 KiB loads per producer), the 128 x 64 tile of packed int4 weights
//     (one 1 KiB load per producer: its own 32 rows), and the scales and zero-point words of those 32 rows (one 4-byte
//     per lane load); then each producer lane reads back its 16 bytes of packed weights (32 columns of one row),
//     dequantises them -- (q - z) * s in fp32, exactly the oracle's value (q * s + (-z * s) is exact and the fma
//     rounds nothing), rounded once to bf16 / fp16 -- and stores them into the stage's weight rows.
// So the dequantisation VALU of one wavefront runs while the other wavefront of its SIMD keeps the matrix core busy,
// instead of both wavefronts alternating the two under one barrier (the all-rounder w4_big_kernel, fg_w4_big.hip).
//
// Ring schedule, slice t in stage t % 3 (iteration t ends with the workgroup barrier that publishes stage t + 1):
//   producers, iteration t: x of slice t + 2 -> stage (t + 2) % 3 (consumed in t - 1); packed weights, scales and
//     zero words of slice t + 3 -> the staging areas of stage t % 3 (read by the producers in t - 1); wait until
//     slice t + 1's staging loads have landed, dequantise slice t + 1 into stage (t + 1) % 3's weight rows (consumed
//     in t - 2); wait until slice t + 1's x rows have landed; barrier.
//   consumers, iteration t: BM / 4 MFMAs (64 at 256 rows) over the two k-steps of stage t % 3; barrier.
// Every producer issues the same loads in the same order each iteration (slices past the end re-read the last one,
// into areas no one reads again), so `s_waitcnt vmcnt(N)` with a constant N is exactly "these loads have landed"
// (loads complete in issue order); the direct-to-LDS loads are invisible to the compiler's wait analysis, so those
// waits are explicit.  Packed weights and scales get two slices (~2 us at full rate) to arrive, x two as well.
//
// LDS per stage: x BM rows x 128 B (16-byte unit c of row r at c ^ (r & 7): conflict-free fragment reads), weight
// rows 128 x 128 B (same swizzle), packed-weight staging 4 KiB (producer p's lane l at p * 1024 + 16 l), scale and
// zero staging 1 KiB (producer p: 32 fp16 scales at p * 256, its 4 zero words at p * 256 + 64, and 128 bytes further the
// same of the group of the slice's second 32 columns); with pc_exact the fp32 scales of the two halves, 1 KiB, which the
// consumers read beside the weight rows.  Three stages: 162816 bytes at BM = 256, 113664 and 89088 below.
//
// Split-K (gridDim.y > 1): each split covers `kchunk` columns and writes fp32 partials [S, M, N] to the caller's
// workspace; w4_splitk_reduce_kernel (fg_w4_mfma.hip) sums them in a fixed order and adds the bias.
//
// A K that ends inside a slice (K % 64 == 32; TAIL) reads zeros in place of x past K and scales the weights there by zero.
//
// Requirements (w4_pc_ok): K % 32 == 0, group a multiple of 32 (or one group), N % 8 == 0, 16-bit scales with an even
// row stride, 16-byte aligned x (ldx % 8 == 0) and qweight (ldq % 4 == 0), 4-byte aligned scales, no act-order perm.
// Rows past M and channels past N read row M - 1 / channel N - 1 and are not stored.
#include <algorithm>

#include "fg_device.h"

namespace fg {

typedef __bf16 bf16x8_pc_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_pc_t __attribute__((ext_vector_type(8)));
typedef float f32x4_pc_t __attribute__((ext_vector_type(4)));
typedef float f32x2_pc_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_pc_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_pc_t __attribute__((ext_vector_type(2)));

constexpr int kPcBN = 128, kPcBK = 64, kPcRow = 128, kPcThreads = 512;
constexpr int kPcWBytes = kPcBN * kPcRow;                      // dequantised weight rows
constexpr int pc_q_bytes(int wb) { return kPcBN * kPcBK * wb / 8; }  // packed weights of the slice (WB bits each)
constexpr int kPcSBytes = 4 * 256;                             // scales and zero words
constexpr int pc_x_bytes(int bm) { return bm * kPcRow; }       // x rows
constexpr bool pc_exact(int wb, bool tail) { return wb == 8 && tail; }
constexpr int kPcFBytes = 2 * kPcBN * 4;                       // fp32 scales of the slice's two 32-column halves (pc_exact)
constexpr int pc_stage(int bm, int wb, bool exact) {
  return pc_x_bytes(bm) + kPcWBytes + pc_q_bytes(wb) + kPcSBytes + (exact ? kPcFBytes : 0);
}
constexpr int pc_lds(int bm, int wb, bool exact) { return 3 * pc_stage(bm, wb, exact); }
static_assert(pc_lds(256, 4, false) <= 160 * 1024 && pc_lds(128, 8, true) <= 160 * 1024, "the ring exceeds the LDS");
// direct-to-LDS loads one producer issues per slice: x rows, packed weights, scales + zero words
constexpr int pc_xi(int bm) { return pc_x_bytes(bm) / 1024 / 4; }
constexpr int pc_qi(int wb) { return pc_q_bytes(wb) / 1024 / 4; }
constexpr int kPcSI = 1;
static_assert(pc_xi(256) == 8, "eight x loads per producer and slice");

// What a TAIL launch reads in place of the 16-byte x units past K: zeros, which meet weights scaled to zero.
static __device__ __align__(16) const uint16_t g_pc_zero[8] = {};

struct PcArgs {
  const uint16_t* x;
  int64_t ldx;
  const void* qw;
  int64_t ldq;  // 4-bit weights: int32 words per row; 8-bit: bytes
  const uint16_t* scales;
  int64_t lds;
  const int32_t* zeros;  // qweight when symmetric (a valid address, never used)
  int64_t ldz;
  const void* bias;
  float* ws;
  uint16_t* y;
  int64_t ldy;
  int M, N, K;
  int kchunk;        // columns per K split (a multiple of 64)
  uint32_t gdiv;     // 32-column chunks per group (0: one group)
  uint32_t gmul;     // chunk / gdiv = umulhi(chunk, gmul) (gdiv > 1)
  int hasz, sbf16, bdt;
};

template <bool XBF16>
__device__ __forceinline__ f32x4_pc_t pc_mfma(uint4 a, uint4 b, f32x4_pc_t c) {
  if constexpr (XBF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_pc_t, a),
                                                   __builtin_bit_cast(bf16x8_pc_t, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_pc_t, a),
                                                  __builtin_bit_cast(f16x8_pc_t, b), c, 0, 0, 0);
  }
}

// two fp32 values as one packed 16-bit pair, each rounded to nearest even
template <bool XBF16>
__device__ __forceinline__ uint32_t pc_pack(float lo, float hi) {
  if constexpr (XBF16) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_pc_t{lo, hi}, bf16x2_pc_t));
  } else {
    return (uint32_t)f32_to_f16_bits(lo) | ((uint32_t)f32_to_f16_bits(hi) << 16);
  }
}

// 16-byte fragment of one swizzled 128-byte LDS row for k-step s: unit 4 s + lane / 16
__device__ __forceinline__ uint4 pc_frag(const uint8_t* rp, int r16, int lane, int s) {
  const int c = (4 * s + (lane >> 4)) ^ (r16 & 7);
  return *reinterpret_cast<const uint4*>(rp + c * 16);
}

template <int BM, bool XBF16, int WB, bool TAIL>
__device__ __forceinline__ void w4_pc_body(const PcArgs& a) {
  constexpr bool kExact = pc_exact(WB, TAIL);
  constexpr int kPcBM = BM, kPcXBytes = pc_x_bytes(BM), kPcStage = pc_stage(BM, WB, kExact), kPcXI = pc_xi(BM);
  constexpr int kPcQI = pc_qi(WB), kPcQBytes = pc_q_bytes(WB);
  constexpr int kF = kPcWBytes + kPcQBytes + kPcSBytes;  // offset of a stage's fp32 scales from its weight rows
  constexpr int TM = BM / 32;  // 16-row blocks of a consumer
  extern __shared__ __align__(16) uint8_t smem[];
  const int ntm = (a.M + kPcBM - 1) / kPcBM, ntn = (a.N + kPcBN - 1) / kPcBN;
  int tm, tn;
  tile_of(blockIdx.x, ntm, ntn, tm, tn);
  const int m0 = tm * kPcBM, n0 = tn * kPcBN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kbeg = blockIdx.y * a.kchunk;
  const int nk = (min(a.K, kbeg + a.kchunk) - kbeg + (TAIL ? kPcBK - 1 : 0)) / kPcBK;

  if (wave < 4) {
    // ------------------------------------------------------------------------------------------- consumers
    // Below 256 rows the weights are the MFMA's first operand: a lane's four results are four consecutive channels of one
    // row of x (row lane % 16 of the block, channels 4 (lane / 16) .. + 3), stored as one unit, which shortens a split
    // launch's partial stores (K=N=2048, M=384 with four splits 24.0 -> 22.0 us).  With 256 rows x comes first (rows 4
    // (lane / 16) .. + 3 of channel lane % 16): the other order measured 3-5% slower at row counts that leave most of the
    // last tile empty (K=14336, N=4096, M=300 62.1 -> 64.4).
    constexpr bool kWFirst = BM < 256;
    static_assert(kWFirst || !kExact, "the scales of a lane's results are those of four channels in a row");
    const int wm = wave >> 1, wn = wave & 1, r16 = lane & 15;
    f32x4_pc_t acc[TM][4];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_pc_t{0.f, 0.f, 0.f, 0.f};
    asm volatile("s_barrier" ::: "memory");  // slice 0 is in stage 0
    // Fragments of k-step 0 of a slice (f0) and of k-step 1 (f1), in registers.  The loop is software-pipelined
    // around the barrier: k-step 0 of slice t + 1 is read right after the barrier that ends slice t, while the last
    // eight MFMAs of slice t (whose fragments are already in registers) run, so a consumer -- the only MFMA issuer of
    // its SIMD -- does not sit out the LDS latency at the top of every slice.
    uint4 fa0[TM], fb0[4], fa1[TM], fb1[4];
    f32x4_pc_t sc0[4], sc1[4];  // pc_exact: scales of the lane's four channels of each column block
    auto read_ks = [&](const uint8_t* st, int s, uint4 (&fa)[TM], uint4 (&fb)[4], f32x4_pc_t (&sc)[4])
                       __attribute__((always_inline)) {
      const uint8_t* sA = st + (wm * (BM / 2) + r16) * kPcRow;
      const uint8_t* sB = st + kPcXBytes + (wn * 64 + r16) * kPcRow;
#pragma unroll
      for (int j = 0; j < 4; ++j) fb[j] = pc_frag(sB + j * 16 * kPcRow, r16, lane, s);
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i] = pc_frag(sA + i * 16 * kPcRow, r16, lane, s);
      if constexpr (kExact) {
        const float* f = reinterpret_cast<const float*>(st + kPcXBytes + kF) + s * kPcBN + wn * 64 + 4 * (lane >> 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) sc[j] = *reinterpret_cast<const f32x4_pc_t*>(f + j * 16);
      }
    };
    auto mfma_rows = [&](int i0, int i1, const uint4 (&fa)[TM], const uint4 (&fb)[4], const f32x4_pc_t (&sc)[4])
                         __attribute__((always_inline)) {
#pragma unroll
      for (int i = i0; i < i1; ++i) {
        if constexpr (kExact) {
          f32x4_pc_t part[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) part[j] = pc_mfma<XBF16>(fb[j], fa[i], f32x4_pc_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fmaf(part[j][e], sc[j][e], acc[i][j][e]);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[i][j] = kWFirst ? pc_mfma<XBF16>(fb[j], fa[i], acc[i][j]) : pc_mfma<XBF16>(fa[i], fb[j], acc[i][j]);
        }
      }
    };
    const uint8_t* st = smem;
    read_ks(st, 0, fa0, fb0, sc0);
    for (int t = 0; t < nk; ++t) {
      read_ks(st, 1, fa1, fb1, sc1);
      mfma_rows(0, TM, fa0, fb0, sc0);
      mfma_rows(0, TM - 2, fa1, fb1, sc1);
      // this stage's fragments are in registers before the barrier lets the producers refill it
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      st = st == smem + 2 * kPcStage ? smem : st + kPcStage;
      read_ks(st, 0, fa0, fb0, sc0);  // slice t + 1 (past the last slice: a stage no one writes any more, unused)
      __builtin_amdgcn_sched_barrier(0);
      mfma_rows(TM - 2, TM, fa1, fb1, sc1);
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_barrier" ::: "memory");  // the producers' last loads have drained: the ring is free

    const int mw = m0 + wm * (BM / 2), nw = n0 + wn * 64, n4 = 4 * (lane >> 4);
    if (gridDim.y > 1) {  // fp32 partials of this split
      // a unit of four lies in one row, 16-byte aligned
      const bool v4 = kWFirst && a.N % 4 == 0 && reinterpret_cast<uintptr_t>(a.ws) % 16 == 0;
      float* const part = a.ws + (int64_t)blockIdx.y * a.M * a.N;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int m = mw + i * 16 + (kWFirst ? r16 : n4), n = nw + j * 16 + (kWFirst ? n4 : r16);
          if (v4) {
            if (m < a.M && n < a.N) *reinterpret_cast<f32x4_pc_t*>(part + (int64_t)m * a.N + n) = acc[i][j];
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int me = m + (kWFirst ? 0 : e), ne = n + (kWFirst ? e : 0);
              if (me < a.M && ne < a.N) part[(int64_t)me * a.N + ne] = acc[i][j][e];
            }
          }
        }
      return;
    }
    // 16-bit output through a per-wavefront LDS slab of 16 rows x 64 columns, stored as 16-byte row segments
    constexpr int SP = 64 + 8;
    uint16_t* slab = reinterpret_cast<uint16_t*>(smem) + wave * 16 * SP;
    float cb[4][kWFirst ? 4 : 1];  // bias of the lane's channels
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < (kWFirst ? 4 : 1); ++e)
        cb[j][e] = a.bias ? load_f(a.bias, a.bdt, min(nw + j * 16 + (kWFirst ? n4 + e : r16), a.N - 1)) : 0.f;
    const bool vec_ok = (a.ldy % 8) == 0 && (reinterpret_cast<uintptr_t>(a.y) % 16) == 0;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = a.bias ? acc[i][j][e] + cb[j][kWFirst ? e : 0] : acc[i][j][e];
          h[e] = XBF16 ? f32_to_bf16_bits(v) : f32_to_f16_bits(v);
        }
        if constexpr (kWFirst) {
          *reinterpret_cast<uint2*>(slab + r16 * SP + j * 16 + n4) = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) slab[(n4 + e) * SP + j * 16 + r16] = (uint16_t)h[e];
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's slab writes are done before it reads them
#pragma unroll
      for (int u0 = 0; u0 < 16 * 64 / 8; u0 += 64) {
        const int u = u0 + lane, r = u / 8, c8 = u % 8;
        const int m = mw + i * 16 + r, n = nw + c8 * 8;
        const uint4 v = *reinterpret_cast<const uint4*>(slab + r * SP + c8 * 8);
        if (m < a.M) {
          uint16_t* yr = a.y + (int64_t)m * a.ldy;
          if (n + 8 <= a.N && vec_ok) {
            *reinterpret_cast<uint4*>(yr + n) = v;
          } else {
            const uint16_t h[8] = {(uint16_t)v.x, (uint16_t)(v.x >> 16), (uint16_t)v.y, (uint16_t)(v.y >> 16),
                                   (uint16_t)v.z, (uint16_t)(v.z >> 16), (uint16_t)v.w, (uint16_t)(v.w >> 16)};
            for (int q = 0; q < 8 && n + q < a.N; ++q) yr[n + q] = h[q];
          }
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // reads done before the next slab overwrites the buffer
    }
    return;
  }

  // --------------------------------------------------------------------------------------------- producers
  const int p = wave - 4;
  // x: load i of producer p fills tile rows (XI p + i) * 8 .. + 8; lane l writes position l % 8 of row
  // (XI p + i) * 8 + l / 8, i.e. global unit (l % 8) ^ (l / 8) (the row's swizzle key is l / 8)
  const int lrow = lane >> 3, lcol = ((lane & 7) ^ (lane >> 3)) * 8;
  const uint16_t* xr[kPcXI];
#pragma unroll
  for (int i = 0; i < kPcXI; ++i) xr[i] = a.x + (int64_t)min(m0 + (kPcXI * p + i) * 8 + lrow, a.M - 1) * a.ldx + lcol;
  // packed weights: lane l owns tile row 32 p + l / 2, columns 32 (l % 2) .. + 32 of each slice (16 or 32 bytes)
  const int wr = 32 * p + (lane >> 1), wh = lane & 1;
  const uint8_t* wq = static_cast<const uint8_t*>(a.qw) + (int64_t)min(n0 + wr, a.N - 1) * a.ldq * (WB == 4 ? 4 : 1);
  // scales and zero words of the producer's 32 channels, of the group of the slice's first 32 columns in lanes 0-31 and
  // of its second 32 in lanes 32-63 (the same group when the group size is a multiple of 64): lanes 0-15 of each half
  // read scale pairs, lanes 16-19 zero words, the rest repeat lane 0's pair (every lane of a direct-to-LDS load writes
  // its 4 bytes)
  const uint8_t* szb;
  int64_t szstride;  // bytes per group
  {
    const int c0 = n0 + 32 * p, l32 = lane & 31;
    if (l32 >= 16 && l32 < 20 && a.hasz) {
      const int w = min(c0 / 8 + (l32 - 16), (a.N - 1) / 8);
      szb = reinterpret_cast<const uint8_t*>(a.zeros + w);
      szstride = a.ldz * 4;
    } else {
      const int c = min(c0 + 2 * (l32 < 16 ? l32 : 0), a.N - 2);
      szb = reinterpret_cast<const uint8_t*>(a.scales + c);
      szstride = a.lds * 2;
    }
  }
  // chunks (32 columns) of a local slice's two halves (slices past the last read it again; past K, the last chunk), the
  // same for the whole wavefront, and the lane's own
  auto chunk0 = [&](int t) { return (kbeg + min(t, nk - 1) * kPcBK) / 32; };
  auto chunk1 = [&](int t) { return TAIL ? min(chunk0(t) + 1, a.K / 32 - 1) : chunk0(t) + 1; };
  auto group_of = [&](int c) -> uint32_t {
    return a.gdiv == 0 ? 0u : (a.gdiv == 1 ? (uint32_t)c : __umulhi((uint32_t)c, a.gmul));
  };
  // x rows of slice t into a stage's x area
  auto issue_x = [&](int t, uint8_t* dst) __attribute__((always_inline)) {
    const int k0 = kbeg + min(t, nk - 1) * kPcBK;
    dst += p * kPcXI * 1024;
#pragma unroll
    for (int i = 0; i < kPcXI; ++i) {
      const uint16_t* src = xr[i] + k0;
      if (TAIL) src = k0 + lcol < a.K ? src : g_pc_zero;
      __builtin_amdgcn_global_load_lds(src, dst + i * 1024, 16, 0, 0);
    }
  };
  // packed weights, scales and zero words of slice t into a stage's staging areas (base: the stage's packed-weight
  // area, the scale area follows it)
  auto issue_q = [&](int t, uint8_t* dst) __attribute__((always_inline)) {
    const int c0 = chunk0(t), c1 = chunk1(t);
    const uint32_t g0 = group_of(c0), g1 = group_of(c1);
#pragma unroll
    for (int h = 0; h < kPcQI; ++h)
      __builtin_amdgcn_global_load_lds(wq + (wh ? c1 : c0) * (4 * WB) + 16 * h, dst + (p * kPcQI + h) * 1024, 16, 0, 0);
    __builtin_amdgcn_global_load_lds(szb + (int64_t)(lane < 32 ? g0 : g1) * szstride, dst + kPcQBytes + p * 256, 4, 0, 0);
  };
  uint32_t nmask = 0x0F0F0F0Fu;
  asm("" : "+v"(nmask));  // hidden from known-bits analysis: bytes of masked words convert with v_cvt_f32_ubyte{k}
  const uint32_t zsel = a.hasz ? 0xffffffffu : 0u;
  // one slice's weights from a stage's staging areas (q) into its weight rows (w).  Past K (TAIL) they take a scale of
  // zero: a weight that overflows 16 bits, times the zeros read for x there, would be a NaN
  auto dequant = [&](int t, const uint8_t* __restrict__ q, uint8_t* __restrict__ w) __attribute__((always_inline)) {
    const bool past = TAIL && wh && chunk0(t) + 1 >= a.K / 32;
    const uint4 qv = *reinterpret_cast<const uint4*>(q + p * kPcQI * 1024 + lane * 16);
    const uint8_t* sz = q + kPcQBytes + p * 256 + wh * 128;
    const uint32_t sraw = past ? 0u : *reinterpret_cast<const uint16_t*>(sz + (lane >> 1) * 2);
    const uint32_t zw = (*reinterpret_cast<const uint32_t*>(sz + 64 + ((lane >> 1) >> 3) * 4) & zsel) |
                        (0x88888888u & ~zsel);  // symmetric: zero-point 8
    const float sc = a.sbf16 ? bf16_bits_to_f32(sraw) : f16_bits_to_f32((uint16_t)sraw);
    if constexpr (WB == 8) {  // u = q ^ 0x80 = q + 128: q * s = u * s - 128 s, exact in fp32, rounded once (pc_exact: s = 1)
      const uint4 qv2 = *reinterpret_cast<const uint4*>(q + (p * kPcQI + 1) * 1024 + lane * 16);
      const uint32_t wd[8] = {qv.x, qv.y, qv.z, qv.w, qv2.x, qv2.y, qv2.z, qv2.w};
      if constexpr (kExact) *reinterpret_cast<float*>(w + kF + (wh * kPcBN + wr) * 4) = sc;
      const float ws = kExact ? 1.f : sc, c128 = -128.f * ws;
      uint8_t* row = w + wr * kPcRow;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float d[8];
#pragma unroll
        for (int b = 0; b < 8; ++b)
          d[b] = __builtin_fmaf((float)(((wd[2 * i + b / 4] ^ 0x80808080u) >> (8 * (b % 4))) & 0xFFu), ws, c128);
        *reinterpret_cast<uint4*>(row + (((4 * wh + i) ^ (wr & 7)) * 16)) =
            make_uint4(pc_pack<XBF16>(d[0], d[1]), pc_pack<XBF16>(d[2], d[3]), pc_pack<XBF16>(d[4], d[5]),
                       pc_pack<XBF16>(d[6], d[7]));
      }
      return;
    }
    const float c = -(float)nibble(zw, (lane >> 1) & 7) * sc;
    const uint32_t wd[4] = {qv.x, qv.y, qv.z, qv.w};
    uint8_t* rp = w + wr * kPcRow;
    if (!XBF16 && !a.sbf16) {
      // fp16 x and scales: 1024 + q by bits, minus 1024 + z (exact), times s in packed fp16 -- the exact product rounded
      // once, as the fp32 form rounds it -- in 17 instructions per 8 values instead of 23
      const uint32_t zb = 0x6400u + nibble(zw, (lane >> 1) & 7);
      const f16x2_pc_t z2 = __builtin_bit_cast(f16x2_pc_t, zb | zb << 16);
      const f16x2_pc_t s2 = __builtin_bit_cast(f16x2_pc_t, sraw | sraw << 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t h = wd[i] >> 4;
        uint32_t o[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {  // byte b: nibbles 2 b and 2 b + 1 into the two halves
          const uint32_t t = __builtin_amdgcn_perm(h, wd[i], 0x0c040c00u + 0x00010001u * b);
          const f16x2_pc_t m = __builtin_bit_cast(f16x2_pc_t, (t & 0x000F000Fu) | 0x64006400u);
          o[b] = __builtin_bit_cast(uint32_t, (m - z2) * s2);
        }
        *reinterpret_cast<uint4*>(rp + (((4 * wh + i) ^ (wr & 7)) * 16)) = make_uint4(o[0], o[1], o[2], o[3]);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // word i = columns 8 i .. 8 i + 7 of the lane's 32 = unit 4 wh + i of the row
      const uint32_t lo = wd[i] & nmask, hi = (wd[i] >> 4) & nmask;  // nibbles 0,2,4,6 / 1,3,5,7
      float d[8];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        d[2 * b] = __builtin_fmaf((float)((lo >> (8 * b)) & 0xFFu), sc, c);
        d[2 * b + 1] = __builtin_fmaf((float)((hi >> (8 * b)) & 0xFFu), sc, c);
      }
      const uint4 v = make_uint4(pc_pack<XBF16>(d[0], d[1]), pc_pack<XBF16>(d[2], d[3]), pc_pack<XBF16>(d[4], d[5]),
                                 pc_pack<XBF16>(d[6], d[7]));
      *reinterpret_cast<uint4*>(rp + (((4 * wh + i) ^ (wr & 7)) * 16)) = v;
    }
  };
  constexpr int kQ = kPcXBytes + kPcWBytes;  // offset of a stage's staging areas
  // Iteration t.  The four regions reach the body as __restrict__ pointers: without them the compiler cannot tell
  // the direct-to-LDS loads from the staging reads and weight-row stores, and waits for every outstanding load.
  auto body = [&](int t, const uint8_t* __restrict__ q_rd, uint8_t* __restrict__ w_wr, uint8_t* __restrict__ x_dst,
                  uint8_t* __restrict__ q_dst) __attribute__((always_inline)) {
    issue_x(t + 2, x_dst);
    issue_q(t + 3, q_dst);
    // slice t + 1's staging landed (issued two iterations ago; everything after it may still be in flight)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kPcXI + 2 * (kPcQI + kPcSI)) : "memory");
    dequant(t + 1, q_rd, w_wr);
    // slice t + 1's x rows landed and this wave's weight stores are done; then the barrier publishes stage t + 1
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kPcXI + 2 * (kPcQI + kPcSI)) : "memory");
  };

  uint8_t* const s0 = smem;
  uint8_t* const s1 = smem + kPcStage;
  uint8_t* const s2 = smem + 2 * kPcStage;
  // prologue, in the steady state's issue order: [q0] [x0 q1] [x1 q2]
  issue_q(0, s0 + kQ);
  issue_x(0, s0);
  issue_q(1, s1 + kQ);
  issue_x(1, s1);
  issue_q(2, s2 + kQ);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kPcXI + 2 * (kPcQI + kPcSI)) : "memory");  // slice 0's staging
  dequant(0, s0 + kQ, s0 + kPcXBytes);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kPcXI + 2 * (kPcQI + kPcSI)) : "memory");
  // stage of slice t: t % 3; rotate (a, b, c) = stages of (t, t + 1, t + 2)
  uint8_t *sa = s0, *sb = s1, *sc = s2;
  for (int t = 0; t < nk; ++t) {
    body(t, sb + kQ, sb + kPcXBytes, sc, sa + kQ);
    uint8_t* tmp = sa;
    sa = sb;
    sb = sc;
    sc = tmp;
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");  // drain before the consumers reuse the ring
}

template <int BM, bool XBF16, int WB, bool TAIL>
__global__ void __launch_bounds__(kPcThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) w4_pc_kernel(const PcArgs a) {
  w4_pc_body<BM, XBF16, WB, TAIL>(a);
}

// W8A16 (int8 weights, ldq in bytes): as w4_pc_ok without zero words.
bool w8_pc_ok(const void* x, int64_t ldx, const int8_t* qw, int64_t ldq, const void* scales, int sdt, int64_t lds,
              int64_t N, int64_t K, int gs, int64_t G) {
  return (K % 32) == 0 && ((gs % 32) == 0 || G == 1) && (N % 2) == 0 && sdt != FG_F32 && (lds % 2) == 0 &&
         (reinterpret_cast<uintptr_t>(scales) % 4) == 0 && (ldx % 8) == 0 &&
         (reinterpret_cast<uintptr_t>(x) % 16) == 0 && (ldq % 16) == 0 && (reinterpret_cast<uintptr_t>(qw) % 16) == 0 &&
         group_div_exact(K, gs, G, 32);
}

bool w4_pc_ok(const void* x, int64_t ldx, const int32_t* qw, int64_t ldq, const int32_t* perm, const void* scales,
              int sdt, int64_t lds, int64_t N, int64_t K, int gs, int64_t G) {
  return perm == nullptr && (K % 32) == 0 && ((gs % 32) == 0 || G == 1) && (N % 8) == 0 && N >= 8 &&
         sdt != FG_F32 && (lds % 2) == 0 && (reinterpret_cast<uintptr_t>(scales) % 4) == 0 && (ldx % 8) == 0 &&
         (reinterpret_cast<uintptr_t>(x) % 16) == 0 && (ldq % 4) == 0 && (reinterpret_cast<uintptr_t>(qw) % 16) == 0 &&
         group_div_exact(K, gs, G, 32);
}

// Row tile (64, 128 or 256) and K splits: the cheapest by a cost in ns fitted to graph replays over five shapes (N =
// 2048..28672, K = 2048..14336, 5..1500 rows): a launch takes the slices of its workgroups times the tile's time per
// slice, plus 4.6 us, for every round of workgroups over the CUs; a split launch 2.7 us and 0.42 us per MB of partials
// more.  The choice lies within 0.5% (geometric mean) of the best of tile and split measured.  The time per slice hardly
// falls below 128 rows: a producer's chain of staging read, dequantisation and stores is what a slice takes there.
// Rows of 64 / 128 / 256 measured (us, fp16 x, groups of 64): K=4096, N=28672 M=64 46 / 52 / -, M=128 89 / 53 / 69,
// M=200 175 / 99 / 71; K=N=2048 M=300 17.8 / 19.2 / 22.7.  The all-rounder, which took these before: M=64 54, M=128 62,
// M=200 89, and 22.5.
// Returns that cost.
int64_t w4_pc_plan(bool w8, int M, int N, int K, int split_k, int* bm, int* splits, int* kchunk) {
  static const struct { int bm, ns; } kTile[] = {{64, 614}, {128, 726}, {256, 880}};
  const uint32_t cus = (uint32_t)device_cus(), slices = ((uint32_t)K + kPcBK - 1) / kPcBK;
  int64_t best = -1;
  for (const auto& t : kTile) {
    if (w8 && t.bm == 256) continue;  // three stages with 8-bit staging exceed the LDS
    const uint32_t tiles = (uint32_t)((M + t.bm - 1) / t.bm) * (uint32_t)((N + kPcBN - 1) / kPcBN);
    const uint32_t most = split_k > 0 ? (uint32_t)split_k
                                      : std::max(1u, std::min(std::min(16u, (uint32_t)K / 256), cus / tiles));
    uint32_t last = 0;
    for (uint32_t s = split_k > 0 ? most : 1; s <= most; ++s) {
      const uint32_t per = (slices + s - 1) / s;
      if (per == last) continue;  // one split more, no shorter ones
      last = per;
      const uint32_t used = (slices + per - 1) / per, rounds = (tiles * used + cus - 1) / cus;
      const int64_t cost = (int64_t)rounds * ((int64_t)per * t.ns + 4600) + (used > 1 ? 2700 + (int64_t)used * M * N / 600 : 0);
      if (best < 0 || cost < best) {
        best = cost;
        *bm = t.bm;
        *splits = (int)used;
        *kchunk = (int)per * kPcBK;
      }
    }
  }
  return best;
}

size_t w4_pc_workspace_bytes(bool w8, int M, int N, int K, int split_k) {
  int bm, s, kc;
  w4_pc_plan(w8, M, N, K, split_k, &bm, &s, &kc);
  return s > 1 ? (size_t)s * (size_t)M * (size_t)N * sizeof(float) : 0;
}

template <bool XBF16>
hipError_t launch_w4_splitk_reduce(const float* ws, int S, int M, int N, const void* bias, int bdt, void* y,
                                   int64_t ldy, hipStream_t s);

template <int WB>
static hipError_t launch_pc(const void* x, int64_t ldx, bool xbf16, const void* qw, int64_t ldq, const void* scales,
                            int sdt, int64_t lds, const int32_t* zeros, int64_t ldz, const void* bias, int bdt, void* y,
                            int64_t ldy, float* ws, int M, int N, int K, int gs, bool single_group, int split_k,
                            hipStream_t s) {
  int bm, splits, kchunk;
  w4_pc_plan(WB == 8, M, N, K, split_k, &bm, &splits, &kchunk);
  PcArgs a;
  a.x = static_cast<const uint16_t*>(x);
  a.ldx = ldx;
  a.qw = qw;
  a.ldq = ldq;
  a.scales = static_cast<const uint16_t*>(scales);
  a.lds = lds;
  a.hasz = zeros != nullptr;
  a.zeros = zeros ? zeros : static_cast<const int32_t*>(qw);
  a.ldz = zeros ? ldz : 0;
  a.bias = bias;
  a.bdt = bdt;
  a.ws = ws;
  a.y = static_cast<uint16_t*>(y);
  a.ldy = ldy;
  a.M = M;
  a.N = N;
  a.K = K;
  a.kchunk = kchunk;
  a.gdiv = single_group ? 0u : (uint32_t)(gs / 32);
  a.gmul = a.gdiv > 1 ? 0xffffffffu / a.gdiv + 1u : 0u;
  a.sbf16 = sdt == FG_BF16;
  if (splits > 1 && ws == nullptr) return hipErrorInvalidValue;
  auto go = [&](auto bm_tag) -> hipError_t {
    constexpr int BM = decltype(bm_tag)::value;
    auto kern = K % kPcBK ? (xbf16 ? w4_pc_kernel<BM, true, WB, true> : w4_pc_kernel<BM, false, WB, true>)
                          : (xbf16 ? w4_pc_kernel<BM, true, WB, false> : w4_pc_kernel<BM, false, WB, false>);
    const int lds_bytes = pc_lds(BM, WB, pc_exact(WB, K % kPcBK != 0));
    const hipError_t err =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (err != hipSuccess) return err;
    const int tiles = ((M + BM - 1) / BM) * ((N + kPcBN - 1) / kPcBN);
    note_kernel("w4_pc_kernel<%s%s> %dx128 splits=%d%s", xbf16 ? "bf16" : "f16", WB == 8 ? ",w8" : "", BM, splits,
                splits > 1 ? " + w4_splitk_reduce_kernel" : "");
    hipLaunchKernelGGL(kern, dim3(tiles, splits), dim3(kPcThreads), lds_bytes, s, a);
    return hipGetLastError();
  };
  hipError_t e;
  if (bm == 64) e = go(std::integral_constant<int, 64>{});
  else if (WB == 8 || bm == 128) e = go(std::integral_constant<int, 128>{});
  else e = go(std::integral_constant<int, WB == 8 ? 128 : 256>{});
  if (e != hipSuccess || splits == 1) return e;
  return xbf16 ? launch_w4_splitk_reduce<true>(ws, splits, M, N, bias, bdt, y, ldy, s)
               : launch_w4_splitk_reduce<false>(ws, splits, M, N, bias, bdt, y, ldy, s);
}

hipError_t launch_w4_pc(const void* x, int64_t ldx, bool xbf16, const int32_t* qw, int64_t ldq, const void* scales,
                        int sdt, int64_t lds, const int32_t* zeros, int64_t ldz, const void* bias, int bdt, void* y,
                        int64_t ldy, float* ws, int M, int N, int K, int gs, bool single_group, int split_k,
                        hipStream_t s) {
  return launch_pc<4>(x, ldx, xbf16, qw, ldq, scales, sdt, lds, zeros, ldz, bias, bdt, y, ldy, ws, M, N, K, gs,
                      single_group, split_k, s);
}

hipError_t launch_w8_pc(const void* x, int64_t ldx, bool xbf16, const int8_t* qw, int64_t ldq, const void* scales,
                        int sdt, int64_t lds, const void* bias, int bdt, void* y, int64_t ldy, float* ws, int M, int N,
                        int K, int gs, bool single_group, int split_k, hipStream_t s) {
  return launch_pc<8>(x, ldx, xbf16, qw, ldq, scales, sdt, lds, nullptr, 0, bias, bdt, y, ldy, ws, M, N, K, gs,
                      single_group, split_k, s);
}

}  // namespace fg
