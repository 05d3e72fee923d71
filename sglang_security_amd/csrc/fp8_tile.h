// Scaled fp8 products of many rows (gfx950): out[M, N] = (a[M, K] . b[N, K]^T) * sa[m] * sb[n] (+ bias), e4m3 codes.
//
// A block of WM x WN waves owns a BM x BN tile and walks K in steps of 128 bytes through a ring of ST LDS stages.  Rows arrive by
// LDS-DMA in 16-byte chunks, chunk c of row r in slot c ^ ((r >> 1) & 7) ^ 4 (r & 1) of its 128 bytes: the 8 (and the
// 16) consecutive rows that an operand read takes at once lie in different banks.  Products are formed on
// v_mfma_f32_32x32x64_f8f6f4, twice the rate of the 16-bit-era fp8 forms; the weights are operand A, so that a lane's
// accumulators are four consecutive output columns of one row, which leave through LDS in whole row pieces.
//
// Bound: 256 x 256 by the matrix unit and the LDS (96 KiB read and 64 KiB written per 2048 matrix cycles of a SIMD);
// the small tiles by the trip of a stage from memory, hence the deeper rings.  Measured (bf16 out): 2048 x 28672 x 4096
// 214 us = 2.25 PFLOP/s, 2048 x 4096 x 14336 110 us = 2.19 PFLOP/s, each launched alone; the register kernel, every wave
// fetching its own operands, 1190 and 593 us (0.40 PFLOP/s).  In a layer's sequence, under the profiler, its two 256 x 256
// products (6144 and 28672 columns) take 304 us, 1.9 PFLOP/s, its two 128 x 128 ones 180 us, 1.7 PFLOP/s.
#pragma once
#include "common.h"

namespace sglk {

typedef int int8v __attribute__((ext_vector_type(8)));

struct Fp8TileArgs {
  const uint8_t *a, *b;
  const float *sa, *sb;
  const void* bias;
  void* out;
  int M, N, K, mt, nt;  // mt x nt tiles
  int64_t a_stride, b_stride, out_stride;
};

__device__ __forceinline__ int fp8_slot(int r, int c) { return c ^ ((r >> 1) & 7) ^ ((r & 1) << 2); }

// two 1-KiB pieces to lds .. lds + 2 KiB: lane's 16 bytes of piece i come from base + off[i] (off[i] < 2^32 - 1024); the
// instruction offset is added to both addresses, so off[1] arrives lowered by 1024 against base - 1024
__device__ __forceinline__ void fp8_dma2(const uint8_t* base, uint32_t lds, uint32_t off0, uint32_t off1) {
  const uint8_t* src = base - 1024;
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %3\n\t"
      "global_load_lds_dwordx4 %2, %3 offset:1024" ::"s"(lds),
      "v"(off0 + 1024), "v"(off1), "s"(src)
      : "memory", "m0");
}

template <typename TO, int BM, int BN, int WM, int WN, int ST>
__global__ void __launch_bounds__(64 * WM * WN, 2) fp8_tile_kernel(Fp8TileArgs p) {
  constexpr int NW = WM * WN, MI = BM / WM / 32, NJ = BN / WN / 32;
  constexpr int kStage = (BM + BN) * 128;
  constexpr int U = (BM + BN) / 16 / NW;  // units of 16 rows (two pieces) a wave fetches per stage: rows of a, then of b
  static_assert(U * 16 * NW == BM + BN && BM % 16 == 0, "whole units per wave");
  static_assert(2 * U * (ST - 2) <= 63, "outstanding requests are counted in six bits");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int l31 = lane & 31, hi = lane >> 5;
  // blocks go to the eight dies in turn: a die takes a run of neighbouring tiles (all row tiles of a weight strip)
  const int total = p.mt * p.nt, q = total >> 3, rem = total & 7, xcd = blockIdx.x & 7;
  const int tile = xcd * q + min(xcd, rem) + ((int)blockIdx.x >> 3);
  const int m0 = tile % p.mt * BM, n0 = tile / p.mt * BN;

  const int nk = p.K / 128;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
  const int wq = __builtin_amdgcn_readfirstlane(wid);
  const uint8_t* base[U];
  uint32_t off[U][2];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int r0 = (wq * U + u) * 16;  // of the stage: wave-uniform
    const bool isa = r0 < BM;
    const int first = isa ? m0 : n0 - BM, last = (isa ? p.M : p.N) - 1;
    const uint32_t stride = (uint32_t)(isa ? p.a_stride : p.b_stride);
    base[u] = isa ? p.a + (int64_t)m0 * p.a_stride : p.b + (int64_t)n0 * p.b_stride;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = r0 + 8 * j + (lane >> 3);  // rows past the end: the last one, never stored
      off[u][j] = (uint32_t)(min(first + r, last) - (isa ? m0 : n0)) * stride + 16 * fp8_slot(r, lane & 7);
    }
  }
  auto issue = [&](int kb) {
    const uint32_t st = lds0 + kb % ST * kStage + wq * U * 2048;
    const int64_t k0 = (int64_t)min(kb, nk - 1) * 128;  // past the end: the last block again, so that the counted waits hold
#pragma unroll
    for (int u = 0; u < U; ++u) fp8_dma2(base[u] + k0, st + u * 2048, off[u][0], off[u][1]);
  };

  const int wm = wid / WN * (32 * MI), wn = wid % WN * (32 * NJ);
  float16v acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  auto operand = [&](const char* rows, int r, int ks) {
    const char* row = rows + r * 128;
    const int4v x = *reinterpret_cast<const int4v*>(row + 16 * fp8_slot(r, 4 * ks + 2 * hi));
    const int4v y = *reinterpret_cast<const int4v*>(row + 16 * fp8_slot(r, 4 * ks + 2 * hi + 1));
    return int8v{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
  };

#pragma unroll
  for (int i = 0; i < ST - 1; ++i) issue(i);
  for (int kb = 0; kb < nk; ++kb) {
    // this wave's pieces of the stage have landed and its operands of the stage before have arrived; behind the barrier
    // everyone's have, and the stage before is free
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * U * (ST - 2)) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (ST > 2 || kb + 1 < nk) issue(kb + ST - 1);
    const char* al = lds + kb % ST * kStage;
    const char* bl = al + BM * 128;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      int8v af[MI], bf[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) bf[j] = operand(bl, wn + 32 * j + l31, ks);
#pragma unroll
      for (int i = 0; i < MI; ++i) af[i] = operand(al, wm + 32 * i + l31, ks);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bf[j], af[i], acc[i][j], 0, 0, 0, 0, 0, 0);
    }
  }

  // lane (m, hi) holds columns 32 j + 8 g + 4 hi + 0 .. 3 of row wm + 32 i + m
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  constexpr int kPitch = 64 * NJ + 16, kOutBytes = 32 * kPitch;  // one 32-row tile row of the wave at a time
  static_assert(NW * kOutBytes <= ST * kStage, "the stages hold the rows on their way out");
  char* ol = lds + wid * kOutBytes;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const float sa = p.sa[min(m0 + wm + 32 * i + l31, p.M - 1)];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = min(n0 + wn + 32 * j + 8 * g + 4 * hi, p.N - 4);  // N % 4 == 0: a quad lies inside or outside whole
        const float4v sb = *reinterpret_cast<const float4v*>(p.sb + n);
        short4v v, bias = {0, 0, 0, 0};
        if (p.bias) bias = *reinterpret_cast<const short4v*>(reinterpret_cast<const uint16_t*>(p.bias) + n);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float bn = p.bias ? Conv<TO>::to_f32((uint16_t)bias[r]) : 0.f;
          v[r] = (short)Conv<TO>::from_f32(scaled_sum(acc[i][j][4 * g + r], sa, sb[r], bn));
        }
        *reinterpret_cast<short4v*>(ol + l31 * kPitch + (32 * j + 8 * g + 4 * hi) * 2) = v;
      }
    __builtin_amdgcn_wave_barrier();  // the wave's own LDS rows: in order, no block barrier
    constexpr int kPer = 8 * NJ / 2;  // lanes (16-byte pieces) per row
    static_assert(64 % kPer == 0, "");
#pragma unroll
    for (int t = 0; t < 32 * kPer / 64; ++t) {
      const int row = t * (64 / kPer) + lane / kPer, c = lane % kPer;
      const int4v v = *reinterpret_cast<const int4v*>(ol + row * kPitch + c * 16);
      const int m = m0 + wm + 32 * i + row, n = n0 + wn + c * 8;
      if (m < p.M && n < p.N)
        *reinterpret_cast<int4v*>(reinterpret_cast<uint16_t*>(p.out) + (int64_t)m * p.out_stride + n) = v;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

}  // namespace sglk
