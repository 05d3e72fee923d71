// 16-bit products of at most 32 rows, those that gemm_dense.hip's rules leave to this kernel, on the streaming weight layout
// (sglk_dense_repack) and, with the same bits, on row-major weights (included by gemm_dense.hip).
//
// Bound by the weights' way from memory.  The staged kernel shares x through LDS and meets at a barrier every 128 of k, two to
// four k-blocks a wave on their way; with so few rows x is a fraction of the weights, so nothing is staged here: a block's
// waves take its k-blocks in turn, straight into registers, and meet once.  Four to sixteen waves of 4 to 16 KiB keep a unit's
// requests going without a deeper ring a wave (two k-blocks ahead were slower on every shape), and far fewer splits
// fill the units, so that the kernels that consume the sums read less.
// us a launch, weights from memory (staged -> direct, splits):
//   rows             1                       16                      32
//   2560 x 2560      6.8 -> 4.2 (5, 3)       6.9 -> 4.5              7.0 -> 5.3
//   6912 x 2560      13.3 -> 7.5 (8, 3)      13.4 -> 8.4             13.9 -> 10.2
//   2560 x 11008     17.0 -> 11.3 (5, 1)     17.4 -> 13.2            18.2 -> 15.8
//   2560 x 13824     18.4 -> 13.2 (5, 1)     19.4 -> 14.3            21.7 -> 16.6
//   2560 x 65536     61.0 -> 53.7 (1, 1)     61.4 -> 57.5
//   4096 x 128256    186 -> 156 (1, 1)       185 -> 164              (6.7 and 6.4 TB/s)
#pragma once
#include "common.h"

namespace sglk {

struct DenseDirectArgs {
  const uint16_t* x;
  const uint16_t* w;
  const uint16_t* bias;
  uint16_t* out;
  float* partial;  // raw sums [split][Mpad][N], or nullptr
  int M, Mpad, N, K, kb_per_split;
  int64_t x_stride, w_stride, out_stride;
};

// MT tiles of 16 rows, CS strips of 16 columns, WAYS waves that take the k-blocks of 128 in turn, one at a time.
template <int MT, int CS, int WAYS>
constexpr int dense_direct_lds() {
  return WAYS * 16 * MT * (16 * CS + 4) * 4;
}
template <typename T, int MT, int CS, int WAYS, bool PACKED>
__global__ void __launch_bounds__(64 * WAYS, WAYS / 4) dense_direct_kernel(const DenseDirectArgs a) {
  constexpr int kCols = 16 * CS, kPitch = kCols + 4, kRows = 16 * MT;
  extern __shared__ __attribute__((aligned(16))) float sums[];
  const int lane = threadIdx.x & 63, way = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i16 = lane & 15, g = lane >> 4;
  const int kblocks = a.K / 128, first = blockIdx.y * a.kb_per_split, kb0 = first + way;
  const int n = (min(a.kb_per_split, kblocks - first) - way + WAYS - 1) / WAYS;  // k-blocks of this wave
  const uint16_t* wsrc[CS];
#pragma unroll
  for (int c = 0; c < CS; ++c)  // strips past the last repeat it
    wsrc[c] = PACKED ? a.w + ((int64_t)min((int)blockIdx.x * CS + c, a.N / 16 - 1) * kblocks + kb0) * 2048 + 8 * lane
                     : a.w + (int64_t)(min((int)blockIdx.x * CS + c, a.N / 16 - 1) * 16 + i16) * a.w_stride + 128 * kb0 + 8 * g;
  const uint16_t* xsrc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xsrc[t] = a.x + (int64_t)min(16 * t + i16, a.M - 1) * a.x_stride + 128 * kb0 + 8 * g;

  float4v acc[CS][MT];
#pragma unroll
  for (int s = 0; s < CS; ++s)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[s][t] = float4v{0.f, 0.f, 0.f, 0.f};
  int4v w[CS][4], xf[MT][4];
  auto load = [&](int i) {
    const int j = WAYS * i;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int c = 0; c < 4; ++c) xf[t][c] = *reinterpret_cast<const int4v*>(xsrc[t] + 128 * j + 32 * c);
#pragma unroll
    for (int s = 0; s < CS; ++s)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        w[s][c] = PACKED ? __builtin_nontemporal_load(reinterpret_cast<const int4v*>(wsrc[s] + (int64_t)2048 * j + 512 * c))
                         : *reinterpret_cast<const int4v*>(wsrc[s] + 128 * j + 32 * c);  // (lines shared by four loads)
    __builtin_amdgcn_sched_barrier(0);  // every request leaves before the first product waits
  };
  auto multiply = [&]() {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int s = 0; s < CS; ++s)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[s][t] = DenseMma<T>::mma(xf[t][c], w[s][c], acc[s][t]);
  };
  if (n > 0) {
    load(0);
    for (int i = 1; i < n; ++i) {
      multiply();
      load(i);
    }
    multiply();
  }
  // register r of tile (s, t): row 16 t + 4 g + r, column 16 s + i16
#pragma unroll
  for (int s = 0; s < CS; ++s)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) sums[(way * kRows + 16 * t + 4 * g + r) * kPitch + 16 * s + i16] = acc[s][t][r];
  __syncthreads();
  for (int e = threadIdx.x; e < kRows * kCols; e += 64 * WAYS) {
    const int m = e / kCols, c = e % kCols, col = blockIdx.x * kCols + c;
    if (m >= a.M || col >= a.N) continue;
    float v = sums[m * kPitch + c];
#pragma unroll
    for (int k = 1; k < WAYS; ++k) v += sums[(k * kRows + m) * kPitch + c];
    if (a.partial)
      __hip_atomic_store(&a.partial[((int64_t)blockIdx.y * a.Mpad + m) * a.N + col], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
      a.out[(int64_t)m * a.out_stride + col] = Conv<T>::from_f32(v + (a.bias ? Conv<T>::to_f32(a.bias[col]) : 0.f));
  }
}

}  // namespace sglk
