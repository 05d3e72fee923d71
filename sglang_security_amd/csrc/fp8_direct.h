// fp8 products of at most 64 rows on the streaming weight layout (sglk_fp8_repack), per-token x per-channel scales
// (included by fp8.hip).
//
// Bound by the weights' way from memory, and on a decode step's shapes (16 to 117 MB over 256 units) by how much of it is
// asked for at once.  Both kernels multiply whole k-blocks: a lane's 32 bytes of a row and of a strip are the operands of one
// 16x16x128 f8f6f4 instruction as they stand, at twice the rate of the four 16x16x32 ones it replaces.  It aligns and adds 128
// products at once where those round in between, so last bits differ; the error against 64-bit sums does not (normal values, 512
// to 14336 of k: 1.2e-5 to 1.5e-5 of the result with either, and the same to 1 % for positive ones, for outliers 300 times the
// rest, and for values or blocks of 32 spread over 2^12 to 2^18).
//
// Up to 32 rows (direct): no staging and no barrier in the loop.  A block's waves take its k-blocks in turn, ask for their bytes
// of x and of the weights straight into registers and meet once in LDS; x is a fraction of the weights' bytes, or, under a
// strip a block, what the caches still carry.
// From 33 rows on (staged) x outweighs a strip: it goes through LDS, four k-blocks a stage, asked for two stages and put
// down one stage ahead, one barrier a stage; the weights keep to registers, PW stages ahead.
//
// us a launch, weights from memory, four waves and a barrier a k-block before (with its reduction launch where it split):
//   rows            1               16               32               64
//   4096 x 6144     12.4 -> 6.3     12.9 -> 6.7      13.6 -> 8.3      15.4 -> 10.2
//   4096 x 4096     10.2 -> 4.8     10.5 -> 5.7      11.0 -> 7.0      12.5 -> 7.2 + 2
//   4096 x 28672    29.5 -> 21.5    29.6 -> 21.6     30.4 -> 23.3     33.8 -> 28.9
//   14336 x 4096    18.8 -> 11.8    18.9 -> 14.7     19.7 -> 14.7 + 2 23.7 -> 16.0 + 2
#pragma once
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace sglk {

struct Fp8DirectArgs {
  const uint8_t* x;
  const uint8_t* wp;
  const float* sa;
  const float* sb;
  const void* bias;
  void* out;
  float* partial;  // raw sums [split][M][N], or nullptr
  int M, N, K, kb_per_split;
  int64_t x_stride, out_stride;
};

typedef int int8v __attribute__((ext_vector_type(8)));
__device__ __forceinline__ float4v fp8_block_mma(int4v x0, int4v x1, int4v w0, int4v w1, float4v c) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(int8v{x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w},
                                                          int8v{w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w}, c, 0, 0, 0, 0, 0, 0);
}

// The waves' tiles in LDS, [WAYS][ROWS][pitch], added up and stored.
template <typename TO, int ROWS, int COLS, int WAYS, int THREADS>
__device__ __forceinline__ void fp8_direct_store(const Fp8DirectArgs& a, const float* red) {
  constexpr int kPitch = COLS + 4;
  for (int e = threadIdx.x; e < ROWS * COLS; e += THREADS) {
    const int m = e / COLS, c = e % COLS, col = blockIdx.x * COLS + c;
    if (m >= a.M || col >= a.N) continue;
    float v = red[m * kPitch + c];
#pragma unroll
    for (int k = 1; k < WAYS; ++k) v += red[(k * ROWS + m) * kPitch + c];
    if (a.partial)
      __hip_atomic_store(&a.partial[((int64_t)blockIdx.y * a.M + m) * a.N + col], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
      st<TO>(a.out, (int64_t)m * a.out_stride + col, v * a.sa[m] * a.sb[col] + (a.bias ? ld<TO>(a.bias, col) : 0.f));
  }
}

// MT tiles of 16 rows, CS strips of 16 columns, WAYS waves, R k-blocks of a wave on their way.
template <int MT, int CS, int WAYS>
constexpr int fp8_direct_lds() {
  return WAYS * 16 * MT * (16 * CS + 4) * 4;
}
template <typename TO, int MT, int CS, int WAYS, int R>
__global__ void __launch_bounds__(64 * WAYS, WAYS / 4) fp8_direct_kernel(const Fp8DirectArgs a) {
  constexpr int kPitch = 16 * CS + 4, kRows = 16 * MT;
  extern __shared__ __attribute__((aligned(16))) float sums[];
  const int lane = threadIdx.x & 63, way = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i16 = lane & 15, g = lane >> 4;
  const int kblocks = a.K / 128, first = blockIdx.y * a.kb_per_split, kb0 = first + way;
  const int n = (min(a.kb_per_split, kblocks - first) - way + WAYS - 1) / WAYS;  // k-blocks of this wave
  const uint8_t* wsrc[CS];
#pragma unroll
  for (int c = 0; c < CS; ++c)  // strips past the last repeat it
    wsrc[c] = a.wp + ((int64_t)min((int)blockIdx.x * CS + c, a.N / 16 - 1) * kblocks + kb0) * 2048 + 16 * lane;
  const uint8_t* xsrc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xsrc[t] = a.x + (int64_t)min(16 * t + i16, a.M - 1) * a.x_stride + 128 * kb0 + 32 * g;

  int4v w[R][CS][2], xf[R][MT][2];
  auto load = [&](int i, int slot) {
    const int j = WAYS * min(i, n - 1);
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) xf[slot][t][h] = *reinterpret_cast<const int4v*>(xsrc[t] + 128 * j + 16 * h);
#pragma unroll
    for (int c = 0; c < CS; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        w[slot][c][h] = __builtin_nontemporal_load(reinterpret_cast<const int4v*>(wsrc[c] + (int64_t)2048 * j + 1024 * h));
  };
  float4v acc[CS][MT];
#pragma unroll
  for (int c = 0; c < CS; ++c)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[c][t] = float4v{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int slot) {
#pragma unroll
    for (int c = 0; c < CS; ++c)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[c][t] = fp8_block_mma(xf[slot][t][0], xf[slot][t][1], w[slot][c][0], w[slot][c][1], acc[c][t]);
  };
  if (n > 0) {
#pragma unroll
    for (int u = 0; u < R; ++u) load(u, u);
    __builtin_amdgcn_sched_barrier(0);  // every request leaves before the first product waits
    int i0 = 0;
    for (; i0 + R < n; i0 += R) {
#pragma unroll
      for (int u = 0; u < R; ++u) {
        multiply(u);
        load(i0 + R + u, u);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int u = 0; u < R; ++u)
      if (i0 + u < n) multiply(u);
  }
  // register r of tile (c, t): row 16 t + 4 g + r, column 16 c + i16
#pragma unroll
  for (int c = 0; c < CS; ++c)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) sums[(way * kRows + 16 * t + 4 * g + r) * kPitch + 16 * c + i16] = acc[c][t][r];
  __syncthreads();
  fp8_direct_store<TO, kRows, 16 * CS, WAYS, 64 * WAYS>(a, sums);
}

// 64 rows; SB strips a block, a wave one strip and 4 / WAYS of a stage's four k-blocks; PW stages of weights on their way.
template <int SB>
constexpr int fp8_staged_lds() {
  return std::max(2 * 4 * 64 * 128, 8 / SB * 64 * (16 * SB + 4) * 4);
}
template <typename TO, int SB, int PW>
__global__ void __launch_bounds__(512, 4) fp8_staged_kernel(const Fp8DirectArgs a) {
  constexpr int WAYS = 8 / SB, KW = 4 / WAYS, kTile = 64 * 128;  // bytes of a k-block of x
  extern __shared__ __attribute__((aligned(16))) char lds[];     // [2 stages][4][kTile], then the sums
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15, g = lane >> 4;
  const int way = wid / SB, strip = blockIdx.x * SB + wid % SB;
  const int kblocks = a.K / 128, kb0 = blockIdx.y * a.kb_per_split, nkb = min(a.kb_per_split, kblocks - kb0), nst = (nkb + 3) / 4;
  const uint8_t* wsrc = a.wp + ((int64_t)min(strip, a.N / 16 - 1) * kblocks + kb0) * 2048 + 16 * lane;
  // x: a thread takes one 16-byte chunk of a row in each of the stage's k-blocks; chunk c of row r lies in slot c ^ (r / 2 % 8)
  // of its 128 bytes, so that an operand read meets every bank group four times, the least there is
  const int xrow = tid >> 3, xc = tid & 7;
  const uint8_t* xsrc = a.x + (int64_t)min(xrow, a.M - 1) * a.x_stride + (int64_t)128 * kb0 + 16 * xc;
  auto off = [](int r, int c) { return r * 128 + ((c ^ ((r >> 1) & 7)) << 4); };
  int4v xr[4], w[PW][KW][2];
  auto x_ask = [&](int s) {
#pragma unroll
    for (int b = 0; b < 4; ++b) xr[b] = *reinterpret_cast<const int4v*>(xsrc + 128 * min(4 * s + b, nkb - 1));
  };
  auto x_put = [&](int buf) {
#pragma unroll
    for (int b = 0; b < 4; ++b) *reinterpret_cast<int4v*>(lds + (buf * 4 + b) * kTile + off(xrow, xc)) = xr[b];
  };
  auto w_ask = [&](int s, int slot, int j) {
    const int kb = min(4 * s + way * KW + j, nkb - 1);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      w[slot][j][h] = __builtin_nontemporal_load(reinterpret_cast<const int4v*>(wsrc + (int64_t)2048 * kb + 1024 * h));
  };
  float4v acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = float4v{0.f, 0.f, 0.f, 0.f};
  x_ask(0);
#pragma unroll
  for (int p = 0; p < PW; ++p)
#pragma unroll
    for (int j = 0; j < KW; ++j) w_ask(p, p, j);
  x_put(0);
  x_ask(1);
  __syncthreads();
  auto stage = [&](int s, int p, auto more) {
    const int buf = p & 1;
#pragma unroll
    for (int j = 0; j < KW; ++j) {
      if (4 * s + way * KW + j < nkb) {
        const char* xt = lds + (buf * 4 + way * KW + j) * kTile;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int4v x0 = *reinterpret_cast<const int4v*>(xt + off(16 * t + i16, 2 * g));
          const int4v x1 = *reinterpret_cast<const int4v*>(xt + off(16 * t + i16, 2 * g + 1));
          acc[t] = fp8_block_mma(x0, x1, w[p][j][0], w[p][j][1], acc[t]);
        }
      }
      if constexpr (decltype(more)::value) w_ask(s + PW, p, j);
    }
    if (s + 1 < nst) {
      x_put(buf ^ 1);  // its readers met at the end of the stage before
      x_ask(s + 2);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // not what is on its way from memory, as __syncthreads() may
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
  };
  static_assert(PW % 2 == 0, "the halves of LDS go by the parity of the stage");
  int s0 = 0;
  for (; s0 + PW < nst; s0 += PW) {
#pragma unroll
    for (int p = 0; p < PW; ++p) stage(s0 + p, p, std::true_type());
  }
#pragma unroll
  for (int p = 0; p < PW; ++p)
    if (s0 + p < nst) stage(s0 + p, p, std::false_type());
  __syncthreads();
  float* sums = reinterpret_cast<float*>(lds);
  constexpr int kPitch = 16 * SB + 4;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) sums[(way * 64 + 16 * t + 4 * g + r) * kPitch + 16 * (wid % SB) + i16] = acc[t][r];
  __syncthreads();
  fp8_direct_store<TO, 64, 16 * SB, WAYS, 512>(a, sums);
}

}  // namespace sglk
