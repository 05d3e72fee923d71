// int4 products of at most 16 activation rows (included by awq.hip, whose header describes the packed layout).
//
// Such a product is a stream over the packed weights, and on the shapes of a decode step a short one: 32 KiB (4096 x 4096)
// to 256 KiB (4096 x 28672) a CU.  What bounds it is how early its requests leave and how little follows the last answer.
// So nothing is staged: a wave asks for weights, scales, zeros and rows of x straight into registers, before its first
// product, and no barrier stands in its loop.  A block is the wide kernel's, 128 columns x the groups of a split, so split
// sums keep that kernel's count and places; its waves take the block's groups in turn, S strips of 16 columns
// each, and meet once in LDS.  x . (OFF + q) runs on 16x16x32 tiles (32-row tiles would double the matrix work for rows that are
// not there); the sum of x that the zero point needs is the same product with a column of ones, so the block sums
// of x are not read.
// x . (OFF + q) - (OFF + z) . sum(x) is in fp16 (OFF is 1024) a hundredth of either term and carries the roundings of both:
// there a group is two halves, whose sums are smaller (16 rows, 4096 x 4096: 1.23e-5 of the result whole, 9.0e-6 so, 1.22e-5
// in the wide kernel).
// Rows that a batch does not have repeat its last one: switching their lanes off costs more than it saves (one row, 4096 x 28672,
// taken before the launches' last shapes: 15.9 against 15.3 us, two halves of a block 29 against 16).  All figures here: weights
// from memory, us a launch.
#pragma once
#include "awq_common.h"

namespace sglk {

struct AwqRows16 {
  static constexpr int kRows = 16;
  static constexpr int kRowStride = 132;  // floats of a row of the waves' tiles in LDS
  static constexpr int kTile = kRows * kRowStride;
};

template <typename T>
struct AwqRows16Args {
  const uint16_t* x;
  const int32_t* packed;
  const uint16_t* scales;
  const int32_t* qzeros;
  const uint16_t* bias;
  uint16_t* out;
  float* partial;    // split sums [split][M][N], or the slabs [tile][split][16][128] behind tickets
  int* tickets;
  float* xsum_out;   // gated activation: sums of 64 of its outputs, added per 128 of them
  int64_t x_stride, out_stride, xs_out_stride;
  int M, N, K, groups_per_split, splits, partial_mode, act_mode;
};

// S: 16-column strips of a wave; R: 128-k groups of a wave that are on their way at once
template <typename T, int S, int R, int NW>
__global__ void __launch_bounds__(64 * NW, NW / 4) awq_rows16_kernel(const AwqRows16Args<T> a) {
  using P = AwqRows16;
  constexpr int kTurns = NW * S / 8;
  constexpr int kParts = AwqMagic<T>::kOff == 128.f ? 1 : 2;  // of a group, each with its zero point taken off by itself
  extern __shared__ __attribute__((aligned(16))) float red[];
  __shared__ int last_block;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15, g = lane >> 4;
  const int turn = S == 8 ? wid : wid >> 1, half = S == 8 ? 0 : wid & 1;
  const int M = a.M, N = a.N;
  const int n0 = blockIdx.x * 128 + half * 64;
  const int nstrips = N / 16, qcols = N / 8;
  const int g0 = blockIdx.y * a.groups_per_split;
  const int ng = min(a.groups_per_split, a.K / 128 - g0);  // groups of the block
  const int n = (ng - turn + kTurns - 1) / kTurns;         // of this wave: turn, turn + kTurns, ..
  // this lane's part of group kb: weights of strip t at wp + kb * nstrips * 256 words + t * 256
  const int32_t* wp = a.packed + ((int64_t)(g0 + turn) * nstrips + n0 / 16) * 256 + lane * 4;
  const uint16_t* xp = a.x + (int64_t)min(i16, M - 1) * a.x_stride + (g0 + turn) * 128 + 8 * g;
  const uint16_t* sp = a.scales + (int64_t)(g0 + turn) * N + n0 + lane;           // lane = column of the half
  const int32_t* zp = a.qzeros + (int64_t)(g0 + turn) * qcols + (n0 + lane) / 8;
  const int zsh = 4 * (((lane & 7) >> 1) + 4 * (lane & 1));  // AWQ order {0,4,1,5,2,6,3,7}

  int4v w[R][S], xf[R][4];
  uint32_t s[R][S / 4], z[R][S / 4];
  auto load = [&](int i, int slot) {
    const int j = kTurns * min(i, n - 1);  // a request past the wave's last group repeats it
#pragma unroll
    for (int c = 0; c < S / 4; ++c) {
      s[slot][c] = sp[(int64_t)j * N + 64 * c];
      z[slot][c] = (uint32_t)zp[(int64_t)j * qcols + 8 * c];
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) xf[slot][d] = *reinterpret_cast<const int4v*>(xp + j * 128 + 32 * d);
#pragma unroll
    for (int t = 0; t < S; ++t) w[slot][t] = *reinterpret_cast<const int4v*>(wp + (int64_t)j * nstrips * 256 + t * 256);
  };
  float4v acc[S];
#pragma unroll
  for (int t = 0; t < S; ++t) acc[t] = float4v{0.f, 0.f, 0.f, 0.f};
  constexpr uint32_t kOne = (uint32_t)(AwqMagic<T>::kOff == 128.f ? 0x3F803F80u : 0x3C003C00u);
  const int4v ones = int4v{(int)kOne, (int)kOne, (int)kOne, (int)kOne};
  auto multiply = [&](int slot) {
    // scale and zero of this lane's column, one word; strip t's are lanes 16 t .. 16 t + 15's
    int sz[S / 4];
#pragma unroll
    for (int c = 0; c < S / 4; ++c) sz[c] = (int)((s[slot][c] << 16) | ((z[slot][c] >> zsh) & 0xF));
    float4v X[kParts];
#pragma unroll
    for (int h = 0; h < kParts; ++h) X[h] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < 4; ++d) X[d * kParts / 4] = AwqMagic<T>::mma(xf[slot][d], ones, X[d * kParts / 4]);
#pragma unroll
    for (int t = 0; t < S; ++t) {
      const uint32_t v = (uint32_t)__builtin_amdgcn_ds_bpermute((16 * (t & 3) + i16) * 4, sz[t >> 2]);
      float4v p[kParts];
#pragma unroll
      for (int h = 0; h < kParts; ++h) p[h] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint32_t q = (uint32_t)w[slot][t][d];
        int4v b;
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = (int)(((q >> (4 * e)) & 0x000F000Fu) | AwqMagic<T>::kOr);
        p[d * kParts / 4] = AwqMagic<T>::mma(xf[slot][d], b, p[d * kParts / 4]);
      }
      const float sc = Conv<T>::to_f32((uint16_t)(v >> 16)), nz = -(AwqMagic<T>::kOff + (float)(v & 0xF));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float s = fmaf(nz, X[0][e], p[0][e]);
        if constexpr (kParts == 2) s += fmaf(nz, X[1][e], p[1][e]);
        acc[t][e] = fmaf(sc, s, acc[t][e]);
      }
    }
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

  // the four turns of a column meet: register e of strip t is row 4 g + e, column 16 t + i16 of the half
  float* mine = red + turn * P::kTile + half * 64;
#pragma unroll
  for (int t = 0; t < S; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) mine[(4 * g + e) * P::kRowStride + 16 * t + i16] = acc[t][e];
  __syncthreads();
  auto total = [&](int row, int c) {
    const float* p = red + row * P::kRowStride + c;
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < kTurns; ++k) v += p[k * P::kTile];
    return v;
  };

  if (a.act_mode) {
    // columns 0..63 are gate columns, 64..127 the matching up columns: the values that the product and silu_and_mul store
    // one after the other.  A wave is a row; its sum is one of two addends of a 128-column block sum.
    for (int row = wid; row < M; row += NW) {
      const float gb = Conv<T>::to_f32(Conv<T>::from_f32(total(row, lane)));
      const float ub = Conv<T>::to_f32(Conv<T>::from_f32(total(row, 64 + lane)));
      const float sv = Conv<T>::to_f32(Conv<T>::from_f32(gb / (1.0f + __expf(-gb))));
      const uint16_t ob = Conv<T>::from_f32(sv * ub);
      a.out[(int64_t)row * a.out_stride + blockIdx.x * 64 + lane] = ob;
      if (a.xsum_out) {
        float v = Conv<T>::to_f32(ob);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) atomicAdd(&a.xsum_out[(int64_t)(blockIdx.x >> 1) * a.xs_out_stride + row], v);
      }
    }
    return;
  }
  const int c = tid & 127, col = blockIdx.x * 128 + c;
  if (a.partial_mode) {
    float* dst = a.partial + (int64_t)blockIdx.y * M * N + col;
    for (int row = tid >> 7; row < M; row += NW / 2)
      __hip_atomic_store(&dst[(int64_t)row * N], total(row, c), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  const float bv = a.bias ? Conv<T>::to_f32(a.bias[col]) : 0.f;
  if (a.splits == 1) {
    for (int row = tid >> 7; row < M; row += NW / 2) a.out[(int64_t)row * a.out_stride + col] = Conv<T>::from_f32(total(row, c) + bv);
    return;
  }
  // splits meet through slabs: agent-scope stores, and the block that draws the last ticket adds them up in split order
  float* slab = a.partial + (int64_t)blockIdx.x * a.splits * (P::kRows * 128) + c;
  for (int row = tid >> 7; row < M; row += NW / 2)
    __hip_atomic_store(&slab[(int64_t)blockIdx.y * (P::kRows * 128) + row * 128], total(row, c), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    const int ticket = __hip_atomic_fetch_add(&a.tickets[blockIdx.x], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last_block = ticket == a.splits - 1;
    if (last_block) __hip_atomic_store(&a.tickets[blockIdx.x], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last_block) return;
  // eight splits of a row are asked for at once, in row order: one after the other each is a trip to memory (16 rows, 14336 x 128 in
  // 28 splits: 18.9 us -> 9.8; 8192 x 1280 in 16: 14.2 -> 8.7)
  for (int row = tid >> 7; row < M; row += NW / 2) {
    const float* p = slab + row * 128;
    float sum = 0.f;
    for (int q0 = 0; q0 < a.splits; q0 += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        v[u] = __hip_atomic_load(&p[(int64_t)min(q0 + u, a.splits - 1) * (P::kRows * 128)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (q0 + u < a.splits) sum += v[u];
    }
    a.out[(int64_t)row * a.out_stride + col] = Conv<T>::from_f32(sum + bv);
  }
}

}  // namespace sglk
