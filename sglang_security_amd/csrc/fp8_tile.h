// Scaled fp8 products of many rows (gfx950): out[M, N] = (a[M, K] . b[N, K]^T) * sa[m] * sb[n] (+ bias), e4m3 codes.
//
// A block of WM x WN waves owns a BM x BN tile and walks K in steps of 128 bytes through a ring of ST LDS stages.  Rows arrive by
// LDS-DMA in 16-byte chunks, chunk c of row r in slot c ^ ((r >> 1) & 7) ^ 4 (r & 1) of its 128 bytes: the 8 (and the
// 16) consecutive rows that an operand read takes at once lie in different banks.  Products are formed on
// v_mfma_f32_32x32x64_f8f6f4, twice the rate of the 16-bit-era fp8 forms; the weights are operand A, so that a lane's
// accumulators are four consecutive output columns of one row, which leave through LDS in whole row pieces.
//
// Two kernels.  fp8_tile4_kernel, four waves of 128 x 64, 128 x 96 or 128 x 128 sums, is bound by a wave's own issue and by the
// matrix unit (busy two thirds of a wave's life; counters), a launch also by its start and by the results that all units store at once.
// fp8_tile_kernel's smaller tiles are bound by the trip of a stage from memory, hence their deeper rings.  Measured (bf16 out,
// weights from memory, both on one card): 2048 x 28672 x 4096 222 us (eight waves) -> 199 = 2.42 PFLOP/s (181 to 202 from card to card);
// 2048 x 4096 x 14336 125 (128 x 128 tiles) -> 97 = 2.48 PFLOP/s; 2048 x 6144 x 4096 50 -> 43, 2048 x 4096 x 4096 39 -> 33.  Of that, the
// rows on their way out without a branch per quad for the bias are a twentieth to a tenth of the largest, in every form.
#pragma once
#include <type_traits>

#include "common.h"

namespace sglk {

typedef int int8v __attribute__((ext_vector_type(8)));

struct Fp8TileArgs {
  const uint8_t *a, *b;
  const float *sa, *sb;
  const void* bias;
  void* out;
  int M, N, K, mt, nt;  // mt x nt tiles
  int nt_tail, tail;    // fp8_tile4_kernel: narrower strips behind them, and their columns
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

constexpr int fp8_out_bytes(int nj) { return 32 * (64 * nj + 16); }  // a wave's 32 rows of 32 nj results

// A wave's sums from row m0, column n0 on, scaled and rounded: lane (m, hi) holds columns 32 j + 8 g + 4 hi + 0 .. 3 of row
// 32 i + m; they leave through LDS, one 32-row tile row at a time, in whole row pieces
template <typename TO, int MI, int NJ>
__device__ __forceinline__ void fp8_tile_store(const Fp8TileArgs& p, const float16v (&acc)[MI][NJ], char* ol, int m0, int n0,
                                               int lane) {
  constexpr int kPitch = 64 * NJ + 16;
  const int l31 = lane & 31, hi = lane >> 5;
  float sa[MI];
  float4v sb[NJ][4];
#pragma unroll
  for (int i = 0; i < MI; ++i) sa[i] = p.sa[min(m0 + 32 * i + l31, p.M - 1)];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g)  // N % 4 == 0: a quad lies inside or outside whole
      sb[j][g] = *reinterpret_cast<const float4v*>(p.sb + min(n0 + 32 * j + 8 * g + 4 * hi, p.N - 4));
  auto rows = [&](auto with_bias) {
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          short4v v, bias = {0, 0, 0, 0};
          if constexpr (decltype(with_bias)::value)
            bias = *reinterpret_cast<const short4v*>(reinterpret_cast<const uint16_t*>(p.bias) +
                                                     min(n0 + 32 * j + 8 * g + 4 * hi, p.N - 4));
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = (short)Conv<TO>::from_f32(scaled_sum(acc[i][j][4 * g + r], sa[i], sb[j][g][r],
                                                        decltype(with_bias)::value ? Conv<TO>::to_f32((uint16_t)bias[r]) : 0.f));
          *reinterpret_cast<short4v*>(ol + l31 * kPitch + (32 * j + 8 * g + 4 * hi) * 2) = v;
        }
      __builtin_amdgcn_wave_barrier();  // the wave's own LDS rows: in order, no block barrier
      constexpr int kPer = 4 * NJ;      // 16-byte pieces per row
#pragma unroll
      for (int t = 0; t < 32 * kPer / 64; ++t) {
        const int piece = t * 64 + lane, row = piece / kPer, c = piece % kPer;
        const int4v v = *reinterpret_cast<const int4v*>(ol + row * kPitch + c * 16);
        const int m = m0 + 32 * i + row, n = n0 + c * 8;
        if (m < p.M && n < p.N)
          *reinterpret_cast<int4v*>(reinterpret_cast<uint16_t*>(p.out) + (int64_t)m * p.out_stride + n) = v;
      }
      __builtin_amdgcn_wave_barrier();
    }
  };
  if (p.bias)
    rows(std::true_type{});
  else
    rows(std::false_type{});
}

// 16 bytes twice: the operand of one matrix instruction, 64 bytes of row r from k-step ks on
__device__ __forceinline__ int8v fp8_operand(const char* rows, int r, int ks, int hi) {
  const char* row = rows + r * 128;
  const int4v x = *reinterpret_cast<const int4v*>(row + 16 * fp8_slot(r, 4 * ks + 2 * hi));
  const int4v y = *reinterpret_cast<const int4v*>(row + 16 * fp8_slot(r, 4 * ks + 2 * hi + 1));
  return int8v{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
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
      for (int j = 0; j < NJ; ++j) bf[j] = fp8_operand(bl, wn + 32 * j + l31, ks, hi);
#pragma unroll
      for (int i = 0; i < MI; ++i) af[i] = fp8_operand(al, wm + 32 * i + l31, ks, hi);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bf[j], af[i], acc[i][j], 0, 0, 0, 0, 0, 0);
    }
  }

  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  static_assert(NW * fp8_out_bytes(NJ) <= ST * kStage, "the stages hold the rows on their way out");
  fp8_tile_store<TO, MI, NJ>(p, acc, lds + wid * fp8_out_bytes(NJ), m0 + wm, n0 + wn, lane);
}

// The same product on four waves of 128 x (BN / 2) sums each, one a SIMD, 512 registers: an operand read from LDS serves four
// products where eight waves have it serve two to four.  Activations and weights have rings of their own, SA and SA + 1 stages
// deep: weights come from memory and are asked for a stage earlier (256 x 256 tiles of two whole stages: 4096 columns at 512 rows, an
// idle chip, 58 -> 44 us).  A stage's barrier lies between its two k-steps, when a wave holds the second one's operands; requests
// are spread one by one among the products, since all waves share one address unit (in pairs at the start of a half: a ninth more for
// 2048 x 28672 x 4096).
template <typename TO, int BN, int SA>
__device__ __forceinline__ void fp8_tile4(const Fp8TileArgs& p, char* lds, int m0, int n0) {
  constexpr int BM = 256, MI = 4, NJ = BN / 64, SB = SA + 1, kA = BM * 128, kB = BN * 128, kRingB = SA * kA;
  constexpr int NA = BM / 32, NB = BN / 32;  // requests (1 KiB, 8 rows) of a wave per stage
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l31 = lane & 31, hi = lane >> 5;
  const int nk = p.K / 128;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
  const uint8_t* const abase = p.a + (int64_t)m0 * p.a_stride;
  const uint8_t* const bbase = p.b + (int64_t)n0 * p.b_stride;
  uint32_t aoff[NA], boff[NB];
#pragma unroll
  for (int d = 0; d < NA; ++d) {  // rows past the end: the last one, never stored
    const int r = (wid * NA + d) * 8 + (lane >> 3);
    aoff[d] = (uint32_t)min(r, p.M - 1 - m0) * (uint32_t)p.a_stride + 16 * fp8_slot(r, lane & 7);
  }
#pragma unroll
  for (int d = 0; d < NB; ++d) {
    const int r = (wid * NB + d) * 8 + (lane >> 3);
    boff[d] = (uint32_t)min(r, p.N - 1 - n0) * (uint32_t)p.b_stride + 16 * fp8_slot(r, lane & 7);
  }
  auto dma = [&](uint32_t dst, uint32_t off, const uint8_t* src) {
    asm volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(src)
        : "memory", "m0");
  };
  // past the end: the last block again, so that the counted waits hold
  auto issue_a = [&](int kb, int at, int d) { dma(lds0 + at * kA + (wid * NA + d) * 1024, aoff[d], abase + (int64_t)min(kb, nk - 1) * 128); };
  auto issue_b = [&](int kb, int at, int d) {
    dma(lds0 + kRingB + at * kB + (wid * NB + d) * 1024, boff[d], bbase + (int64_t)min(kb, nk - 1) * 128);
  };

  const int wm = (wid >> 1) * 128, wn = (wid & 1) * (BN / 2);
  float16v acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  int8v af[2][MI], bf[2][NJ];
  auto product = [&](int t, int ks) {
    const int i = t / NJ, j = t % NJ;
    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bf[ks][j], af[ks][i], acc[i][j], 0, 0, 0, 0, 0, 0);
  };
  // the operands of a k-step, one behind each of the first products of the one before
  auto read_part = [&](int at_a, int at_b, int ks, int t) {
    if (t < NJ)
      bf[ks][t] = fp8_operand(lds + kRingB + at_b * kB, wn + 32 * t + l31, ks, hi);
    else if (t < NJ + MI)
      af[ks][t - NJ] = fp8_operand(lds + at_a * kA, wm + 32 * (t - NJ) + l31, ks, hi);
  };

#pragma unroll
  for (int i = 0; i < SA; ++i) {
#pragma unroll
    for (int d = 0; d < NB; ++d) issue_b(i, i, d);
#pragma unroll
    for (int d = 0; d < NA; ++d) issue_a(i, i, d);
  }
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((SA - 1) * (NA + NB)) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int t = 0; t < MI * NJ; ++t) read_part(0, 0, 0, t);
  int ia = 0, ib = 0, pb = SB - 1;  // slots of this stage, and of the weights of the stage before
  for (int kb = 0; kb < nk; ++kb) {
    const int na = ia + 1 == SA ? 0 : ia + 1, nb = ib + 1 == SB ? 0 : ib + 1;
#pragma unroll
    for (int t = 0; t < MI * NJ; ++t) {
      // into the slot that the stage before has left; evenly among the products, since four waves share one address unit
#pragma unroll
      for (int d = t * NB / (MI * NJ); d < (t + 1) * NB / (MI * NJ); ++d) issue_b(kb + SB - 1, pb, d);
      read_part(ia, ib, 1, t);
      product(t, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    // this wave holds the rest of the stage and its pieces of the next one have landed; behind the barrier everyone's have, and
    // this stage is free
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NB + (SA - 2) * (NA + NB)) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int t = 0; t < MI * NJ; ++t) {
#pragma unroll
      for (int d = t * NA / (MI * NJ); d < (t + 1) * NA / (MI * NJ); ++d) issue_a(kb + SA, ia, d);
      read_part(na, nb, 0, t);
      product(t, 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    ia = na;
    pb = ib;
    ib = nb;
  }

  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  static_assert(4 * fp8_out_bytes(NJ) <= SA * kA, "the stages hold the rows on their way out");
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // what depends on the lane is formed again: kept over the loop it would go out to memory
  fp8_tile_store<TO, MI, NJ>(p, acc, lds + wid * fp8_out_bytes(NJ), m0 + wm, n0 + wn, tid & 63);
}

// Strips of 256 columns, then narrower ones (`tail` columns) for what would be a last round that leaves units idle: 2048 x 28672
// in three rounds and one of half strips instead of four, an eighth less; 2048 x 6144 in one of 192 columns, a fifth
template <typename TO>
__global__ void __launch_bounds__(256, 1) fp8_tile4_kernel(Fp8TileArgs p) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int whole = p.mt * p.nt;
  const bool main = (int)blockIdx.x < whole;
  // a die takes a run of neighbouring tiles (all row tiles of a weight strip)
  const int total = main ? whole : p.mt * p.nt_tail, i = blockIdx.x - (main ? 0 : whole);
  const int q = total >> 3, rem = total & 7, xcd = i & 7;
  const int tile = xcd * q + min(xcd, rem) + (i >> 3);
  const int m0 = tile % p.mt * 256, strip = tile / p.mt;
  if (main)
    fp8_tile4<TO, 256, 2>(p, lds, m0, strip * 256);
  else if (p.tail == 192)
    fp8_tile4<TO, 192, 2>(p, lds, m0, p.nt * 256 + strip * 192);
  else
    fp8_tile4<TO, 128, 2>(p, lds, m0, p.nt * 256 + strip * 128);
}

}  // namespace sglk
