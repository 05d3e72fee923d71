// Products of many rows with 16-bit activations (gfx950): out[M, N] = x[M, K] @ W (+ bias), W as packed int4 words or as 16-bit rows.
//
// A block of four waves, one a SIMD with up to 512 registers, owns 64 MI rows and 64 NJ columns, a wave a quarter of them (32 MI x 32 NJ
// sums on v_mfma_f32_32x32x16), and walks K in stages of 64.  Rows (and 16-bit weights) arrive by LDS-DMA; int4 words go straight to
// registers, two k-blocks of 128 ahead, and leave them as finished 16-bit weights in LDS, each dequantised once for all rows of the
// block.  A stage's barrier lies between its halves: by then a wave holds the operands of the second half, so behind it the next
// stage's first operands are read, the stage after next's rows asked for and its weights written while products run.
//
// Bound: one wave's issue.  A half stage of 128 x 128 sums is 32 matrix instructions of 32 cycles, beside which a wave issues 100
// vector instructions for its weights, 20 for LDS and 10 requests, at 4 cycles each (8 for a matrix one): nothing may wait for the
// instruction before, and nothing may gather.  So a pair of weights takes three steps, one behind each second product, and the
// products are pinned where they stand.  2048 x 28672 x 4096, one card: 16-bit weights 374 us (1.29 PFLOP/s; the library 367), int4 395 (each
// step's instructions in a row: a twelfth more), where the library behind a dequantisation takes 381; 1152 rows 246 and 292.
#pragma once
#include <type_traits>

#include "common.h"

namespace sglk {

// acc += a . b.  PINNED: where the text stands.  Left to the compiler, products gather behind the requests and conversions that are
// to run under them.  The instruction itself is the compiler's, which knows how long its sums take: written out as text, a copy of an
// accumulator that it places behind one would read them too early.
template <typename T, bool PINNED>
__device__ __forceinline__ void prefill_mma(float16v& acc, int4v a, int4v b) {
  if constexpr (std::is_same<T, bf16_t>::value)
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bfloat8, a), __builtin_bit_cast(bfloat8, b), acc, 0, 0, 0);
  else
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), acc, 0, 0, 0);
  if constexpr (PINNED) asm volatile("" : "+a"(acc));
}

// two numbers, each rounded to nearest
template <typename T>
__device__ __forceinline__ int prefill_pair(float a, float b) {
  typedef float float2v __attribute__((ext_vector_type(2)));
  using H = typename std::conditional<std::is_same<T, bf16_t>::value, __bf16, _Float16>::type;
  typedef H pair __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(int, __builtin_convertvector(float2v{a, b}, pair));
}

struct PrefillArgs {
  const uint16_t* x;
  const void* w;  // packed words, or rows of K
  const uint16_t* scales;
  const int32_t* qzeros;
  const uint16_t* bias;
  uint16_t* out;
  int M, N, K, group_size;
  int64_t x_stride, w_stride, out_stride;
  int gated;                    // blocks of 64 columns alternate between gate and up: out = silu(gate) * up, N / 2 columns
  int mt, whole, tail, narrow;  // row tiles, strips of 256 columns, strips of `narrow` columns behind them
};

// 16-byte chunk c of a row's 128 bytes (64 numbers): 16 consecutive rows of one chunk lie in 16 different slots
__device__ __forceinline__ int pf_slot(int r, int c) { return c ^ ((r >> 1) & 7) ^ ((r & 1) << 2); }

template <typename T, bool AWQ, int MI, int NJ>
__device__ __forceinline__ void prefill_tile(const PrefillArgs& p, char* lds, int m0, int n0) {
  constexpr int BM = 64 * MI, BN = 64 * NJ, SA = 2, SB = AWQ ? 2 : 3, kA = BM * 128, kB = BN * 128;
  constexpr int kRingB = SA * kA, kSz = kRingB + SB * kB;
  constexpr int NA = BM / 32, NB = BN / 32;      // requests (1 KiB, 8 rows) of a wave per stage
  constexpr int SW = 2;  // k-blocks of weights in registers
  constexpr int P = 2 * MI * NJ, kOps = 2 * (MI + NJ);  // products and operands of half a stage
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l31 = lane & 31, hi = lane >> 5;
  const int nkb = p.K / 128, ns = 2 * nkb;  // a stage: 64 of K
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);

  // request j of a group of four, to dst + 1024 j: the instruction's offset moves both addresses, so `off` arrives lowered by
  // 1024 j against src, which is 3072 too low; the first of a group sets the LDS address for all
  auto dma = [&](int j, uint32_t dst, uint32_t off, const char* src) {
    if (j == 0)
      asm volatile(
          "s_mov_b32 m0, %0\n\t"
          "s_nop 0\n\t"
          "global_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(src)
          : "memory", "m0");
    else if (j == 1)
      asm volatile("global_load_lds_dwordx4 %0, %1 offset:1024" ::"v"(off), "s"(src) : "memory");
    else if (j == 2)
      asm volatile("global_load_lds_dwordx4 %0, %1 offset:2048" ::"v"(off), "s"(src) : "memory");
    else
      asm volatile("global_load_lds_dwordx4 %0, %1 offset:3072" ::"v"(off), "s"(src) : "memory");
  };
  // rows past the end: the last one, never stored; stages past the end: the last one again, so that the counted waits hold
  const char* const abase = reinterpret_cast<const char*>(p.x + (int64_t)m0 * p.x_stride) - 3072;
  uint32_t aoff[NA];
#pragma unroll
  for (int d = 0; d < NA; ++d) {
    const int r = (wid * NA + d) * 8 + (lane >> 3);
    aoff[d] = (uint32_t)min(r, p.M - 1 - m0) * (uint32_t)(2 * p.x_stride) + 16 * pf_slot(r, lane & 7) + 3072 - 1024 * (d % 4);
  }
  auto issue_a = [&](int s, int at, int d) { dma(d % 4, lds0 + at * kA + (wid * NA + d) * 1024, aoff[d], abase + (int64_t)min(s, ns - 1) * 128); };
  const char* const bbase = AWQ ? nullptr : reinterpret_cast<const char*>(p.w) + (int64_t)n0 * p.w_stride * 2 - 3072;
  uint32_t boff[AWQ ? 1 : NB];
  if constexpr (!AWQ)
#pragma unroll
    for (int d = 0; d < NB; ++d) {
      const int r = (wid * NB + d) * 8 + (lane >> 3);
      boff[d] = (uint32_t)min(r, p.N - 1 - n0) * (uint32_t)(2 * p.w_stride) + 16 * pf_slot(r, lane & 7) + 3072 - 1024 * (d % 4);
    }
  auto issue_b = [&](int s, int at, int d) {
    dma(d % 4, lds0 + kRingB + at * kB + (wid * NB + d) * 1024, boff[d], bbase + (int64_t)min(s, ns - 1) * 128);
  };

  // ---- int4: a wave dequantises NJ strips of 16 columns.  Strip t of k-block kb is 1 KiB; word d of lane (i, g) holds the eight
  // weights k = 32 d + 8 g .. + 7 of column i: a 16-byte chunk of that column's row.
  const int i16 = lane & 15, g4 = lane >> 4;
  const int first = n0 / 16 + wid * NJ, nstrips = p.N / 16;  // (strips past the last: the last one again)
  int4v wreg[SW][NJ];
  uint32_t woff[NJ];
#pragma unroll
  for (int t = 0; t < NJ; ++t) woff[t] = (uint32_t)min(first + t, nstrips - 1) * 1024 + lane * 16;
  auto load_w = [&](int kb, int set, int t) {
    const char* src = reinterpret_cast<const char*>(p.w) + (int64_t)min(kb, nkb - 1) * nstrips * 1024;
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(wreg[set][t]) : "v"(woff[t]), "s"(src) : "memory");
  };
  // scales and zeros of strip t lie behind those of the wave's first one.  Of 48 columns the last 16 or 32 may lie past N: their
  // lanes ask for nothing, and what is made of them is never stored.  A wave that has no column takes the last ones.
  const int col0 = first < nstrips ? first * 16 : p.N - 16 * NJ;
  const int live = min(NJ, nstrips - col0 / 16);
  auto load_sz = [&](int kb, int slot, int which) {
    const int gq = min(kb, nkb - 1) * 128 / p.group_size;
    const char* src = which == 0 ? reinterpret_cast<const char*>(p.scales + (int64_t)gq * p.N + col0)
                                 : reinterpret_cast<const char*>(p.qzeros + (int64_t)gq * (p.N / 8) + col0 / 8);
    const uint64_t mask = (1ull << (which == 0 ? 8 * live : 2 * live)) - 1;
    uint64_t saved;
    asm volatile(
        "s_mov_b32 m0, %1\n\t"
        "s_and_saveexec_b64 %0, %4\n\t"
        "global_load_lds_dword %2, %3\n\t"
        "s_mov_b64 exec, %0"
        : "=&s"(saved)
        : "s"(lds0 + kSz + (slot * 4 + wid) * 256 + which * 128), "v"(4 * lane), "s"(src), "s"(mask)
        : "memory", "m0", "scc");
  };
  float sc[NJ];
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
  half2v zh[NJ];  // 1024 + z twice
  uint32_t or_const = 0x64006400u, nib_mask = 0x000F000Fu;
  float minus_zero = -0.f;  // added, it changes nothing; a sum of products is what takes a half as it stands
  asm volatile("" : "+v"(or_const));
  asm volatile("" : "+s"(nib_mask));
  asm volatile("" : "+s"(minus_zero));
  uint32_t raw_s[NJ], raw_z[NJ];
  auto read_sz = [&](int slot) {
    const char* s = lds + kSz + (slot * 4 + wid) * 256;
#pragma unroll
    for (int t = 0; t < NJ; ++t) {
      raw_s[t] = *reinterpret_cast<const uint16_t*>(s + 2 * (16 * t + i16));
      raw_z[t] = *reinterpret_cast<const uint32_t*>(s + 128 + 4 * ((16 * t + i16) >> 3));
    }
  };
  const int zshift = 4 * (((i16 & 7) >> 1) + 4 * (i16 & 1));  // AWQ nibble order {0, 4, 1, 5, 2, 6, 3, 7}
  auto take_sz = [&]() {
#pragma unroll
    for (int t = 0; t < NJ; ++t) {
      sc[t] = Conv<T>::to_f32((uint16_t)raw_s[t]);
      zh[t] = __builtin_bit_cast(half2v, ((raw_z[t] >> zshift) & 0xF) * 0x10001u | 0x64006400u);
    }
  };
  const int bwrite = kRingB + (16 * NJ * wid + i16) * 128 + 16 * pf_slot(i16, g4);
  // Words n0w .. of the k-block in `set` (of 2 NJ a stage: strip n >> 1, d = 2 half + (n & 1)) into B slot `at`, a pair of weights a
  // step in three parts, one step apart, so that no instruction waits for the one before: step k begins pair k, multiplies pair k - 1
  // and rounds pair k - 2.  E pairs take E + 2 steps.
  constexpr int E = 4 * NJ;
  half2v begun;
  float part[2];
  int4v park;
  auto dequant = [&](int set, int half, int at, int n0w, int k) {
    if (k >= 2) {
      const int n = n0w + (k - 2) / 4, q = (k - 2) % 4;
      int word = prefill_pair<T>(part[0], part[1]);
      asm volatile("" : "+v"(word));  // here, not where it is written
      park[q] = word;
      if (q == 3) *reinterpret_cast<int4v*>(lds + at * kB + (bwrite ^ ((n & 1) << 6)) + (n >> 1) * 2048) = park;
    }
    if (k >= 1 && k <= E) {  // times the scale in fp32
      const int t = (n0w + (k - 1) / 4) >> 1;
#pragma unroll
      for (int e = 0; e < 2; ++e) part[e] = __builtin_fmaf((float)begun[e], sc[t], minus_zero);
      asm volatile("" : "+v"(part[0]), "+v"(part[1]));
    }
    if (k < E) {  // 1024 + nibble as a half, minus 1024 + z: exact
      const int n = n0w + k / 4;
      const uint32_t pair = (((uint32_t)wreg[set][n >> 1][2 * half + (n & 1)] >> (4 * (k % 4))) & nib_mask) | or_const;
      uint32_t v = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2v, pair) - zh[n >> 1]);
      asm volatile("" : "+v"(v));
      begun = __builtin_bit_cast(half2v, v);
    }
  };

  const int wm = (wid >> 1) * (32 * MI), wn = (wid & 1) * (32 * NJ);
  float16v acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  int4v af[2][2][MI], bf[2][2][NJ];
  const int arow = (wm + l31) * 128, brow = kRingB + (wn + l31) * 128;  // (32 rows on: the same slots)
  auto read_part = [&](int at_a, int at_b, int half, int f) {  // operand f of the half: k-step f / (MI + NJ)
    if (f >= kOps) return;
    const int k2 = f / (MI + NJ), u = f % (MI + NJ);
    const int c = 16 * pf_slot(l31, 2 * (2 * half + k2) + hi);
    if (u < NJ)
      bf[half][k2][u] = *reinterpret_cast<const int4v*>(lds + at_b * kB + brow + c + u * 4096);
    else
      af[half][k2][u - NJ] = *reinterpret_cast<const int4v*>(lds + at_a * kA + arow + c + (u - NJ) * 4096);
  };
  auto product = [&](int t, int half) {
    const int k2 = t / (MI * NJ), i = t / NJ % MI, j = t % NJ;
    prefill_mma<T, AWQ>(acc[i][j], bf[half][k2][j], af[half][k2][i]);
  };
  auto landed = [&](int set) {
#pragma unroll
    for (int t = 0; t < NJ; ++t) asm volatile("" : "+v"(wreg[set][t]));
  };

  // ---- prologue
  if constexpr (AWQ) {
#pragma unroll
    for (int t = 0; t < NJ; ++t) load_w(0, 0, t);
    load_sz(0, 0, 0);
    load_sz(0, 0, 1);
#pragma unroll
    for (int s = 0; s < SA; ++s)
#pragma unroll
      for (int d = 0; d < NA; ++d) issue_a(s, s, d);
#pragma unroll
    for (int kb = 1; kb < SW; ++kb) {
#pragma unroll
      for (int t = 0; t < NJ; ++t) load_w(kb, kb, t);
      load_sz(kb, kb, 0);
      load_sz(kb, kb, 1);
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(SA * NA + (SW - 1) * (NJ + 2)) : "memory");
    landed(0);
    read_sz(0);
    take_sz();
#pragma unroll
    for (int part3 = 0; part3 < 3; ++part3)  // the first stage, and the first half of the second one
#pragma unroll
      for (int k = 0; k < E + 2; ++k) dequant(0, part3 >> 1, part3 >> 1, part3 == 1 ? NJ : 0, k);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((SA - 1) * NA + (SW - 1) * (NJ + 2)) : "memory");
  } else {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int d = 0; d < NB; ++d) issue_b(s, s, d);
#pragma unroll
      for (int d = 0; d < NA; ++d) issue_a(s, s, d);
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NA + NB) : "memory");
  }
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int f = 0; f < kOps; ++f) read_part(0, 0, 0, f);

  int pb = 2;  // dense: B slots of the stage two on, of this one and of the next
  int ib = 0, ia = 0;  // slots of this stage
  for (int kb0 = 0; kb0 < nkb; kb0 += SW) {
#pragma unroll
    for (int u = 0; u < 2 * SW; ++u) {  // stages 2 kb0 + u
      const int s = 2 * kb0 + u, at = u & 1, half_k = u & 1, set = u >> 1;
      const int na = ia + 1 == SA ? 0 : ia + 1, nb = ib + 1 == SB ? 0 : ib + 1;
      const int this_b = AWQ ? at : ib, next_b = AWQ ? at ^ 1 : nb;
      const int later = (set + 1) % SW;
      if (u > 0 && half_k == 0 && kb0 + set >= nkb) break;
      // first half: what is left of the stage after next's weights (the k-block's other words), the second half's operands
#pragma unroll
      for (int t = 0; t < P; ++t) {
        if constexpr (!AWQ)
#pragma unroll
          for (int d = t * NB / P; d < (t + 1) * NB / P; ++d) issue_b(s + 2, pb, d);
        if constexpr (AWQ)
#pragma unroll
          for (int k = t * (E + 2) / P; k < (t + 1) * (E + 2) / P; ++k)
            dequant(half_k ? later : set, half_k ^ 1, at ^ 1, NJ, k);
        read_part(ia, this_b, 1, t);
        product(t, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      // the next stage's rows have landed (and, behind an even stage, the next k-block's weights); this wave holds the rest of the
      // stage, and its weights for the next one are written: behind the barrier this stage is free and that one whole
      if constexpr (AWQ) {
        if (half_k)
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NJ + 2) : "memory");
        else
          asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NB) : "memory");
      }
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if constexpr (AWQ)
        if (!half_k) {
          landed(later);
          read_sz(later);
        }
      // second half: rows of the stage after next, weights of the k-block after next, the first half of the stage after next's
      // weights dequantised, the next stage's first operands
      constexpr int kReqs = NA + (AWQ ? NJ + 2 : 0), kLate = P / 8;  // the new scales are on their way from LDS at first
      auto from = [&](int t, int odd) { return odd ? t * (E + 2) / P : t <= kLate ? 0 : (t - kLate) * (E + 2) / (P - kLate); };
#pragma unroll
      for (int t = 0; t < P; ++t) {
        const int reqs = half_k ? NA : kReqs;
#pragma unroll
        for (int d = t * reqs / P; d < (t + 1) * reqs / P; ++d) {
          if (d < NA)
            issue_a(s + SA, ia, d);
          else if (d < NA + NJ)
            load_w(kb0 + set + SW, set, d - NA);
          else
            load_sz(kb0 + set + SW, set, d - NA - NJ);
        }
        if (AWQ && !half_k && t == kLate) take_sz();
        if constexpr (AWQ)
#pragma unroll
          for (int k = from(t, half_k); k < from(t + 1, half_k); ++k) dequant(later, half_k, at, 0, k);
        read_part(na, next_b, 0, t);
        product(t, 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      pb = ib;
      ib = nb;
      ia = na;
    }
  }
  (void)pb;

  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < SW; ++i) landed(i);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // lane (m, hi) holds columns 32 j + 8 g + 4 hi + 0 .. 3 of row 32 i + m; rows leave through the wave's own LDS in whole pieces
  constexpr int kPitch = 64 * NJ + 16, kPer = 4 * NJ;
  static_assert(4 * 32 * kPitch <= SA * kA + SB * kB, "the stages hold the rows on their way out");
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // what depends on the lane is formed again: kept over the loop it would go out to memory
  const int ln = tid & 63, row31 = ln & 31, up = ln >> 5;
  char* ol = lds + (tid >> 6) * 32 * kPitch;
  auto rows = [&](auto kind) {  // 0: plain, 1: with a bias, 2: gated
    constexpr int kKind = decltype(kind)::value;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          short4v v, bias = {0, 0, 0, 0};
          if constexpr (kKind == 1)
            bias = *reinterpret_cast<const short4v*>(p.bias + min(n0 + wn + 32 * j + 8 * g + 4 * up, p.N - 4));
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = (short)Conv<T>::from_f32(acc[i][j][4 * g + r] + (kKind == 1 ? Conv<T>::to_f32((uint16_t)bias[r]) : 0.f));
          *reinterpret_cast<short4v*>(ol + row31 * kPitch + (32 * j + 8 * g + 4 * up) * 2) = v;
        }
      if constexpr (kKind == 2) {
        // the rounding points of the product followed by silu_and_mul; a wave of 128 columns holds a gate block and its up
        // block, of 64 columns one of them: there the two waves of a row take half the rows each
        if constexpr (NJ == 2)
          __syncthreads();
        else
          __builtin_amdgcn_wave_barrier();
        constexpr int kPieces = 32 * 8 / (NJ == 2 ? 2 : 1);
        const char* gl = NJ == 2 ? lds + ((tid >> 6) & ~1) * 32 * kPitch : ol;
        const char* ul = NJ == 2 ? gl + 32 * kPitch : ol + 128;
#pragma unroll
        for (int t = 0; t < kPieces / 64; ++t) {
          const int piece = t * 64 + ln + (NJ == 2 ? (tid >> 6 & 1) * kPieces : 0), row = piece >> 3, c = piece & 7;
          const short8 gate = *reinterpret_cast<const short8*>(gl + row * kPitch + c * 16);
          const short8 upper = *reinterpret_cast<const short8*>(ul + row * kPitch + c * 16);
          short8 o;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float x = Conv<T>::to_f32((uint16_t)gate[e]);
            const float sv = Conv<T>::to_f32(Conv<T>::from_f32(x / (1.0f + __expf(-x))));
            o[e] = (short)Conv<T>::from_f32(sv * Conv<T>::to_f32((uint16_t)upper[e]));
          }
          const int m = m0 + wm + 32 * i + row, n = n0 + (NJ == 2 ? 0 : wn);  // N % 256 == 0
          if (m < p.M && n < p.N) *reinterpret_cast<short8*>(p.out + (int64_t)m * p.out_stride + n / 2 + 8 * c) = o;
        }
        if constexpr (NJ == 2)
          __syncthreads();
        else
          __builtin_amdgcn_wave_barrier();
        continue;
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int t = 0; t < 32 * kPer / 64; ++t) {
        const int piece = t * 64 + ln, row = piece / kPer, c = piece % kPer;
        const int4v v = *reinterpret_cast<const int4v*>(ol + row * kPitch + c * 16);
        const int m = m0 + wm + 32 * i + row, n = n0 + wn + c * 8;
        if (m < p.M && n < p.N) *reinterpret_cast<int4v*>(p.out + (int64_t)m * p.out_stride + n) = v;
      }
      __builtin_amdgcn_wave_barrier();
    }
  };
  if constexpr (AWQ && NJ != 3)
    if (p.gated) return rows(std::integral_constant<int, 2>{});
  if (p.bias)
    rows(std::integral_constant<int, 1>{});
  else
    rows(std::integral_constant<int, 0>{});
}

template <typename T, bool AWQ, int MI>
__global__ void __launch_bounds__(256, 1) prefill_tile_kernel(PrefillArgs p) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int whole = p.mt * p.whole;
  const bool main = (int)blockIdx.x < whole;
  // a die takes a run of neighbouring tiles (all row tiles of a weight strip)
  const int total = main ? whole : p.mt * p.tail, i = blockIdx.x - (main ? 0 : whole);
  const int q = total >> 3, rem = total & 7, xcd = i & 7;
  const int tile = xcd * q + min(xcd, rem) + (i >> 3);
  const int m0 = tile % p.mt * (64 * MI), strip = tile / p.mt;
  if (main)
    prefill_tile<T, AWQ, MI, 4>(p, lds, m0, strip * 256);
  else if (p.narrow == 192)
    prefill_tile<T, AWQ, MI, 3>(p, lds, m0, p.whole * 256 + strip * 192);
  else
    prefill_tile<T, AWQ, MI, 2>(p, lds, m0, p.whole * 256 + strip * 128);
}

}  // namespace sglk
