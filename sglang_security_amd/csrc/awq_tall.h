// Fused int4 GEMM for more than 64 rows (gfx950): the wide kernel's arithmetic (awq.hip) on blocks of 96 or 128 rows.
//
// Eight waves, two a SIMD: two 64-column chunks x four 128-k groups; a stage is 512 k, in two halves of 64 k a group.  A wave
// multiplies its 64 columns by ALL rows of the block, so a weight is fetched and dequantised once for 128 rows instead of once
// for 64: 112 + 128 vector instructions (dequantisation, change of unit) beside 72 matrix instructions of 32 cycles a group,
// where the wide kernel has 112 + 64 beside 36.
//
//   x  : half a stage = 4 tiles of 32 RT rows x 64 k by LDS-DMA, two halves;
//   sz : per wave and stage one 256-byte LDS-DMA piece (scale pairs + zero words), two stages;
//   w  : 4 x 16 bytes per lane straight into registers, requested a whole stage ahead (two register sets);
//   X  : block sums of x, from the producer of x by LDS-DMA, or formed here from the operands on their way to the matrix unit.
//
// A barrier each half, before its last k-step: by then a wave holds that k-step's operands, so behind the barrier the half's
// buffer is free for the next stage's and the other half's rows are there, while products are left to issue.  In the last k-step of a
// stage a row tile's products are followed by its change to the next group's unit, under the products of the tile after it.
//
// With the producer's sums a group begins with its zero-point term, as in the wide kernel, and whole sums are that kernel's to the bit,
// those left for the next product too.  Sums formed here are there only behind the group's last k-step, and so is its term.
#pragma once
#include "awq_common.h"

namespace sglk {

struct AwqTallArgs {
  const uint16_t* x;
  const int32_t* packed;
  const uint16_t* scales;
  const int32_t* qzeros;
  const uint16_t* bias;
  uint16_t* out;
  float* partial;
  int* tickets;
  const float* xsum_in;
  float* xsum_out;
  int64_t x_stride, out_stride, xs_stride, xs_out_stride;
  int M, N, K, stages_per_split, splits, act_mode;
  int wide_out;  // act_mode: out rows take 16-byte stores
};

static constexpr int64_t kTallMaxStride = 1 << 24;  // elements from row to row: 128 rows stay below 2^32 bytes

struct TallPlan {
  bool ok;
  int rt, tiles, splits, stages_per_split, mblocks;
};
// gated: the gated activation behind the product (whole sums in one block), else finished rows; sums: with the block sums of x;
// slab_bytes: room for the sums of a split product
TallPlan plan_awq_tall(int M, int N, int K, int group_size, int dtype, bool gated, bool sums, int64_t slab_bytes = 0);
int launch_awq_tall(const TallPlan& p, AwqTallArgs a, hipStream_t s);
int prepare_awq_tall();

struct AwqTall {
  static constexpr int kStageK = 512;
  static constexpr int kSz = 2 * 8 * 256, kXs = 2 * 8 * 128 * 4;
  static constexpr int x_half(int rt) { return 4 * rt * 32 * 128; }
  static constexpr int lds(int rt) { return 2 * x_half(rt) + kSz + kXs + 16; }
};

template <bool XS, int RT>
__global__ void __launch_bounds__(512, 2) awq_tall_kernel(AwqTallArgs a) {
  using T = bf16_t;
  constexpr int kX = AwqTall::x_half(RT), kSzOff = 2 * kX, kXsOff = kSzOff + AwqTall::kSz;
  constexpr int kRest = 6 + (XS ? 2 : 0);  // requests of a stage that are younger than its second half of x
  extern __shared__ __attribute__((aligned(16))) char smem[];
  int* flag = reinterpret_cast<int*>(smem + kXsOff + AwqTall::kXs);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw = wid & 3, nw = wid >> 2;
  const int i16 = lane & 15, r32 = lane & 31, h = lane >> 5;
  const int m0 = blockIdx.z * 32 * RT, n0 = blockIdx.x * 128 + nw * 64;
  const int st0 = blockIdx.y * a.stages_per_split;
  const int nst = min(a.stages_per_split, a.K / AwqTall::kStageK - st0);
  const int64_t nstrips = a.N / 16;
  const int qcols = a.N / 8;

  // ---- requests; those past the split's end go out with every lane switched off, so the counted waits hold for every stage
  auto live_mask = [&](int stage) -> uint64_t {
    const uint32_t c = (uint32_t)__builtin_amdgcn_readfirstlane(stage < nst ? -1 : 0);
    uint64_t m = ((uint64_t)c << 32) | c;
    asm volatile("" : "+s"(m));
    return m;
  };
  auto lds_address = [&](const char* p) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p);
  };
  // x: a wave fills half a tile, piece j = rows 16 RT (wid & 1) + 8 j + 0 .. 7; 16-byte chunk c of row r in slot c ^ (r >> 1 & 7).
  // Offsets are formed anew for every request: kept, they would push other registers out to memory.
  const int xlast = min(32 * RT, a.M - m0) - 1;  // rows past it: that one again
  const uint32_t xpitch = (uint32_t)(2 * a.x_stride), xend = xlast * xpitch;  // 32 RT rows span less than 2^32 bytes
  const uint32_t xfirst = (16 * RT * (wid & 1) + (lane >> 3)) * xpitch;
  const char* const xbase = reinterpret_cast<const char*>(a.x + (int64_t)m0 * a.x_stride + 128 * (wid >> 1)) - 1024;
  uint32_t xchunk[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) xchunk[j] = 16 * ((lane & 7) ^ ((lane >> 4) + 4 * j)) + 1024 - 1024 * j;
  auto issue_x = [&](int stage, int half) {
    const char* src = xbase + ((int64_t)(st0 + min(stage, nst - 1)) * AwqTall::kStageK + 64 * half) * 2;
    const uint32_t dst = lds_address(smem + half * kX + wid * 2 * RT * 1024);
    const uint64_t live = live_mask(stage);
    uint32_t at = xfirst;
    asm volatile("" : "+v"(at));
#pragma unroll
    for (int q = 0; q < RT; ++q) {
      uint64_t saved;
      uint32_t off[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) off[j] = min(at + (uint32_t)(16 * q + 8 * j) * xpitch, xend) + xchunk[j];
      asm volatile(
          "s_mov_b32 m0, %1\n\t"
          "s_and_saveexec_b64 %0, %5\n\t"
          "global_load_lds_dwordx4 %2, %4\n\t"
          "global_load_lds_dwordx4 %3, %4 offset:1024\n\t"
          "s_mov_b64 exec, %0"
          : "=&s"(saved)
          : "s"(dst + q * 2048), "v"(off[0]), "v"(off[1]), "s"(src), "s"(live)
          : "memory", "m0", "scc");
    }
  };
  const uint32_t wvoff = (uint32_t)((((int64_t)kw * nstrips + (n0 >> 4) + (r32 >> 4)) * 64 + i16 + 16 * h) * 16);
  int4v wreg[2][4];
  auto issue_rest = [&](int stage, int set) {  // scales and zeros, weights, block sums
    const int at = st0 + min(stage, nst - 1);
    const int gq = at * 4 + kw;
    const uint64_t live = live_mask(stage);
    uint64_t saved;
    uint32_t lane4 = 4 * lane;
    asm volatile("" : "+v"(lane4));
    asm volatile(  // 32 scale pairs of the wave's 64 columns, 8 zero words behind them
        "s_mov_b32 m0, %1\n\t"
        "s_and_saveexec_b64 %0, %5\n\t"
        "global_load_lds_dword %2, %3\n\t"
        "s_mov_b64 exec, %6\n\t"
        "s_add_u32 m0, m0, 128\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dword %2, %4\n\t"
        "s_mov_b64 exec, %0"
        : "=&s"(saved)
        : "s"(lds_address(smem + kSzOff + (set * 8 + wid) * 256)), "v"(lane4), "s"(a.scales + (int64_t)gq * a.N + n0),
          "s"(a.qzeros + (int64_t)gq * qcols + (n0 >> 3)), "s"(live & 0xFFFFFFFFu), "s"(live & 0xFFu)
        : "memory", "m0", "scc");
    const char* src = reinterpret_cast<const char*>(a.packed) + (int64_t)at * 4 * nstrips * 1024;
    asm volatile(
        "s_and_saveexec_b64 %4, %7\n\t"
        "global_load_dwordx4 %0, %5, %6\n\t"
        "global_load_dwordx4 %1, %5, %6 offset:512\n\t"
        "global_load_dwordx4 %2, %5, %6 offset:2048\n\t"
        "global_load_dwordx4 %3, %5, %6 offset:2560\n\t"
        "s_mov_b64 exec, %4"
        : "=&v"(wreg[set][0]), "=&v"(wreg[set][1]), "=&v"(wreg[set][2]), "=&v"(wreg[set][3]), "=&s"(saved)
        : "v"(wvoff), "s"(src), "s"(live)
        : "memory", "scc");
    if constexpr (XS) {
      const float* xs = a.xsum_in + (int64_t)gq * a.xs_stride + m0;
      asm volatile(
          "s_mov_b32 m0, %1\n\t"
          "s_and_saveexec_b64 %0, %5\n\t"
          "global_load_lds_dword %2, %4\n\t"
          "s_add_u32 m0, m0, 256\n\t"
          "s_nop 0\n\t"
          "global_load_lds_dword %3, %4\n\t"
          "s_mov_b64 exec, %0"
          : "=&s"(saved)
          : "s"(lds_address(smem + kXsOff + (set * 8 + wid) * 512)), "v"(min(lane4, 4u * xlast)),
            "v"(min(lane4 + 256, 4u * xlast)), "s"(xs), "s"(live)
          : "memory", "m0", "scc");
    }
  };

  // R[ct][rt]: running sums in units of the current group's scale (see wide_body)
  float16v R[2][RT];
#pragma unroll
  for (int ct = 0; ct < 2; ++ct)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int e = 0; e < 16; ++e) R[ct][rt][e] = 0.f;
  float s_cur[2] = {1.f, 1.f};
  const int zsh = 4 * (((r32 & 7) >> 1) + 4 * (r32 & 1));
  uint32_t or_const = AwqMagic<T>::kOr, nib_mask = 0x000F000Fu;
  asm volatile("" : "+v"(or_const));
  asm volatile("" : "+s"(nib_mask));
  uint32_t orc[2] = {or_const, or_const};
  uint32_t bz[2];  // -(OFF + z), the zero-point k-step's B operand (0: this group adds nothing)
  struct Unit {
    uint32_t scale[2], zeros[2];
  };
  auto read_unit = [&](int slot, Unit& un) {  // scales and zeros of a stage (after its wait)
    const char* szp = smem + kSzOff + (slot * 8 + wid) * 256;
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      un.scale[ct] = *reinterpret_cast<const uint16_t*>(szp + 2 * (32 * ct + r32));
      un.zeros[ct] = *reinterpret_cast<const uint32_t*>(szp + 128 + 4 * ((32 * ct + r32) >> 3));
    }
  };
  // The factors that take R to the new unit.  A zero (or denormal) scale cannot become the unit: the column keeps its own and
  // this group adds nothing to it.  `none`: no such stage.
  auto prep = [&](const Unit& un, bool none, int set, float(&ratio)[2]) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      const float s_in = Conv<T>::to_f32((uint16_t)un.scale[ct]);
      const bool skip = none || !(fabsf(s_in) >= 1.17549435e-38f);
      const float sg = skip ? s_cur[ct] : s_in;
      ratio[ct] = none ? 1.f : s_cur[ct] * __builtin_amdgcn_rcpf(sg);
      s_cur[ct] = sg;
      const uint32_t z = (un.zeros[ct] >> zsh) & 0xF;
      orc[ct] = skip ? 0u : or_const;
      if (__builtin_expect(__any(skip), 0)) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int d = 0; d < 4; ++d) wreg[set][2 * ct + j][d] = skip ? 0 : wreg[set][2 * ct + j][d];
      }
      const uint32_t nzb = ((AwqMagic<T>::kOr & 0xFFFFu) | 0x8000u) | z;
      bz[ct] = !skip && h == 0 ? nzb : 0;  // k-slots 0..2 belong to the lower half-wave
    }
  };
  // A operand of k-step s: 16 bytes at row 32 rt + r, chunk 2 (s & 3) + h of this wave's tile of half s >> 2
  const int abase = kw * RT * 4096 + r32 * 128 + ((h ^ ((r32 >> 1) & 7)) << 4);
  auto read_a = [&](int s, int4v(&af)[RT]) {
    const char* p = smem + (s >> 2) * kX + (abase ^ ((s & 3) << 5));
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) af[rt] = *reinterpret_cast<const int4v*>(p + rt * 4096);
  };
  auto dequant = [&](int set, int s, int4v(&bf)[2]) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
      const uint32_t w = (uint32_t)wreg[set][2 * ct + (s & 1)][s >> 1];
#pragma unroll
      for (int e = 0; e < 4; ++e) bf[ct][e] = (int)(((w >> (4 * e)) & nib_mask) | orc[ct]);
    }
  };
  auto change_unit = [&](int rt, const float(&ratio)[2]) {
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) {
#pragma unroll
      for (int e = 0; e < 16; ++e) R[ct][rt][e] *= ratio[ct];
      asm volatile("" : "+v"(R[ct][rt]));  // here, not where the next product needs it
    }
  };
  // R + (a + b + c) bz, X = a + b + c exactly, three values of the operand type
  auto zero_point = [&](int rt, float X, const uint32_t(&z)[2]) {
    const uint32_t xa = __float_as_uint(X) & 0xFFFF0000u;
    const float r1 = X - __uint_as_float(xa);
    const uint32_t xb = __float_as_uint(r1) & 0xFFFF0000u;
    const float r2 = r1 - __uint_as_float(xb);
    const int4v ax = int4v{(int)((xa >> 16) | xb), (int)(__float_as_uint(r2) >> 16), 0, 0};
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
      R[ct][rt] = AwqMagic<T>::mma32(ax, int4v{(int)(z[ct] * 0x10001u), (int)z[ct], 0, 0}, R[ct][rt]);
  };
  auto given_sum = [&](int slot, int rt) {
    return reinterpret_cast<const float*>(smem + kXsOff + (slot * 8 + wid) * 512)[32 * rt + r32];
  };
  float xacc[RT];  // this lane's part of the block sums of the group (without XS)
  auto add_sums = [&](const int4v(&af)[RT]) {
    if constexpr (!XS)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int e = 0; e < 4; ++e) xacc[rt] = AwqMagic<T>::pair_sum((uint32_t)af[rt][e], xacc[rt]);
  };
  auto barrier = [&]() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // ---- prologue
  issue_rest(0, 0);
  issue_x(0, 0);
  issue_x(0, 1);
  issue_rest(1, 1);
  asm volatile("s_waitcnt vmcnt(%4)"
               : "+v"(wreg[0][0]), "+v"(wreg[0][1]), "+v"(wreg[0][2]), "+v"(wreg[0][3])
               : "n"(kRest + 2 * RT)
               : "memory");
  barrier();
  int4v af[2][RT], bf[2][2];
  float ratio[2];
  Unit un;
  read_unit(0, un);
  prep(un, false, 0, ratio);
  read_a(0, af[0]);
  dequant(0, 0, bf[0]);
  if constexpr (XS)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) zero_point(rt, given_sum(0, rt), bz);

  const int npad = (nst + 1) / 2 * 2;
  for (int i0 = 0; i0 < npad; i0 += 2) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i = i0 + u;
      const bool last = i + 1 >= nst;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) xacc[rt] = 0.f;
#pragma unroll
      for (int s = 0; s < 7; ++s) {
        __builtin_amdgcn_sched_barrier(0);
        if (s == 3) {  // the other half's rows are there, nobody reads this half's any more
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kRest) : "memory");
          barrier();
          issue_x(i + 1, 0);
        }
        read_a(s + 1, af[(s + 1) & 1]);
        dequant(u, s + 1, bf[(s + 1) & 1]);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int ct = 0; ct < 2; ++ct) R[ct][rt] = AwqMagic<T>::mma32(af[s & 1][rt], bf[s & 1][ct], R[ct][rt]);
        add_sums(af[s & 1]);
        // an operand read and two vector instructions behind every matrix instruction
#pragma unroll
        for (int q = 0; q < 2 * RT; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, XS ? 2 : 5, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      add_sums(af[1]);
      float X[RT];
      if constexpr (!XS)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) X[rt] = xacc[rt] + __shfl_xor(xacc[rt], 32, 64);
      // everything has landed: the next stage's first half, its weights, scales and sums
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)"
                   : "+v"(wreg[u ^ 1][0]), "+v"(wreg[u ^ 1][1]), "+v"(wreg[u ^ 1][2]), "+v"(wreg[u ^ 1][3])::"memory");
      barrier();
      issue_x(i + 1, 1);
      issue_rest(i + 2, u);
      read_unit(u ^ 1, un);
      if constexpr (XS)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) X[rt] = last ? 0.f : given_sum(u ^ 1, rt);
      const uint32_t bzo[2] = {bz[0], bz[1]};
      int4v na[RT], nb[2];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) R[ct][rt] = AwqMagic<T>::mma32(af[1][rt], bf[1][ct], R[ct][rt]);
        if constexpr (!XS) zero_point(rt, X[rt], bzo);
        na[rt] = *reinterpret_cast<const int4v*>(smem + abase + rt * 4096);
        if (rt == 0) {
          prep(un, last, u ^ 1, ratio);
        } else {
          change_unit(rt - 1, ratio);
          if constexpr (XS) zero_point(rt - 1, X[rt - 1], bz);
        }
        if (rt == RT - 1) dequant(u ^ 1, 0, nb);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, XS ? 18 : 9, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      change_unit(RT - 1, ratio);
      if constexpr (XS) zero_point(RT - 1, X[RT - 1], bz);
      if (last) goto done;
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) af[0][rt] = na[rt];
      bf[0][0] = nb[0], bf[0][1] = nb[1];
    }
  }
done:
  // nothing may land in the stages any more (requests past the end fetch nothing)
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  barrier();

  // ---- the four k-waves of a column chunk, a column tile at a time: wave kw finishes row tile kw
  float4v* red = reinterpret_cast<float4v*>(smem);  // [wave][rt][j][lane]
  float4v fin[2][4];
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    if (ct) __syncthreads();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float4v v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = R[ct][rt][4 * j + e] * s_cur[ct];
        red[((wid * RT + rt) * 4 + j) * 64 + lane] = v;
      }
    __syncthreads();
    if (kw < RT)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        fin[ct][j] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) fin[ct][j] += red[(((4 * nw + k2) * RT + kw) * 4 + j) * 64 + lane];
      }
  }
  // lane (r, h) of a wave kw < RT now holds rows 32 kw + e + 8 j + 4 h of columns 128 bx + 64 nw + 32 ct + r
  if (a.act_mode) {
    // The first 64 columns are gate columns, the last 64 the matching up columns (see wide_body): wave nw forms the
    // activation of column tile nw and hands the other one's numbers over.
    constexpr int kOutPitch = 64 * 2 + 16;
    float4v* ex = red;  // [wave][j][lane]
    char* tile = reinterpret_cast<char*>(ex + 8 * 4 * 64);
    static_assert(8 * 4096 + 32 * RT * kOutPitch <= 2 * kX, "the stages hold the epilogue");
    __syncthreads();
    if (kw < RT)
#pragma unroll
      for (int j = 0; j < 4; ++j) ex[(wid * 4 + j) * 64 + lane] = nw ? fin[0][j] : fin[1][j];
    __syncthreads();
    if (kw < RT)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4v o = ex[((wid ^ 4) * 4 + j) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float gb = Conv<T>::to_f32(Conv<T>::from_f32(nw ? o[e] : fin[0][j][e]));
          const float ub = Conv<T>::to_f32(Conv<T>::from_f32(nw ? fin[1][j][e] : o[e]));
          const float sv = Conv<T>::to_f32(Conv<T>::from_f32(gb / (1.0f + __expf(-gb))));
          *reinterpret_cast<uint16_t*>(tile + (32 * kw + e + 8 * j + 4 * h) * kOutPitch + 2 * (32 * nw + r32)) =
              Conv<T>::from_f32(sv * ub);
        }
      }
    __syncthreads();
    // Four threads a row, 8 of every 16 columns each: its pieces, and its sum for the next product's zero-point term, in the wide
    // kernel's order (a column tile's numbers 16, 8, 4, 2 and 1 apart, then the two tiles)
    const int row = tid >> 2, ctile = tid >> 1 & 1, odd = tid & 1;
    if (row < 32 * RT && m0 + row < a.M) {
      const int at = 32 * ctile + 8 * odd;
      const char* src = tile + row * kOutPitch + 2 * at;
      uint16_t* dst = a.out + (int64_t)(m0 + row) * a.out_stride + blockIdx.x * 64 + at;
      float sum[8];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int4v v = *reinterpret_cast<const int4v*>(src + 32 * c);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint16_t o = (uint16_t)((uint32_t)v[e >> 1] >> (16 * (e & 1)));
          sum[e] = c ? sum[e] + Conv<T>::to_f32(o) : Conv<T>::to_f32(o);
          if (!a.wide_out) dst[16 * c + e] = o;
        }
        if (a.wide_out) *reinterpret_cast<int4v*>(dst + 16 * c) = v;
      }
      if (a.xsum_out) {
#pragma unroll
        for (int e = 0; e < 8; ++e) sum[e] += __shfl_xor(sum[e], 1, 64);
#pragma unroll
        for (int d = 4; d > 0; d >>= 1)
#pragma unroll
          for (int e = 0; e < d; ++e) sum[e] += sum[e + d];
        sum[0] += __shfl_xor(sum[0], 2, 64);
        if ((tid & 3) == 0) atomicAdd(&a.xsum_out[(int64_t)(blockIdx.x >> 1) * a.xs_out_stride + m0 + row], sum[0]);
      }
    }
    return;
  }
  const int n = n0 + r32;
  const int mrow = m0 + 32 * kw + 4 * h;
  if (a.splits > 1) {
    // slabs and tickets as in wide_body
    constexpr int kTile = 32 * RT * 128;
    const int tile = (int)(blockIdx.z * gridDim.x + blockIdx.x);
    float* const tslab = a.partial + (int64_t)tile * a.splits * kTile;
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(tslab, 0, a.splits * kTile * 4, 0x00020000);
    constexpr int kSc1 = 16;
    const int voff = ((nw * RT + kw) * 8 * 64 + lane) * 16;
    if (kw < RT)
#pragma unroll
      for (int ct = 0; ct < 2; ++ct)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, fin[ct][j]), rsrc, voff + (ct * 4 + j) * 1024,
                                                 blockIdx.y * kTile * 4, kSc1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (tid == 0) {
      const int ticket = __hip_atomic_fetch_add(&a.tickets[tile], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int is_last = ticket == a.splits - 1;
      if (is_last) __hip_atomic_store(&a.tickets[tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *flag = is_last;
    }
    __syncthreads();
    if (*flag == 0 || kw >= RT) return;
#pragma unroll
    for (int ct = 0; ct < 2; ++ct)
#pragma unroll
      for (int j = 0; j < 4; ++j) fin[ct][j] = float4v{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < a.splits; s0 += 2) {  // two slabs asked for at a time
      float4v v[2][2][4];
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            v[q][ct][j] = __builtin_bit_cast(
                float4v, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff + (ct * 4 + j) * 1024,
                                                               min(s0 + q, a.splits - 1) * kTile * 4, kSc1));
#pragma unroll
      for (int q = 0; q < 2; ++q)
        if (s0 + q < a.splits)
#pragma unroll
          for (int ct = 0; ct < 2; ++ct)
#pragma unroll
            for (int j = 0; j < 4; ++j) fin[ct][j] += v[q][ct][j];
    }
  }
  if (kw >= RT) return;
#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
    const float bv = a.bias ? Conv<T>::to_f32(a.bias[n + 32 * ct]) : 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = mrow + 8 * j + e;
        if (m < a.M) a.out[(int64_t)m * a.out_stride + n + 32 * ct] = Conv<T>::from_f32(fin[ct][j][e] + bv);
      }
  }
}

}  // namespace sglk
