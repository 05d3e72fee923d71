// Absorbed latent decode over 576-element rows (the first 512 are the values), 32 query heads or more a latent head (gfx950).
//
// A block owns a tile of 32 query heads of one request and walks its tokens with four waves that do not wait for each other:
// a wave takes every fourth tile of 16 tokens through two LDS stages of its own (LDS-DMA, counted waits, no block barrier),
// holds the whole queries (144 registers) and all 512 output rows of its 32 heads (256 accumulators), and the four states meet
// once, at the end.  S^T = K . Q^T on 16x16x32; two half-row exchanges turn the rounded probabilities into the operand of
// O^T += V^T . P^T on 32x32x16.
//
// Bound: a tile is 1600 cycles of a SIMD's matrix unit (36 products of 16 and, with probabilities in two parts, 32 of 32) and, for the
// four waves, 1088 of operand reads; a wave alone on its SIMD gets to 2900 a tile.  A block's start (plan, queries, slots: 6000
// cycles) and end (256 KiB through the LDS: 7500) are the rest.  Blocks of a request read the same rows, so they sit on one die.
// The kernel before dealt the k-steps of a 32-token tile to four waves, which met at three block barriers a tile, and left partials
// of every split in memory.  Measured (bf16, 128 heads, calls with the pool's write and the merge, replayed over the same rows,
// which stay in the cache behind the dies), before -> now: 64 requests of 43 to 64 / 768 to 1152 / 2731 to 4096 tokens 27.2 / 71.2 / 191 -> 16.2
// / 43.6 / 115 us; 32 of them 18.0 / 46.0 / 103 -> 13.4 / 38.9 / 82; 16 of the longest 62 -> 49.
//
// The maximum may lag far behind the scores (rescaling 256 accumulators costs more than a tile's products).  A probability is then
// rounded wherever it falls, and not against a largest one of exactly 1: with one 16-bit number a probability the rows were
// 0.00210 off the 64-bit result (64 requests of 768 to 1152 tokens; the kernel before 0.00204), so it is carried as the sum of two
// (0.00166, what rounding the result leaves).
#pragma once
#include <algorithm>
#include <type_traits>

#include "attention_mla.h"
#include "extend_tile.h"

namespace sglk {

static constexpr int kMinBlockKV = 32;  // decode_attention.py:40 (_MIN_BLOCK_KV)

__host__ __device__ __forceinline__ int cdiv_i(int a, int b) { return (a + b - 1) / b; }

// How many ways request b's context is split: as the caller says, or, where `fewer` names a number for that many and a batch
// of such a mean context (64 tokens and up, by powers of two), as it says (mla_fewer_splits).  A request twice as long as
// the mean keeps what it was given: alone in the last round, it would end the launch.
constexpr int kMeans = 7;
struct FewerSplits {
  int batch;  // 0: always as the caller says
  uint64_t pick[kMeans];  // four bits a number of splits, 1 .. 16; 0: as the caller says
};
__device__ __forceinline__ int splits_of(int given, int total, int len, int max_splits, const FewerSplits& fewer) {
  const int most = max(given, 1);
  if (fewer.batch == 0 || most > min(max_splits, 16)) return most;  // (fewer: fewer than 2^20 requests)
  uint64_t picks = fewer.pick[0];
#pragma unroll
  for (int k = 1; k < kMeans; ++k) picks = (uint32_t)total < (uint32_t)(64 << k) * (uint32_t)fewer.batch ? picks : fewer.pick[k];
  const int n = (int)(picks >> (4 * (most - 1))) & 15;
  return total < 64 * fewer.batch || (uint64_t)len * (uint32_t)fewer.batch > 2 * (uint64_t)total || n == 0 ? most : n;
}

struct LatentArgs {
  const uint16_t *q, *kv;
  const int32_t *kv_indptr, *kv_indices, *num_kv_splits, *gate;
  float *part, *lse;  // [B, Hq, max_splits, 512] and [B, Hq, max_splits]
  void* o;
  int B, Hq, Hkv, head_tiles, group, max_splits;
  int direct, units;  // of a head tile: blocks that every request has a place for, places (latent_places)
  float per_b;        // 1 / B
  int64_t q_sb, q_sh, k_sn, k_sh, o_sb, o_sh;
  float sm_scale, logit_cap;
};

constexpr int kLatTok = 16;                          // tokens per tile
constexpr int kLatTile = kLatTok * kMlaD * 2;        // 18432 bytes: two halves of 8 rows, each nine 1-KiB pieces of 8 x 128 bytes
constexpr int kLatTurn = 4 * kLatTok;                 // tokens of a tile for each of a block's waves
constexpr int kLatFold = 8;                          // most splits a block folds
constexpr int kLatRing = 4 * 2 * kLatTile;           // 147456
static_assert(32 * 1088 <= 2 * kLatTile, "a wave's 256 output rows fit its ring");
constexpr int kLatState = 4 * 32 * 8;                // a maximum and a sum per wave and head
constexpr int kLatLds = kLatRing + (kLatFold + 1) * kLatState + 4 * 1024;  // and a corner a wave: 160768

// How a request's splits fall to blocks.  A split is what the caller's partials are counted in (each leaves its log-sum-exp);
// a block folds neighbouring ones: there are 256 units for one block each, and a second round of blocks costs a start and an
// end (8 us), so a request gets its share of 256 by its tokens (rounded down where it is short: the longest block then walks
// little more, and a block less has its rows merged), and a block 64 tokens where there are as many.
struct LatentPlan {
  int start, len, per, live, fold, blocks;
};
// Blocks a request would have, whatever the splits.  (The share is a rounded number before anything is added to it: block and merge
// kernel have to agree to the last bit.)
__device__ __forceinline__ int latent_share(const LatentArgs& a, int len, int total) {
  float share = 256.f * (float)len * __builtin_amdgcn_rcpf((float)max(total, 1) * (float)(a.Hkv * a.head_tiles));
  asm("" : "+v"(share));
  return max(min((int)fminf(share + (len >= 512 ? 0.4f : 0.01f), 65536.f), len / kLatTurn), 1);
}
__device__ __forceinline__ LatentPlan latent_plan(const LatentArgs& a, int b, const FewerSplits& fewer) {
  // (five loads that wait for nothing but the arguments: one trip; a division is 200 cycles on the way to the first request)
  const int first = a.kv_indptr[0], begin = a.kv_indptr[b], end = a.kv_indptr[b + 1], last = a.kv_indptr[a.B], given = a.num_kv_splits[b];
  LatentPlan p;
  p.start = begin;
  p.len = end - begin;
  const int blocks = latent_share(a, p.len, last - first), n = splits_of(given, last - first, p.len, a.max_splits, fewer);
  p.per = cdiv_i(n == 1 ? p.len : cdiv_i(p.len, n), kMinBlockKV) * kMinBlockKV;
  p.live = p.len > 0 ? min(n == 1 ? 1 : cdiv_i(p.len, p.per), a.max_splits) : 0;  // (slots for more there are not)
  p.fold = 1;
  p.blocks = p.live;
  if (p.live > blocks) {
    p.fold = blocks == 1 ? min(p.live, kLatFold) : min(cdiv_i(p.live, blocks), kLatFold);
    p.blocks = p.live <= p.fold ? 1 : cdiv_i(p.live, p.fold);
  }
  return p;
}

// The blocks of a head tile: `direct` of every request, which find it by their number, and behind them the further ones without
// gaps, those that every request has first; for these a lane looks at a request.  Dies take the blocks in turn, so each gets as
// many, and there are few blocks without work: one holds a unit's LDS for 1 us all the same.  (A place for each of max_splits blocks
// a request, 1800 of 2048 without work at 64 requests and 8 splits, and the end's stores under a condition each: calls of 64 requests
// of up to 64 / 300 / 1152 tokens 23.9 / 31.3 / 49.8 us, now 16.2 / 23.4 / 43.6; of 24 requests of up to 200 / 800, whose blocks fell
// unevenly on the dies, 26.3 / 35.5, now 19.8 / 30.6.)
__device__ __forceinline__ bool latent_block(const LatentArgs& a, const FewerSplits& fewer, int unit, int& b, int& z, LatentPlan& p) {
  if (unit < a.B * a.direct) {
    z = __builtin_amdgcn_readfirstlane((int)(((float)unit + 0.5f) * a.per_b));  // (fewer than 2^19 units)
    b = unit - z * a.B;
    p = latent_plan(a, b, fewer);
    return z < p.blocks;
  }
  int more = unit - a.B * a.direct;
  const int lane = threadIdx.x & 63, total = a.kv_indptr[a.B] - a.kv_indptr[0];
  for (int j = 0; j < a.B; j += 64) {
    const int r = min(j + lane, a.B - 1);
    const bool several = j + lane < a.B && (latent_share(a, a.kv_indptr[r + 1] - a.kv_indptr[r], total) > a.direct || a.max_splits > kLatFold * a.direct);
    if (__ballot(several) == 0) continue;
    const LatentPlan q = latent_plan(a, r, fewer);
    const int blocks = several ? q.blocks : 0;
    for (int i = a.direct;; ++i) {  // every request's block i, those that have one
      const uint64_t on = __ballot(blocks > i);
      const int n = __popcll(on);
      if (n == 0) break;
      if (more < n) {
        const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(on >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)on, 0u));
        const int l = __builtin_ctzll(__ballot(blocks > i && rank == more));
        auto of = [&](int v) { return __builtin_amdgcn_readlane(v, l); };
        b = j + l;
        z = i;
        p = LatentPlan{of(q.start), of(q.len), of(q.per), of(q.live), of(q.fold), of(q.blocks)};
        return true;
      }
      more -= n;
    }
  }
  return false;
}
// On the host.  A request's blocks exceed its share of the chip by less than one, or are what folding forces.  `direct`: what a request
// has of requests of one length, and four at most (eight splits make four blocks where a share is five to seven).
inline void latent_places(LatentArgs& a) {
  const int64_t room = 256 / ((int64_t)a.Hkv * a.head_tiles), forced = (a.max_splits + kLatFold - 1) / kLatFold;
  a.direct = (int)std::max<int64_t>(std::min<int64_t>(std::min<int64_t>(room / a.B, 4), a.max_splits), 1);
  a.units = (int)((int64_t)a.B * a.direct + std::min<int64_t>((int64_t)a.B * (a.max_splits - a.direct), room + 1 + a.B * std::max<int64_t>(forced - a.direct, 0)));
  a.per_b = 1.f / (float)a.B;
}

// nine 1-KiB pieces of eight rows: lane's 16 bytes of piece j come from src + 128 j and land at lds + 1024 j + 16 lane (the
// instruction's offset is added to both addresses); this wave's reads of the stage before have arrived by then
__device__ __forceinline__ void latent_dma(const char* src, uint32_t lds) {
  asm volatile(
      "s_waitcnt lgkmcnt(0)\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
      "s_add_u32 m0, m0, 0x380\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:128\n\t"
      "s_add_u32 m0, m0, 0x380\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:256\n\t"
      "s_add_u32 m0, m0, 0x380\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:384\n\t"
      "s_add_u32 m0, m0, 0x380\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:512\n\t"
      "s_add_u32 m0, m0, 0x380\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:640\n\t"
      "s_add_u32 m0, m0, 0x380\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:768\n\t"
      "s_add_u32 m0, m0, 0x380\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:896\n\t"
      "s_add_u32 m0, m0, 0x380\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:1024" ::"s"(lds),
      "v"(src)
      : "memory", "m0", "scc");
}

// odd 16-lane rows of a change places with the even ones of b
__device__ __forceinline__ void swap_rows16(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// sum and maximum over the four 16-lane rows, in every lane (register swaps: a shuffle is a trip through the LDS)
__device__ __forceinline__ float rows_sum(float v) {
  uint32_t a = __float_as_uint(v), b = a;
  swap_rows16(a, b);
  a = __float_as_uint(__uint_as_float(a) + __uint_as_float(b));
  const auto r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float rows_max(float v) {
  uint32_t a = __float_as_uint(v), b = a;
  swap_rows16(a, b);
  a = __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
  const auto r = __builtin_amdgcn_permlane32_swap(a, a, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

template <typename T, bool CAP>
__global__ void __launch_bounds__(256, 1) latent_decode_kernel(LatentArgs a, FewerSplits fewer) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  if (a.gate && *a.gate != 0) return;
  constexpr float LOG2E = 1.4426950408889634f, LN2 = 0.6931471805599453f;
  // the head tiles of one (request, block) differ by multiples of eight: they share a die and its cache
  const int unit = (int)(blockIdx.x + 8 * blockIdx.z), y = blockIdx.y;
  if (unit >= a.units) return;
  int b, z;
  LatentPlan p;
  if (!latent_block(a, fewer, unit, b, z, p)) return;  // block-uniform
  const int kvh = a.Hkv == 1 ? 0 : y / a.head_tiles, ht = y - kvh * a.head_tiles, group = a.group;
  const int sp0 = z * p.fold, sp1 = min(sp0 + p.fold, p.live);
  const int end = min(sp1 * p.per, p.len);               // tokens sp0 * per .. end
  const int t0 = sp0 * (p.per / kLatTok), t1 = (end + kLatTok - 1) / kLatTok;  // tiles
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hl = lane & 15, g = lane >> 4;

  float m[2] = {-INFINITY, -INFINITY}, lcur[2] = {0.f, 0.f}, ldone[2] = {0.f, 0.f};  // log2 domain; this lane's share of the sums

  const int32_t* idx = a.kv_indices + p.start;
  const char* kb = reinterpret_cast<const char*>(a.kv + (int64_t)kvh * a.k_sh);
  const int64_t row_bytes = a.k_sn * 2;
  char* ring = lds + wid * 2 * kLatTile;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
  const uint32_t ring0 = lds0 + wid * 2 * kLatTile;
  float2v* state = reinterpret_cast<float2v*>(lds + kLatRing);  // [1 + fold][4 waves][32 heads]

  // row r of a tile, 16-byte chunk c: half r >> 3, piece c >> 3, row r & 7 of it, place (c & 7) ^ (r >> 1): 16 rows of a chunk (a K
  // operand) fall on 16 different slots of 256 bytes
  const int k_row = (hl >> 3) * 9216 + (hl & 7) * 128;
  const int k_even = k_row + ((g ^ (hl >> 1)) << 4), k_odd = k_row + (((4 + g) ^ (hl >> 1)) << 4);
  int v_at[2][2];  // [second half of the eight tokens][odd 64 bytes]
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int odd = 0; odd < 2; ++odd) {
      const int kh = lane >> 5, r7 = 4 * j + (hl >> 2), x = 4 * kh + (r7 >> 1);
      const int c7 = 4 * odd + 2 * (g & 1) + ((hl >> 1) & 1);
      v_at[j][odd] = kh * 9216 + r7 * 128 + ((c7 ^ x) << 4) + 8 * (hl & 1);
    }
  const uint32_t src_at[2] = {(uint32_t)(((lane & 7) ^ (lane >> 4)) << 4), (uint32_t)(((lane & 7) ^ (4 + (lane >> 4))) << 4)};

  // slots of sixteen of the wave's tiles: word j of lane 16 i + r has token r of tile t + 4 (4 j + i) (tokens past the end: the last)
  int slots[4];
  auto ask_slots = [&](int t) {
#pragma unroll
    for (int j = 0; j < 4; ++j) slots[j] = idx[min((t + 16 * j + 4 * g) * kLatTok + hl, end - 1)];
  };
  auto load_slots = [&](int t) {
    ask_slots(t);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), once in sixteen tiles: the loop then counts its own requests
  };
  auto issue = [&](int nth, int stage) {
    const int s0 = slots[0], s1 = slots[1], s2 = slots[2], s3 = slots[3];
    const int from = nth & 8 ? (nth & 4 ? s3 : s2) : (nth & 4 ? s1 : s0);
#pragma unroll
    for (int rh = 0; rh < 2; ++rh) {
      const int slot = __shfl(from, 16 * (nth & 3) + 8 * rh + (lane >> 3), 64);
      latent_dma(kb + (int64_t)slot * row_bytes + src_at[rh], ring0 + stage * kLatTile + rh * 9216);
    }
  };
  int split = sp0;
  auto leave_split = [&]() {  // this wave's part of the split's sum
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const float l = rows_sum(lcur[t]);
      if (g == t) state[((1 + split - sp0) * 4 + wid) * 32 + 16 * t + hl] = float2v{m[t], l};
      ldone[t] += lcur[t];
      lcur[t] = 0.f;
    }
    ++split;
  };

  // what the maximum may lag behind by: probabilities stay far below the type's largest number
  constexpr float kLag = std::is_same<T, bf16_t>::value ? 20.f : 8.f;
  float4v* corner = reinterpret_cast<float4v*>(lds + kLatRing + (kLatFold + 1) * kLatState + wid * 1024);
  bool any = false;
  const float qk_scale = CAP ? a.sm_scale : a.sm_scale * LOG2E;
  int t = t0 + wid;
  // slots and queries are on their way while the accumulators are cleared (256 registers, 1024 cycles)
  ask_slots(t);
  // the queries (as a tile of keys: sixteen heads in the second stage of the first and of the second wave), then the first tile
  {
    const int th = wid >> 1, rh = wid & 1;
    const int h = min(ht * 32 + 16 * th + 8 * rh + (lane >> 3), group - 1);  // heads past the group: the last one, never stored
    const uint32_t at = lds0 + (2 * th + 1) * kLatTile + rh * 9216;
    latent_dma(reinterpret_cast<const char*>(a.q + (int64_t)b * a.q_sb + (int64_t)(kvh * group + h) * a.q_sh) + src_at[rh], at);
  }
  float16v oacc[16];
#pragma unroll
  for (int n = 0; n < 16; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[n][r] = 0.f;
#pragma unroll
  for (int n = 0; n < 16; ++n) asm volatile("" : "+a"(oacc[n]));
  __builtin_amdgcn_s_waitcnt(0x0F70);
  if (t < t1) issue(0, 0);
  __syncthreads();
  short8 qf[2][18];  // Q^T operand: column hl of heads 16 u, elements 32 ks + 8 g .. + 7
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int ks = 0; ks < 18; ++ks)
      qf[u][ks] = *reinterpret_cast<const short8*>(lds + (2 * u + 1) * kLatTile + (ks & 1 ? k_odd : k_even) + (ks >> 1) * 1024);
  __syncthreads();
  // tile t, the i-th of the wave's: the next one's rows are requested, then this one's awaited
  for (int i = 0; t < t1; ++i, t += 4) {
    if (t + 4 < t1) {
      if (((i + 1) & 15) == 0) load_slots(t + 4);
      issue((i + 1) & 15, (i + 1) & 1);
      asm volatile("s_waitcnt vmcnt(18)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    while (t * kLatTok >= (split + 1) * p.per) leave_split();
    const char* tile = ring + (i & 1) * kLatTile;
#pragma unroll
    for (int n = 0; n < 16; ++n) asm("" : "+a"(oacc[n]));
    __builtin_amdgcn_sched_barrier(0);
    float4v s[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) s[u][0] = s[u][1] = float4v{0.f, 0.f, 0.f, 0.f};
    // operand reads run a few k-steps ahead of the matrix unit (left to itself the compiler waits for each)
    auto key = [&](int ks) { return *reinterpret_cast<const short8*>(tile + (ks & 1 ? k_odd : k_even) + (ks >> 1) * 1024); };
    constexpr int kAhead = 4;
    short8 kf[18 + kAhead];
#pragma unroll
    for (int ks = 0; ks < kAhead; ++ks) kf[ks] = key(ks);
#pragma unroll
    for (int ks = 0; ks < 18; ++ks) {
      __builtin_amdgcn_sched_barrier(0);
      if (ks + kAhead < 18) kf[ks + kAhead] = key(ks + kAhead);
#pragma unroll
      for (int u = 0; u < 2; ++u) s[u][ks & 1] = Mfma16<T>::mma(kf[ks], qf[u][ks], s[u][ks & 1]);
    }
    __builtin_amdgcn_sched_barrier(0);
    // lane (hl, g): tokens 4 g + r of head 16 u + hl
    float sc[2][4];
    bool more = false;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = (s[u][0][r] + s[u][1][r]) * qk_scale;
        if constexpr (CAP) v = a.logit_cap * tanhf(v / a.logit_cap) * LOG2E;
        if (t * kLatTok + 4 * g + r >= end) v = -INFINITY;
        sc[u][r] = v;
        more |= v > m[u] + kLag;
      }
    if (__any(more)) {
      float alpha[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float top = rows_max(fmaxf(fmaxf(sc[u][0], sc[u][1]), fmaxf(sc[u][2], sc[u][3])));
        const float m_new = fmaxf(m[u], top);
        alpha[u] = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m[u] - m_new);
        m[u] = m_new;
        lcur[u] *= alpha[u];
        ldone[u] *= alpha[u];
      }
      if (any) {  // (a wave's first tile has nothing to rescale)
        const float al = g & 1 ? alpha[1] : alpha[0];
#pragma unroll
        for (int n = 0; n < 16; ++n) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float4v* at = corner + lane;
            *at = float4v{oacc[n][4 * q], oacc[n][4 * q + 1], oacc[n][4 * q + 2], oacc[n][4 * q + 3]};
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            float4v v = *at;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] *= al;
            *at = v;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            v = *at;
#pragma unroll
            for (int r = 0; r < 4; ++r) oacc[n][4 * q + r] = v[r];
          }
          asm("" : "+a"(oacc[n]));
        }
      }
    }
    any = true;
    // probabilities as the sum of two 16-bit numbers: [hi, lo][head tile][pair]
    uint32_t w[2][2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float from = m[u] == -INFINITY ? 0.f : m[u];  // nothing but scores of -inf so far: they weigh nothing
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint16_t first[2], second[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float x = __builtin_amdgcn_exp2f(sc[u][2 * h + e] - from);
          lcur[u] += x;
          first[e] = Conv<T>::from_f32(x);
          second[e] = Conv<T>::from_f32(x - Conv<T>::to_f32(first[e]));
        }
        w[0][u][h] = (uint32_t)first[0] | ((uint32_t)first[1] << 16);
        w[1][u][h] = (uint32_t)second[0] | ((uint32_t)second[1] << 16);
      }
    }
    // P^T operands: lane holds head lane & 31, tokens 8 (lane >> 5) .. + 7
    short8 pf[2];
#pragma unroll
    for (int part = 0; part < 2; ++part) {
#pragma unroll
      for (int h = 0; h < 2; ++h) swap_rows16(w[part][0][h], w[part][1][h]);
      pf[part] = __builtin_bit_cast(short8, uint4v{w[part][0][0], w[part][0][1], w[part][1][0], w[part][1][1]});
    }
    auto value = [&](int n) {
      const short4v lo = lds_read_tr16(tile + v_at[0][n & 1] + (n >> 1) * 1024);
      const short4v hi = lds_read_tr16(tile + v_at[1][n & 1] + (n >> 1) * 1024);
      return short8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    constexpr int kAheadV = 3;
    short8 vf[16 + kAheadV];
#pragma unroll
    for (int n = 0; n < kAheadV; ++n) vf[n] = value(n);
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      __builtin_amdgcn_sched_barrier(0);
      if (n + kAheadV < 16) vf[n + kAheadV] = value(n + kAheadV);
      oacc[n] = Mfma32<T>::mma(vf[n], pf[0], oacc[n]);
      oacc[n] = Mfma32<T>::mma(vf[n], pf[1], oacc[n]);
      asm("" : "+a"(oacc[n]));
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  while (split < sp1) leave_split();

  // ---- the four waves' states meet; 256 output rows at a time go through the LDS, a wave's through its own ring (nobody else reads
  // that any more, and its last tile was waited for), where a thread sums the waves' parts of four rows of a head: eight lanes take
  // 32 rows of one, at a pitch that puts their reads on different banks.  (A quarter of the rows a wave, its own part left in
  // registers, moves 25 % less, but leaves in 16-byte pieces a head: 1.4 us slower.)
  const int l31 = lane & 31, hi = lane >> 5;
  auto leave_rows = [&](int half) {
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float16v& x = oacc[8 * half + n];
        *reinterpret_cast<float4v*>(ring + (4 * n + q) * 1088 + hi * 544 + l31 * 16) = float4v{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
      }
  };
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const float l = rows_sum(ldone[u]);
    if (g == u) state[wid * 32 + 16 * u + hl] = float2v{m[u], l};
  }
  leave_rows(0);
  __syncthreads();
  // the states of one head: maximum and sum over the waves (a wave without tokens has neither)
  auto meet = [&](const float2v* st, float& top, float& sum) {
    top = -INFINITY;
    sum = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) top = fmaxf(top, st[w * 32][0]);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float2v x = st[w * 32];
      sum += x[1] == 0.f ? 0.f : x[1] * __builtin_amdgcn_exp2f(x[0] - top);  // (the maximum of a wave without a weight is not asked)
    }
  };
  const int hd = 8 * wid + (lane >> 3), in_group = ht * 32 + hd, head = kvh * group + in_group;  // this thread's on the way out
  const int64_t row = ((int64_t)b * a.Hq + head) * a.max_splits;
  const int piece = lane & 7;
  float share[4];
  {
    float top, sum;
    meet(state + hd, top, sum);
    // where nothing weighs anything: NaN if this is the request, nothing if other blocks may have what does (log-sum-exps of -inf)
    const float inv = sum == 0.f && p.blocks > 1 ? 0.f : 1.f / sum;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float2v own = state[w * 32 + hd];
      share[w] = (own[1] == 0.f ? 0.f : __builtin_amdgcn_exp2f(own[0] - top)) * inv;
    }
  }
  if (in_group < group && sp0 + (lane & 7) < sp1) {  // the splits' log-sum-exps
    float top, sum;
    meet(state + (1 + (lane & 7)) * 4 * 32 + hd, top, sum);
    a.lse[row + sp0 + (lane & 7)] = (top + log2f(sum)) * LN2;
  }
  auto rows_of = [&](int n) {  // 8 heads x 32 rows
    float4v v = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float4v x = *reinterpret_cast<const float4v*>(lds + w * 2 * kLatTile + (4 * n + (piece >> 1)) * 1088 + (piece & 1) * 544 + hd * 16);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = fmaf(x[r], share[w], v[r]);
    }
    return v;
  };
  const bool mine = in_group < group;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    if (half) {
      __syncthreads();
      leave_rows(1);
      __syncthreads();
    }
    const int d = 256 * half + 4 * piece;
    if (p.blocks > 1) {
      float* dst = a.part + (row + sp0) * kMlaDv + d;
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        const float4v v = rows_of(n);
        if (mine) *reinterpret_cast<float4v*>(dst + 32 * n) = v;
      }
      continue;
    }
    uint16_t* dst = reinterpret_cast<uint16_t*>(a.o) + (int64_t)b * a.o_sb + (int64_t)head * a.o_sh + d;
    short4v x[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      const float4v v = rows_of(n);
#pragma unroll
      for (int r = 0; r < 4; ++r) x[n][r] = (short)Conv<T>::from_f32(v[r]);
    }
    if (!mine) continue;
    if ((reinterpret_cast<uintptr_t>(dst) & 7) == 0) {
#pragma unroll
      for (int n = 0; n < 8; ++n) *reinterpret_cast<short4v*>(dst + 32 * n) = x[n];
    } else {
#pragma unroll
      for (int n = 0; n < 8; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[32 * n + r] = (uint16_t)x[n][r];
    }
  }
}

// Requests of several blocks: their partials (and rows of requests without tokens, NaN as an empty sum's).  A wave a head, its
// weights before its rows: three dependent trips to memory whatever the number of blocks.
template <typename T>
__global__ void __launch_bounds__(256) latent_merge_kernel(LatentArgs a, FewerSplits fewer) {
  if (a.gate && *a.gate != 0) return;
  const int b = blockIdx.x, lane = threadIdx.x & 63;
  const LatentPlan p = latent_plan(a, b, fewer);
  if (p.blocks == 1) return;
  const int h = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (h >= a.Hq) return;
  const int64_t row = ((int64_t)b * a.Hq + h) * a.max_splits;
  float top = -INFINITY;
  for (int s = lane; s < p.live; s += 64) top = fmaxf(top, a.lse[row + s]);
  top = wave_max(top);
  float total = 0.f;
  float4v acc[2] = {float4v{0.f, 0.f, 0.f, 0.f}, float4v{0.f, 0.f, 0.f, 0.f}};
  for (int z0 = 0; z0 < p.blocks; z0 += 64) {
    float w = 0.f;  // of block z0 + lane
    for (int s = (z0 + lane) * p.fold; s < min((z0 + lane + 1) * p.fold, p.live); ++s) w += expf(a.lse[row + s] - top);
    total += wave_sum(w);
    const int nz = min(p.blocks - z0, 64);
#pragma unroll 4
    for (int z = 0; z < nz; ++z) {
      const float wz = __shfl(w, z, 64);
      const float* v = a.part + (row + (z0 + z) * p.fold) * kMlaDv + 4 * lane;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float4v x = *reinterpret_cast<const float4v*>(v + 256 * i);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][r] = fmaf(wz, x[r], acc[i][r]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) st<T>(a.o, (int64_t)b * a.o_sb + (int64_t)h * a.o_sh + 256 * i + 4 * lane + r, acc[i][r] / total);
}

}  // namespace sglk
