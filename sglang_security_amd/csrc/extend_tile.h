// Extend attention over 16-bit K / V rows, head sizes 64 and 128 (gfx950).
//
// Rows are (token, query head) pairs of one kv head, token-major: a block owns 128 consecutive ones, a wave 32.  The
// query heads that share a kv head so sit in one block whatever their number, every wave of a block sees nearly the
// same tokens, and the K / V rows are fetched once for all of them.  Scores are formed transposed on the 32x32x16
// matrix instruction, S^T = K . Q^T: a lane's accumulators are 16 tokens of ONE row, so a row's maximum takes one
// exchange between the two half waves, and the same registers, rounded, are the P^T operand of O^T += V^T . P^T (the
// order of the tokens inside a k-step is free as long as V is read in the same order).
//
// Bound: the issue port.  A tile of 64 tokens x 128 rows is 1024 matrix cycles per SIMD beside 32 KiB written to and 128 KiB
// read from the LDS, but the matrix pipe is busy a third of the time (counters; no bank conflicts): maxima, exponentials and
// conversions stand between the products, and two blocks per CU do not hide them.  Head size 64
// carries its probabilities as the sum of two 16-bit numbers (the wave-per-row kernel it replaces kept them in fp32:
// 0.00166 off the 64-bit result both, 0.0023 with one number); head size 128 rounds them once and divides by the sum of the
// rounded ones, whose errors cancel in part (700 tokens, 32 / 8 heads: 0.00196 off; 0.00198 over the sum of the others, and
// 0.00197 with that on tiles of 32 tokens, which had more probabilities of exactly one).
//
// Measured (bf16, launch alone): 8 prompts of 768 to 1152 tokens, 32 / 8 heads of 128: 264 us (one block per 64 rows of
// one head, 32-token tiles on 16x16x32) -> 113 us, 576 TFLOP/s; one prompt of 1152 tokens: 69 -> 36 us; 128 tokens over
// 1024 cached, split 8 ways: 20.1 -> 14.6 us; 4 prompts of 667 to 1000 tokens over 683 to 1024 cached, 14 / 2 heads of
// 64: 3.24 ms (wave per row) -> 0.052 ms.  Operand reads are spelled out ahead of the products that use them: the
// compiler's own order waits for each (8 prompts: 137.5 -> 134.5 us of a call with its copies, one box).
#pragma once
#include <type_traits>

#include "attention_tile.h"

namespace sglk {

template <typename T>
struct Mfma32;
template <>
struct Mfma32<bf16_t> {
  static __device__ __forceinline__ float16v mma(short8 a, short8 b, float16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bfloat8, a), __builtin_bit_cast(bfloat8, b), c, 0, 0, 0);
  }
};
template <>
struct Mfma32<f16_t> {
  static __device__ __forceinline__ float16v mma(short8 a, short8 b, float16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
  }
};

// acc + the two numbers of a word
template <typename T>
__device__ __forceinline__ float add_pair(short lo, short hi, float acc) {
  typedef short short2v __attribute__((ext_vector_type(2)));
  const short2v v = {lo, hi};
  if constexpr (std::is_same<T, bf16_t>::value) {
    typedef __bf16 two __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(two, v), two{(__bf16)1.f, (__bf16)1.f}, acc, false);
  } else {
    typedef _Float16 two __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(two, v), two{(_Float16)1.f, (_Float16)1.f}, acc, false);
  }
}

template <typename T>
struct Special {  // the type's infinity and one
  static constexpr uint16_t kInf = std::is_same<T, bf16_t>::value ? 0x7F80 : 0x7C00, kOne = std::is_same<T, bf16_t>::value ? 0x3F80 : 0x3C00;
};

struct ExtendArgs {
  const uint16_t *q, *ke, *ve, *kb, *vb;  // ke == nullptr: every token is in the pool (paged form)
  uint16_t* o;
  const int32_t *qo_indptr, *kv_indptr, *kv_indices;
  int Hq, Hkv;
  int64_t q_st, q_sh, ke_sh, ve_sh, o_st, o_sh, kb_sh, vb_sh;
  uint32_t ke_row, ve_row, kb_row, vb_row;  // bytes from row to row (below 2^32: one 32 x 32 + 64-bit product an address)
  float sm_scale, logit_cap;
  int causal, kv_splits;
  int wide_rows;  // rows leave whole: not split, and they start at multiples of 16 bytes
  int last_block, z_blocks;  // of rows, over the grid's second dimension and, unsplit, its third (blocks a step of it has, else 0)
  float *part_o, *part_lse;  // kv_splits > 1: [T, Hq, kv_splits, D] and [T, Hq, kv_splits]
};

constexpr int kExtTokens = 64;  // per tile
constexpr int kExtRows = 128;   // per block

// 16-byte chunk c of K row r: 16 rows of one chunk (an operand read) fall on 16 different slots of 256 bytes
template <int D>
__device__ __forceinline__ int ext_k_off(int r, int c) {
  return D == 128 ? r * 256 + ((c ^ (r & 15)) << 4) : r * 128 + ((c ^ ((r >> 1) & 7)) << 4);
}
// 64-byte granule of V row r: the four rows of a transposed read fall on four different granules
template <int D>
__device__ __forceinline__ int ext_v_off(int r, int byte) {
  const int sw = D == 128 ? (r & 3) : ((r >> 1) & 1);
  return r * 2 * D + ((((byte >> 6) ^ sw) << 6) | (byte & 63));
}

// kv_splits > 1: blockIdx.z is the split; split s walks its slice of the cached prefix, the last one also the new
// tokens, and leaves normalised fp32 rows + log-sum-exps (a short extend over a long prefix has too few rows to fill
// the chip otherwise).
// PRE: scores are finished (scale, cap) before their maximum is taken: a capped call, or a scale that is not positive.
// A block's walk over its ranges: rows leave where `mine`, unless a result of theirs is not finite; returns whether one of
// this lane's row is not.  CAREFUL: values that are not finite stay out of the matrix products, and all rows leave.
template <typename T, int D, bool PRE, bool CAREFUL>
__device__ __forceinline__ bool extend_walk(const ExtendArgs& a, const int tid, bool mine) {
  constexpr int KS = D / 16, NV = D / 32, NP = D / 32;  // k-steps, 32-wide value blocks, 16-byte pieces per thread
  constexpr int kStage = kExtTokens * 2 * D;            // K (or V) bytes of a stage
  constexpr int kTpr = D / 8;                           // threads (chunks) per row
  constexpr float LOG2E = 1.4426950408889634f;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int kvh = blockIdx.x % a.Hkv, b = blockIdx.x / a.Hkv;
  const int share = a.Hq / a.Hkv;
  const int q0 = a.qo_indptr[b], ext = a.qo_indptr[b + 1] - q0;
  const int nrows = ext * share;
  const int split = a.z_blocks ? 0 : blockIdx.z;
  const int R0 = (a.last_block - (int)blockIdx.y - a.z_blocks * (int)blockIdx.z) * kExtRows;  // the rows that see most start first
  if (R0 >= nrows) return false;  // block-uniform
  const int lane = tid & 63, wid = tid >> 6;
  const int l31 = lane & 31, hi = lane >> 5;
  const bool paged = a.ke == nullptr;
  const int pstart = a.kv_indptr[b], plen = a.kv_indptr[b + 1] - pstart;
  const int shift = paged ? plen - ext : 0;

  // this lane's row
  const int R = R0 + 32 * wid + l31;
  const bool row_ok = R < nrows;
  const int Rc = min(R, nrows - 1);
  const int tok = Rc / share, head = kvh * share + Rc - tok * share;
  // the new tokens this lane, and any lane of this wave, may see (as positions of the causal stage)
  const int w_first = min(R0 + 32 * wid, nrows - 1) / share + shift;
  const int w_last = min(R0 + 32 * wid + 31, nrows - 1) / share + shift;
  const bool w_idle = R0 + 32 * wid >= nrows;
  const int b_last = min(R0 + kExtRows - 1, nrows - 1) / share;

  short8 qf[KS];
  {
    const uint16_t* qr = a.q + (int64_t)(q0 + tok) * a.q_st + (int64_t)head * a.q_sh + 8 * hi;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const short8*>(qr + 16 * ks);
  }

  // ranges: tokens p0 .. p1 of the index list, then tokens 0 .. e1 of the new ones
  int p0 = 0, p1 = plen, e1 = 0;
  if (paged) {
    if (a.causal) p1 = min(plen, shift + b_last + 1);
  } else {
    if (a.kv_splits > 1) {
      const int per = (((plen + a.kv_splits - 1) / a.kv_splits) + 31) / 32 * 32;
      p0 = min(per * split, plen);
      p1 = min(p0 + per, plen);
    }
    if (split == a.kv_splits - 1) e1 = a.causal ? b_last + 1 : ext;
  }
  const int nt1 = p1 > p0 ? (p1 - p0 + kExtTokens - 1) / kExtTokens : 0;
  const int nt = nt1 + (e1 + kExtTokens - 1) / kExtTokens;

  const uint16_t* kb = a.kb + (int64_t)kvh * a.kb_sh;
  const uint16_t* vb = a.vb + (int64_t)kvh * a.vb_sh;
  const uint16_t* ke = paged ? nullptr : a.ke + (int64_t)q0 * (a.ke_row >> 1) + (int64_t)kvh * a.ke_sh;
  const uint16_t* ve = paged ? nullptr : a.ve + (int64_t)q0 * (a.ve_row >> 1) + (int64_t)kvh * a.ve_sh;
  const int32_t* idx = a.kv_indices + pstart;

  // a thread moves 16-byte piece `chunk` of rows frow + i * 256 / kTpr
  const int frow = tid / kTpr, chunk = tid % kTpr;
  int4v kreg[NP], vreg[NP];
  int slot[NP];
  auto fetch_idx = [&](int j) {  // pool rows of tile j (rows past the end re-read the last one; their scores are masked)
    if (j < nt1) {
#pragma unroll
      for (int i = 0; i < NP; ++i) slot[i] = idx[min(p0 + j * kExtTokens + frow + i * (256 / kTpr), p1 - 1)];
    }
  };
  // D = 64 has half the work per tile to hide the addresses behind: a whole tile of new tokens has a uniform base and one
  // 32-bit offset a lane there (4 prompts of 667 to 1000 tokens, 14 / 2 heads: a call 62 -> 57 us; at D = 128 the same form gains nothing)
  const uint32_t ke_off = (uint32_t)frow * a.ke_row + chunk * 16, ve_off = (uint32_t)frow * a.ve_row + chunk * 16;
  auto fetch = [&](int j) {
    const int t0 = (j - nt1) * kExtTokens;
    if (D == 64 && j >= nt1 && t0 + kExtTokens <= e1) {
      const char* kp = reinterpret_cast<const char*>(ke) + (uint64_t)(uint32_t)t0 * a.ke_row;
      const char* vp = reinterpret_cast<const char*>(ve) + (uint64_t)(uint32_t)t0 * a.ve_row;
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        kreg[i] = *reinterpret_cast<const int4v*>(kp + (uint64_t)(i * (256 / kTpr)) * a.ke_row + ke_off);
        vreg[i] = *reinterpret_cast<const int4v*>(vp + (uint64_t)(i * (256 / kTpr)) * a.ve_row + ve_off);
      }
      return;
    }
    const bool pool = j < nt1;  // block-uniform
    const char* kp = reinterpret_cast<const char*>(pool ? kb : ke);
    const char* vp = reinterpret_cast<const char*>(pool ? vb : ve);
    const uint32_t ks = pool ? a.kb_row : a.ke_row, vs = pool ? a.vb_row : a.ve_row;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const uint32_t r = pool ? slot[i] : min(t0 + frow + i * (256 / kTpr), e1 - 1);
      kreg[i] = *reinterpret_cast<const int4v*>(kp + ((uint64_t)r * ks + chunk * 16));
      vreg[i] = *reinterpret_cast<const int4v*>(vp + ((uint64_t)r * vs + chunk * 16));
    }
  };

  const float c = PRE ? 1.f : a.sm_scale * LOG2E;
  if (!CAREFUL) mine = row_ok;
  float m = -INFINITY, lsum = 0.f;  // running maximum (log2 domain) and this lane's share of the running sum
  float16v oacc[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[n][r] = 0.f;

  if (!CAREFUL && nt > 0) {
    fetch_idx(0);
    fetch(0);
    fetch_idx(1);
  }
  for (int j = 0; j < nt; ++j) {
    if constexpr (CAREFUL) {  // none ahead: the registers are needed below
      fetch_idx(j);
      fetch(j);
    }
    char* kl = lds + (j & 1) * 2 * kStage;
    char* vl = kl + kStage;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int r = frow + i * (256 / kTpr);
      *reinterpret_cast<int4v*>(kl + ext_k_off<D>(r, chunk)) = kreg[i];
      *reinterpret_cast<int4v*>(vl + ext_v_off<D>(r, chunk * 16)) = vreg[i];
    }
    __syncthreads();  // also: nobody reads the other stage any more once the next tile is parked
    if (!CAREFUL && j + 1 < nt) {
      fetch(j + 1);
      fetch_idx(j + 2);
    }
    const bool pool = j < nt1;
    const int t0 = pool ? p0 + j * kExtTokens : (j - nt1) * kExtTokens;
    const int t_end = pool ? p1 : e1;
    const bool diag = a.causal && (paged || !pool);
    if (w_idle || (diag && t0 > w_last)) continue;  // wave-uniform: nothing of this tile is visible here

    float16v s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[u][r] = 0.f;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const short8 kf = *reinterpret_cast<const short8*>(kl + ext_k_off<D>(32 * u + l31, 2 * ks + hi));
        s[u] = Mfma32<T>::mma(kf, qf[ks], s[u]);
      }
    // operand reads run kAhead products ahead of the matrix unit (left to itself the compiler waits for each)
    constexpr int kAhead = 4;
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
    for (int i = 0; i < 2 * KS - kAhead; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x8, kAhead, 0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (PRE) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float v = s[u][r] * a.sm_scale;
          s[u][r] = (a.logit_cap > 0.f ? a.logit_cap * tanhf(v / a.logit_cap) : v) * LOG2E;
        }
    }
    [[maybe_unused]] uint32_t hidden = 0;
    if (t0 + kExtTokens > t_end || (diag && t0 + kExtTokens - 1 > w_first)) {  // wave-uniform
      const int lim = diag ? min(tok + shift, t_end - 1) : t_end - 1;          // last token this row sees
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (t0 + 32 * u + 8 * (r >> 2) + 4 * hi + (r & 3) > lim) {
            s[u][r] = -INFINITY;
            if constexpr (CAREFUL) hidden |= 1u << (16 * u + r);
          }
    }
    float tmax = s[0][0];
#pragma unroll
    for (int r = 1; r < 16; ++r) tmax = fmaxf(tmax, s[0][r]);
#pragma unroll
    for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s[1][r]);
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64)) * c;
    // The maximum only keeps the exponentials in range.  Probabilities that are rounded to 16 bits need it exact (the
    // largest one is then 1 and has no rounding error); split ones let it lag by 2^8 and save most of the rescaling.
    constexpr bool P2 = D == 64;
    if (__any(tmax > m + (P2 && !CAREFUL ? 8.f : 0.f))) {
      const float m_new = fmaxf(m, tmax);
      const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
      lsum *= alpha;
#pragma unroll
      for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[n][r] *= alpha;
    }
    const float m_use = m == -INFINITY ? 0.f : m;  // nothing visible yet: everything stays zero
    short8 pf[4], pl[P2 ? 4 : 1];
    float psum = 0.f;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[u][r], c, -m_use));
        if constexpr (P2) psum += p;
        if constexpr (CAREFUL) {
          s[u][r] = p;
          continue;
        }
        const uint16_t ph = Conv<T>::from_f32(p);
        pf[2 * u + (r >> 3)][r & 7] = (short)ph;
        if constexpr (P2) pl[2 * u + (r >> 3)][r & 7] = (short)Conv<T>::from_f32(p - Conv<T>::to_f32(ph));
      }
    // two rounded probabilities an instruction, added as exactly as one
    if constexpr (!P2 && !CAREFUL)
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int e = 0; e < 8; e += 2) psum = add_pair<T>(pf[k][e], pf[k][e + 1], psum);
    if constexpr (!CAREFUL) lsum += psum;
    if constexpr (CAREFUL) {
      // A value that is not finite counts as zero in the product; two more products count those of a row's 16 tokens on
      // either side (a NaN, and an infinity of weight zero, is one on both), and one infinity stands for a side.
      auto value = [&](int k, int n) {  // V^T operand: 16 tokens from 16 k on, elements 32 n .. 32 n + 31
        const int row = 16 * k + 4 * hi + ((lane & 15) >> 2);
        const int byte = 64 * n + 32 * ((lane >> 4) & 1) + 8 * (lane & 3);
        const short4v lo = lds_read_tr16(vl + ext_v_off<D>(row, byte));
        const short4v up = lds_read_tr16(vl + ext_v_off<D>(row + 8, byte));
        return short8{lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]};
      };
      constexpr int kInf = Special<T>::kInf, kOne = Special<T>::kOne;
      if (m == -INFINITY) hidden = ~0u;  // (nothing of weight so far: the row takes nothing)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        short8 hp, lp, on, off;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float p = s[k >> 1][8 * (k & 1) + e];
          const int seen = hidden >> (8 * k + e) & 1 ? 0 : kOne;
          const uint16_t ph = Conv<T>::from_f32(p);
          hp[e] = (short)ph;
          lp[e] = (short)Conv<T>::from_f32(p - Conv<T>::to_f32(ph));
          on[e] = (short)(p == 0.f ? 0 : seen);
          off[e] = (short)(p == 0.f ? seen : 0);
        }
        if constexpr (!P2)
#pragma unroll
          for (int e = 0; e < 8; e += 2) psum = add_pair<T>(hp[e], hp[e + 1], psum);  // in the first walk's order
#pragma unroll
        for (int n = 0; n < NV; ++n) {
          __builtin_amdgcn_sched_barrier(0);
          const short8 vf = value(k, n);
          short8 fin, any, side[2];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int sign = vf[e] >> 15, mag = vf[e] & 0x7FFF;
            const int odd = (kInf - 1 - mag) >> 31, nan = (kInf - mag) >> 31;  // all ones or zeros
            fin[e] = (short)(vf[e] & ~odd);
            any[e] = (short)(odd & kOne);
            side[0][e] = (short)((nan | (odd & ~sign)) & kOne);
            side[1][e] = (short)((nan | (odd & sign)) & kOne);
          }
          oacc[n] = Mfma32<T>::mma(fin, hp, oacc[n]);
          if constexpr (P2) oacc[n] = Mfma32<T>::mma(fin, lp, oacc[n]);
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            float16v count;
#pragma unroll
            for (int r = 0; r < 16; ++r) count[r] = 0.f;
            count = Mfma32<T>::mma(side[t], on, Mfma32<T>::mma(any, off, count));
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[n][r] += count[r] == 0.f ? 0.f : t == 0 ? INFINITY : -INFINITY;
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      lsum += psum;
      continue;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        const int row = 16 * k + 4 * hi + ((lane & 15) >> 2);
        const int byte = 64 * n + 32 * ((lane >> 4) & 1) + 8 * (lane & 3);
        const short4v lo = lds_read_tr16(vl + ext_v_off<D>(row, byte));
        const short4v up = lds_read_tr16(vl + ext_v_off<D>(row + 8, byte));
        const short8 vf = short8{lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]};
        oacc[n] = Mfma32<T>::mma(vf, pf[k], oacc[n]);
        if constexpr (P2) oacc[n] = Mfma32<T>::mma(vf, pl[k], oacc[n]);
      }
    constexpr int kPer = P2 ? 2 : 1, kAheadV = 3;  // products a value operand, operands read ahead
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kAheadV, 1);
#pragma unroll
    for (int i = 0; i < 4 * NV - kAheadV; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x8, kPer, 1);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
    }
    __builtin_amdgcn_sched_group_barrier(0x8, kPer * kAheadV, 1);
  }

  const float tot = lsum + __shfl_xor(lsum, 32, 64);
  const float inv = tot == 0.f ? 0.f : 1.0f / tot;
  float zero[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r) zero[r & 3] = fmaf(oacc[n][r], 0.f, zero[r & 3]);
  const float nan = (zero[0] + zero[1]) + (zero[2] + zero[3]);
  const float nan_other = __shfl_xor(nan, 32, 64);  // by all lanes, whatever their own is
  const bool odd = nan != 0.f || nan_other != 0.f;
  if constexpr (!CAREFUL && D == 128) {
    if (a.wide_rows) {
      // Whole rows, turned in the stage that the last tile does not use: a lane's own pieces of 8 bytes are 16 requests a wave,
      // each of 16 bytes of 32 rows.  8 prompts of 512 tokens 41.4 -> 37.5 us, of 1024 108 -> 102, 8 of 768 to 1152 in a call with its
      // copies 120.3 -> 115.5.  Stored past the caches they are 3 us faster still, and the product that reads them 7 slower.  Head size
      // 64 has half the bytes a row and gains nothing (52.3 -> 52.9 for 4 prompts over cached prefixes).
      char* ol = lds + (nt & 1) * 2 * kStage + wid * (64 * D);
      auto out_off = [&](int r, int piece) { return r * 2 * D + ((piece ^ (r & 15)) << 4); };
#pragma unroll
      for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          short4v v;
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = (short)Conv<T>::from_f32(oacc[n][4 * g + r] * inv);
          *reinterpret_cast<short4v*>(ol + out_off(l31, 4 * n + g) + 8 * hi) = v;
        }
      __builtin_amdgcn_wave_barrier();  // the wave's own LDS rows: in order, no block barrier
      const uint64_t leave = __ballot(mine && !odd);
      const int64_t off = (int64_t)(q0 + tok) * a.o_st + (int64_t)head * a.o_sh;
#pragma unroll
      for (int t = 0; t < 32 * kTpr / 64; ++t) {
        const int r = t * (64 / kTpr) + lane / kTpr, piece = lane % kTpr;
        const int4v v = *reinterpret_cast<const int4v*>(ol + out_off(r, piece));
        const int64_t to = __shfl(off, r, 64);
        if (leave >> r & 1) *reinterpret_cast<int4v*>(a.o + to + piece * 8) = v;
      }
      return mine && odd;
    }
  }
  if (!mine || (odd && !CAREFUL)) return mine && odd;
  // lane (row, hi) holds elements 32 n + 8 g + 4 hi + 0 .. 3 of its row
  if (a.kv_splits > 1) {
    const int64_t row = ((int64_t)(q0 + tok) * a.Hq + head) * a.kv_splits + split;
    float* dst = a.part_o + row * D + 4 * hi;
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float4v v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = oacc[n][4 * g + r] * inv;
        *reinterpret_cast<float4v*>(dst + 32 * n + 8 * g) = v;
      }
    if (hi == 0) a.part_lse[row] = tot == 0.f ? -INFINITY : (m + log2f(tot)) * 0.6931471805599453f;
    return false;
  }
  uint16_t* dst = a.o + (int64_t)(q0 + tok) * a.o_st + (int64_t)head * a.o_sh + 4 * hi;
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      short4v v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = (short)Conv<T>::from_f32(oacc[n][4 * g + r] * inv);
      *reinterpret_cast<short4v*>(dst + 32 * n + 8 * g) = v;
    }
  return false;
}

template <typename T, int D, bool PRE>
__global__ void __launch_bounds__(256, 2) extend_tile_kernel(ExtendArgs a) {
  // A value that is not finite spoils, times a probability of zero, the rows that do not see it as well (and, at head size
  // 64, times the second part of a probability, those that do; there also sums that overflow under a lagging maximum).
  // Rows whose result is not finite are walked once more.  To the others that costs a multiplication a result and a
  // barrier at the end: 0.2 us of a launch alone, 118.2 -> 118.9 us for the 8 prompts above.
  int tid = threadIdx.x;
  const bool again = extend_walk<T, D, PRE, false>(a, tid, false);
  __shared__ int spoilt[4];
  if ((tid & 63) == 0) spoilt[tid >> 6] = 0;
  if (again) spoilt[tid >> 6] = 1;
  __syncthreads();  // also: nobody reads a stage any more
  if (__builtin_expect((spoilt[0] | spoilt[1] | spoilt[2] | spoilt[3]) == 0, 1)) return;
  // the second walk takes everything from the arguments again: what the first keeps in registers for it slows its loop
  // (head size 128: by a quarter)
  auto args = __builtin_amdgcn_kernarg_segment_ptr();  // the kernel's one argument
  asm volatile("" : "+s"(args), "+v"(tid));
  extend_walk<T, D, PRE, true>(*(const ExtendArgs*)args, tid, again);
}

}  // namespace sglk
