// Probability filters and inverse-CDF sampling for the sampler's GPU path (top-k / top-p / min-p): a block
// per row, or a row spread over several.
//
// A threshold (the k-th largest value; the smallest value whose cumulative mass reaches a target) is found by radix
// selection on the float bit pattern in digits of 12, 10 and 9 bits.  What bounds it is one unit's trips over its row
// (513 KB at 128256 entries) and the LDS atomics: a float addition there takes three cycles a LANE, an integer one hides
// behind the loads.  So a bin holds its count and its mass in one 64-bit integer, the mass in fixed point (2^-44 of the
// row's at this length: finer than fp32 sums, and the same in any order).  Values that cannot hold either threshold are
// only added up (a value below (1 - p) / n of the mass lies below the top-p cut, however many there are); the first digit
// is wide enough (sixteen bins an octave) that the chosen bins fit an LDS list, and the other digits are taken from
// there; rows are read in 16-byte pieces, eight in flight a thread.
//
// Measured, 64 rows of 128256 out of memory, top-k and top-p together: sampling 555 us (256 bins for four 8-bit digits each, a
// float atomic on a handful of exponents for every element, a thread's elements 500 bytes from the next thread's) -> 81 us
// with a block a row, 46.5 with its rows spread over four blocks in four launches, 36 in three; top-p renormalisation 390 -> 66 ->
// 41.6 -> 37.  (One row of 32000: 28.5 -> 24 and 21.4 -> 19.)  The last step: an element's bin word is bits that it has, where
// its fixed-point mass took fifteen instructions; the slice is asked for before the cuts are looked for; lists of candidates
// are counted by the whole block, not walked by a wave (two thousand of them: 6 us); scans run on DPP operands, not through
// LDS; the chunks' masses are added up beside the search for candidates, a launch less.
// Rows that the guess does not hold for are done over by one block behind the spread launches: sampling from 64 rows of one certain
// token each (fewer than k above the mean) 615 us at first, 99 unspread, 118 spread; of nearly equal values (bins beyond the
// lists) 674, 148, 175; one certain row among 64 574, 92, 124.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace sglk {
namespace {

constexpr int kSampThreads = 1024;
constexpr int kBins = 4096;   // first digit: exponent and four mantissa bits
constexpr int kList = 2048;   // elements of a chosen bin that are kept in LDS
typedef unsigned long long u64;

struct SampShared {
  union {
    u64 bin[kBins];  // count << mass bits | mass
    float chunk[kBins];
  };
  uint32_t list[2][kList];  // bit patterns: candidates of the top-k cut, of the top-p cut
  u64 digit[2][128];
  uint32_t cut[2];
  float red[16];
  u64 ured[16];
  uint32_t fill[2];
  int pick;
  u64 below;
  uint32_t need;
};

constexpr int kNoMass = -400;  // a scale at which every mass is zero

// Mass in fixed point: v 2^scale, rounded down.  bits: of the mass in a bin's word (the count has the rest).
struct Fixed {
  int bits, scale;
  __device__ __forceinline__ u64 of(uint32_t b) const {  // b: pattern of a non-negative float
    const int down = 190 - scale - (int)(b >> 23);        // from the 24 leading bits at the top of the word
    const u64 top = (u64)(((b & 0x7FFFFFu) | 0x800000u) << 8) << 32;
    return down > 63 ? 0 : top >> (down & 63);
  }
  __device__ __forceinline__ u64 mass(u64 w) const { return w & ((1ull << bits) - 1); }
  __device__ __forceinline__ uint32_t count(u64 w) const { return (uint32_t)(w >> bits); }
};

__device__ __forceinline__ float bsum(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < 16; ++w) t += red[w];
  __syncthreads();
  return t;
}
__device__ __forceinline__ float bmax(float v, float* red) {
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = red[0];
#pragma unroll
  for (int w = 1; w < 16; ++w) t = fmaxf(t, red[w]);
  __syncthreads();
  return t;
}
// sum over the block's threads in front of this one; total: over all
template <typename V>
__device__ __forceinline__ V bscan(V v, V* red, V& total) {
  V incl = v;
  if constexpr (std::is_same_v<V, u64>) {
    incl = wave_scan(v);
  } else {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const V u = __shfl_up(incl, o, 64);
      if ((int)(threadIdx.x & 63) >= o) incl += u;
    }
  }
  if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = incl;
  __syncthreads();
  V base = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    if (w < (int)(threadIdx.x >> 6)) base += red[w];
    total += red[w];
  }
  __syncthreads();
  return base + incl - v;
}

// f(value) for every element of the row, U loads in flight
template <bool VEC, int U = 8, typename F>
__device__ __forceinline__ void each(const float* __restrict__ x, int n, F f) {
  if constexpr (VEC) {
    const int n4 = n >> 2;
    for (int i0 = threadIdx.x; i0 < n4; i0 += U * kSampThreads) {
      float4v r[U];
#pragma unroll
      for (int u = 0; u < U; ++u) r[u] = *reinterpret_cast<const float4v*>(x + 4 * (int64_t)min(i0 + u * kSampThreads, n4 - 1));
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (i0 + u * kSampThreads < n4) {
#pragma unroll
          for (int e = 0; e < 4; ++e) f(r[u][e]);
        }
    }
    if ((int)threadIdx.x < (n & 3)) f(x[(n & ~3) + threadIdx.x]);
  } else {
    for (int i = threadIdx.x; i < n; i += kSampThreads) f(x[i]);
  }
}

__device__ __forceinline__ uint32_t value_bits(float v) { return __float_as_uint(fmaxf(v, 0.f)); }  // NaN counts as zero

// bin (of PER * 1024) that holds the k-th largest of the counted elements; sh.need: its rank inside the bin
template <int PER>
__device__ __forceinline__ int pick_count(SampShared& sh, const Fixed& fx, uint32_t k) {
  uint32_t c[PER];
  u64 own = 0, total;
#pragma unroll
  for (int j = 0; j < PER; ++j) own += c[j] = fx.count(sh.bin[threadIdx.x * PER + j]);
  const u64 before = bscan<u64>(own, sh.ured, total);
  u64 above = total - before - own;  // in the bins behind this thread's
#pragma unroll
  for (int j = PER - 1; j >= 0; --j) {
    if (above < k && k <= above + c[j]) {
      sh.pick = threadIdx.x * PER + j;
      sh.need = k - (uint32_t)above;
    }
    above += c[j];
  }
  __syncthreads();
  return sh.pick;
}

// first bin with mass at which the mass, `below` included, reaches `target`; if the target lies beyond the total, the last
// bin with mass (0 if there is none).  sh.below: the mass in front of the bin
template <int PER>
__device__ __forceinline__ int pick_mass(SampShared& sh, const Fixed& fx, u64 below, u64 target) {
  u64 m[PER], own = 0, total;
#pragma unroll
  for (int j = 0; j < PER; ++j) own += m[j] = fx.mass(sh.bin[threadIdx.x * PER + j]);
  u64 run = below + bscan<u64>(own, sh.ured, total);
  if (target == 0) target = 1;
  if (below + total >= target) {  // block-uniform: whole numbers, one bin passes the target
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      if (m[j] > 0 && (run < target || run == below) && run + m[j] >= target) {
        sh.pick = threadIdx.x * PER + j;
        sh.below = run;
      }
      run += m[j];
    }
    __syncthreads();
    return sh.pick;
  }
  if (threadIdx.x == 0) sh.pick = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if (m[j] > 0) atomicMax(&sh.pick, (int)threadIdx.x * PER + j);
  if (threadIdx.x == 0) sh.below = below;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (m[j] > 0 && sh.pick == (int)threadIdx.x * PER + j) sh.below = run;
    run += m[j];
  }
  __syncthreads();
  return sh.pick;
}

__device__ __forceinline__ void clear_bins(SampShared& sh, int bins) {
  for (int i = threadIdx.x; i < bins; i += kSampThreads) sh.bin[i] = 0;
  __syncthreads();
}

// The remaining 19 bits of a threshold whose first digit is `bin`: among the elements of the bin from bit pattern `lo` on,
// from the LDS list when they fit, else from the row.  COUNT: the rank-th largest; else: the mass cut.
template <bool VEC, bool COUNT>
__device__ uint32_t refine(const float* __restrict__ x, int n, SampShared& sh, const Fixed& fx, const uint32_t* list, int listed,
                           int bin, uint32_t rank, u64 below, u64 target, uint32_t lo) {
  uint32_t prefix = (uint32_t)bin << 19;
  int bits = 19;
#pragma unroll
  for (int digit = 0; digit < 2; ++digit) {
    const int take = digit == 0 ? 10 : 9, shift = bits - take;
    clear_bins(sh, 1024);
    auto add = [&](uint32_t b) {
      if ((b >> bits) != (prefix >> bits) || b < lo) return;
      atomicAdd(&sh.bin[(b >> shift) & ((1u << take) - 1)], (1ull << fx.bits) + fx.of(b));
    };
    if (listed <= kList)
      for (int i = threadIdx.x; i < listed; i += kSampThreads) add(list[i]);
    else
      each<VEC>(x, n, [&](float v) { add(value_bits(v)); });
    __syncthreads();
    int d;
    if (COUNT) {
      d = pick_count<1>(sh, fx, rank);
      rank = sh.need;
    } else {
      d = pick_mass<1>(sh, fx, below, target);
      below = sh.below;
    }
    __syncthreads();
    prefix |= (uint32_t)d << shift;
    bits = shift;
  }
  return prefix;
}

// One digit of the same, by one wave from 64 or 128 bins, two a lane, which it leaves at zero.  Returns the digit; rank and
// below go on into it.
template <bool COUNT>
__device__ __forceinline__ int pick_digit(u64* bins, const Fixed& fx, uint32_t& rank, u64& below, u64 target) {
  const int lane = threadIdx.x & 63;
  const u64 w0 = bins[2 * lane], w1 = bins[2 * lane + 1];
  bins[2 * lane] = bins[2 * lane + 1] = 0;
  const u64 incl = wave_scan(w0 + w1), total = __shfl(incl, 63, 64), before = incl - (w0 + w1);
  int d = -1;
  if (COUNT) {
    const uint32_t c0 = fx.count(w0), c1 = fx.count(w1);
    uint32_t above = fx.count(total) - fx.count(before) - c0 - c1;
    uint32_t need = 0;
    if (above < rank && rank <= above + c1) d = 2 * lane + 1, need = rank - above;
    above += c1;
    if (above < rank && rank <= above + c0) d = 2 * lane, need = rank - above;
    const u64 who = __ballot(d >= 0);
    const int src = who ? __ffsll(who) - 1 : 0;
    d = max(__shfl(d, src, 64), 0);
    rank = __shfl(need, src, 64);
  } else {
    const u64 m0 = fx.mass(w0), m1 = fx.mass(w1);
    const bool reach = below + fx.mass(total) >= target;  // else: the last bin with mass
    u64 at = below + fx.mass(before), run = at;
    if (m0 > 0 && (reach ? run + m0 >= target : true)) d = 2 * lane, at = run;
    run += m0;
    if (m1 > 0 && (reach ? d < 0 && run + m1 >= target : true)) d = 2 * lane + 1, at = run;
    const u64 who = __ballot(d >= 0);
    const int src = !who ? 0 : reach ? __ffsll(who) - 1 : 63 - __clzll(who);
    d = max(__shfl(d, src, 64), 0);
    if (who) below = __shfl(at, src, 64);
  }
  return d;
}

struct RowParams {
  int top_k;      // <= 0 or >= n: no top-k filter
  float top_p;    // >= 1: no top-p filter
  float min_p;    // <= 0: no min-p filter
  int joint;      // 1: both filters on the original distribution; 0: top-p on the top-k renormalised one
};

// Threshold of the kept set {x >= thr} for the row's filters.  kept: its mass where one filter was applied and the chosen
// bin's elements were listed, else negative.  FILTER: the call may have a top-k or top-p
template <bool VEC, bool FILTER>
__device__ float row_threshold(const float* __restrict__ x, int n, const RowParams& rp, SampShared& sh, float& kept) {
  constexpr int PER = kBins / kSampThreads;
  const bool use_k = FILTER && rp.top_k > 0 && rp.top_k < n, use_p = FILTER && rp.top_p < 1.0f;
  float thr = 0.f, vmax = 0.f;
  kept = -1.f;
  if (use_k || use_p) {
    const bool p_first = use_p && !(use_k && !rp.joint);  // the top-p cut is taken over the whole row
    // A row of mass about one is guessed and checked: values below `least` are only added up (they must not reach the
    // top-p target, and enough must be left for k), masses have to fit their words; else the row is binned once more.
    const float share = 0.999f * (1.0f - rp.top_p) / (float)n;
    float least = p_first ? (use_k ? fminf(1.0f / (float)n, share) : share) : 1.0f / (float)n;
    if (!(least >= 0.f)) least = 0.f;
    Fixed fx;
    fx.bits = 32 + __clz(n) - 1;  // counts up to n fit above
    fx.scale = fx.bits - 2;       // masses below two
    double total = 0.0;
    float under = 0.f;
    for (int guess = 0;; ++guess) {
      clear_bins(sh, kBins);
      float s = 0.f, o = 0.f, mx = 0.f;
      each<VEC>(x, n, [&](float raw) {
        const float v = fmaxf(raw, 0.f);
        const uint32_t b = __float_as_uint(v);
        const bool in = v >= least;
        mx = fmaxf(mx, v);
        s += in ? 0.f : v;
        o += in ? v : 0.f;
        if (in) atomicAdd(&sh.bin[b >> 19], (1ull << fx.bits) + fx.of(b));
      });
      vmax = bmax(mx, sh.red);  // also: the bins are complete
      under = bsum(s, sh.red);
      total = (double)under + (double)bsum(o, sh.red);
      if (!(total < 3e38)) {  // an infinite mass: counts only
        if (fx.scale == kNoMass || guess == 2) break;
        fx.scale = kNoMass;
        least = 0.f;
        continue;
      }
      const double unit = exp2((double)(fx.bits - 2 - fx.scale));
      const bool fits = total == 0.0 || (total < 2.0 * unit && total > 0.2 * unit);
      uint32_t left = 0;
      u64 all;
#pragma unroll
      for (int j = 0; j < PER; ++j) left += fx.count(sh.bin[threadIdx.x * PER + j]);
      bscan<u64>(left, sh.ured, all);
      if (guess == 2 || (fits && (!(least > 0.f) || (all > 0 && (!use_k || (int)all >= rp.top_k) &&
                                                    (!p_first || (double)under < (double)(1.0f - rp.top_p) * total)))))
        break;
      if (fits || guess == 1) least = 0.f;
      if (!fits) {
        int e;
        frexp(total, &e);
        fx.scale = fx.bits - 1 - e;  // total < 2^e
        least *= (float)total;
      }
    }
    const uint32_t from = __float_as_uint(least);
    int kbin = -1, pbin = -1;
    uint32_t rank = 0;
    u64 below = 0, target = 0;
    if (use_k) {
      kbin = pick_count<PER>(sh, fx, (uint32_t)rp.top_k);
      rank = sh.need;
      __syncthreads();
    }
    const bool finite = total < 3e38;  // beyond: the target is out of reach of any finite value
    auto goal = [&](u64 mass) { return (u64)fmin(ceil((double)(1.0f - rp.top_p) * (double)mass), 4e18); };
    auto mass_of = [&](int first_bin) {  // of the bins from first_bin on
      u64 own = 0, all;
#pragma unroll
      for (int j = 0; j < PER; ++j)
        if ((int)threadIdx.x * PER + j >= first_bin) own += fx.mass(sh.bin[threadIdx.x * PER + j]);
      bscan<u64>(own, sh.ured, all);
      return all;
    };
    if (p_first && finite) {
      const u64 low = (u64)ldexp((double)under, fx.scale);
      target = goal(low + mass_of(0));
      pbin = pick_mass<PER>(sh, fx, low, target);
      below = sh.below;
      __syncthreads();
    }
    const int kcount = kbin >= 0 ? (int)fx.count(sh.bin[kbin]) : 0;
    int pcount = pbin >= 0 ? (int)fx.count(sh.bin[pbin]) : 0;
    // the counted elements of the chosen bins
    auto collect = [&](int a, int na, int b, int nb) {
      if (threadIdx.x < 2) sh.fill[threadIdx.x] = 0;
      __syncthreads();
      if ((a >= 0 && na <= kList) || (b >= 0 && nb <= kList))
        each<VEC>(x, n, [&](float raw) {
          const uint32_t bits = value_bits(raw);
          const int d = bits >= from ? (int)(bits >> 19) : -2;
          if (d == a && na <= kList) sh.list[0][atomicAdd(&sh.fill[0], 1u)] = bits;
          if (d == b && nb <= kList) sh.list[1][atomicAdd(&sh.fill[1], 1u)] = bits;
        });
      __syncthreads();
    };
    collect(kbin, kcount, pbin, pcount);
    const bool single = finite && use_k != use_p && !(rp.min_p > 0.f) && (use_k ? kcount : pcount) <= kList;
    u64 above = 0;
    if (single)
      above = mass_of((use_k ? kbin : pbin) + 1);
    else if (use_p && !p_first && finite)
      above = mass_of(kbin + 1);
    uint32_t kbits = 0;
    if (use_k) kbits = refine<VEC, true>(x, n, sh, fx, sh.list[0], kcount, kbin, rank, 0, 0, from);
    thr = __uint_as_float(kbits);
    if (use_p && !finite) {
      thr = vmax;
    } else if (p_first) {
      thr = fmaxf(thr, __uint_as_float(refine<VEC, false>(x, n, sh, fx, sh.list[1], pcount, pbin, 0u, below, target, from)));
    } else if (use_p) {
      // top-p over the k largest: the k bin counts from the cut on, bins in front of it not at all.  The first 1024 bins
      // (values below 2^-63) have been used for digits: if the k bin is one of them the row is binned again.
      u64 part = 0, all;
      auto add = [&](uint32_t b) {
        if ((int)(b >> 19) == kbin && b >= kbits) part += fx.of(b);
      };
      if (kcount <= kList)
        for (int i = threadIdx.x; i < kcount; i += kSampThreads) add(sh.list[0][i]);
      else
        each<VEC>(x, n, [&](float v) { add(value_bits(v)); });
      bscan<u64>(part, sh.ured, all);
      part = all;
      if (kbin < 1024) {
        clear_bins(sh, 1024);
        each<VEC>(x, n, [&](float v) {
          const uint32_t b = value_bits(v);
          if (b >= kbits && (b >> 19) < 1024) atomicAdd(&sh.bin[b >> 19], (1ull << fx.bits) + fx.of(b));
        });
        __syncthreads();
      }
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const int d = threadIdx.x * PER + j;
        if (d <= kbin) sh.bin[d] = d == kbin ? ((u64)kcount << fx.bits) + part : 0;
      }
      __syncthreads();
      target = goal(above + part);
      pbin = pick_mass<PER>(sh, fx, 0, target);
      below = sh.below;
      __syncthreads();
      int plist = 0;
      pcount = kcount;
      if (pbin != kbin) {
        pcount = (int)fx.count(sh.bin[pbin]);
        plist = 1;
        collect(-1, 0, pbin, pcount);
      }
      thr = fmaxf(thr, __uint_as_float(refine<VEC, false>(x, n, sh, fx, sh.list[plist], pcount, pbin, 0u, below, target, kbits)));
    }
    if (single) {
      u64 part = 0, all;
      for (int i = threadIdx.x; i < (use_k ? kcount : pcount); i += kSampThreads) {
        const uint32_t b = sh.list[use_k ? 0 : 1][i];
        if (__uint_as_float(b) >= thr) part += fx.of(b);
      }
      bscan<u64>(part, sh.ured, all);
      kept = (float)ldexp((double)(above + all), -fx.scale);
    }
  } else if (rp.min_p > 0.f) {
    each<VEC>(x, n, [&](float v) { vmax = fmaxf(vmax, v); });
    vmax = bmax(vmax, sh.red);
  }
  if (rp.min_p > 0.f) thr = fmaxf(thr, rp.min_p * vmax);
  return thr;
}

template <bool VEC>
__device__ __forceinline__ void write_renormed(const float* __restrict__ x, float* __restrict__ o, int n, float thr, float inv) {
  if constexpr (VEC) {
    for (int i = threadIdx.x; i < n >> 2; i += kSampThreads) {
      float4v v = *reinterpret_cast<const float4v*>(x + 4 * (int64_t)i);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] >= thr ? v[e] * inv : 0.f;
      *reinterpret_cast<float4v*>(o + 4 * (int64_t)i) = v;
    }
    const int i = (n & ~3) + threadIdx.x;
    if (i < n) o[i] = x[i] >= thr ? x[i] * inv : 0.f;
  } else {
    for (int i = threadIdx.x; i < n; i += kSampThreads) o[i] = x[i] >= thr ? x[i] * inv : 0.f;
  }
}

template <bool VEC, bool FILTER>
__device__ void renorm_row(const float* __restrict__ x, float* __restrict__ o, int n, const RowParams& rp, SampShared& sh) {
  float kept;
  const float thr = row_threshold<VEC, FILTER>(x, n, rp, sh, kept);
  if (!(kept > 0.f)) {
    float s = 0.f;
    each<VEC>(x, n, [&](float v) { s += v >= thr ? v : 0.f; });
    kept = bsum(s, sh.red);
  }
  write_renormed<VEC>(x, o, n, thr, 1.0f / kept);
}

// kept values of elements i .. i + 3
template <bool VEC>
__device__ __forceinline__ float4v kept_four(const float* __restrict__ x, int n, int64_t i, float thr) {
  float4v v = {0.f, 0.f, 0.f, 0.f};
  if (VEC && i + 4 <= n) {
    v = *reinterpret_cast<const float4v*>(x + i);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (i + e < n) v[e] = x[i + e];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = v[e] >= thr ? v[e] : 0.f;
  return v;
}

// elements a chunk has: at most kBins chunks a row
__host__ __device__ inline int64_t chunk_of(int64_t n) { return 256 * ((n + 256 * kBins - 1) / (256 * kBins)); }

// masses of the kept elements of chunks c0 .. c1 - 1, whole waves at a time
template <bool VEC>
__device__ __forceinline__ void sum_chunks(const float* __restrict__ x, int n, float thr, int64_t chunk, int first, int last,
                                           float* __restrict__ sums) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int c0 = first + wid; c0 < last; c0 += 64) {
    float s[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      s[u] = 0.f;
      const int64_t c = c0 + 16 * u;
      if (c < last)
        for (int64_t i = c * chunk; i < (c + 1) * chunk; i += 256) {
          const float4v v = kept_four<VEC>(x, n, i + 4 * lane, thr);
          s[u] += (v[0] + v[1]) + (v[2] + v[3]);
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      s[u] = wave_sum(s[u]);
      if (lane == 0 && c0 + 16 * u < last) sums[c0 + 16 * u] = s[u];
    }
  }
}

// Inverse CDF over the kept elements in index order: the first kept index whose running sum exceeds u * total.  One wave
// walks the chunk that holds the target from the mass in front of it; c < 0: none does.
template <bool VEC>
__device__ void walk_chunk(const float* __restrict__ x, int n, float thr, int64_t chunk, int c, float run, float target,
                           int32_t* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  int pick = -1;
  if (c >= 0) {
    int last = -1;
    for (int64_t i = c * chunk; i < (c + 1) * chunk && pick < 0; i += 256) {
      const float4v v = kept_four<VEC>(x, n, i + 4 * lane, thr);
      const float sum = (v[0] + v[1]) + (v[2] + v[3]);
      float incl = sum;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const float w = __shfl_up(incl, o, 64);
        if (lane >= o) incl += w;
      }
      float r = run + (incl - sum);
      int at = 1 << 30, mine = -1;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (v[e] > 0.f) {
          r += v[e];
          mine = (int)(i + 4 * lane + e);
          if (r > target) at = min(at, mine);
        }
      }
      // lanes are in the elements' order: the first lane that has one past the target, the last that has one at all
      const u64 past = __ballot(at < (1 << 30)), some = __ballot(mine >= 0);
      if (past) pick = __builtin_amdgcn_readlane(at, __ffsll(past) - 1);
      if (some) last = __builtin_amdgcn_readlane(mine, 63 - __clzll(some));
      run += __shfl(incl, 63, 64);
    }
    if (pick < 0) pick = last;  // rounding at the chunk's end: its last kept element
  }
  if (lane == 0) {
    if (pick < 0) {  // u * total fell on a boundary lost to rounding: the last kept element of the row
      for (int i = n - 1; i >= 0 && pick < 0; --i)
        if (x[i] >= thr) pick = i;
      if (pick < 0) pick = 0;
    }
    *out = pick;
  }
}

// The chunks' masses stand in sh.chunk (zeros behind the last).
template <bool VEC>
__device__ void choose(const float* __restrict__ x, int n, float thr, int64_t chunk, float u, int32_t* __restrict__ out, SampShared& sh) {
  if (threadIdx.x == 0) sh.pick = kBins;
  __syncthreads();
  constexpr int PER = kBins / kSampThreads;
  float m[PER], own = 0.f, total;
#pragma unroll
  for (int j = 0; j < PER; ++j) own += m[j] = sh.chunk[threadIdx.x * PER + j];
  float run = bscan<float>(own, sh.red, total);
  const float target = u * total;
  int first = kBins;
  float at_first = 0.f;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (m[j] > 0.f && first == kBins && target < run + m[j]) first = threadIdx.x * PER + j, at_first = run;
    run += m[j];
  }
  if (first < kBins) atomicMin(&sh.pick, first);
  __syncthreads();
  const int c = sh.pick;
  if (c == first && first < kBins) sh.red[0] = at_first;
  __syncthreads();
  if (threadIdx.x >= 64) return;
  walk_chunk<VEC>(x, n, thr, chunk, c < kBins ? c : -1, sh.red[0], target, out);
}

template <bool VEC, bool FILTER>
__device__ void sample_row(const float* __restrict__ x, int n, const RowParams& rp, float u, int32_t* __restrict__ out, SampShared& sh) {
  float kept;
  const float thr = row_threshold<VEC, FILTER>(x, n, rp, sh, kept);
  const int64_t chunk = chunk_of(n);
  __syncthreads();
  for (int i = threadIdx.x; i < kBins; i += kSampThreads) sh.chunk[i] = 0.f;
  __syncthreads();
  sum_chunks<VEC>(x, n, thr, chunk, 0, (int)((n + chunk - 1) / chunk), sh.chunk);
  __syncthreads();
  choose<VEC>(x, n, thr, chunk, u, out, sh);
}

struct SampArgs {
  const float* probs;
  float* out;               // renormalised rows, or nullptr
  const float* uniform;
  int32_t* ids;
  int n;
  int64_t in_stride, out_stride;
  const int32_t* k_arr;
  const float *p_arr, *m_arr;
  int k_val;
  float p_val, m_val;
  int joint;
  int slices, slice;        // blocks a row is spread over, elements each
  char* ws;
};

__device__ __forceinline__ RowParams load_params(const SampArgs& a, int row) {
  RowParams rp;
  rp.top_k = a.k_arr ? a.k_arr[row] : a.k_val;
  rp.top_p = a.p_arr ? a.p_arr[row] : a.p_val;
  rp.min_p = a.m_arr ? a.m_arr[row] : a.m_val;
  rp.joint = a.joint;
  return rp;
}

// One block per row.  Calls without a top-k or top-p have a kernel of their own: the selection's 128 registers leave room for
// one block a unit (512 rows of 4096, sampling without a filter: 17 us with them, 8.3 without).
template <bool VEC, bool FILTER>
__global__ void __launch_bounds__(kSampThreads) filter_rows_kernel(SampArgs a) {
  __shared__ SampShared sh;
  const int row = blockIdx.x;
  const float* x = a.probs + (int64_t)row * a.in_stride;
  const RowParams rp = load_params(a, row);
  if (a.out)
    renorm_row<VEC, FILTER>(x, a.out + (int64_t)row * a.out_stride, a.n, rp, sh);
  else
    sample_row<VEC, FILTER>(x, a.n, rp, a.uniform[row], a.ids + row, sh);
}

// Short rows without a selection: a block of four waves, a chunk of 256 elements a wave at a time, the choice by one wave of
// a lane a chunk.  Such a row is a handful of loads, and what a block of 1024 threads starts, clears and meets for is most of
// its launch (sampling without a filter, 1024 threads and 256: 512 rows of 4096 8.5 and 5.0 us, with a min-p 11.2 and 5.9;
// one row 5.8 and 4.2.  From 16384 elements on four waves are too few for a row: 64 rows 7.4 and 8.3 us).
constexpr int kShort = 8192;
template <bool VEC>
__global__ void __launch_bounds__(256) short_rows_kernel(SampArgs a) {
  __shared__ float chunk[64], red[4];
  const int row = blockIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6, n = a.n, chunks = (n + 255) / 256;
  const float* x = a.probs + (int64_t)row * a.in_stride;
  const float min_p = load_params(a, row).min_p;
  float thr = 0.f;
  if (threadIdx.x < 64) chunk[threadIdx.x] = 0.f;
  if (min_p > 0.f) {  // block-uniform
    float mx = 0.f;
    for (int c0 = wid; c0 < chunks; c0 += 16) {
      float4v v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = kept_four<VEC>(x, n, (c0 + 4 * j) * 256 + 4 * lane, 0.f);
#pragma unroll
      for (int j = 0; j < 4; ++j) mx = fmaxf(fmaxf(mx, fmaxf(v[j][0], v[j][1])), fmaxf(v[j][2], v[j][3]));
    }
    mx = wave_max(mx);
    if (lane == 0) red[wid] = mx;
  }
  __syncthreads();
  if (min_p > 0.f) thr = fmaxf(0.f, min_p * fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
  for (int c0 = wid; c0 < chunks; c0 += 16) {
    float4v v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = kept_four<VEC>(x, n, (c0 + 4 * j) * 256 + 4 * lane, thr);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float sum = wave_sum((v[j][0] + v[j][1]) + (v[j][2] + v[j][3]));
      if (lane == 0 && c0 + 4 * j < chunks) chunk[c0 + 4 * j] = sum;
    }
  }
  __syncthreads();
  const float m = chunk[lane];
  float incl = m;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float w = __shfl_up(incl, o, 64);
    if (lane >= o) incl += w;
  }
  const float total = __shfl(incl, 63, 64);
  if (a.out) {
    float* o = a.out + (int64_t)row * a.out_stride;
    const float inv = 1.0f / total;
    for (int i = threadIdx.x; i < n; i += 256) o[i] = x[i] >= thr ? x[i] * inv : 0.f;
    return;
  }
  if (wid) return;
  const float target = a.uniform[row] * total;
  const u64 past = __ballot(m > 0.f && target < incl);
  const int c = past ? __ffsll(past) - 1 : -1;
  walk_chunk<VEC>(x, n, thr, 256, c, __shfl(incl - m, max(c, 0), 64), target, a.ids + row);
}

// ---- rows spread over several blocks --------------------------------------------------------------------------------
// A unit streams about 20 bytes a clock of a row that the caches do not hold, and a batch of 64 rows leaves three of four
// units idle.  The same selection in launches that meet at their ends: bins per slice; every block adds its row's bins up
// and collects its slice's candidates; every block finishes the threshold and writes its slice, or, sampling, one block per
// row finishes it and picks.  The first digit has a window of 1024 bins (2^64 of the least value binned).  Rows the guess of mass one does
// not hold for, or whose candidates overflow a list, are done whole by one block of the last launch.
constexpr int kWindow = 1024;
constexpr int kMaxSlices = 16;
struct SliceStat {
  float under, over, vmax, pad;
};
struct RowState {
  u64 below, target, above;
  int valid, kbin, pbin, kcount, pcount;
  uint32_t rank;
  float vmax;
};
struct SampWs {  // of one row
  u64* bins;        // [slices][kWindow]
  SliceStat* stat;  // [slices]
  RowState* state;
  uint32_t* list;   // [2][kList]
  uint32_t* place;  // [2][kList]: where in the row (sampling)
  float* chunk;     // [kBins]
};
__host__ __device__ inline int64_t samp_ws_row(int slices) {
  return (int64_t)slices * (kWindow * 8 + 16) + 128 + 4 * kList * 4 + kBins * 4;
}
__device__ __forceinline__ SampWs samp_ws(const SampArgs& a, int row) {
  char* w = a.ws + (int64_t)row * samp_ws_row(a.slices);
  SampWs r;
  r.bins = reinterpret_cast<u64*>(w);
  w += (int64_t)a.slices * kWindow * 8;
  r.state = reinterpret_cast<RowState*>(w);
  w += 128;
  r.stat = reinterpret_cast<SliceStat*>(w);
  w += a.slices * 16;
  r.list = reinterpret_cast<uint32_t*>(w);
  w += 2 * kList * 4;
  r.place = reinterpret_cast<uint32_t*>(w);
  w += 2 * kList * 4;
  r.chunk = reinterpret_cast<float*>(w);
  return r;
}
static_assert(sizeof(RowState) <= 128, "");

struct Guess {  // what a row of mass one can leave unbinned
  bool use_k, use_p;
  float least;
  Fixed fx;
  int base;
};
__device__ __forceinline__ Guess guess_of(const RowParams& rp, int n) {
  Guess g;
  g.use_k = rp.top_k > 0 && rp.top_k < n;
  g.use_p = rp.top_p < 1.0f;
  const float share = 0.999f * (1.0f - rp.top_p) / (float)n, mean = 1.0f / (float)n;
  g.least = g.use_p ? (g.use_k ? fminf(mean, share) : share) : mean;
  if (!(g.least >= 0.f)) g.least = 0.f;
  g.fx.bits = 32 + __clz(n) - 1;
  g.fx.scale = g.fx.bits - 2;
  g.base = (int)(__float_as_uint(g.least) >> 19);
  return g;
}

// A slice in pieces of four elements, piece u of a thread the (threadIdx.x + 1024 u)-th: a wave's piece is a chunk of 256.
// The first eight are asked for by hold(), before whatever the block has to find out first, and are there when it has; longer
// slices go on from memory.
constexpr int kHeld = 8;
// A wave's piece of rows that cannot be read so holds its elements 64 apart: every load is 64 consecutive elements, not one of four
// of each lane (one row of 50257: renormalised 27.6 us -> 23.8, 64 rows 35.8 -> 28.9).
template <bool VEC>
__device__ __forceinline__ int piece_element(int i, int e) {
  return VEC ? 4 * i + e : 4 * (i & ~63) + 64 * e + (i & 63);
}
template <bool VEC>
__device__ __forceinline__ float4v slice_piece(const float* __restrict__ x, int n, int i) {
  float4v v = {0.f, 0.f, 0.f, 0.f};
  if (VEC && 4 * i + 4 <= n) {
    v = *reinterpret_cast<const float4v*>(x + 4 * i);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (piece_element<VEC>(i, e) < n) v[e] = x[piece_element<VEC>(i, e)];
  }
  return v;
}
// (A slice has 8192 - 15 x 255 elements at least, the last one too.  What does not lie in a whole wave of pieces is read again below.  No branch, so
// that what was asked for before can be waited for without these.)
template <bool VEC>
__device__ __forceinline__ void hold(const float* __restrict__ x, int n, float4v (&r)[kHeld]) {
#pragma unroll
  for (int u = 0; u < kHeld; ++u)
    if constexpr (VEC)
      r[u] = *reinterpret_cast<const float4v*>(x + 4 * min((int)threadIdx.x + u * kSampThreads, (n >> 2) - 1));
  __builtin_amdgcn_sched_barrier(0);
}
// f(piece, its place, elements of it): whole waves, with pieces of no elements behind the slice's end.  Where a wave's pieces are
// whole (a scalar question) they are not asked again element by element: these loops are bound by their instructions, and
// 25 an element instead of ten cost as much as the trip to memory.
template <bool VEC, typename F>
__device__ __forceinline__ void each_piece(const float* __restrict__ x, int n, float4v (&r)[kHeld], F f) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x) & ~63, lane = threadIdx.x & 63;
  int first = wave;
  if constexpr (VEC) {
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
      const int at = wave + u * kSampThreads;
      if (4 * at + 256 <= n) {
        f(r[u], at + lane, 4);
        first = at + kSampThreads;
      }
    }
  }
#pragma unroll 1
  for (; 4 * first < n; first += 4 * kSampThreads) {
    float4v v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = slice_piece<VEC>(x, n, first + lane + u * kSampThreads);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int at = first + u * kSampThreads, i = at + lane;
      if (4 * at < n) f(v[u], i, max(min(VEC ? n - 4 * i : (n - 4 * at - lane + 63) >> 6, 4), 0));
    }
  }
}

// A bin's word: count << 40 | the sum of the 19 bits below its digit.  All its elements share the bits above, so that is their
// exact mass, and adding an element is one 64-bit add of bits that it has already.
constexpr int kCountAt = 40;
__device__ __forceinline__ u64 word_sum(u64 w, int digit) {  // in units of 2^(max(digit / 16, 1) - 150)
  return (w >> kCountAt) * (u64)((digit >> 4 ? 0x800000u : 0u) | ((uint32_t)(digit & 15) << 19)) + (w & ((1ull << kCountAt) - 1));
}

// Draws without a top-k or top-p (FILTER: the call may have one) need no bins, and this launch only for a min-p's largest value.
template <bool VEC, bool FILTER>
__global__ void __launch_bounds__(kSampThreads) slice_bins_kernel(SampArgs a) {
  __shared__ u64 bins[kWindow];
  __shared__ float red[3][16];
  const int slice = blockIdx.x, row = blockIdx.y, lo = slice * a.slice, n = min(a.slice, a.n - lo);
  const float* x = a.probs + (int64_t)row * a.in_stride + lo;
  float4v held[kHeld];
  hold<VEC>(x, n, held);
  const RowParams rp = load_params(a, row);
  const Guess g = guess_of(rp, a.n);
  const SampWs w = samp_ws(a, row);
  bins[threadIdx.x] = 0;
  __syncthreads();
  float s = 0.f, mx = 0.f;
  const bool bin = FILTER && (g.use_k || g.use_p);
  const float least = bin ? g.least : __uint_as_float(0x7FC00000u);  // without a filter nothing is binned
  each_piece<VEC>(x, n, held, [&](const float4v& piece, int, int have) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float raw = e < have ? piece[e] : -1.f, v = fmaxf(raw, 0.f);
      const bool in = FILTER && raw >= least;
      mx = fmaxf(mx, v);
      s += in ? 0.f : v;
      if (in) {
        const uint32_t b = __float_as_uint(raw);
        atomicAdd(&bins[min((int)(b >> 19) - g.base, kWindow - 1)], (1ull << kCountAt) | (b & 0x7FFFFu));
      }
    }
  });
  __syncthreads();
  const u64 word = bins[threadIdx.x];
  // the window's last bin takes what lies beyond it: no mass of such a row is known
  float o = threadIdx.x < kWindow - 1 ? ldexpf((float)word_sum(word, g.base + threadIdx.x), max((g.base + (int)threadIdx.x) >> 4, 1) - 150) : word ? __uint_as_float(0x7F800000u) : 0.f;
  s = wave_sum(s), o = wave_sum(o), mx = wave_max(mx);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) red[0][wid] = s, red[1][wid] = o, red[2][wid] = mx;
  if (bin) w.bins[slice * kWindow + threadIdx.x] = word;
  __syncthreads();
  if (threadIdx.x == 0) {
    SliceStat st{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 16; ++t) st.under += red[0][t], st.over += red[1][t], st.vmax = fmaxf(st.vmax, red[2][t]);
    w.stat[slice] = st;
  }
}

// SUM (sampling): also the masses of the chunks, of what is kept whatever the cut inside its bin turns out to be; the
// bin's own elements are listed with their places and added by the last launch.
template <bool VEC, bool SUM, bool FILTER>
__global__ void __launch_bounds__(kSampThreads) slice_collect_kernel(SampArgs a) {
  __shared__ u64 bins[kWindow];
  __shared__ u64 ured[16];
  __shared__ uint32_t list[2][kList], place[SUM ? 2 : 1][SUM ? kList : 1];
  __shared__ uint32_t cut[2], fill[2], start[2], need;
  __shared__ u64 below;
  const int slice = blockIdx.x, row = blockIdx.y, lo = slice * a.slice, n = min(a.slice, a.n - lo);
  const float* x = a.probs + (int64_t)row * a.in_stride + lo;
  const RowParams rp = load_params(a, row);
  const SampWs w = samp_ws(a, row);
  const Guess g = guess_of(rp, a.n);
  const bool bin = FILTER && (g.use_k || g.use_p);
  // what the slices left (a lane a slice for the sums), then the slice itself: it arrives while the cuts are found
  const int lane = threadIdx.x & 63;
  float4v stat, held[kHeld];
  u64 word = 0;
  uint32_t ahead = 0;  // elements of this thread's bin in the slices in front
  auto ask = [&](auto most) {
    u64 part[decltype(most)::value];
    stat = *reinterpret_cast<const float4v*>(w.stat + min(lane, a.slices - 1));
#pragma unroll
    for (int t = 0; t < most; ++t) part[t] = w.bins[min(t, a.slices - 1) * kWindow + threadIdx.x];  // (not written without a filter)
    __builtin_amdgcn_sched_barrier(0);
    hold<VEC>(x, n, held);
#pragma unroll
    for (int t = 0; t < most; ++t) {
      word += t < a.slices ? part[t] : 0;
      ahead += t < slice ? (uint32_t)(part[t] >> kCountAt) : 0;
    }
  };
  if constexpr (!FILTER) {
    stat = *reinterpret_cast<const float4v*>(w.stat + min(lane, a.slices - 1));  // (not written without a min-p)
    hold<VEC>(x, n, held);
  } else if (a.slices <= 4)
    ask(std::integral_constant<int, 4>());
  else
    ask(std::integral_constant<int, kMaxSlices>());
  if (lane >= a.slices) stat = float4v{0.f, 0.f, 0.f, 0.f};
  RowState st{};
  double under = stat[0], total = (double)stat[0] + (double)stat[1];  // the first row of lanes has them all
  auto ror = [](double v, auto ctrl) {
    const u64 b = __builtin_bit_cast(u64, v);
    return __builtin_bit_cast(double, ((u64)dpp<decltype(ctrl)::value>((uint32_t)(b >> 32)) << 32) | dpp<decltype(ctrl)::value>((uint32_t)b));
  };
  auto turn = [&](auto ctrl) {
    under += ror(under, ctrl);
    total += ror(total, ctrl);
    st.vmax = fmaxf(st.vmax, __uint_as_float(dpp<decltype(ctrl)::value>(__float_as_uint(st.vmax))));
  };
  st.vmax = stat[2];
  turn(std::integral_constant<int, kDppRor8>());
  turn(std::integral_constant<int, kDppRor4>());
  turn(std::integral_constant<int, kDppXor2>());
  turn(std::integral_constant<int, kDppXor1>());
  auto first_lane = [](double v) {
    const u64 b = __builtin_bit_cast(u64, v);
    return __builtin_bit_cast(double, ((u64)(uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32) |
                                          (uint32_t)__builtin_amdgcn_readfirstlane((int)b));
  };
  under = first_lane(under), total = first_lane(total);
  st.vmax = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(st.vmax)));
  st.valid = 1;
  st.kbin = st.pbin = -1;
  if (bin) {
    // counts and masses in front of this thread's bin in one scan of packed words (masses that do not fit are no valid row's)
    const int digit = g.base + threadIdx.x, up = max(digit >> 4, 1) - 150 + g.fx.scale;
    const u64 whole = word_sum(word, digit), mass = up >= 0 ? whole << (up & 63) : up > -64 ? whole >> (-up & 63) : 0;
    const u64 sum = ((word >> kCountAt) << g.fx.bits) + mass;
    bins[threadIdx.x] = sum;
    u64 words;
    const u64 before = bscan<u64>(sum, ured, words);
    const uint32_t all = g.fx.count(words), c = g.fx.count(sum), behind = all - g.fx.count(before) - c;
    const u64 low = (u64)ldexp(under, g.fx.scale), m = g.fx.mass(sum), run = low + g.fx.mass(before);
    st.target = max((u64)fmin(ceil((double)(1.0f - rp.top_p) * (double)(low + g.fx.mass(words))), 4e18), (u64)1);
    // the whole-row form's checks, and the window's
    st.valid = total > 0.2 && total < 1.99 && all > 0 && (!g.use_k || (int)all >= rp.top_k) &&
               (!g.use_p || (under < (double)(1.0f - rp.top_p) * total && low + g.fx.mass(words) >= st.target && low < st.target));
    if (st.valid && g.use_k && behind < (uint32_t)rp.top_k && (uint32_t)rp.top_k <= behind + c) {
      cut[0] = threadIdx.x;
      start[0] = ahead;
      need = rp.top_k - behind;
    }
    if (st.valid && g.use_p && m > 0 && run < st.target && run + m >= st.target) {
      cut[1] = threadIdx.x;
      start[1] = ahead;
      below = run;
    }
    __syncthreads();
    if (st.valid && g.use_k) {
      st.kbin = cut[0];
      st.rank = need;
      st.kcount = (int)g.fx.count(bins[st.kbin]);
    }
    if (st.valid && g.use_p) {
      st.pbin = cut[1];
      st.below = below;
      st.pcount = (int)g.fx.count(bins[st.pbin]);
    }
    if (st.kcount > kList || st.pcount > kList) st.valid = 0;
    // for the kept mass: of the bins behind the cut
    if (st.valid && (int)threadIdx.x == (g.use_k ? st.kbin : st.pbin)) ured[0] = g.fx.mass(words) - g.fx.mass(before) - m;
    if (threadIdx.x < 2) fill[threadIdx.x] = 0;
    __syncthreads();
    st.above = ured[0];
  }
  if (slice == 0 && threadIdx.x == 0) *w.state = st;
  if ((!bin && !SUM) || !st.valid) return;  // block-uniform, the same in every block of the row
  // the elements of a bin: bit patterns of one range (negative values and what is no number lie outside), from `least` on
  const uint32_t from = __float_as_uint(g.least);
  auto range = [&](int d, uint32_t& lo_bits, uint32_t& span) {
    const uint32_t first = (uint32_t)(d + g.base) << 19;
    lo_bits = max(first, from);
    span = d < 0 ? 0u : first + (1u << 19) - lo_bits;
  };
  uint32_t klo, kspan, plo, pspan;
  range(st.kbin, klo, kspan);
  range(st.pbin, plo, pspan);
  // kept for certain: what lies behind the bins, and from the min-p threshold on
  const int last = max(st.kbin, st.pbin);
  const float sure = fmaxf(bin ? __uint_as_float((uint32_t)(last + 1 + g.base) << 19) : 0.f, rp.min_p > 0.f ? rp.min_p * st.vmax : 0.f);
  each_piece<VEC>(x, n, held, [&](const float4v& piece, int at, int have) {
    float sums[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float raw = e < have ? piece[e] : -1.f;
      const uint32_t b = __float_as_uint(raw);
      if (b - klo < kspan) {
        const uint32_t to = atomicAdd(&fill[0], 1u);
        list[0][to] = b;
        if (SUM) place[0][to] = lo + piece_element<VEC>(at, e);
      }
      if (b - plo < pspan) {
        const uint32_t to = atomicAdd(&fill[1], 1u);
        list[1][to] = b;
        if (SUM) place[SUM][to] = lo + piece_element<VEC>(at, e);
      }
      sums[e] = raw >= sure ? raw : 0.f;
    }
    if (SUM) {
      const float mass = wave_sum((sums[0] + sums[1]) + (sums[2] + sums[3]));
      if (lane == 0) w.chunk[(lo >> 8) + (at >> 6)] = mass;
    }
  });
  if (!bin) return;
  __syncthreads();
  // behind what the slices in front have in the bins (in any order: what is taken from the lists does not depend on it)
#pragma unroll
  for (int t = 0; t < 2; ++t)
    for (int i = threadIdx.x; i < (int)fill[t]; i += kSampThreads) {
      w.list[t * kList + start[t] + i] = list[t][i];
      if (SUM) w.place[t * kList + start[t] + i] = place[SUM ? t : 0][i];
    }
}

struct HeldLists {
  uint32_t got[2][kList / kSampThreads];
  __device__ __forceinline__ void load(const uint32_t* from) {  // whatever stands behind the lists' ends is not looked at
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < kList / kSampThreads; ++j) got[t][j] = from[t * kList + threadIdx.x + j * kSampThreads];
  }
};

// The row's threshold from its candidates, which lie two a thread and list in registers: digits of 6, 6 and 7 bits, counted by the
// whole block and picked by a wave a list (a wave that walks a list of two thousand by itself takes 6 us).  Block-uniform.
__device__ __forceinline__ float finish_threshold(SampShared& sh, const HeldLists& lists, const RowParams& rp, const Guess& g,
                                                  const RowState& st) {
  float thr = 0.f;
  if (g.use_k || g.use_p) {
    const int wid = threadIdx.x >> 6;
    constexpr int kOwn = kList / kSampThreads;
    if (wid < 2) sh.digit[wid][threadIdx.x & 63] = sh.digit[wid][64 + (threadIdx.x & 63)] = 0;
    uint32_t prefix[2] = {(uint32_t)(st.kbin + g.base) << 19, (uint32_t)(st.pbin + g.base) << 19};
    const int listed[2] = {g.use_k ? st.kcount : 0, g.use_p ? st.pcount : 0};
    u64 word[2][kOwn];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < kOwn; ++j) word[t][j] = (1ull << g.fx.bits) + g.fx.of(lists.got[t][j]);
    uint32_t rank = st.rank;
    u64 below = st.below;
    int bits = 19;
    __syncthreads();
#pragma unroll
    for (int digit = 0; digit < 3; ++digit) {
      const int take = digit < 2 ? 6 : 7, shift = bits - take;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < kOwn; ++j) {
          const uint32_t b = lists.got[t][j];
          if ((int)threadIdx.x + j * kSampThreads < listed[t] && (b >> bits) == (prefix[t] >> bits))
            atomicAdd(&sh.digit[t][(b >> shift) & ((1u << take) - 1)], word[t][j]);
        }
      __syncthreads();
      if (wid < 2) {
        u64 unused = 0;
        const int d = wid ? pick_digit<false>(sh.digit[1], g.fx, rank, below, max(st.target, (u64)1))
                          : pick_digit<true>(sh.digit[0], g.fx, rank, unused, 0);
        sh.cut[wid] = d;
      }
      __syncthreads();
      prefix[0] |= sh.cut[0] << shift, prefix[1] |= sh.cut[1] << shift;
      bits = shift;
    }
    thr = fmaxf(g.use_k ? __uint_as_float(prefix[0]) : 0.f, g.use_p ? __uint_as_float(prefix[1]) : 0.f);
  }
  return rp.min_p > 0.f ? fmaxf(thr, rp.min_p * st.vmax) : thr;
}

template <bool VEC>
__global__ void __launch_bounds__(kSampThreads) slice_apply_kernel(SampArgs a) {
  __shared__ SampShared sh;
  const int slice = blockIdx.x, row = blockIdx.y, lo = slice * a.slice, n = min(a.slice, a.n - lo);
  const float* x = a.probs + (int64_t)row * a.in_stride + lo;
  const SampWs w = samp_ws(a, row);
  const RowState st = *w.state;
  HeldLists lists;
  lists.load(w.list);
  float4v held[kHeld];
  hold<VEC>(x, n, held);
  const RowParams rp = load_params(a, row);
  const Guess g = guess_of(rp, a.n);
  if (!st.valid) return;  // block-uniform
  const float thr = finish_threshold(sh, lists, rp, g, st);
  float kept = -1.f;
  if (g.use_k != g.use_p) {
    u64 part = 0, all;
#pragma unroll
    for (int j = 0; j < kList / kSampThreads; ++j) {
      const uint32_t b = g.use_k ? lists.got[0][j] : lists.got[1][j];
      if ((int)threadIdx.x + j * kSampThreads < (g.use_k ? st.kcount : st.pcount) && __uint_as_float(b) >= thr) part += g.fx.of(b);
    }
    bscan<u64>(part, sh.ured, all);
    kept = (float)ldexp((double)(st.above + all), -g.fx.scale);
  }
  if (!(kept > 0.f)) {  // no filter: the whole row's mass
    kept = 0.f;
    for (int t = 0; t < a.slices; ++t) kept += w.stat[t].under + w.stat[t].over;
  }
  const float inv = 1.0f / kept;
  float* o = a.out + (int64_t)row * a.out_stride + lo;
  each_piece<VEC>(x, n, held, [&](const float4v& piece, int at, int have) {
    float4v v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = piece[e] >= thr ? piece[e] * inv : 0.f;
    if (VEC && have == 4) {
      *reinterpret_cast<float4v*>(o + 4 * at) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e < have) o[piece_element<VEC>(at, e)] = v[e];
    }
  });
}

// Renormalised rows that the guess did not hold for, a block a row (48 rows of 256000 nearly equal values 126 us; 132 in the
// kernel that samples, whose registers it shared).
template <bool VEC>
__global__ void __launch_bounds__(kSampThreads) slice_redo_kernel(SampArgs a) {
  __shared__ SampShared sh;
  const int row = blockIdx.x;
  if (samp_ws(a, row).state->valid) return;
  renorm_row<VEC, true>(a.probs + (int64_t)row * a.in_stride, a.out + (int64_t)row * a.out_stride, a.n, load_params(a, row), sh);
}

// A block a row that is sampled from: the choice, and all of it where the guess did not hold.
template <bool VEC, bool FILTER>
__global__ void __launch_bounds__(kSampThreads) slice_choose_kernel(SampArgs a) {
  __shared__ SampShared sh;
  const int row = blockIdx.x;
  const float* x = a.probs + (int64_t)row * a.in_stride;
  const SampWs w = samp_ws(a, row);
  const RowParams rp = load_params(a, row);
  constexpr int PER = kBins / kSampThreads;
  const int chunks = (a.n + 255) / 256;
  HeldLists lists, places;
  if constexpr (FILTER) {
    lists.load(w.list);
    places.load(w.place);
  }
  float mass[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) mass[j] = w.chunk[min((int)threadIdx.x + j * kSampThreads, chunks - 1)];
  const RowState st = *w.state;
  float thr;
  if constexpr (FILTER) {
    if (!st.valid) {
      sample_row<VEC, true>(x, a.n, rp, a.uniform[row], a.ids + row, sh);
      return;
    }
    const Guess g = guess_of(rp, a.n);
    for (int i = threadIdx.x; i < min(chunks, kBins); i += kSampThreads) sh.bin[i] = 0;
    thr = finish_threshold(sh, lists, rp, g, st);  // a block barrier, or no elements to add
    // the cut bin's kept elements, in whole numbers: the same in any order
    const int which = st.kbin >= st.pbin ? 0 : 1, listed = which ? st.pcount : st.kcount;
    if (g.use_k || g.use_p) {
#pragma unroll
      for (int j = 0; j < kList / kSampThreads; ++j) {
        const uint32_t b = which ? lists.got[1][j] : lists.got[0][j], at = which ? places.got[1][j] : places.got[0][j];
        if ((int)threadIdx.x + j * kSampThreads < listed && __uint_as_float(b) >= thr) atomicAdd(&sh.bin[at >> 8], g.fx.of(b));
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int i = threadIdx.x + j * kSampThreads;
      mass[j] = i < chunks ? mass[j] + (float)ldexp((double)sh.bin[i], -g.fx.scale) : 0.f;
    }
    __syncthreads();  // the masses take the place of the sums
  } else {
    thr = rp.min_p > 0.f ? fmaxf(0.f, rp.min_p * st.vmax) : 0.f;
#pragma unroll
    for (int j = 0; j < PER; ++j) mass[j] = (int)threadIdx.x + j * kSampThreads < chunks ? mass[j] : 0.f;
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) sh.chunk[threadIdx.x + j * kSampThreads] = mass[j];
  __syncthreads();
  choose<VEC>(x, a.n, thr, 256, a.uniform[row], a.ids + row, sh);
}

// Blocks a row is spread over: at least 8192 elements each, and one block a unit at most (what a block scans and waits for
// does not shrink with its share: 64 rows over 512 blocks took 155 us for sampling and renormalisation, over 256 85 us,
// unspread 152 us).
static int samp_slices(int64_t batch, int64_t n) {
  if (batch <= 0 || n > 256 * kBins) return 1;
  const int64_t s = std::min<int64_t>({kMaxSlices, n / 8192, 256 / batch});
  return (int)std::max<int64_t>(s, 1);
}

static int launch_filters(SampArgs a, int batch, void* workspace, int64_t workspace_bytes, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  const bool vec = aligned16(a.probs) && a.in_stride % 4 == 0 && (!a.out || (aligned16(a.out) && a.out_stride % 4 == 0));
  const bool both_in_turn = !a.joint && (a.k_arr || a.k_val > 0) && (a.p_arr || a.p_val < 1.f);  // top-p over the k largest
  const bool filter = a.k_arr || (a.k_val > 0 && a.k_val < a.n) || a.p_arr || a.p_val < 1.f;
  a.slices = samp_slices(batch, a.n);
  // Without a selection to share out, one block a row is the faster one up to 32768 elements (us, a block and spread: 64 rows of
  // 16384 8.4 and 9.9, of 32000 11.5 and 10.3, with a min-p 12.2 and 13.7; of 50304 14.6 and 11.7, 15.5 and 15.9; of 128256 25.2
  // and 14.5, 29.0 and 20.0; one row of 50304 10.8 and 9.6, 13.1 and 13.3, of 128256 19.4 and 9.3, 22.7 and 12.7).
  if (a.slices < 2 || (!filter && a.n <= 32768) || both_in_turn || batch > 65535 || !workspace || (reinterpret_cast<uintptr_t>(workspace) & 15) ||
      workspace_bytes < samp_ws_row(a.slices) * batch) {
    if (!filter && a.n <= kShort) {
      hipLaunchKernelGGL(vec ? short_rows_kernel<true> : short_rows_kernel<false>, dim3(batch), dim3(256), 0, s, a);
      SGLK_LAUNCH_CHECK();
      return SGLK_OK;
    }
    const auto kernel = filter ? (vec ? filter_rows_kernel<true, true> : filter_rows_kernel<false, true>)
                               : (vec ? filter_rows_kernel<true, false> : filter_rows_kernel<false, false>);
    hipLaunchKernelGGL(kernel, dim3(batch), dim3(kSampThreads), 0, s, a);
    SGLK_LAUNCH_CHECK();
    return SGLK_OK;
  }
  a.slice = (int)(((int64_t)a.n + a.slices * 256 - 1) / (a.slices * 256) * 256);
  a.slices = (a.n + a.slice - 1) / a.slice;
  a.ws = (char*)workspace;
  const dim3 grid(a.slices, batch), block(kSampThreads);
  if (!filter && !a.out) {
    if (a.m_arr || a.m_val > 0.f)
      hipLaunchKernelGGL((vec ? slice_bins_kernel<true, false> : slice_bins_kernel<false, false>), grid, block, 0, s, a);
    hipLaunchKernelGGL((vec ? slice_collect_kernel<true, true, false> : slice_collect_kernel<false, true, false>), grid, block, 0, s, a);
    hipLaunchKernelGGL((vec ? slice_choose_kernel<true, false> : slice_choose_kernel<false, false>), dim3(batch), block, 0, s, a);
    SGLK_LAUNCH_CHECK();
    return SGLK_OK;
  }
  hipLaunchKernelGGL((vec ? slice_bins_kernel<true, true> : slice_bins_kernel<false, true>), grid, block, 0, s, a);
  if (a.out) {
    hipLaunchKernelGGL((vec ? slice_collect_kernel<true, false, true> : slice_collect_kernel<false, false, true>), grid, block, 0, s, a);
    hipLaunchKernelGGL(vec ? slice_apply_kernel<true> : slice_apply_kernel<false>, grid, block, 0, s, a);
    hipLaunchKernelGGL(vec ? slice_redo_kernel<true> : slice_redo_kernel<false>, dim3(batch), block, 0, s, a);
  } else {
    hipLaunchKernelGGL((vec ? slice_collect_kernel<true, true, true> : slice_collect_kernel<false, true, true>), grid, block, 0, s, a);
    hipLaunchKernelGGL((vec ? slice_choose_kernel<true, true> : slice_choose_kernel<false, true>), dim3(batch), block, 0, s, a);
  }
  SGLK_LAUNCH_CHECK();
  return SGLK_OK;
}

}  // namespace
}  // namespace sglk

using namespace sglk;

extern "C" {

int64_t sglk_sampling_workspace_bytes(int batch, int vocab) {
  const int slices = vocab > 0 ? samp_slices(batch, vocab) : 1;
  return slices < 2 ? 0 : samp_ws_row(slices) * batch;
}

int sglk_top_k_renorm_probs_ws(const float* probs, float* out, const int32_t* top_k_arr, int top_k_val, int batch, int vocab,
                               int64_t in_stride, int64_t out_stride, void* workspace, int64_t workspace_bytes, void* stream) {
  SGLK_CHECK(batch >= 0 && vocab > 0 && in_stride >= vocab && out_stride >= vocab, "top_k_renorm_probs: bad shape");
  if (batch == 0) return SGLK_OK;
  SGLK_CHECK(probs && out, "top_k_renorm_probs: null pointer");
  SampArgs a{};
  a.probs = probs, a.out = out, a.n = vocab, a.in_stride = in_stride, a.out_stride = out_stride;
  a.k_arr = top_k_arr, a.k_val = top_k_val, a.p_val = 1.0f, a.joint = 1;
  return launch_filters(a, batch, workspace, workspace_bytes, stream);
}

int sglk_top_k_renorm_probs(const float* probs, float* out, const int32_t* top_k_arr, int top_k_val, int batch, int vocab,
                            int64_t in_stride, int64_t out_stride, void* stream) {
  return sglk_top_k_renorm_probs_ws(probs, out, top_k_arr, top_k_val, batch, vocab, in_stride, out_stride, nullptr, 0, stream);
}

int sglk_top_p_renorm_probs_ws(const float* probs, float* out, const float* top_p_arr, float top_p_val, int batch, int vocab,
                               int64_t in_stride, int64_t out_stride, void* workspace, int64_t workspace_bytes, void* stream) {
  SGLK_CHECK(batch >= 0 && vocab > 0 && in_stride >= vocab && out_stride >= vocab, "top_p_renorm_probs: bad shape");
  if (batch == 0) return SGLK_OK;
  SGLK_CHECK(probs && out, "top_p_renorm_probs: null pointer");
  SampArgs a{};
  a.probs = probs, a.out = out, a.n = vocab, a.in_stride = in_stride, a.out_stride = out_stride;
  a.p_arr = top_p_arr, a.p_val = top_p_val, a.joint = 1;
  return launch_filters(a, batch, workspace, workspace_bytes, stream);
}

int sglk_top_p_renorm_probs(const float* probs, float* out, const float* top_p_arr, float top_p_val, int batch, int vocab,
                            int64_t in_stride, int64_t out_stride, void* stream) {
  return sglk_top_p_renorm_probs_ws(probs, out, top_p_arr, top_p_val, batch, vocab, in_stride, out_stride, nullptr, 0, stream);
}

int sglk_sampling_from_probs_ws(const float* probs, const float* uniform, int32_t* out, const int32_t* top_k_arr, int top_k_val,
                                const float* top_p_arr, float top_p_val, const float* min_p_arr, float min_p_val, int joint,
                                int batch, int vocab, int64_t in_stride, void* workspace, int64_t workspace_bytes, void* stream) {
  SGLK_CHECK(batch >= 0 && vocab > 0 && in_stride >= vocab, "sampling_from_probs: bad shape");
  if (batch == 0) return SGLK_OK;
  SGLK_CHECK(probs && uniform && out, "sampling_from_probs: null pointer");
  SampArgs a{};
  a.probs = probs, a.uniform = uniform, a.ids = out, a.n = vocab, a.in_stride = in_stride;
  a.k_arr = top_k_arr, a.k_val = top_k_val, a.p_arr = top_p_arr, a.p_val = top_p_val, a.m_arr = min_p_arr, a.m_val = min_p_val;
  a.joint = joint ? 1 : 0;
  return launch_filters(a, batch, workspace, workspace_bytes, stream);
}

int sglk_sampling_from_probs(const float* probs, const float* uniform, int32_t* out, const int32_t* top_k_arr, int top_k_val,
                             const float* top_p_arr, float top_p_val, const float* min_p_arr, float min_p_val, int joint,
                             int batch, int vocab, int64_t in_stride, void* stream) {
  return sglk_sampling_from_probs_ws(probs, uniform, out, top_k_arr, top_k_val, top_p_arr, top_p_val, min_p_arr, min_p_val, joint,
                                     batch, vocab, in_stride, nullptr, 0, stream);
}
}
