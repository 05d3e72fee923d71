// Probability filters and inverse-CDF sampling for the sampler's GPU path (top-k / top-p / min-p): one block per row.
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
// Measured, 64 rows of 128256, top-k and top-p together: sampling 555 -> 81 us, top-p renormalisation 390 -> 66 us (256
// bins for four 8-bit digits each, a float atomic on a handful of exponents for every element, and a thread's elements
// 500 bytes from the next thread's).
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
  float red[16];
  u64 ured[16];
  uint32_t fill[2];
  int pick, last;
  u64 below, below_last;
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
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const V u = __shfl_up(incl, o, 64);
    if ((int)(threadIdx.x & 63) >= o) incl += u;
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

// f(value) for every element of the row
template <bool VEC, typename F>
__device__ __forceinline__ void each(const float* __restrict__ x, int n, F f) {
  if constexpr (VEC) {
    const int n4 = n >> 2;
    constexpr int U = 8;  // loads in flight
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
// bin with mass.  sh.below: the mass in front of the bin
template <int PER>
__device__ __forceinline__ int pick_mass(SampShared& sh, const Fixed& fx, u64 below, u64 target) {
  if (threadIdx.x == 0) {
    sh.pick = kBins;
    sh.last = -1;
  }
  u64 m[PER], own = 0, total;
#pragma unroll
  for (int j = 0; j < PER; ++j) own += m[j] = fx.mass(sh.bin[threadIdx.x * PER + j]);
  u64 run = below + bscan<u64>(own, sh.ured, total);  // also: pick and last are set
  int first = kBins, last = -1;
  u64 at_first = run, at_last = run;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (m[j] > 0) {
      if (run + m[j] >= target && first == kBins) first = threadIdx.x * PER + j, at_first = run;
      last = threadIdx.x * PER + j, at_last = run;
    }
    run += m[j];
  }
  if (first < kBins) atomicMin(&sh.pick, first);
  if (last >= 0) atomicMax(&sh.last, last);
  __syncthreads();
  if (sh.pick == first && first < kBins) sh.below = at_first;
  if (sh.last == last && last >= 0) sh.below_last = at_last;
  __syncthreads();
  const bool found = sh.pick < kBins;
  const int d = found ? sh.pick : max(sh.last, 0);
  if (!found && threadIdx.x == 0) sh.below = sh.last >= 0 ? sh.below_last : below;
  __syncthreads();
  return d;
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

struct RowParams {
  int top_k;      // <= 0 or >= n: no top-k filter
  float top_p;    // >= 1: no top-p filter
  float min_p;    // <= 0: no min-p filter
  int joint;      // 1: both filters on the original distribution; 0: top-p on the top-k renormalised one
};

// Threshold of the kept set {x >= thr} for the row's filters.  kept: its mass where one filter was applied and the chosen
// bin's elements were listed, else negative
template <bool VEC>
__device__ float row_threshold(const float* __restrict__ x, int n, const RowParams& rp, SampShared& sh, float& kept) {
  constexpr int PER = kBins / kSampThreads;
  const bool use_k = rp.top_k > 0 && rp.top_k < n, use_p = rp.top_p < 1.0f;
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

__device__ __forceinline__ RowParams load_params(int row, const int32_t* k_arr, int k_val, const float* p_arr, float p_val,
                                                 const float* m_arr, float m_val, int joint) {
  RowParams rp;
  rp.top_k = k_arr ? k_arr[row] : k_val;
  rp.top_p = p_arr ? p_arr[row] : p_val;
  rp.min_p = m_arr ? m_arr[row] : m_val;
  rp.joint = joint;
  return rp;
}

template <bool VEC>
__global__ void __launch_bounds__(kSampThreads) renorm_kernel(const float* __restrict__ probs, float* __restrict__ out,
                                                             int n, int64_t in_stride, int64_t out_stride,
                                                             const int32_t* k_arr, int k_val, const float* p_arr,
                                                             float p_val) {
  __shared__ SampShared sh;
  const int row = blockIdx.x;
  const float* x = probs + (int64_t)row * in_stride;
  const RowParams rp = load_params(row, k_arr, k_val, p_arr, p_val, nullptr, 0.f, 1);
  float kept;
  const float thr = row_threshold<VEC>(x, n, rp, sh, kept);
  if (!(kept > 0.f)) {
    float s = 0.f;
    each<VEC>(x, n, [&](float v) { s += v >= thr ? v : 0.f; });
    kept = bsum(s, sh.red);
  }
  const float inv = 1.0f / kept;
  float* o = out + (int64_t)row * out_stride;
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

// Inverse CDF over the kept elements in index order: the first kept index whose running sum exceeds u * total.  The row
// is summed in chunks of whole waves; the chunk that holds the target is walked again by one wave.
template <bool VEC>
__global__ void __launch_bounds__(kSampThreads) sample_kernel(const float* __restrict__ probs,
                                                             const float* __restrict__ uniform, int32_t* __restrict__ out,
                                                             int n, int64_t in_stride, const int32_t* k_arr, int k_val,
                                                             const float* p_arr, float p_val, const float* m_arr,
                                                             float m_val, int joint) {
  __shared__ SampShared sh;
  const int row = blockIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const float* x = probs + (int64_t)row * in_stride;
  const RowParams rp = load_params(row, k_arr, k_val, p_arr, p_val, m_arr, m_val, joint);
  float kept;
  const float thr = row_threshold<VEC>(x, n, rp, sh, kept);
  auto four = [&](int64_t i) {  // kept values of elements i .. i + 3
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
  };
  const int64_t chunk = 256 * (((int64_t)n + 256 * kBins - 1) / (256 * kBins));  // at most kBins chunks
  const int chunks = (int)((n + chunk - 1) / chunk);
  __syncthreads();
  for (int i = threadIdx.x; i < kBins; i += kSampThreads) sh.chunk[i] = 0.f;
  __syncthreads();
  for (int c0 = wid; c0 < chunks; c0 += 64) {
    float s[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      s[u] = 0.f;
      const int64_t c = c0 + 16 * u;
      if (c < chunks)
        for (int64_t i = c * chunk; i < (c + 1) * chunk; i += 256) {
          const float4v v = four(i + 4 * lane);
          s[u] += (v[0] + v[1]) + (v[2] + v[3]);
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      s[u] = wave_sum(s[u]);
      if (lane == 0 && c0 + 16 * u < chunks) sh.chunk[c0 + 16 * u] = s[u];
    }
  }
  if (threadIdx.x == 0) sh.pick = kBins;
  __syncthreads();
  constexpr int PER = kBins / kSampThreads;
  float m[PER], own = 0.f, total;
#pragma unroll
  for (int j = 0; j < PER; ++j) own += m[j] = sh.chunk[threadIdx.x * PER + j];
  float run = bscan<float>(own, sh.red, total);
  const float target = uniform[row] * total;
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
  if (wid != 0) return;
  int pick = -1;
  if (c < kBins) {
    run = sh.red[0];
    int last = -1;
    for (int64_t i = c * chunk; i < (c + 1) * chunk && pick < 0; i += 256) {
      const float4v v = four(i + 4 * lane);
      const float sum = (v[0] + v[1]) + (v[2] + v[3]);
      float incl = sum;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const float u = __shfl_up(incl, o, 64);
        if (lane >= o) incl += u;
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
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        at = min(at, __shfl_xor(at, o, 64));
        mine = max(mine, __shfl_xor(mine, o, 64));
      }
      if (at < (1 << 30)) pick = at;
      last = max(last, mine);
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
    out[row] = pick;
  }
}

}  // namespace
}  // namespace sglk

using namespace sglk;

extern "C" {

int sglk_top_k_renorm_probs(const float* probs, float* out, const int32_t* top_k_arr, int top_k_val, int batch, int vocab,
                            int64_t in_stride, int64_t out_stride, void* stream) {
  SGLK_CHECK(batch >= 0 && vocab > 0 && in_stride >= vocab && out_stride >= vocab, "top_k_renorm_probs: bad shape");
  if (batch == 0) return SGLK_OK;
  SGLK_CHECK(probs && out, "top_k_renorm_probs: null pointer");
  const bool vec = aligned16(probs) && aligned16(out) && in_stride % 4 == 0 && out_stride % 4 == 0;
  hipLaunchKernelGGL(vec ? renorm_kernel<true> : renorm_kernel<false>, dim3(batch), dim3(kSampThreads), 0, (hipStream_t)stream,
                     probs, out, vocab, in_stride, out_stride, top_k_arr, top_k_val, (const float*)nullptr, 1.0f);
  SGLK_LAUNCH_CHECK();
  return SGLK_OK;
}

int sglk_top_p_renorm_probs(const float* probs, float* out, const float* top_p_arr, float top_p_val, int batch, int vocab,
                            int64_t in_stride, int64_t out_stride, void* stream) {
  SGLK_CHECK(batch >= 0 && vocab > 0 && in_stride >= vocab && out_stride >= vocab, "top_p_renorm_probs: bad shape");
  if (batch == 0) return SGLK_OK;
  SGLK_CHECK(probs && out, "top_p_renorm_probs: null pointer");
  const bool vec = aligned16(probs) && aligned16(out) && in_stride % 4 == 0 && out_stride % 4 == 0;
  hipLaunchKernelGGL(vec ? renorm_kernel<true> : renorm_kernel<false>, dim3(batch), dim3(kSampThreads), 0, (hipStream_t)stream,
                     probs, out, vocab, in_stride, out_stride, (const int32_t*)nullptr, 0, top_p_arr, top_p_val);
  SGLK_LAUNCH_CHECK();
  return SGLK_OK;
}

int sglk_sampling_from_probs(const float* probs, const float* uniform, int32_t* out, const int32_t* top_k_arr,
                             int top_k_val, const float* top_p_arr, float top_p_val, const float* min_p_arr,
                             float min_p_val, int joint, int batch, int vocab, int64_t in_stride, void* stream) {
  SGLK_CHECK(batch >= 0 && vocab > 0 && in_stride >= vocab, "sampling_from_probs: bad shape");
  if (batch == 0) return SGLK_OK;
  SGLK_CHECK(probs && uniform && out, "sampling_from_probs: null pointer");
  const bool vec = aligned16(probs) && in_stride % 4 == 0;
  hipLaunchKernelGGL(vec ? sample_kernel<true> : sample_kernel<false>, dim3(batch), dim3(kSampThreads), 0, (hipStream_t)stream,
                     probs, uniform, out, vocab, in_stride, top_k_arr, top_k_val, top_p_arr, top_p_val, min_p_arr, min_p_val, joint ? 1 : 0);
  SGLK_LAUNCH_CHECK();
  return SGLK_OK;
}
}
