// Large-M GEMM for the extend (prefill) step: out[M, N] = x[M, K] @ W (+ bias), 16-bit activations, for
//   * AWQ int4 weights in the packed layout of sglk_awq_repack, dequantised on the way into LDS
//     ((q - z) * scale rounded to the activation type: the very weights the reference's
//     awq_dequantize-then-matmul multiplies by, python/sglang/srt/layers/quantization/awq.py:197-215), and
//   * dense 16-bit weights [N, K] (bf16 / fp16 checkpoints: layers/linear.py UnquantizedLinearMethod).
// prefill_tile.h holds the kernel.  The one below serves rows whose pitch is beyond its 32-bit offsets, and scales and biases that do not
// start where it loads them from, at a multiple of 4 and of 8 bytes: a block of four waves owns a 256 x 128 output tile and walks K in steps of 32 through two LDS stages (A: 256 rows x 64 bytes, B: 128 columns x 64 bytes, k
// contiguous in both, 16-byte chunks XOR-swizzled by (row >> 2) & 3); rows travel global -> registers while the current stage is
// multiplied, and are parked (the int4 words dequantised first) before the one barrier per stage.
#include <algorithm>

#include "prefill_tile.h"

namespace sglk {

static constexpr int kPfBM = 256, kPfBN = 128, kPfBK = 32;
static constexpr int kPfABytes = kPfBM * 64, kPfBBytes = kPfBN * 64;
static constexpr int kPfStage = kPfABytes + kPfBBytes;  // 24 KiB
static constexpr int kPfLds = 2 * kPfStage;             // 48 KiB: two blocks per CU

// 16-byte chunk c (k = 8c .. 8c + 7 of the stage) of row / column r
__device__ __forceinline__ int pf_off(int r, int c) { return r * 64 + ((c ^ ((r >> 2) & 3)) << 4); }

template <typename T, bool AWQ>
__global__ void __launch_bounds__(256, 2) prefill_gemm_kernel(
    const uint16_t* __restrict__ x, const void* __restrict__ wptr, const uint16_t* __restrict__ scales,
    const int32_t* __restrict__ qzeros, const uint16_t* __restrict__ bias, uint16_t* __restrict__ out, int M, int N, int K,
    int group_size, int64_t x_stride, int64_t w_stride, int64_t out_stride) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int wm = wid >> 1, wn = wid & 1;
  const int m0 = blockIdx.x * kPfBM, n0 = blockIdx.y * kPfBN;
  const int nk = K / kPfBK;

  // ---- global -> register roles
  // A: chunk q = tid + 256 i (i < 4): row q >> 2, chunk q & 3
  const uint16_t* asrc[4];
  bool aok[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = tid + 256 * i, row = q >> 2, c = q & 3;
    aok[i] = m0 + row < M;
    asrc[i] = x + (int64_t)(aok[i] ? m0 + row : 0) * x_stride + 8 * c;
  }
  // B: (column q >> 2, chunk q & 3) for q = tid + 256 i (i < 2)
  const uint16_t* bsrc[2] = {nullptr, nullptr};  // dense: row n0 + col of W [N, K]
  const int32_t* psrc[2] = {nullptr, nullptr};   // AWQ: the lane's four words of a 128-k block
  int bcol[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int q = tid + 256 * i, col = q >> 2, c = q & 3;
    bcol[i] = n0 + col;
    if (AWQ) {
      // word d of lane (i16, g) of strip s holds k = 128 kb + 32 d + 8 g + e of column 16 s + i16: chunk c <-> g
      psrc[i] = reinterpret_cast<const int32_t*>(wptr) + ((int64_t)(bcol[i] >> 4) * 64 + (bcol[i] & 15) + 16 * c) * 4;
    } else {
      bsrc[i] = reinterpret_cast<const uint16_t*>(wptr) + (int64_t)bcol[i] * w_stride + 8 * c;
    }
  }
  const int nstrips = N >> 4;

  int4v areg[4], breg[2];
  int4v wq[2];         // AWQ: the words of the current 128-k block
  float sc[2];         // ... scale and zero point of this thread's two columns in the current group
  int zp[2];
  auto fetch_a = [&](int kt) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      areg[i] = aok[i] ? *reinterpret_cast<const int4v*>(asrc[i] + kPfBK * kt) : int4v{0, 0, 0, 0};
  };
  auto fetch_b = [&](int kt) {
    if (AWQ) {
      if ((kt & 3) == 0) {
        const int kb = kt >> 2;
        const int gq = (128 * kb) / group_size;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          wq[i] = *reinterpret_cast<const int4v*>(psrc[i] + (int64_t)kb * nstrips * 256);
          sc[i] = Conv<T>::to_f32(scales[(int64_t)gq * N + bcol[i]]);
          const uint32_t zw = (uint32_t)qzeros[(int64_t)gq * (N >> 3) + (bcol[i] >> 3)];
          const int j = bcol[i] & 7;
          zp[i] = (int)((zw >> (4 * ((j >> 1) + 4 * (j & 1)))) & 0xF);  // AWQ nibble order {0, 4, 1, 5, 2, 6, 3, 7}
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) breg[i] = *reinterpret_cast<const int4v*>(bsrc[i] + kPfBK * kt);
    }
  };
  auto park = [&](int kt, int buf) {
    char* a = lds + buf * kPfStage;
    char* b = a + kPfABytes;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int q = tid + 256 * i;
      *reinterpret_cast<int4v*>(a + pf_off(q >> 2, q & 3)) = areg[i];
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int q = tid + 256 * i;
      int4v v;
      if (AWQ) {
        const uint32_t w = (uint32_t)wq[i][kt & 3];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          // k offsets e = 2p (nibble p) and e = 2p + 1 (nibble p + 4)
          const float v0 = (float)((int)((w >> (4 * p)) & 0xF) - zp[i]) * sc[i];
          const float v1 = (float)((int)((w >> (4 * p + 16)) & 0xF) - zp[i]) * sc[i];
          v[p] = (int)((uint32_t)Conv<T>::from_f32(v0) | ((uint32_t)Conv<T>::from_f32(v1) << 16));
        }
      } else {
        v = breg[i];
      }
      *reinterpret_cast<int4v*>(b + pf_off(q >> 2, q & 3)) = v;
    }
  };

  float16v acc[4][2];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.f;

  fetch_a(0);
  fetch_b(0);
  park(0, 0);
  __syncthreads();

  const int r32 = lane & 31, h = lane >> 5;
  for (int kt = 0; kt < nk; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nk) {
      fetch_a(kt + 1);
      fetch_b(kt + 1);
    }
    const char* a = lds + buf * kPfStage;
    const char* b = a + kPfABytes;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      int4v af[4], bf[2];
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
        af[mt] = *reinterpret_cast<const int4v*>(a + pf_off(128 * wm + 32 * mt + r32, 2 * ks + h));
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
        bf[nt] = *reinterpret_cast<const int4v*>(b + pf_off(64 * wn + 32 * nt + r32, 2 * ks + h));
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) prefill_mma<T, false>(acc[mt][nt], af[mt], bf[nt]);
    }
    if (kt + 1 < nk) park(kt + 1, buf ^ 1);
    __syncthreads();
  }

  // ---- epilogue: every wave transposes its 32 x 32 tiles through 2.5 KiB of LDS of its own (rows padded to 80 bytes)
  // and stores 16-byte row pieces.  Accumulator register r of lane (c, h) is D[(r & 3) + 8 (r >> 2) + 4 h][c].
  char* tl = lds + wid * 2560;
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int col0 = n0 + 64 * wn + 32 * nt;
      const float bv = bias ? Conv<T>::to_f32(bias[min(col0 + r32, N - 1)]) : 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = (r & 3) + 8 * (r >> 2) + 4 * h;
        *reinterpret_cast<uint16_t*>(tl + row * 80 + r32 * 2) = Conv<T>::from_f32(acc[mt][nt][r] + bv);
      }
      __builtin_amdgcn_wave_barrier();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int q = lane + 64 * i, row = q >> 2, c = q & 3;
        const int m = m0 + 128 * wm + 32 * mt + row, n = col0 + 8 * c;
        const int4v v = *reinterpret_cast<const int4v*>(tl + row * 80 + c * 16);
        if (m < M && n < N) *reinterpret_cast<int4v*>(out + (int64_t)m * out_stride + n) = v;
      }
      __builtin_amdgcn_wave_barrier();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
}

// ---- which blocks a product takes
// Microseconds of a round of blocks of 64 mi rows: its start and end, and a stage of 64 of K in strips of 128, 192 or 256 columns
// (half the second index + 1), with up to 200 and with more blocks at once.  Fitted to the four projections of Llama-3-8B, int4
// and bf16, weights from memory, 129 to 2048 rows.
static constexpr double kRound = 6.0;
static constexpr double kStage[3][3][2] = {
    {{0.55, 0.61}, {0.67, 0.84}, {0.86, 1.08}}, {{0.65, 0.82}, {0.91, 1.14}, {1.04, 1.30}}, {{0.76, 0.97}, {1.07, 1.33}, {1.32, 1.62}}};

struct PrefillPlan {
  int mi, mt, whole, tail, narrow;
  double cost;
};

// Strips of 256 columns while they fill whole rounds of 256 units; what is left over, if it would fill no more than three quarters
// of a round, in strips of 192 or 128 (1152 x 28672 x 4096, 192 rows a block: two rounds and 216 blocks of 192 columns, 254 us).
static PrefillPlan prefill_strips(int64_t M, int64_t N, int64_t K, int mi, bool gated) {
  auto up = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  const int64_t mt = up(M, 64 * mi), all = up(N, 256), stages = K / 64;
  auto rounds = [&](int64_t blocks, int strip) {
    const int64_t full = blocks / 256, rest = blocks % 256;
    const double* c = kStage[mi - 2][strip];
    return full * (kRound + stages * c[1]) + (rest ? kRound + stages * c[rest > 200] : 0.0);
  };
  PrefillPlan p{mi, (int)mt, (int)all, 0, 128, rounds(mt * all, 2)};
  const int64_t whole = mt * all / 256 * 256 / mt;
  for (int strip = 0; strip < (gated ? 1 : 2); ++strip) {  // (a gate block and its up block: strips of whole 128s)
    const int narrow = 128 + 64 * strip;
    const int64_t tail = up(N - whole * 256, narrow);
    if (whole < all && mt * tail <= 256)
      return {mi, (int)mt, (int)whole, (int)tail, narrow, rounds(mt * whole, 2) + rounds(mt * tail, strip)};
  }
  return p;
}

// Rows a block: whatever wastes least of the last round and of the last block (1152 rows: six of 192).  16-bit weights, which are
// not dequantised on the way, keep 512 registers only up to 192 rows.
static PrefillPlan prefill_plan(int64_t M, int64_t N, int64_t K, bool awq, bool gated = false) {
  PrefillPlan best = prefill_strips(M, N, K, 2, gated);
  for (int mi = 3; mi <= (awq ? 4 : 3); ++mi) {
    const PrefillPlan p = prefill_strips(M, N, K, mi, gated);
    if (p.cost < best.cost) best = p;
  }
  return best;
}

template <typename T, bool AWQ, int MI>
static int launch_prefill(const PrefillArgs& a, hipStream_t s) {
  constexpr int lds = (2 * 64 * MI + (AWQ ? 2 : 3) * 256) * 128 + (AWQ ? 2048 : 0);
  if (int rc = ensure_lds<&prefill_tile_kernel<T, AWQ, MI>>(lds)) return rc;
  hipLaunchKernelGGL((prefill_tile_kernel<T, AWQ, MI>), dim3((unsigned)(a.mt * (a.whole + a.tail))), dim3(256), lds, s, a);
  SGLK_LAUNCH_CHECK();
  return SGLK_OK;
}

static constexpr int64_t kPrefillPitch = 1 << 23;  // 256 rows of less than that span less than 2^32 bytes
static bool starts_at(const void* p, uintptr_t multiple) { return reinterpret_cast<uintptr_t>(p) % multiple == 0; }

template <typename T, bool AWQ>
static int launch_prefill_any(const PrefillArgs& a, hipStream_t s) {
  if (a.x_stride >= kPrefillPitch || a.w_stride >= kPrefillPitch || !starts_at(a.scales, 4) || !starts_at(a.bias, 8)) {
    const dim3 grid((a.M + kPfBM - 1) / kPfBM, a.N / kPfBN);
    hipLaunchKernelGGL((prefill_gemm_kernel<T, AWQ>), grid, dim3(256), kPfLds, s, a.x, a.w, a.scales, a.qzeros, a.bias, a.out, a.M,
                       a.N, a.K, a.group_size, a.x_stride, a.w_stride, a.out_stride);
    SGLK_LAUNCH_CHECK();
    return SGLK_OK;
  }
  const PrefillPlan pl = prefill_plan(a.M, a.N, a.K, AWQ, a.gated);
  PrefillArgs b = a;
  b.mt = pl.mt, b.whole = pl.whole, b.tail = pl.tail, b.narrow = pl.narrow;
  if (pl.mi == 2) return launch_prefill<T, AWQ, 2>(b, s);
  if constexpr (AWQ)
    if (pl.mi == 4) return launch_prefill<T, AWQ, 4>(b, s);
  return launch_prefill<T, AWQ, 3>(b, s);
}

static int prefill_checks(const void* x, const void* w, const void* out, int M, int N, int K, int64_t x_stride,
                          int64_t out_stride, const char* what) {
  SGLK_CHECK(x && w && out, "%s: null pointer", what);
  SGLK_CHECK(M > 0 && N > 0 && K > 0, "%s: bad shape", what);
  SGLK_CHECK(K % 128 == 0 && N % 128 == 0, "%s: K=%d and N=%d must be multiples of 128", what, K, N);
  SGLK_CHECK(aligned16(x) && aligned16(w) && aligned16(out) && x_stride % 8 == 0 && out_stride % 8 == 0,
             "%s: rows must be 16-byte aligned", what);
  return SGLK_OK;
}

}  // namespace sglk

using namespace sglk;

extern "C" {

int sglk_awq_gemm_prefill(const void* x, const int32_t* packed, const void* scales, const int32_t* qzeros,
                          const void* bias, void* out, int M, int N, int K, int group_size, int64_t x_stride,
                          int64_t out_stride, int dtype, void* stream) {
  if (int rc = prefill_checks(x, packed, out, M, N, K, x_stride, out_stride, "awq_gemm_prefill")) return rc;
  SGLK_CHECK(scales && qzeros, "awq_gemm_prefill: null pointer");
  SGLK_CHECK(group_size > 0 && group_size % 128 == 0 && K % group_size == 0,
             "awq_gemm_prefill: group size %d must be a multiple of 128 that divides K", group_size);
  const PrefillArgs a{(const uint16_t*)x, packed, (const uint16_t*)scales, qzeros, (const uint16_t*)bias, (uint16_t*)out, M, N, K,
                      group_size, x_stride, 0, out_stride, 0, 0, 0, 0, 0};
  SGLK_DISPATCH_HALF(dtype, T, { return (launch_prefill_any<T, true>(a, (hipStream_t)stream)); });
  return SGLK_OK;
}

int sglk_awq_gemm_prefill_silu_mul(const void* x, const int32_t* packed, const void* scales, const int32_t* qzeros, void* out,
                                   int M, int N, int K, int group_size, int64_t x_stride, int64_t out_stride, int dtype,
                                   void* stream) {
  if (int rc = prefill_checks(x, packed, out, M, N, K, x_stride, out_stride, "awq_gemm_prefill_silu_mul")) return rc;
  SGLK_CHECK(scales && qzeros, "awq_gemm_prefill_silu_mul: null pointer");
  SGLK_CHECK(N % 256 == 0 && out_stride >= N / 2, "awq_gemm_prefill_silu_mul: N=%d must be a multiple of 256, out rows hold N / 2", N);
  SGLK_CHECK(group_size > 0 && group_size % 128 == 0 && K % group_size == 0,
             "awq_gemm_prefill_silu_mul: group size %d must be a multiple of 128 that divides K", group_size);
  SGLK_CHECK(x_stride < kPrefillPitch, "awq_gemm_prefill_silu_mul: rows %lld elements apart", (long long)x_stride);
  SGLK_CHECK(starts_at(scales, 4), "awq_gemm_prefill_silu_mul: scales must be 4-byte aligned");
  const PrefillArgs a{(const uint16_t*)x, packed, (const uint16_t*)scales, qzeros, nullptr, (uint16_t*)out, M, N, K,
                      group_size, x_stride, 0, out_stride, 1, 0, 0, 0, 0};
  SGLK_DISPATCH_HALF(dtype, T, { return (launch_prefill_any<T, true>(a, (hipStream_t)stream)); });
  return SGLK_OK;
}

int sglk_awq_gemm_prefill_tiles(int M, int N, int K, int gated, int* tiles) {
  SGLK_CHECK(tiles && M > 0 && N > 0 && K > 0, "awq_gemm_prefill_tiles: bad argument");
  const PrefillPlan p = prefill_plan(M, N, K, true, gated != 0);
  const int all[5] = {64 * p.mi, p.mt, p.whole, p.tail, p.narrow};
  std::copy(all, all + 5, tiles);
  return SGLK_OK;
}

// The other way, in microseconds: the weight dequantised to memory and the library's product, whose tiles round M up and whose chain
// along K is never shorter than that.  Fitted to what follows, within a tenth for half of it: choices of the library's own move its
// products by a quarter either way, so the entries below draw lines around the estimate.
static double prefill_library(int M, int N, int K) {
  const double weights = (double)N * K;
  return 14 + 0.22e-6 * weights + std::max(2e-9 / 1.52 * weights * (M + 336), 0.0049 * K);
}

// Timed both ways, one launch behind the other on weights from memory, over 28 weights of 1B to 70B models and eight of their ranks,
// 257 to 4096 rows in bf16; captured over 32, 1 to 8192 rows, bf16 and fp16.  Of the calls that these lines take none is more than 3 % slower
// than the library behind a dequantisation (captured, without the gap between two launches, four are, by 4 to 8 %: 4096 x 4096 at 1536
// rows, 5120 x 5120 at 1152, 8192 x 8192 and 3584 at 640), and they take a fifth less on average: 28672 x 4096, 257 rows 136 -> 83 us, 500 rows 158 -> 105, 1152
// rows 288 -> 244; 6144 x 4096, 500 rows 49 -> 42, 1152 rows 67 -> 62.  Left to the library: 4096 x 14336 at 640 rows 117 and here 137,
// 7168 x 8192 at 800 116 and 124, 28672 x 4096 at 4096 675 and 781, and a long K with so few rows as other kernels take, 100 of 8192 x
// 8192 63 and 78.
int sglk_awq_prefill_fused(int M, int N, int K) {
  if (M <= 0 || K <= 0 || K % 128 != 0 || N % 128 != 0 || (int64_t)N * K < (4 << 20)) return 0;
  const bool wide = N >= 8192;
  if (N < 4096 || M > 1700 || (M < 256 && !wide) || (K > 5120 && (M < 256 || !wide))) return 0;
  return prefill_plan(M, N, K, true).cost < (wide ? 1.0 : 0.95) * prefill_library(M, N, K);
}

// With the activation behind it, against the library and a launch of the activation: twelve weights, 257 to 8192 rows, captured; none
// taken is more than 3 % slower.  28672 x 4096, 2048 rows 426 -> 409 us, 27648 x 5120, 1300 rows 387 -> 352; left to the library: 16384
// x 3072, 3000 rows 254 and here 268.
int sglk_awq_prefill_silu_mul_fused(int M, int N, int K) {
  if (M < 256 || M > 2112 || N < 8192 || K <= 0 || K % 128 != 0 || N % 256 != 0) return 0;
  const double activation = 3 + 0.61e-6 * M * N;
  return prefill_plan(M, N, K, true, true).cost < prefill_library(M, N, K) + activation;
}

int sglk_dense_gemm_prefill(const void* x, const void* w, const void* bias, void* out, int M, int N, int K,
                            int64_t x_stride, int64_t w_stride, int64_t out_stride, int dtype, void* stream) {
  if (int rc = prefill_checks(x, w, out, M, N, K, x_stride, out_stride, "dense_gemm_prefill")) return rc;
  SGLK_CHECK(w_stride % 8 == 0, "dense_gemm_prefill: weight rows must be 16-byte aligned");
  const PrefillArgs a{(const uint16_t*)x, w, nullptr, nullptr, (const uint16_t*)bias, (uint16_t*)out, M, N, K, 128, x_stride,
                      w_stride, out_stride, 0, 0, 0, 0, 0};
  SGLK_DISPATCH_HALF(dtype, T, { return (launch_prefill_any<T, false>(a, (hipStream_t)stream)); });
  return SGLK_OK;
}
}
