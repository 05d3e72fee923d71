// Fused int4 GEMM of more than 64 rows: plan and launches of the kernel in awq_tall.h.
#include "awq_tall.h"

#include <algorithm>
#include <cstdlib>

namespace sglk {

// Which kernel takes a product of more than 64 rows, in microseconds: a round's start and end, and a stage with up to 128 and with 256
// blocks at once; blocks of 96 and of 128 rows and the wide kernel's of 64, without and with the producer's sums.  Fitted to 780
// products in each form (2048 to 32768 columns, 2 to 56 stages, bf16, cold weights, captured), which they tell within a tenth; the bound
// of nineteen twentieths leaves none that is taken more than 2 % slower than on the wide kernel.  A split product's sums cost 1.5 and 0.9 a split
// on both.  Measured, wide and here: 4096 x 28672 with its activation and the producer's sums 96 rows 42.8 and 34.1, 128 rows 42.3 and 40.3,
// without sums 47.4 and 38.6, 46.0 and 44.3; finished rows 5120 x 15360 at 192 rows 56.8 and 41.6, 8192 x 10240 at 96 (three splits) 41.4
// and 33.0, 28672 x 8192 at 192 (two) 134 and 115; left to the wide one: 13824 x 5120 at 80 rows 30.1 and 34.5 (four splits), 26624 x 12160 at 255 210 and 245, 4096 x 6144 at 128 14.2 and 15.3 (a launch's start and end, with twice the sums to add
// up and to leave, outweigh few stages).
struct TallCost {
  float round, few, full;
};
static constexpr TallCost kTallCost[2][3] = {{{7.5f, 3.08f, 3.65f}, {8.4f, 3.98f, 4.65f}, {6.4f, 1.96f, 2.3f}},
                                             {{7.3f, 2.68f, 3.4f}, {8.2f, 3.48f, 4.15f}, {6.4f, 1.78f, 2.1f}}};

TallPlan plan_awq_tall(int M, int N, int K, int group_size, int dtype, bool gated, bool sums, int64_t slab_bytes) {
  TallPlan p{};
  if (dtype != SGLK_BF16 || M <= kGemmBM || getenv("SGLK_AWQ_WIDE") || getenv("SGLK_AWQ_WIDE_SPS")) return p;  // (test hooks)
  const WidePlan wide = plan_awq_wide(M, N, K, group_size, gated);
  if (!wide.ok) return p;
  const int row_tiles = (M + 31) / 32;
  p.mblocks = (row_tiles + 3) / 4;
  p.rt = (row_tiles + p.mblocks - 1) / p.mblocks;
  p.tiles = (N / 128) * p.mblocks;
  const int total = K / AwqTall::kStageK;
  const int64_t slab = (int64_t)p.tiles * p.rt * 32 * 128 * 4;
  auto cost = [&](int tiles, int sps, const TallCost& c) {
    const int splits = (total + sps - 1) / sps, blocks = tiles * splits, whole = blocks / 256, rest = blocks % 256;
    const float last = rest == 0 ? 0.f : c.few + (c.full - c.few) * std::max(0, rest - 128) / 128.f;
    return (whole + (rest > 0)) * c.round + sps * (whole * c.full + last) + (splits > 1 ? 1.5f + 0.9f * splits : 0.f);
  };
  float least = 1e30f;
  for (int sps = gated ? total : 1; sps <= total; ++sps) {
    const int splits = (total + sps - 1) / sps;
    if (splits > 1 && slab * splits > slab_bytes) continue;
    const float c = cost(p.tiles, sps, kTallCost[sums][p.rt - 3]);
    if (c < least) {
      least = c;
      p.stages_per_split = sps;
      p.splits = splits;
    }
  }
  p.ok = least < 0.95f * cost(wide.tiles, gated ? total : wide.stages_per_split, kTallCost[sums][2]);
  return p;
}

int launch_awq_tall(const TallPlan& p, AwqTallArgs a, hipStream_t s) {
  a.stages_per_split = p.stages_per_split;
  a.splits = p.splits;
  a.wide_out = aligned16(a.out) && a.out_stride % 8 == 0;
  const dim3 grid(a.N / 128, p.splits, p.mblocks);
#define SGLK_TALL(XS, RT)                                                                   \
  {                                                                                         \
    if (int rc = ensure_lds<&awq_tall_kernel<XS, RT>>(AwqTall::lds(RT))) return rc;         \
    hipLaunchKernelGGL((awq_tall_kernel<XS, RT>), grid, dim3(512), AwqTall::lds(RT), s, a); \
  }
  if (p.rt == 3) {
    if (a.xsum_in) SGLK_TALL(true, 3) else SGLK_TALL(false, 3)
  } else {
    if (a.xsum_in) SGLK_TALL(true, 4) else SGLK_TALL(false, 4)
  }
#undef SGLK_TALL
  SGLK_LAUNCH_CHECK();
  return SGLK_OK;
}

// LDS limits of every form, for callers that launch under capture
int prepare_awq_tall() {
  if (int rc = ensure_lds<&awq_tall_kernel<true, 3>>(AwqTall::lds(3))) return rc;
  if (int rc = ensure_lds<&awq_tall_kernel<false, 3>>(AwqTall::lds(3))) return rc;
  if (int rc = ensure_lds<&awq_tall_kernel<true, 4>>(AwqTall::lds(4))) return rc;
  return ensure_lds<&awq_tall_kernel<false, 4>>(AwqTall::lds(4));
}

}  // namespace sglk
