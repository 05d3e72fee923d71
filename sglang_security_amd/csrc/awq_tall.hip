// Fused int4 GEMM of more than 64 rows: plan and launches of the kernel in awq_tall.h.  A source of its own because it is compiled
// with the sums of the matrix instructions in vector registers (the accumulation registers hold the weights on their way).
#include "awq_tall.h"

#include <algorithm>
#include <cstdlib>

namespace sglk {

// Which kernel takes a product of more than 64 rows, in microseconds fitted to the four projections of Llama-3-8B (bf16, cold
// weights, captured) at 80 to 384 rows.  A launch here costs 8.4 (96 rows a block) or 9.9 (128) and 2.45 or 2.75 a stage, 3.3
// and 4.1 where more than 192 blocks run at once; the wide kernel's rounds of 64 rows 5.5 and 1.95 or 2.4.  Within a microsecond the
// wide kernel, whose sums are those of fewer rows to the bit.  Measured, wide and here: 4096 x 28672 with its activation
// 96 rows 49.6 and 34.8, 128 rows 49.1 and 41.9, 192 rows 71 and 66, 255 rows 94 and 80; left to the wide one: 128 rows of
// 4096 x 6144 14.2 and 15.3, of 14336 x 4096 22.1 and 27.4, of 4096 x 4096 11.9 and 14.2 (a launch's start and end, with twice
// the sums to add up and to leave, outweigh few stages).
TallPlan plan_awq_tall(int M, int N, int K, int group_size, int dtype, bool gated, int64_t slab_bytes) {
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
  auto cost = [&](int tiles, int sps, float start, float one, float full) {
    const int splits = (total + sps - 1) / sps, blocks = tiles * splits;
    return start + (blocks + 255) / 256 * sps * (blocks > 192 ? full : one) + (splits > 1 ? 0.5f * splits : 0.f);
  };
  float least = 1e30f;
  for (int sps = gated ? total : 1; sps <= total; ++sps) {
    const int splits = (total + sps - 1) / sps;
    if (splits > 1 && slab * splits > slab_bytes) continue;
    const float c = p.rt == 3 ? cost(p.tiles, sps, 8.4f, 2.45f, 3.3f) : cost(p.tiles, sps, 9.9f, 2.75f, 4.1f);
    if (c < least) {
      least = c;
      p.stages_per_split = sps;
      p.splits = splits;
    }
  }
  p.ok = least + 1.f < cost(wide.tiles, gated ? total : wide.stages_per_split, 5.5f, 1.95f, 2.4f);
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
