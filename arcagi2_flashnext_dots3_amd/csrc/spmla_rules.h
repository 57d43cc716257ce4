// Rules of sizes by which the launchers choose a kernel (plain host code).
#pragma once

namespace spmla {
namespace rules {

constexpr int WIDE_ROWS = 2048;       // longest list that the prefill kernel takes

// Whether an attention launch without the split merge takes fwd_kernel (spmla_attn.hip: 128 heads per workgroup) or the
// head-group kernel (spmla_attn_hg.hip: 32 heads per workgroup, any K); both run one workgroup per compute unit, whole
// rounds of 256. Fitted in tenths of a us to graphed launches of both formats with 1 to 64 tiles of 32 rows per list: a
// round of the head-group kernel takes 10.2 + 0.6 per tile, one of fwd_kernel 10 + 2.3 per tile and its first 7 more.
// Measured (us, head-group / fwd_kernel), Row656, K = 2048: H = 128: T = 129 142 / 169, 192 164 / 169, 224 195 / 172, 300
// 253 / 319, 400 345 / 325, 900 759 / 676, 2048 1618 / 1406; T = 1500, H = 32 384 / 874; T = 512, H = 160 523 / 645. Shorter
// lists: H = 128: T = 129, K = 1024 86 / 94, K = 128 39 / 31, T = 300, K = 512 100 / 108, K = 128 65 / 54, T = 400, K = 1024
// 209 / 187; T = 2000, H = 64, K = 128 233 / 184; T = 512, H = 160, K = 256 160 / 144. Row576 lies the same way (H = 128, K =
// 2048: T = 192 147 / 150, 224 176 / 153, 400 316 / 292, 2048 1458 / 1258). Of 546 such points the rule misses two by
// more than 5 % (Row576, K = 128: 8 %).
inline bool attn_wide(int T, int H, int K, int S) {
  const long long tiles = ((K + S - 1) / S + 31) / 32, ts = (long long)T * S;
  const long long r32 = (ts * ((H + 31) / 32) + 255) / 256, r128 = (ts * ((H + 127) / 128) + 255) / 256;
  return 32 * tiles <= WIDE_ROWS && r32 * (102 + 6 * tiles) > 72 + r128 * (100 + 23 * tiles);
}

// Model (us) of a merged launch of s splits over Row656 or Row576 rows: ts = T * ceil(H / 32) workgroups a split; see the
// fit in kernels.py, whose _split_cost this is.
inline double split_cost(long long ts, int K, int s, bool r576) {
  const long long tiles = ((K + s - 1) / s + 31) / 32, wgs = ts * s;
  const double m2 = r576 ? 4.0 : 3.0, m4 = r576 ? 5.0 : 3.6, m8 = r576 ? 7.3 : 6.0;
  const double round = (r576 ? 10.8 : 11.5) + (r576 ? 1.81 : 2.13) * (double)((tiles + 3) / 4);
  return (double)((wgs + 255) / 256) * round + (s == 1 ? 0.0 : s == 2 ? m2 : s <= 4 ? m4 : m8) +
         0.013 * (double)(wgs < 256 ? wgs : 256);
}

// Splits of a merged launch that may take up to S. Up to one round of workgroups as many as are asked for: more are taken
// only where they are faster. us of S splits of 128-head workgroups with f16 partials (the merge before this one) / S
// splits of this kernel / what is chosen, 128 heads: T = 32, K = 2048, S = 8 60 / 79 / 38 (2); T = 64, K = 256, S = 4 34 / 58
// / 18 (1); T = 200, K = 2048, S = 8 279 / 438 / 150 (1).
inline int merged_splits(int T, int H, int K, int S, bool r576) {
  const long long ts = (long long)T * ((H + 31) / 32);
  if (ts * S <= 256) return S;
  if (2 * ts > 256) return 1;
  int best = 1;
  for (int s = 2; s <= S; ++s)
    if (split_cost(ts, K, s, r576) < split_cost(ts, K, best, r576)) best = s;
  return best;
}

}  // namespace rules
}  // namespace spmla
