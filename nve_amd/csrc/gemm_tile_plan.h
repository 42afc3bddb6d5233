// gemm_tile_plan.h -- tile shape and K split of a W4A16 tile GEMM launch (host only).
#pragma once

namespace nve_host {

// shape: 0 = 64 x 128 and 1 = 128 x 128 (iterations of 128 of K), 2 = 96 x 256 and 3 = 128 x 256
// (64 of K); split workgroups per tile of ks iterations each (the last one fewer); us: the
// estimate.
struct TilePlan {
  int shape, split, ks;
  double us;
};

// The plan with the least estimated time:
//   rounds * (fixed + iterations * (it + full * load)) [+ launch + way * 1e-6 split M N]
// rounds of 256 workgroups, one per CU; load grows from 0 to 1 between 128 and 240 workgroups
// (a full chip clocks lower); the second part is the partials' way through memory and the
// reduction's launch.  The constants (us) are fitted to 990 (with AWQ 990) timed launches,
// fp16, 10 layer shapes (N 512-14336, K 2048-14336), M = 40-512, splits 1-16: rms error 3-6%,
// and the plan picked takes 0.6% (AWQ 0.9%) longer on average than the fastest one timed.
inline TilePlan plan_gemm_tile(int M, int N, int K, bool awq, int max_split) {
  static constexpr struct {
    int bm, bn, ik;  // tile, K of an iteration
    double fixed, it, it_awq, full, launch, way;
  } shapes[4] = {{64, 128, 128, 5.3, 0.58, 0.79, 0.06, 1.4, 2.3},
                 {128, 128, 128, 7.3, 0.71, 0.88, 0.16, 1.4, 1.9},
                 {96, 256, 64, 6.7, 0.67, 0.88, 0.06, 1.7, 1.9},
                 {128, 256, 64, 8.1, 0.72, 0.88, 0.16, 3.2, 1.1}};
  const int kit = K / 128;
  TilePlan best{0, 1, 0, 1e30};
  for (int c = 0; c < 4; ++c) {
    const auto& h = shapes[c];
    const long g = (long)((M + h.bm - 1) / h.bm) * ((N + h.bn - 1) / h.bn);
    int last = 0;
    for (int s = 1; s <= max_split && s <= kit; ++s) {
      const int per = (kit + s - 1) / s, used = (kit + per - 1) / per;  // no empty split
      if (used == last) continue;
      last = used;
      const long wgs = g * used, rounds = (wgs + 255) / 256;
      if (used > 1 && rounds > 1) break;
      const double load = wgs <= 128 ? 0.0 : wgs >= 240 ? 1.0 : (double)(wgs - 128) / 112;
      const double it = (awq ? h.it_awq : h.it) + h.full * load;
      double us = (double)rounds * (h.fixed + (double)per * (128 / h.ik) * it);
      if (used > 1) us += h.launch + h.way * 1e-6 * used * M * (double)N;
      if (us < best.us) best = TilePlan{c, used, per * (128 / h.ik), us};
    }
  }
  return best;
}

}  // namespace nve_host
