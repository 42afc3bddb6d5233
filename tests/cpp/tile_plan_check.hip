// Host-only check of the W4A16 tile GEMM's plan (nve_amd/csrc/gemm_tile_plan.h): over a grid of
// products, the split covers K exactly, has no empty part, starts every part on a nibble
// slot (128 of K), stays within the partials offered, and no split launch has more than one
// round of workgroups.
#include <cstdio>
#include <initializer_list>

#include "../../nve_amd/csrc/gemm_tile_plan.h"

int main() {
  const int bm[4] = {64, 128, 96, 128}, bn[4] = {128, 128, 256, 256}, ik[4] = {128, 128, 64, 64};
  long bad = 0, seen[4] = {0, 0, 0, 0}, splits = 0;
  const int Ms[] = {33, 40, 64, 65, 96, 97, 128, 129, 197, 256, 300, 512, 513, 1024, 2048};
  const int Ns[] = {1, 64, 129, 512, 1024, 3072, 4096, 4101, 8192, 14336, 128256};
  for (int M : Ms)
    for (int N : Ns)
      for (int K = 128; K <= 32768; K += K < 2048 ? 128 : 1408)
        for (int awq = 0; awq < 2; ++awq)
          for (int most : {1, 2, 3, 8, 16, 64}) {
            const nve_host::TilePlan p = nve_host::plan_gemm_tile(M, N, K, awq, most);
            if (p.shape < 0 || p.shape > 3) return 1;
            const int T = K / ik[p.shape], per = 128 / ik[p.shape];
            const long g = (long)((M + bm[p.shape] - 1) / bm[p.shape]) * ((N + bn[p.shape] - 1) / bn[p.shape]);
            const bool ok = p.split >= 1 && p.split <= most && p.ks % per == 0 && p.ks >= per &&
                            (long)p.ks * p.split >= T && (long)p.ks * (p.split - 1) < T &&
                            (p.split == 1 || g * p.split <= 256);
            if (!ok && ++bad < 20)
              std::printf("M %d N %d K %d awq %d most %d: shape %d split %d ks %d\n", M, N, K, awq, most, p.shape,
                          p.split, p.ks);
            ++seen[p.shape];
            splits += p.split > 1;
          }
  for (int c = 0; c < 4; ++c)
    if (!seen[c]) ++bad, std::printf("shape %d never planned\n", c);
  if (!splits) ++bad;
  std::printf("%ld bad\n", bad);
  return bad ? 1 : 0;
}
