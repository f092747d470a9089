// Host program for tests/test_gemm_paths.py: answers for the lines on standard
// input, "p M N K sBk sCi" (a pointwise product) or "s K batch cus" (a split one).
#include <cstdio>

#include "gemm_paths.hpp"

using namespace namsa;

int main() {
  char what;
  while (std::scanf(" %c", &what) == 1) {
    if (what == 'p') {
      int M, N, K;
      long long sBk, sCi;
      if (std::scanf("%d %d %d %lld %lld", &M, &N, &K, &sBk, &sCi) != 5) return 1;
      std::printf("%d %d %d\n", pointwise_fits(M, N, K, sBk, sCi), pointwise_mt(M), pointwise_ks(K));
    } else {
      int K, batch, cus;
      if (std::scanf("%d %d %d", &K, &batch, &cus) != 3) return 1;
      const SplitPlan p = split_plan(K, batch, cus);
      long long sum = 0, most = 0, least = K;
      for (int x = 0; x < p.groups; ++x) {
        const long long n = split_len(K, x * p.k_per, p.k_per);
        sum += n;
        most = n > most ? n : most;
        least = n < least ? n : least;
      }
      std::printf("%d %d %lld %lld %lld\n", p.groups, p.k_per, sum, most, least);
    }
  }
  return 0;
}
