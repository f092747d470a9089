// Host program for tests/test_gemm_paths.py: answers for the products on
// standard input, one "M N K sBk sCi" a line.
#include <cstdio>

#include "gemm_paths.hpp"

int main() {
  int M, N, K;
  long long sBk, sCi;
  while (std::scanf("%d %d %d %lld %lld", &M, &N, &K, &sBk, &sCi) == 5)
    std::printf("%d %d %d\n", namsa::pointwise_fits(M, N, K, sBk, sCi), namsa::pointwise_mt(M), namsa::pointwise_ks(K));
  return 0;
}
