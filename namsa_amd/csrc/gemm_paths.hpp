// Which products the special kernels of gemm_mfma.hip can address, in plain
// C++ so that the rules can be checked without a GPU.
#pragma once

#include <climits>

namespace namsa {

// gemm_pointwise_kernel's instance: 32-row blocks of the result, K steps of 16.
constexpr int pointwise_mt(int M) { return M <= 32 ? 1 : 2; }
constexpr int pointwise_ks(int K) { return K <= 16 ? 1 : K <= 32 ? 2 : 4; }
constexpr int kPointwiseCols = 512;  // columns of a workgroup, at most

// gemm_pointwise_kernel forms 32-bit byte offsets for all 32 MT rows of C and
// 16 KS rows of B, those past M and K as well: they have to lie past the
// buffer's end, so none may wrap (a row's pitch below 64 MiB at MT = KS = 1).
// B is also read up to the last workgroup's columns.  At 32 rows that is 16.7
// million columns; wider products take the staged kernel, whose strides are
// 64-bit.
constexpr bool pointwise_fits(int M, int N, int K, long long sBk, long long sCi) {
  return M <= 64 && K <= 64 && sBk >= N && sCi >= N &&
         sBk <= (INT_MAX - 4 * kPointwiseCols) / (64 * pointwise_ks(K)) && sCi <= INT_MAX / (128 * pointwise_mt(M));
}

// gemm_split_kernel's share of K: workgroup x takes split_len(K, x * k_per,
// k_per) values from x * k_per on, in steps of 128 that stay below 2^31 from
// kSplitMaxK down.  One workgroup per CU, each at least one step of 32 k per
// wavefront.
constexpr int kSplitMaxK = INT_MAX - 255;

struct SplitPlan {
  int groups, k_per;
};

constexpr SplitPlan split_plan(int K, int batch, int cus) {
  const long long most = (cus + batch - 1LL) / batch, steps = (K + 127LL) / 128;
  const long long want = steps < most ? steps : most;
  const long long k_per = ((K + want - 1) / want + 127) / 128 * 128;
  return {static_cast<int>((K + k_per - 1) / k_per), static_cast<int>(k_per)};
}

constexpr int split_len(int K, int k_begin, int k_per) { return K - k_begin < k_per ? K - k_begin : k_per; }

}  // namespace namsa
