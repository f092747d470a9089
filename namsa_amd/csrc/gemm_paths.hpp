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

}  // namespace namsa
