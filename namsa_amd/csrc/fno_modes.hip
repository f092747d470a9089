// The y transforms of the corrector network's Fourier layers (16 modes an
// axis) between the row-DFT operands Z / Zp, [(c * B + b) * H + y][32] float,
// and the mode values Xs / Ys, [p * 16 + q][(r, c)][b] float with r the real
// and the imaginary part.  Operands rounded to bf16, FP32 sums.
//
//   forward:  P[(r,p)][(t,q)] = sum_y Fy[(r,p)][y] Z[y][(t,q)],
//             Xs_pq = (P[0p][0q] + P[1p][1q], P[0p][1q] - P[1p][0q])
//   inverse:  E[0p][0q] = E[1p][1q] = Yr_pq, E[0p][1q] = -E[1p][0q] = Yi_pq,
//             Zp[y][(t,q)] = sum_(r,p) Fy[(r,p)][y] E[(r,p)][(t,q)]
//
// One workgroup for a channel of a sample.
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "mfma.hpp"
#include "namsa_hip.h"

namespace namsa {
namespace {

constexpr int kM = 16;                  // modes an axis
constexpr int kM2 = 2 * kM;
constexpr int kSteps = 3;               // steps of 16 y a wavefront has in flight

// Reads past the H rows of this channel and sample give 0, stores there are dropped.
__device__ __forceinline__ Rsrc rows_of(const float* Z, int cb, int H) {
  return buffer_of(Z + static_cast<long long>(cb) * H * kM2, 4 * kM2 * H);
}

// Bound by reading Z once.  The four wavefronts take every fourth step of 16 y,
// all their loads in flight, and their sums meet in LDS in the order of the
// general small product; the first one combines P's quarters between lanes and
// stores the modes.  (As that product, a branch a load, and a kernel that read
// P back: 17 + 5 us for 512 channels of 170 rows, here 7.3.)
__global__ void __launch_bounds__(256) modes_forward_kernel(const float* __restrict__ Z, const __bf16* __restrict__ fy,
                                                            int H, int Hp, int C, int B, float* __restrict__ Xs) {
  __shared__ float part[3][16][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, half = lane >> 5, kh = 8 * half;
  const int cb = blockIdx.x, c = cb / B, b = cb % B;
  const Rsrc rz = rows_of(Z, cb, H);
  f32x16 acc = zero16();
  for (int k0 = 16 * wave; k0 < H; k0 += 64 * kSteps) {
    float z[kSteps][8];
#pragma unroll
    for (int s = 0; s < kSteps; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        z[s][e] = load_b32(rz, 4 * (kM2 * kh + col), 4 * kM2 * (k0 + 64 * s + e));
    bf16x8 a[kSteps];
#pragma unroll
    for (int s = 0; s < kSteps; ++s) a[s] = ld8(fy + col * Hp + min(k0 + 64 * s, Hp - 16) + kh);
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      if (k0 + 64 * s >= H) break;
      bf16x8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = __bf16(z[s][e]);
      acc = mfma(a[s], v, acc);
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int i = 0; i < 16; ++i) part[wave - 1][i][lane] = acc[i];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] += part[0][i][lane] + part[1][i][lane] + part[2][i][lane];
  // rows p and 16 + p are registers i and i + 8, columns q and 16 + q lanes 16
  // apart: the lower 16 columns leave the real parts, the upper the imaginary
  const int q = col & 15, r = col >> 4;
  float* X = Xs + (static_cast<long long>(q) * 2 * C + r * C + c) * B + b;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int p = 8 * (i >> 2) + 4 * half + (i & 3);
    const float other = __shfl_xor(acc[i + 8], 16, 64);
    X[static_cast<long long>(p) * kM * 2 * C * B] = r == 0 ? acc[i] + other : acc[i] - other;
  }
}

// Bound by writing Zp once.  The 512 mode values become the product's operand
// in LDS; each wavefront takes every fourth tile of 32 y, whose transform
// factors it reads in operand order.  (As a kernel that wrote E and the strided
// product, whose 128-row tiles left a third of their rows empty: 4 + 14 us for
// 512 channels of 170 rows, here 5.8.)
__global__ void __launch_bounds__(256) modes_inverse_kernel(const float* __restrict__ Ys,
                                                            const __bf16* __restrict__ fyT, int H, int C, int B,
                                                            float* __restrict__ Zp) {
  __shared__ __align__(16) __bf16 E[kM2][kM2 + 8];  // [column][row]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, half = lane >> 5, kh = 8 * half;
  const int cb = blockIdx.x, c = cb / B, b = cb % B;
  {
    const int p = threadIdx.x / kM, q = threadIdx.x % kM;
    const float* Y = Ys + (static_cast<long long>(threadIdx.x) * 2 * C + c) * B + b;
    const float yr = Y[0], yi = Y[static_cast<long long>(C) * B];
    E[q][p] = __bf16(yr);
    E[q][kM + p] = __bf16(-yi);
    E[kM + q][p] = __bf16(yi);
    E[kM + q][kM + p] = __bf16(yr);
  }
  const Rsrc rz = rows_of(Zp, cb, H);
  __syncthreads();
  const bf16x8 e0 = ld8(&E[col][kh]), e1 = ld8(&E[col][16 + kh]);
  for (int y0 = 32 * wave; y0 < H; y0 += 128) {
    const __bf16* f = fyT + (y0 + col) * kM2 + kh;
    f32x16 acc = mfma(ld8(f), e0, zero16());
    acc = mfma(ld8(f + 16), e1, acc);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      store_b32(acc[i], rz, 4 * (4 * kM2 * half + col), 4 * kM2 * (y0 + 8 * (i >> 2) + (i & 3)));
  }
}

int check_modes(int H, int Hp, int C, int B, const char* who) {
  if (H <= 0 || H > (1 << 20) || Hp < H || Hp % 32 != 0 || C <= 0 || B <= 0 ||
      static_cast<long long>(C) * B > 0x7fffffffLL / 512)
    return fail(kErrArg, "%s: bad shape H=%d Hp=%d C=%d B=%d (Hp a multiple of 32, >= H)", who, H, Hp, C, B);
  return kOk;
}

}  // namespace
}  // namespace namsa

using namespace namsa;

extern "C" {

int namsa_modes_forward(const float* Z, const void* fy, int H, int Hp, int C, int B, float* Xs, void* stream) {
  if (int rc = check_modes(H, Hp, C, B, "namsa_modes_forward")) return rc;
  if (!Z || !fy || !Xs) return fail(kErrArg, "namsa_modes_forward: null argument");
  hipLaunchKernelGGL(modes_forward_kernel, dim3(C * B), dim3(256), 0, as_stream(stream), Z,
                     static_cast<const __bf16*>(fy), H, Hp, C, B, Xs);
  return check_hip(hipGetLastError(), "modes_forward_kernel launch");
}

int namsa_modes_inverse(const float* Ys, const void* fyT, int H, int Hp, int C, int B, float* Zp, void* stream) {
  if (int rc = check_modes(H, Hp, C, B, "namsa_modes_inverse")) return rc;
  if (!Ys || !fyT || !Zp) return fail(kErrArg, "namsa_modes_inverse: null argument");
  hipLaunchKernelGGL(modes_inverse_kernel, dim3(C * B), dim3(256), 0, as_stream(stream), Ys,
                     static_cast<const __bf16*>(fyT), H, C, B, Zp);
  return check_hip(hipGetLastError(), "modes_inverse_kernel launch");
}

}  // extern "C"
