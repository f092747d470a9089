// Channel-last BF16 inference of the corrector network on the matrix cores.
//
// The network's activations are 32 channels per pixel; here they live as
// bf16 [rows][W][32] (rows = B * H, one image row of one sample each), so one
// image row is a W x 32 matrix and every product of a Fourier layer that
// touches the full activation is a row-local MFMA product:
//
//   x_{l+1}[x][o] = gelu( alpha sum_q Fx[x][q] Zp_l[o][q] + sum_c x_l[x][c] W_l[o][c] + b_l[o] )
//   Z_{l+1}[c][q] = sum_x x_{l+1}[x][c] Fx[x][q]
//
// with Fx[x][q] the truncated row DFT ([cos | -sin] of the m retained x modes,
// 2m = 32 columns), Zp_l the row-inverse operand the small mode-space
// products leave (mode mixing, on the strided GEMM, and the y transforms),
// and Z_{l+1} the next layer's row DFT.  One wavefront streams one row in
// 32-pixel tiles: the first product is four v_mfma_f32_32x32x16_bf16 with
// K = 32 modes + 32 channels (both operands read 16 bytes per lane straight
// from memory), the tile goes through LDS once (after bias and GELU, as bf16)
// and leaves as the next activation, and two more MFMAs fold it into the next
// row DFT.
// Each layer therefore reads and writes the activation once: 128 bytes per
// pixel.  The lift (features -> 32 channels) also forms layer 0's row DFT;
// the last layer feeds the pointwise head (32 -> 64 -> 2) instead.
//
// Z / Zp rows are ordered (c, b, y): row (c * B + b) * H + y, 32 floats each,
// the layout of the strided GEMM path's row-DFT output.
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "mfma.hpp"
#include "namsa_hip.h"

namespace namsa {
namespace {

constexpr int kCh = 32;        // channels
constexpr int kQ = 32;         // 2m row-DFT columns
constexpr int kHid = 64;       // head width
constexpr int kTile = 32;      // pixels per tile
constexpr int kPitch = 40;     // LDS row pitch in bf16 (80 bytes: 16-byte aligned rows)
constexpr int kWaves = 4;

// tanh-GELU, x/2 (1 + tanh(u)) = x (1 - 1 / (exp(2u) + 1)), u = sqrt(2/pi) (x + 0.044715 x^3);
// the exponential form differs from tanhf by ~1e-7, far below the bf16 rounding of its result.
// The quotient is one Newton step from the reciprocal's, which rounds as the
// division does (the divisor lies in [1, 2^100], where its scaling steps have
// nothing to do): 5 instructions for 11 of the 25.
__device__ __forceinline__ float gelu_t(float x) {
  const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  const float d = fminf(__expf(2.0f * u) + 1.0f, 0x1p100f);
  const float r = __builtin_amdgcn_rcpf(d), q = x * r;
  return x - fmaf(fmaf(-d, q, x), r, q);
}

__device__ __forceinline__ bf16x8 cvt8(const float* p, float scale) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  const float4 b = *reinterpret_cast<const float4*>(p + 4);
  bf16x8 v;
  v[0] = __bf16(a.x * scale);
  v[1] = __bf16(a.y * scale);
  v[2] = __bf16(a.z * scale);
  v[3] = __bf16(a.w * scale);
  v[4] = __bf16(b.x * scale);
  v[5] = __bf16(b.y * scale);
  v[6] = __bf16(b.z * scale);
  v[7] = __bf16(b.w * scale);
  return v;
}

// What the lanes of a wavefront exchange of a tile.
struct alignas(16) Exchange {
  __bf16 by_channel[kCh][kPitch], by_pixel[kTile][kPitch];
};

struct RowGeom {
  int rows, W, Wp, H, B;
};

// A tile's values, channel 8 (i / 4) + 4 half + i % 4 of pixel x0 + col in v[i],
// leave rounded as the next activation and are added to the row's DFT:
// zacc(c, q) += sum_x v(c, x) fxT[q][x], f holding the tile's rows of fxT.  Both
// pass through LDS: for the DFT the pixels have to lie along k, and the
// activation is stored in whole 1 KiB runs.  (A layer of 64 images of 170 x 170
// took 107 us with 16 bytes of each 64 a store and Z in pieces of 16 bytes.)
__device__ __forceinline__ void tile_out(const f32x16& v, f32x16& zacc, const bf16x8 (&f)[2], int x0, int W,
                                         Exchange& ex, __bf16* __restrict__ row, int lane) {
  const int col = lane & 31, half = lane >> 5, kh = 8 * half;
  const bool in = x0 + col < W;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    bf16x8 h;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int i = 8 * s + e;
      h[e] = __bf16(in ? v[i] : 0.0f);
      ex.by_channel[8 * (i >> 2) + 4 * half + (i & 3)][col] = h[e];
    }
    *reinterpret_cast<bf16x8*>(&ex.by_pixel[col][16 * s + kh]) = rows_to_k(h);
  }
  wave_sync();
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int px = 16 * s + (lane >> 2);
    const bf16x8 h = ld8(&ex.by_pixel[px][8 * (lane & 3)]);
    if (x0 + px < W) *reinterpret_cast<bf16x8*>(row + static_cast<long long>(x0 + px) * kCh + 8 * (lane & 3)) = h;
    zacc = mfma(ld8(&ex.by_channel[col][16 * s + kh]), f[s], zacc);
  }
  wave_sync();
}

// Z's rows of the image row, whole rows of 32 q a store.
__device__ __forceinline__ void store_z(float* __restrict__ Z, const f32x16& zacc, const RowGeom& g, int r,
                                        int lane) {
  const int b = r / g.H, y = r % g.H;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int c = 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
    Z[((static_cast<long long>(c) * g.B + b) * g.H + y) * kQ + (lane & 31)] = zacc[i];
  }
}

// x0 = Wl u + bl (u channel-major [cin][rows * W]) and layer 0's row DFT.
// Per 32-pixel tile one MFMA with K = 16 (cin inputs, the rest zero):
// A(o, k) = Wl[o][k], B(k, x) = u[k][x], the next tile's read while one
// computes.  Bound by the activation's writes and the wavefronts' serial tiles:
// 64 images of 170 x 170 85 -> 43 us (the pixel in the lane throughout, no
// branch around a load).
__global__ void __launch_bounds__(256)
fno_lift_kernel(const float* __restrict__ u, int cin, const float* __restrict__ Wl, const float* __restrict__ bl,
                const __bf16* __restrict__ fxT, RowGeom g, __bf16* __restrict__ xout, float* __restrict__ Z) {
  __shared__ Exchange exchange[kWaves];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = blockIdx.x * kWaves + wave;
  if (r >= g.rows) return;
  const long long n = static_cast<long long>(g.rows) * g.W;
  const int col = lane & 31, half = lane >> 5, kh = 8 * half;
  bf16x8 wop;                                    // A(o = col, k = kh + e)
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float w = Wl[col * cin + min(kh + e, cin - 1)];
    wop[e] = __bf16(kh + e < cin ? w : 0.0f);
  }
  float bias[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) bias[i] = bl[8 * (i >> 2) + 4 * half + (i & 3)];
  // input e at this lane's pixel; the upper half's inputs do not exist (cin <= 8), nor do pixels past the row
  const float* ur = u + static_cast<long long>(r) * g.W;
  auto load_in = [&](int px, float (&v)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = ur[min(e, cin - 1) * n + min(px, g.W - 1)];
  };
  const __bf16* fx_row = fxT + static_cast<long long>(col) * g.Wp + kh;
  f32x16 zacc = zero16();
  float next[8];
  load_in(col, next);
  for (int x0 = 0; x0 < g.W; x0 += kTile) {
    bf16x8 a;
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = __bf16(kh + e < cin ? next[e] : 0.0f);
    const bf16x8 f[2] = {ld8(fx_row + x0), ld8(fx_row + x0 + 16)};
    load_in(x0 + kTile + col, next);
    f32x16 acc = mfma(wop, a, zero16());
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] += bias[i];
    tile_out(acc, zacc, f, x0, g.W, exchange[wave], xout + static_cast<long long>(r) * g.W * kCh, lane);
  }
  store_z(Z, zacc, g, r, lane);
}

// One Fourier layer.  LAST == 0: x_out = gelu(...) and Z_next; LAST == 1: no
// GELU, then the head out[t][p] = Q2 gelu(Q1 x + bq1) + bq2 (out channel-major
// [2][rows * W] float).  The pixel stays in the lane from the first product to
// the last, so a product's result is the next one's operand after an exchange
// between the wavefront's halves.  A layer is bound by its 326 MB (3.7 TB/s),
// the head by the arithmetic of 64 GELUs a pixel.  64 images of 170 x 170: 110 -> 88 us, with
// the head 182 -> 117, against the channel in the lane and each result passed
// through LDS.
template <int LAST>
__global__ void __launch_bounds__(256, 3)
fno_layer_kernel(const __bf16* __restrict__ x_in, const float* __restrict__ Zp, const __bf16* __restrict__ fx,
                 const __bf16* __restrict__ fxT, const float* __restrict__ Wt, const float* __restrict__ bias,
                 float alpha, RowGeom g, __bf16* __restrict__ x_out, float* __restrict__ Z_next,
                 const float* __restrict__ Q1, const float* __restrict__ bq1, const float* __restrict__ Q2,
                 const float* __restrict__ bq2, float* __restrict__ out) {
  __shared__ Exchange exchange[LAST ? 1 : kWaves];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = blockIdx.x * kWaves + wave;
  if (r >= g.rows) return;
  const int b = r / g.H, y = r % g.H;
  const int col = lane & 31, half = lane >> 5, kh = 8 * half;

  // A operands of the layer product, the same for every tile of the row:
  // k < 32: alpha Zp[o][q] (q = k), k >= 32: W[o][c] (c = k - 32), o = col
  bf16x8 aop[4];
  const float* zp_row = Zp + ((static_cast<long long>(col) * g.B + b) * g.H + y) * kQ;
  aop[0] = cvt8(zp_row + kh, alpha);
  aop[1] = cvt8(zp_row + 16 + kh, alpha);
  aop[2] = cvt8(Wt + col * kCh + kh, 1.0f);
  aop[3] = cvt8(Wt + col * kCh + 16 + kh, 1.0f);
  float bo[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) bo[i] = bias[8 * (i >> 2) + 4 * half + (i & 3)];
  bf16x8 q1op[2][2];                            // head operands A(j, k = c) = Q1[j][c], constant per wave
  bf16x8 q2op[4];                               // A(t, k = j) = Q2[t][j] for t = col < 2, else 0
  float b1[LAST ? 2 : 1][16];
  if (LAST) {
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) {
#pragma unroll
      for (int s = 0; s < 2; ++s) q1op[jb][s] = cvt8(Q1 + (32 * jb + col) * kCh + 16 * s + kh, 1.0f);
#pragma unroll
      for (int i = 0; i < 16; ++i) b1[jb][i] = bq1[32 * jb + 8 * (i >> 2) + 4 * half + (i & 3)];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) q2op[s][e] = __bf16(col < 2 ? Q2[col * kHid + 16 * s + kh + e] : 0.0f);
  }

  f32x16 zacc = zero16();
  const long long n = static_cast<long long>(g.rows) * g.W;
  // a tile's operands, modes B(k = 16 s + kh .., x) and channels B(k = 32 + 16 s
  // + kh .., x), are loaded while the tile before computes; pixels past the row
  // read its last one, their results go nowhere
  const __bf16* x_row = x_in + static_cast<long long>(r) * g.W * kCh + kh;
  const __bf16* fx_row = fxT + static_cast<long long>(col) * g.Wp + kh;
  auto load = [&](int x0, bf16x8 (&a)[4]) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      a[s] = ld8(fx + static_cast<long long>(min(x0 + col, g.Wp - 1)) * kQ + 16 * s + kh);
      a[2 + s] = ld8(x_row + static_cast<long long>(min(x0 + col, g.W - 1)) * kCh + 16 * s);
    }
  };
  bf16x8 next[4];
  load(0, next);
  for (int x0 = 0; x0 < g.W; x0 += kTile) {
    const int px = x0 + col;                    // this lane's pixel
    const bf16x8 bop[4] = {next[0], next[1], next[2], next[3]};
    bf16x8 f[2];                                // asked for before the next tile: a wait for it is none for that
    if constexpr (!LAST) {
      f[0] = ld8(fx_row + x0);
      f[1] = ld8(fx_row + x0 + 16);
    }
    load(x0 + kTile, next);
    f32x16 acc = zero16();
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = mfma(aop[s], bop[s], acc);
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] += bo[i];
    if constexpr (!LAST) {
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = gelu_t(acc[i]);
      tile_out(acc, zacc, f, x0, g.W, exchange[wave], x_out + static_cast<long long>(r) * g.W * kCh, lane);
    } else {
      // head: h = gelu(Q1 x + bq1) as two 32-row blocks, out[t] = Q2[t] . h + bq2[t] over K = 64
      bf16x8 xb[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int e = 0; e < 8; ++e) xb[s][e] = __bf16(acc[8 * s + e]);
        xb[s] = rows_to_k(xb[s]);
      }
      f32x16 oacc = zero16();
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) {
        f32x16 hacc = zero16();
#pragma unroll
        for (int s = 0; s < 2; ++s) hacc = mfma(q1op[jb][s], xb[s], hacc);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          bf16x8 h;
#pragma unroll
          for (int e = 0; e < 8; ++e) h[e] = __bf16(gelu_t(hacc[8 * s + e] + b1[jb][8 * s + e]));
          oacc = mfma(q2op[2 * jb + s], rows_to_k(h), oacc);
        }
      }
      if (half == 0 && px < g.W) {              // rows t < 2 of the result
#pragma unroll
        for (int t = 0; t < 2; ++t) out[t * n + static_cast<long long>(r) * g.W + px] = oacc[t] + bq2[t];
      }
    }
  }
  if constexpr (!LAST) store_z(Z_next, zacc, g, r, lane);
}

int check_geom(int B, int H, int W, int Wp, const char* who) {
  if (B <= 0 || H <= 0 || W <= 0 || Wp < W || Wp % kTile != 0 || static_cast<long long>(B) * H > 0x7fffffffLL)
    return fail(kErrArg, "%s: bad geometry B=%d H=%d W=%d Wp=%d (Wp must be a multiple of 32, >= W)", who, B, H,
                W, Wp);
  return kOk;
}

}  // namespace
}  // namespace namsa

using namespace namsa;

extern "C" {

int namsa_fno_lift(const float* u, int cin, const float* Wl, const float* bl, const void* fxT, int B, int H, int W,
                   int Wp, void* x0, float* Z, void* stream) {
  if (int rc = check_geom(B, H, W, Wp, "namsa_fno_lift")) return rc;
  if (!u || !Wl || !bl || !fxT || !x0 || !Z || cin < 1 || cin > 8)
    return fail(kErrArg, "namsa_fno_lift: null argument or cin=%d outside 1..8", cin);
  const RowGeom g{B * H, W, Wp, H, B};
  const unsigned blocks = static_cast<unsigned>((g.rows + kWaves - 1) / kWaves);
  hipLaunchKernelGGL(fno_lift_kernel, dim3(blocks), dim3(256), 0, as_stream(stream), u, cin, Wl, bl,
                     static_cast<const __bf16*>(fxT), g, static_cast<__bf16*>(x0), Z);
  return check_hip(hipGetLastError(), "fno_lift_kernel launch");
}

int namsa_fno_layer(const void* x_in, const float* Zp, const void* fx, const void* fxT, const float* Wt,
                    const float* bias, float alpha, int B, int H, int W, int Wp, void* x_out, float* Z_next,
                    const float* Q1, const float* bq1, const float* Q2, const float* bq2, float* out, void* stream) {
  if (int rc = check_geom(B, H, W, Wp, "namsa_fno_layer")) return rc;
  if (!x_in || !Zp || !fx || !fxT || !Wt || !bias) return fail(kErrArg, "namsa_fno_layer: null operand");
  const bool last = out != nullptr;
  if (last ? (!Q1 || !bq1 || !Q2 || !bq2) : (!x_out || !Z_next))
    return fail(kErrArg, "namsa_fno_layer: a layer needs x_out and Z_next, the last layer Q1, bq1, Q2, bq2 and out");
  const RowGeom g{B * H, W, Wp, H, B};
  const unsigned blocks = static_cast<unsigned>((g.rows + kWaves - 1) / kWaves);
  const auto* xi = static_cast<const __bf16*>(x_in);
  const auto* f = static_cast<const __bf16*>(fx);
  const auto* ft = static_cast<const __bf16*>(fxT);
  if (last)
    hipLaunchKernelGGL(fno_layer_kernel<1>, dim3(blocks), dim3(256), 0, as_stream(stream), xi, Zp, f, ft, Wt, bias,
                       alpha, g, nullptr, nullptr, Q1, bq1, Q2, bq2, out);
  else
    hipLaunchKernelGGL(fno_layer_kernel<0>, dim3(blocks), dim3(256), 0, as_stream(stream), xi, Zp, f, ft, Wt, bias,
                       alpha, g, static_cast<__bf16*>(x_out), Z_next, nullptr, nullptr, nullptr, nullptr, nullptr);
  return check_hip(hipGetLastError(), "fno_layer_kernel launch");
}

}  // extern "C"
