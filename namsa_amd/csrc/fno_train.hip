// The corrector network's Fourier layers in training: FP32 activations,
// channel-major [32][rows * W] (rows = B * H, one image row of one sample
// each), products on the matrix cores with operands rounded to bf16.
//
// A layer's full-width work is local to an image row, forward and backward:
//
//   v[o][x] = alpha sum_q Zp[o][q] Fx[x][q]  +  (sum_c W[o][c] in[c][x] + bias[o])
//   forward:  out = gelu(v), v kept;   backward: out = v gelu'(pre)
//   Z[o][q] = zalpha sum_x out[o][x] Fx[x][q]
//
// (backward with W transposed and no bias; Z is what the next layer, or the
// previous one's gradient, starts from).  The small mode-space products
// between Z and Zp stay on the strided GEMM.
//
// MFMA 32x32x16 operand layout (lane l, 8 bf16 per operand register set):
//   A: row l%32, k = 8*(l/32) + e      B: column l%32, k = 8*(l/32) + e
//   D: 16 floats, register r holds row 8*(r/4) + 4*(l/32) + r%4, column l%32.
// Z / Zp rows are ordered (c, b, y): row (c * B + b) * H + y, 32 floats each.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"
#include "gelu.hpp"
#include "namsa_hip.h"

namespace namsa {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kCh = 32;                 // channels
constexpr int kQ = 32;                  // 2m row-DFT columns
constexpr int kTile = 32;               // pixels per tile
constexpr int kPitch = 40;              // LDS row pitch in bf16 (80 bytes: 16-byte aligned rows)
constexpr int kTiles = 2;               // tiles of a wavefront
constexpr int kRunTiles = 12;           // tiles of a workgroup at a time
constexpr int kTileBytes = 2 * kCh * kPitch + 2 * kQ * kTile;  // a rounded tile and its row-DFT operand
constexpr int kRawBuffer = 0x00020000;  // gfx9 raw-buffer resource word 3
constexpr int kNowhere = 0x7ffffffc;    // a byte offset past every buffer: stores there are dropped

__device__ __forceinline__ bf16x8 ld8(const __bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }

typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Accesses through a buffer resource at a lane's and a scalar byte offset;
// reads past its end give 0, stores there are dropped.
__device__ __forceinline__ float load_b32(Rsrc r, int lane_at, int at) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, lane_at, at, 0));
}
__device__ __forceinline__ void store_b32(float v, Rsrc r, int lane_at, int at) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, lane_at, at, 0);
}
__device__ __forceinline__ bf16x8 load_bf8(Rsrc r, int lane_at, int at) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, lane_at, at, 0));
}
// eight consecutive floats, rounded to bf16
__device__ __forceinline__ bf16x8 load_f8(Rsrc r, int lane_at, int at) {
  const u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(r, lane_at, at, 0);
  const u32x4 b = __builtin_amdgcn_raw_buffer_load_b128(r, lane_at, at + 16, 0);
  bf16x8 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = __bf16(__builtin_bit_cast(float, static_cast<unsigned>(a[e])));
    v[e + 4] = __bf16(__builtin_bit_cast(float, static_cast<unsigned>(b[e])));
  }
  return v;
}

__device__ __forceinline__ f32x16 zero16() {
  f32x16 v;
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = 0.0f;
  return v;
}

// v + alpha x with the product rounded first, as the separate products do
__device__ __forceinline__ float add_scaled(float v, float alpha, float x) {
#pragma clang fp contract(off)
  const float p = alpha * x;
  return v + p;
}

struct RowArgs {
  const float* x;
  int cin;                    // channels of x
  const float* Zp;
  const __bf16* fx;           // [Wp][32]
  const __bf16* fxT;          // [32][Wp], zero from column W on
  const float* Wt;
  int sWo, sWc;
  const float* bias;
  float alpha, zalpha;
  const float* pre_in;
  float* pre_out;
  float* out;
  float* Z;
  int rows, W, Wp, H, B;
  int pitch;                  // bytes from one channel to the next
};

enum Act { kPlain, kGelu, kGeluGrad };

// One workgroup takes one image row, a wavefront two 32-pixel tiles of it (of
// each run of 12 tiles); KS steps of 16 input channels, MODES: the mode
// product joins in, DFT: Z is formed, by the first wavefront from the rounded
// tiles the others leave in LDS.  Bound by the activations read and written,
// each once (a GELU layer 178 MB for 16 images of 170 x 170).  As separate
// products v was also written and read, `out` read again for its row DFT and,
// backward, the gradient read and written for gelu'.  At that size, separate
// -> here: layer 118 -> 49 us (3.6 TB/s), backward 132 -> 52, last layer 60 ->
// 28, lift and row DFT 38 -> 20.  The two products keep an accumulator each and
// every sum its order: the bits are those of the separate products.
//
// Two tiles a wavefront, at two or three wavefronts a SIMD: the weights, Zp and
// bias are fetched once for both and all their pixels' loads are in flight
// together.  One tile 56 and 69 us (the operands' fetches), two within 128
// registers 51 and 63 (the pixels' loads wait for one another), a wavefront to
// a whole row 68 and 67 (too few wavefronts).  Accesses go through buffer
// resources, the channel in the scalar offset: as 64-bit pointers the 16
// channels' addresses took more registers than the data.
template <int KS, bool MODES, bool TRANS, bool BIAS, Act ACT, bool DFT>
__global__ void __launch_bounds__(64 * kRunTiles / kTiles, 2) fno_rows_kernel(RowArgs g) {
  extern __shared__ __align__(16) char tiles[];  // [kTiles * waves][kTileBytes]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = blockDim.x >> 6;
  // neighbouring rows share cache lines: an eighth of the rows to each XCD
  const int xcd = blockIdx.x & 7, each = g.rows >> 3;
  const int r = xcd * each + min(xcd, g.rows & 7) + (blockIdx.x >> 3);
  const int col = lane & 31, half = lane >> 5, kh = 8 * half;
  const int b = r / g.H, y = r % g.H;
  const int zrow = 4 * kQ * ((col * g.B + b) * g.H + y);  // byte offset of channel `col` in Z and Zp
  const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.x), 0, g.cin * g.pitch, kRawBuffer);
  const auto ro = __builtin_amdgcn_make_buffer_rsrc(g.out, 0, kCh * g.pitch, kRawBuffer);
  const auto rp = __builtin_amdgcn_make_buffer_rsrc(ACT == kGelu ? g.pre_out : const_cast<float*>(g.pre_in), 0,
                                                    ACT == kPlain ? 0 : kCh * g.pitch, kRawBuffer);
  const auto rz = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.Zp), 0, MODES ? 4 * kQ * kCh * g.rows : 0,
                                                    kRawBuffer);
  const auto rf = __builtin_amdgcn_make_buffer_rsrc(const_cast<__bf16*>(g.fx), 0, MODES ? 2 * kQ * g.Wp : 0, kRawBuffer);
  const auto rt = __builtin_amdgcn_make_buffer_rsrc(const_cast<__bf16*>(g.fxT), 0, DFT ? 2 * kQ * g.Wp : 0, kRawBuffer);
  const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.Wt), 0, 4 * kCh * g.cin, kRawBuffer);
  const auto rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.bias), 0, BIAS ? 4 * kCh : 0, kRawBuffer);
  const int row = 4 * r * g.W;  // byte offset of the image row in a channel

  f32x16 zacc = zero16();
  for (int t0 = 0; 32 * t0 < g.W; t0 += kTiles * waves) {
    const int first = 32 * (t0 + kTiles * wave);  // this wavefront's first pixel
    // the small operands first, so that rounding them does not wait for the
    // pixels; bias here as well: among the stores a read would wait for them
    float bias[BIAS ? 16 : 1];
    if constexpr (BIAS) {
#pragma unroll
      for (int i = 0; i < 16; ++i) bias[i] = load_b32(rb, 16 * half, 4 * (8 * (i >> 2) + (i & 3)));
    }
    bf16x8 aw[KS], am[2];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if constexpr (KS == 2 && !TRANS) {
        aw[s] = load_f8(rw, 4 * (col * g.sWo + kh), 64 * s);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float w = load_b32(rw, 4 * (col * g.sWo + kh * g.sWc), 4 * (16 * s + e) * g.sWc);
          aw[s][e] = __bf16(16 * s + kh + e < g.cin ? w : 0.0f);
        }
      }
    }
    if constexpr (MODES) {
#pragma unroll
      for (int s = 0; s < 2; ++s) am[s] = load_f8(rz, zrow + 4 * kh, 64 * s);
    }
    float in[kTiles][KS][8], pre[kTiles][16];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      const int px = first + 32 * t + col;
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          in[t][s][e] = load_b32(rx, px < g.W ? kh * g.pitch + 4 * px : kNowhere, (16 * s + e) * g.pitch + row);
    }
    if constexpr (ACT == kGeluGrad) {
#pragma unroll
      for (int t = 0; t < kTiles; ++t) {
        const int px = first + 32 * t + col;
#pragma unroll
        for (int i = 0; i < 16; ++i)
          pre[t][i] = load_b32(rp, px < g.W ? 4 * half * g.pitch + 4 * px : kNowhere,
                               (8 * (i >> 2) + (i & 3)) * g.pitch + row);
      }
    }
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      const int x0 = first + 32 * t, px = x0 + col;
      if (x0 >= g.W) break;
      __bf16 (*tt)[kPitch] = reinterpret_cast<__bf16 (*)[kPitch]>(tiles + (kTiles * wave + t) * kTileBytes);
      if constexpr (DFT) {  // the row DFT's operand of this tile, for the first wavefront
        bf16x8* f = reinterpret_cast<bf16x8*>(reinterpret_cast<char*>(tt) + kCh * kPitch * 2);
#pragma unroll
        for (int s = 0; s < 2; ++s) f[64 * s + lane] = load_bf8(rt, 2 * (col * g.Wp + kh), 2 * (x0 + 16 * s));
      }
      f32x16 acc = zero16(), modes = zero16();
      if constexpr (MODES) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
          modes = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am[s], load_bf8(rf, 2 * (px * kQ + kh), 32 * s), modes, 0, 0,
                                                          0);
      }
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        bf16x8 c;
#pragma unroll
        for (int e = 0; e < 8; ++e) c[e] = __bf16(in[t][s][e]);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(aw[s], c, acc, 0, 0, 0);
      }
      const int at = px < g.W ? 4 * half * g.pitch + 4 * px : kNowhere;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int chan = (8 * (i >> 2) + (i & 3)) * g.pitch + row;
        float v = acc[i];
        if constexpr (BIAS) v += bias[i];
        if constexpr (MODES) v = add_scaled(v, g.alpha, modes[i]);
        if constexpr (ACT == kGelu) {
          store_b32(v, rp, at, chan);
          v = gelu_tanh(v);
        }
        if constexpr (ACT == kGeluGrad) v *= gelu_grad_tanh(pre[t][i]);
        store_b32(v, ro, at, chan);
        if constexpr (DFT) tt[8 * (i >> 2) + 4 * half + (i & 3)][col] = __bf16(px < g.W ? v : 0.0f);
      }
    }
    if constexpr (DFT) {
      // zacc(q, c) += sum_x Fx[x][q] out[c][x] tile by tile, pixels now along k
      __syncthreads();
      if (wave == 0) {
        for (int w = 0; w < kTiles * waves && 32 * (t0 + w) < g.W; ++w) {
          const char* t = tiles + w * kTileBytes;
          const __bf16 (*zt)[kPitch] = reinterpret_cast<const __bf16 (*)[kPitch]>(t);
          const bf16x8* f = reinterpret_cast<const bf16x8*>(t + kCh * kPitch * 2);
#pragma unroll
          for (int s = 0; s < 2; ++s)
            zacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[64 * s + lane], ld8(&zt[col][16 * s + kh]), zacc, 0, 0, 0);
        }
      }
      if (32 * (t0 + kTiles * waves) < g.W) __syncthreads();
    }
  }
  if constexpr (DFT) {
    if (wave > 0) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float4 z;
      z.x = g.zalpha * zacc[4 * i];
      z.y = g.zalpha * zacc[4 * i + 1];
      z.z = g.zalpha * zacc[4 * i + 2];
      z.w = g.zalpha * zacc[4 * i + 3];
      *reinterpret_cast<float4*>(reinterpret_cast<char*>(g.Z) + zrow + 32 * i + 16 * half) = z;
    }
  }
}

template <int KS, bool MODES, bool TRANS, bool BIAS, Act ACT, bool DFT>
int launch_rows(const RowArgs& g, hipStream_t st) {
  // runs of at most kRunTiles tiles (55 KiB of LDS), as equal as they get
  const int need = (g.W + kTiles * kTile - 1) / (kTiles * kTile), runs = (need * kTiles + kRunTiles - 1) / kRunTiles;
  const int waves = (need + runs - 1) / runs;
  const size_t lds = DFT ? static_cast<size_t>(kTileBytes) * kTiles * waves : 0;
  hipLaunchKernelGGL((fno_rows_kernel<KS, MODES, TRANS, BIAS, ACT, DFT>), dim3(g.rows), dim3(64 * waves), lds, st, g);
  return check_hip(hipGetLastError(), "fno_rows_kernel launch");
}

}  // namespace
}  // namespace namsa

using namespace namsa;

extern "C" {

int namsa_fno_rows(const float* x, int cin, const float* Zp, const void* fx, const void* fxT, const float* Wt,
                   int transposed, const float* bias, float alpha, const float* pre_in, float* pre_out,
                   float zalpha, int B, int H, int W, int Wp, float* out, float* Z, void* stream) {
  if (B <= 0 || H <= 0 || W <= 0 || Wp < W || Wp % kTile != 0 ||
      static_cast<long long>(B) * H > 0x7fffffffLL / (4LL * kCh * std::max(W, kQ)))
    return fail(kErrArg, "namsa_fno_rows: bad geometry B=%d H=%d W=%d Wp=%d (Wp a multiple of 32, >= W; 32 channels "
                "below 2 GiB)", B, H, W, Wp);
  if (!x || !Wt || !out || (Zp ? cin != kCh : cin < 1 || cin > 16) || (Zp && !fx) || (Z && !fxT))
    return fail(kErrArg, "namsa_fno_rows: null argument or cin=%d (a layer takes 32, the lift 1..16)", cin);
  const RowArgs g{x,       cin, Zp, static_cast<const __bf16*>(fx), static_cast<const __bf16*>(fxT), Wt,
                  transposed ? 1 : cin, transposed ? kCh : 1, bias,
                  alpha,   zalpha, pre_in, pre_out, out, Z, B * H, W, Wp, H, B, 4 * B * H * W};
  hipStream_t st = as_stream(stream);
  const bool none = !pre_in && !pre_out;
  if (!Zp && Z && bias && none && !transposed) return launch_rows<1, false, false, true, kPlain, true>(g, st);
  if (Zp && Z && bias && pre_out && !pre_in && !transposed)
    return launch_rows<2, true, false, true, kGelu, true>(g, st);
  if (Zp && Z && !bias && pre_in && !pre_out && transposed)
    return launch_rows<2, true, true, false, kGeluGrad, true>(g, st);
  if (Zp && !Z && none && bias && !transposed) return launch_rows<2, true, false, true, kPlain, false>(g, st);
  if (Zp && !Z && none && !bias && transposed) return launch_rows<2, true, true, false, kPlain, false>(g, st);
  return fail(kErrArg, "namsa_fno_rows: no layer has this combination of Zp, Z, bias, pre_in and pre_out");
}

}  // extern "C"
