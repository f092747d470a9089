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
// Z / Zp rows are ordered (c, b, y): row (c * B + b) * H + y, 32 floats each.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"
#include "gelu.hpp"
#include "mfma.hpp"
#include "namsa_hip.h"

namespace namsa {
namespace {

constexpr int kCh = 32;                 // channels
constexpr int kQ = 32;                  // 2m row-DFT columns
constexpr int kTile = 32;               // pixels per tile
constexpr int kPitch = 40;              // LDS row pitch in bf16 (80 bytes: 16-byte aligned rows)
constexpr int kTiles = 2;               // tiles of a wavefront
constexpr int kRunTiles = 12;           // tiles of a workgroup at a time
constexpr int kTileBytes = 2 * kCh * kPitch + 2 * kQ * kTile;  // a rounded tile and its row-DFT operand

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
  const Rsrc rx = buffer_of(g.x, g.cin * g.pitch), ro = buffer_of(g.out, kCh * g.pitch);
  const Rsrc rp = buffer_of(ACT == kGelu ? g.pre_out : g.pre_in, ACT == kPlain ? 0 : kCh * g.pitch);
  const Rsrc rz = buffer_of(g.Zp, MODES ? 4 * kQ * kCh * g.rows : 0);
  const Rsrc rf = buffer_of(g.fx, MODES ? 2 * kQ * g.Wp : 0), rt = buffer_of(g.fxT, DFT ? 2 * kQ * g.Wp : 0);
  const Rsrc rw = buffer_of(g.Wt, 4 * kCh * g.cin), rb = buffer_of(g.bias, BIAS ? 4 * kCh : 0);
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
          modes = mfma(am[s], load_bf8(rf, 2 * (px * kQ + kh), 32 * s), modes);
      }
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        bf16x8 c;
#pragma unroll
        for (int e = 0; e < 8; ++e) c[e] = __bf16(in[t][s][e]);
        acc = mfma(aw[s], c, acc);
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
            zacc = mfma(f[64 * s + lane], ld8(&zt[col][16 * s + kh]), zacc);
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

// ------------------------------------------------------------------ the head
// out = Q2 gelu(Q1 x + bq1) + bq2, 32 -> 64 -> 2 channels, and its gradients.
// The hidden activation, 64 floats a pixel, is never stored: the backward pass
// forms it again from x, 1.9 GFLOP of matrix products (16 images of 170 x 170;
// 2 us at the bf16 rate) for each 118 MB (23 us) that hidden value,
// pre-activation and gradient took each time they were written or read.  At that size, as products of their own -> here:
// forward 129 -> 32 us, backward 340 -> 80 us, and 355 MB less held.

constexpr int kHid = 64;
constexpr int kOut = 2;
constexpr int kHeadTiles = 4;             // 32-pixel tiles of a forward wavefront
constexpr int kHeadWaves = 8;             // wavefronts of a backward workgroup
constexpr int kHPitch = kHid + 8;         // LDS row pitch in bf16 (144 bytes: 16-byte aligned rows)

struct HeadArgs {
  const float* x;                         // [32][n]
  const float *Q1, *bq1, *Q2, *bq2;       // [64][32], [64], [2][64], [2]
  int n;
  float* out;                             // [2][n]
  const float* gout;                      // [2][n]
  float *gx, *gQ1, *gbq1, *gQ2, *gbq2;
};

// 16 channels' steps of a tile, channels 16 s + 8 half + e at this lane's pixel
__device__ __forceinline__ void load_pixels(float (&v)[2][8], Rsrc r, int pitch, int px, int n, int kh) {
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e)
      v[s][e] = load_b32(r, px < n ? kh * pitch + 4 * px : kNowhere, (16 * s + e) * pitch);
}

__device__ __forceinline__ void round_pixels(bf16x8 (&b)[2], const float (&v)[2][8]) {
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) b[s][e] = __bf16(v[s][e]);
}

// Forward: bound by the 64 tanh of a pixel (about 45 instructions each).  The
// hidden block leaves the matrix cores with its pixel in the lane and 4 of
// every 8 units in each half of the wavefront; exchanging half the registers
// between the halves makes it the next product's operand, no LDS.
__global__ void __launch_bounds__(256) fno_head_kernel(HeadArgs g) {
  const int lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5, kh = 8 * half;
  const int pitch = 4 * g.n;
  const Rsrc rx = buffer_of(g.x, kCh * pitch), ro = buffer_of(g.out, kOut * pitch);
  const Rsrc rq1 = buffer_of(g.Q1, 4 * kHid * kCh), rq2 = buffer_of(g.Q2, 4 * kOut * kHid);
  const Rsrc rb1 = buffer_of(g.bq1, 4 * kHid);
  const int first = 32 * kHeadTiles * (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
  bf16x8 q1[2][2], q2[4];  // rows j of Q1, rows t of Q2
  float b1[2][16];
#pragma unroll
  for (int jb = 0; jb < 2; ++jb) {
#pragma unroll
    for (int s = 0; s < 2; ++s) q1[jb][s] = load_f8(rq1, 4 * (col * kCh + kh), 4 * (32 * jb * kCh + 16 * s));
#pragma unroll
    for (int i = 0; i < 16; ++i) b1[jb][i] = load_b32(rb1, 16 * half, 4 * (32 * jb + 8 * (i >> 2) + (i & 3)));
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) q2[s] = load_f8(rq2, col < kOut ? 4 * (col * kHid + kh) : kNowhere, 64 * s);
  const float b2[kOut] = {g.bq2[0], g.bq2[1]};
  float next[2][8];
  load_pixels(next, rx, pitch, first + col, g.n, kh);
  for (int t = 0; t < kHeadTiles; ++t) {
    const int x0 = first + 32 * t, px = x0 + col;
    if (x0 >= g.n) return;
    bf16x8 bx[2];
    round_pixels(bx, next);
    if (t + 1 < kHeadTiles) load_pixels(next, rx, pitch, px + 32, g.n, kh);
    f32x16 out = zero16();
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) {
      f32x16 acc = zero16();
#pragma unroll
      for (int s = 0; s < 2; ++s) acc = mfma(q1[jb][s], bx[s], acc);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        bf16x8 h;
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = __bf16(gelu_tanh(acc[8 * s + e] + b1[jb][8 * s + e]));
        out = mfma(q2[2 * jb + s], rows_to_k(h), out);
      }
    }
#pragma unroll
    for (int c = 0; c < kOut; ++c) store_b32(out[c] + b2[c], ro, half == 0 && px < g.n ? 4 * px : kNowhere, c * pitch);
  }
}

// Backward, one workgroup a CU, its wavefronts striding over the tiles with the
// weight gradients in their accumulators.  The hidden block is formed with its
// unit in the lane and 16 pixels in the registers: that is the operand of
// dQ1 = gh x^T, of dQ2 and of dbq1 as it stands (x and gout read once more, a
// channel a lane, the pixels in the registers' order).  Only gh goes through
// LDS, to become the operand of gx = Q1^T gh.  Bound by the 64 tanh of a pixel
// (one for value and derivative: two took 99 us) and the arithmetic around them.
__global__ void __launch_bounds__(64 * kHeadWaves, 2) fno_head_backward_kernel(HeadArgs g) {
  __shared__ __align__(16) __bf16 tt_all[kHeadWaves][32][kHPitch];
  __shared__ float red[kHid * kCh + kHid + kOut * kHid + kOut];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, half = lane >> 5, kh = 8 * half;
  __bf16 (*tt)[kHPitch] = tt_all[wave];
  const int pitch = 4 * g.n;
  const Rsrc rx = buffer_of(g.x, kCh * pitch), rg = buffer_of(g.gout, kOut * pitch), ro = buffer_of(g.gx, kCh * pitch);
  const Rsrc rq1 = buffer_of(g.Q1, 4 * kHid * kCh), rq2 = buffer_of(g.Q2, 4 * kOut * kHid);
  bf16x8 q1[2][2], q1t[4], q2[2];  // Q1 rows j; Q1^T rows c; Q2^T rows j
  float b1[2];
#pragma unroll
  for (int jb = 0; jb < 2; ++jb) {
    b1[jb] = g.bq1[32 * jb + col];
#pragma unroll
    for (int s = 0; s < 2; ++s) q1[jb][s] = load_f8(rq1, 4 * (col * kCh + kh), 4 * (32 * jb * kCh + 16 * s));
#pragma unroll
    for (int e = 0; e < 8; ++e)
      q2[jb][e] = __bf16(e < kOut ? load_b32(rq2, half == 0 ? 4 * col : kNowhere, 4 * (e * kHid + 32 * jb)) : 0.0f);
  }
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) q1t[s][e] = __bf16(load_b32(rq1, 4 * (kh * kCh + col), 4 * (16 * s + e) * kCh));

  bf16x8 ones;  // row kOut of an operand: sums the other over its pixels
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = __bf16(col == kOut ? 1.0f : 0.0f);
  f32x16 gq1[2] = {zero16(), zero16()}, gq2[2] = {zero16(), zero16()};  // gq2: rows of dQ2, then dbq1
  float gb2[kOut] = {0.0f, 0.0f};
  const int step = 32 * kHeadWaves * gridDim.x;
  int x0 = 32 * (kHeadWaves * blockIdx.x + wave);
  float next[2][8];
  load_pixels(next, rx, pitch, x0 + col, g.n, kh);
  for (; x0 < g.n; x0 += step) {
    const int px = x0 + col;
    bf16x8 bx[2], go, gt[2], xt[2];
    round_pixels(bx, next);
#pragma unroll
    for (int e = 0; e < 8; ++e) go[e] = __bf16(0.0f);
#pragma unroll
    for (int c = 0; c < kOut; ++c) {
      go[c] = __bf16(load_b32(rg, half == 0 && px < g.n ? 4 * px : kNowhere, c * pitch));
      gb2[c] += static_cast<float>(go[c]);
    }
    // a channel of x, or a row of gout, to a lane, at the hidden block's pixels
    // in register order: 8 (i / 4) + 4 half + i % 4
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int p = x0 + 8 * i + 4 * half;
      u32x4 xv, gv;
      if (x0 + 32 <= g.n) {
        xv = __builtin_amdgcn_raw_buffer_load_b128(rx, col * pitch + 4 * p, 0, 0);
        gv = __builtin_amdgcn_raw_buffer_load_b128(rg, col < kOut ? col * pitch + 4 * p : kNowhere, 0, 0);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool in = p + e < g.n;
          xv[e] = __builtin_amdgcn_raw_buffer_load_b32(rx, in ? col * pitch + 4 * (p + e) : kNowhere, 0, 0);
          gv[e] = __builtin_amdgcn_raw_buffer_load_b32(rg, in && col < kOut ? col * pitch + 4 * (p + e) : kNowhere, 0,
                                                       0);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        xt[i >> 1][4 * (i & 1) + e] = __bf16(__builtin_bit_cast(float, static_cast<unsigned>(xv[e])));
        gt[i >> 1][4 * (i & 1) + e] = __bf16(__builtin_bit_cast(float, static_cast<unsigned>(gv[e])));
      }
    }
    load_pixels(next, rx, pitch, px + step, g.n, kh);
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) {
      f32x16 pre = zero16();
#pragma unroll
      for (int s = 0; s < 2; ++s) pre = mfma(bx[s], q1[jb][s], pre);
      const f32x16 gh0 = mfma(go, q2[jb], zero16());
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        bf16x8 h, gh;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int i = 8 * s + e;
          const float v = pre[i] + b1[jb], t = gelu_inner(v);
          h[e] = __bf16(gelu_tanh(v, t));
          gh[e] = __bf16(gh0[i] * gelu_grad_tanh(v, t));
          tt[8 * (i >> 2) + 4 * half + (i & 3)][32 * jb + col] = gh[e];
        }
        gq1[jb] = mfma(gh, xt[s], gq1[jb]);
        gq2[jb] = mfma(gt[s], h, gq2[jb]);
        gq2[jb] = mfma(ones, gh, gq2[jb]);
      }
    }
    wave_sync();
    f32x16 gx = zero16();
#pragma unroll
    for (int s = 0; s < 4; ++s)
      gx = mfma(q1t[s], ld8(&tt[col][16 * s + kh]), gx);
    wave_sync();
    const int at = px < g.n ? 4 * half * pitch + 4 * px : kNowhere;
#pragma unroll
    for (int i = 0; i < 16; ++i) store_b32(gx[i], ro, at, (8 * (i >> 2) + (i & 3)) * pitch);
  }

  // the workgroup's sums, then one atomic a value
  constexpr int kB1 = kHid * kCh, kQ2 = kB1 + kHid, kB2 = kQ2 + kOut * kHid, kAll = kB2 + kOut;
  for (int i = threadIdx.x; i < kAll; i += 64 * kHeadWaves) red[i] = 0.0f;
  __syncthreads();
#pragma unroll
  for (int jb = 0; jb < 2; ++jb) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      atomicAdd(&red[(32 * jb + 8 * (i >> 2) + 4 * half + (i & 3)) * kCh + col], gq1[jb][i]);
    if (half == 0) {
#pragma unroll
      for (int c = 0; c < kOut; ++c) atomicAdd(&red[kQ2 + c * kHid + 32 * jb + col], gq2[jb][c]);
      atomicAdd(&red[kB1 + 32 * jb + col], gq2[jb][kOut]);
    }
  }
#pragma unroll
  for (int c = 0; c < kOut; ++c) {
    float v = gb2[c];  // the upper half's is 0
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (lane == 0) atomicAdd(&red[kB2 + c], v);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kAll; i += 64 * kHeadWaves) {
    float* dst = i < kB1 ? g.gQ1 + i : i < kQ2 ? g.gbq1 + (i - kB1) : i < kB2 ? g.gQ2 + (i - kQ2) : g.gbq2 + (i - kB2);
    atomicAdd(dst, red[i]);
  }
}

int head_size_ok(long long n, const char* who) {
  if (n <= 0 || n > 0x7fffffffLL / (4 * kCh))
    return fail(kErrArg, "%s: n=%lld pixels (32 channels must stay below 2 GiB)", who, n);
  return kOk;
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

int namsa_fno_head(const float* x, const float* Q1, const float* bq1, const float* Q2, const float* bq2, long long n,
                   float* out, void* stream) {
  if (int rc = head_size_ok(n, "namsa_fno_head")) return rc;
  if (!x || !Q1 || !bq1 || !Q2 || !bq2 || !out) return fail(kErrArg, "namsa_fno_head: null argument");
  const HeadArgs g{x, Q1, bq1, Q2, bq2, static_cast<int>(n), out, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  const int per = 4 * 32 * kHeadTiles;
  hipLaunchKernelGGL(fno_head_kernel, dim3((g.n + per - 1) / per), dim3(256), 0, as_stream(stream), g);
  return check_hip(hipGetLastError(), "fno_head_kernel launch");
}

int namsa_fno_head_backward(const float* x, const float* Q1, const float* bq1, const float* Q2, const float* gout,
                            long long n, float* gx, float* gQ1, float* gbq1, float* gQ2, float* gbq2, void* stream) {
  if (int rc = head_size_ok(n, "namsa_fno_head_backward")) return rc;
  if (!x || !Q1 || !bq1 || !Q2 || !gout || !gx || !gQ1 || !gbq1 || !gQ2 || !gbq2)
    return fail(kErrArg, "namsa_fno_head_backward: null argument");
  const HeadArgs g{x, Q1, bq1, Q2, nullptr, static_cast<int>(n), nullptr, gout, gx, gQ1, gbq1, gQ2, gbq2};
  const int per = 32 * kHeadWaves, groups = std::min((g.n + per - 1) / per, device_cu_count());
  hipLaunchKernelGGL(fno_head_backward_kernel, dim3(groups), dim3(64 * kHeadWaves), 0, as_stream(stream), g);
  return check_hip(hipGetLastError(), "fno_head_backward_kernel launch");
}

}  // extern "C"
