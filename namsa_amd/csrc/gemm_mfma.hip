// Strided batched GEMM on CDNA4 matrix cores: BF16 operands, FP32 accumulate.
//
//   C[b](i,j) = alpha * sum_k A[b](i,k) B[b](k,j) + beta * C[b](i,j)  (+ bias, GELU)
//
// Operands live in HBM as FP32 with arbitrary element strides (so transposes
// and the planar complex layouts of the corrector network need no copies).
// A 256-thread workgroup (4 wavefronts) computes a TM x TN tile of C, each
// wavefront one 32 x 32 block with v_mfma_f32_32x32x16_bf16.  The tile shape
// follows the matrix: the corrector's products are skinny (one side is a
// 32-channel or 32-mode dimension), so N <= 32 takes 128 x 32 tiles, M <= 32
// takes 32 x 128 tiles and the rest 64 x 64 -- no wavefront idles on a
// 32-wide side -- and batches of many items that each fit one 32 x 32 block
// take one workgroup per item.  Operand tiles of K = 32 are staged through LDS
// as bf16 with k contiguous: the unit-stride axis is read with 16-byte loads
// (at any 4-byte aligned address), and the next K tile is loaded into registers
// while the matrix cores work on the current one.  MFMA operands come out of
// LDS as 16-byte reads.  Pointwise layers over many columns run without LDS
// (gemm_pointwise_kernel).  With split_k > 1 the K range is divided over
// workgroups and partial products are added to C with FP32 atomics (C must then
// already hold beta*C); gemm_split_kernel takes the small products over a long
// contiguous K.
//
// MFMA 32x32x16 operand layout (lane l, 8 bf16 per operand register set):
//   A: row l%32, k = 8*(l/32) + e      B: column l%32, k = 8*(l/32) + e
//   D: 16 floats, register r holds row 8*(r/4) + 4*(l/32) + r%4, column l%32.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "common.hpp"
#include "gelu.hpp"
#include "gemm_paths.hpp"
#include "namsa_hip.h"

namespace namsa {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct GemmArgs {
  const float* A;
  long long sAb, sAi, sAk;
  const float* B;
  long long sBb, sBk, sBj;
  float* C;
  long long sCb, sCi, sCj;
  int M, N, K, batch, split_k;
  float alpha, beta;
  const float* bias;  // bias_mode 1: bias[i]; 2: bias[j]
  int bias_mode;
  int gelu;           // 1: C = gelu(value), pre-activation stored to P
  float* P;           // same strides as C
};

constexpr int kTK = 32;
constexpr int kLdK = kTK + 8;  // LDS row pitch in bf16: 80 bytes keeps every row 16-byte aligned

// Four consecutive floats at any 4-byte aligned address, one 16-byte load.
struct alignas(4) F4 {
  float v[4];
};

// One operand tile of R rows (i for A, j for B) by kTK k values, element
// (r, k) at base + (r0 + r) * sr + (k0 + k) * sk, valid for r0 + r < rows
// and k0 + k < k_end.  Each thread carries G groups of 4 elements that are
// consecutive along the operand's unit-stride axis (k when kfast).
template <int R>
struct Tile {
  static constexpr int G = R * kTK / 4 / 256;
  float v[G][4];

  __device__ __forceinline__ void load(const float* __restrict__ base, long long sr, long long sk, int r0,
                                       int rows, int k0, int k_end, bool kfast, bool vec) {
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const int grp = threadIdx.x + 256 * q;
      int r, k;
      if (kfast) {
        r = grp / (kTK / 4);
        k = (grp % (kTK / 4)) * 4;
      } else {
        k = grp / (R / 4);
        r = (grp % (R / 4)) * 4;
      }
      const int gr = r0 + r, gk = k0 + k;
      if (vec && (kfast ? (gr < rows && gk + 3 < k_end) : (gr + 3 < rows && gk < k_end))) {
        const F4 f = *reinterpret_cast<const F4*>(base + gr * sr + gk * sk);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[q][e] = f.v[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int er = kfast ? gr : gr + e, ek = kfast ? gk + e : gk;
          v[q][e] = (er < rows && ek < k_end) ? base[er * sr + ek * sk] : 0.0f;
        }
      }
    }
  }

  __device__ __forceinline__ void store(__bf16 (*lds)[kLdK], bool kfast) const {
#pragma unroll
    for (int q = 0; q < G; ++q) {
      const int grp = threadIdx.x + 256 * q;
      if (kfast) {
        const int r = grp / (kTK / 4), k = (grp % (kTK / 4)) * 4;
        bf16x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = __bf16(v[q][e]);
        *reinterpret_cast<bf16x4*>(&lds[r][k]) = h;
      } else {
        const int k = grp / (R / 4), r = (grp % (R / 4)) * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) lds[r + e][k] = __bf16(v[q][e]);
      }
    }
  }
};

template <int WM, int WN>
__global__ void __launch_bounds__(256) gemm_bf16_kernel(GemmArgs g) {
  constexpr int TM = 32 * WM, TN = 32 * WN;
  __shared__ __align__(16) __bf16 As[TM][kLdK];
  __shared__ __align__(16) __bf16 Bs[TN][kLdK];  // transposed: [j][k]

  const int tiles_n = (g.N + TN - 1) / TN;
  const int tm = blockIdx.x / tiles_n, tn = blockIdx.x % tiles_n;
  const int b = blockIdx.y;
  const int split = blockIdx.z;
  const int i0 = tm * TM, j0 = tn * TN;
  const int k_per = ((g.K + g.split_k - 1) / g.split_k + kTK - 1) / kTK * kTK;
  const int k_begin = split * k_per;
  const int k_end = min(g.K, k_begin + k_per);

  const float* A = g.A + b * g.sAb;
  const float* B = g.B + b * g.sBb;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN;

  // A rows are i (stride sAi), B rows are j (stride sBj); k is the column
  const bool a_kfast = g.sAk == 1 || (g.sAi != 1 && g.sAk <= g.sAi);
  const bool b_kfast = g.sBk == 1 || (g.sBj != 1 && g.sBk <= g.sBj);
  const bool a_vec = (a_kfast ? g.sAk : g.sAi) == 1;
  const bool b_vec = (b_kfast ? g.sBk : g.sBj) == 1;

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;

  Tile<TM> ta;
  Tile<TN> tb;
  if (k_begin < k_end) {
    ta.load(A, g.sAi, g.sAk, i0, g.M, k_begin, k_end, a_kfast, a_vec);
    tb.load(B, g.sBj, g.sBk, j0, g.N, k_begin, k_end, b_kfast, b_vec);
  }
  for (int k0 = k_begin; k0 < k_end; k0 += kTK) {
    ta.store(As, a_kfast);
    tb.store(Bs, b_kfast);
    __syncthreads();
    if (k0 + kTK < k_end) {  // next K tile in flight while the matrix cores work
      ta.load(A, g.sAi, g.sAk, i0, g.M, k0 + kTK, k_end, a_kfast, a_vec);
      tb.load(B, g.sBj, g.sBk, j0, g.N, k0 + kTK, k_end, b_kfast, b_vec);
    }
    const int ra = wm * 32 + (lane & 31), rb = wn * 32 + (lane & 31);
#pragma unroll
    for (int ks = 0; ks < kTK; ks += 16) {
      const int kk = ks + 8 * (lane >> 5);
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(&As[ra][kk]);
      const bf16x8 bb = *reinterpret_cast<const bf16x8*>(&Bs[rb][kk]);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bb, acc, 0, 0, 0);
    }
    __syncthreads();
  }

  float* C = g.C + b * g.sCb;
  float* P = g.P ? g.P + b * g.sCb : nullptr;
  const int j = j0 + wn * 32 + (lane & 31);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int i = i0 + wm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
    if (i >= g.M || j >= g.N) continue;
    float* c = C + i * g.sCi + j * g.sCj;
    float v = g.alpha * acc[r];
    if (g.split_k > 1) {
      atomicAdd(c, v);
      continue;
    }
    if (g.beta != 0.0f) v += g.beta * *c;
    if (g.bias_mode == 1) v += g.bias[i];
    if (g.bias_mode == 2) v += g.bias[j];
    if (g.gelu) {
      P[i * g.sCi + j * g.sCj] = v;
      v = gelu_tanh(v);
    }
    *c = v;
  }
}

// Epilogue of one 32 x 32 MFMA block of item b, rows i0 .. i0 + 31 and columns
// j0 .. j0 + 31:
// C = alpha acc + beta C (+ bias), optionally keeping the pre-activation in P
// and applying GELU.  Register r of lane l holds row 8(r/4) + 4(l/32) + r%4,
// column l%32.
__device__ __forceinline__ void store_block(const GemmArgs& g, long long b, const f32x16& acc, int i0, int j0,
                                            int lane) {
  float* C = g.C + b * g.sCb;
  float* P = g.P ? g.P + b * g.sCb : nullptr;
  const int j = j0 + (lane & 31);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int i = i0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
    if (i >= g.M || j >= g.N) continue;
    float* c = C + i * g.sCi + j * g.sCj;
    float v = g.alpha * acc[r];
    if (g.beta != 0.0f) v += g.beta * *c;
    if (g.bias_mode == 1) v += g.bias[i];
    if (g.bias_mode == 2) v += g.bias[j];
    if (g.gelu) {
      P[i * g.sCi + j * g.sCj] = v;
      v = gelu_tanh(v);
    }
    *c = v;
  }
}

// Batched products whose every matrix fits one MFMA block (M <= 32, N <= 32;
// the y transforms of a corrector of other than 16 modes, hundreds of items):
// one workgroup per batch item, its four wavefronts taking every fourth
// K step of 16 with the operands read straight into the MFMA layout, the
// partial accumulators summed through LDS.  Splitting K shortens each
// wavefront's chain of dependent loads and MFMAs fourfold; one wavefront
// per item left the loads' latency exposed (about 0.8 TB/s on the operand).
__global__ void __launch_bounds__(256) gemm_small_kernel(GemmArgs g) {
  __shared__ float part[3][16][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long b = blockIdx.x;
  const float* A = g.A + b * g.sAb;
  const float* B = g.B + b * g.sBb;
  const int row = lane & 31, kh = 8 * (lane >> 5);
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  for (int k0 = 16 * wave; k0 < g.K; k0 += 64) {
    bf16x8 a, bb;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = k0 + kh + e;
      a[e] = __bf16((row < g.M && k < g.K) ? A[row * g.sAi + k * g.sAk] : 0.0f);
      bb[e] = __bf16((row < g.N && k < g.K) ? B[k * g.sBk + row * g.sBj] : 0.0f);
    }
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bb, acc, 0, 0, 0);
  }
  if (wave > 0) {
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave - 1][r][lane] = acc[r];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] += part[0][r][lane] + part[1][r][lane] + part[2][r][lane];
  store_block(g, b, acc, 0, 0, lane);
}

// Eight consecutive k of one operand row as an MFMA register set, rounded to
// bf16; `left` of them exist, the others are 0.  Rows need not be 16-byte
// aligned: the loads only assume 4-byte alignment.
__device__ __forceinline__ bf16x8 load_k8(const float* __restrict__ p, int left) {
  bf16x8 h;
  if (left >= 8) {
    const F4 a = *reinterpret_cast<const F4*>(p), b = *reinterpret_cast<const F4*>(p + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h[e] = __bf16(a.v[e]);
      h[e + 4] = __bf16(b.v[e]);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) h[e] = __bf16(e < left ? p[e] : 0.0f);
  }
  return h;
}

// Split-K products of few rows and columns (M <= 32 MT, N <= 32 NT) over a
// long K with both operands contiguous along it: the weight gradients, sums
// over every pixel of a batch.  Bound by reading the operands once, so a
// workgroup's four wavefronts each take every fourth step of 32 k of its K
// range, with all 32 x 32 blocks of the result in their accumulators and the
// operands read straight into the MFMA layout (a tile staged through LDS left
// three of four wavefronts without a block and one load in flight per
// barrier).  The wavefronts' blocks are summed through LDS and added to C with
// one FP32 atomic per value and workgroup, so one workgroup per CU: two per CU
// were no faster.  Over 462,400 k: 32 x 32 175 -> 30 us (3.9 TB/s), 64 x 32 239
// -> 42, 32 sums 185 -> 22, against 112 staged workgroups.
// SUMS: each row's sum over k (a layer's bias gradient) is formed as well, a
// product with ones, and added to `sums`: 462,400 k, 32 x 32 28 -> 30 us,
// against 23 us more for reading the rows again.
template <int MT, int NT, bool SUMS>
__global__ void __launch_bounds__(256) gemm_split_kernel(GemmArgs g, int k_per, float* __restrict__ sums) {
  __shared__ float part[4][MT * NT][16][64];
  __shared__ float part_sums[4][SUMS ? 32 * MT : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long b = blockIdx.y;
  const int row = lane & 31, kh = 8 * (lane >> 5);
  const int k_begin = blockIdx.x * k_per, k_len = split_len(g.K, k_begin, k_per);
  // lanes past the last row or column read that row: what they add to goes
  // into values that are not stored
  const float* A[MT];
  const float* B[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) A[i] = g.A + b * g.sAb + min(32 * i + row, g.M - 1) * g.sAi + k_begin + kh;
#pragma unroll
  for (int j = 0; j < NT; ++j) B[j] = g.B + b * g.sBb + min(32 * j + row, g.N - 1) * g.sBj + k_begin + kh;
  f32x16 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  f32x16 total[MT];  // in column 0
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = __bf16(row == 0 ? 1.0f : 0.0f);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) total[i][r] = 0.0f;
#pragma unroll 2
  for (int k0 = 32 * wave; k0 < k_len; k0 += 128) {
    bf16x8 a[MT][2], c[NT][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int left = k_len - k0 - kh - 16 * h;
#pragma unroll
      for (int i = 0; i < MT; ++i) a[i][h] = load_k8(A[i] + k0 + 16 * h, left);
#pragma unroll
      for (int j = 0; j < NT; ++j) c[j][h] = load_k8(B[j] + k0 + 16 * h, left);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][h], c[j][h], acc[i][j], 0, 0, 0);
        if constexpr (SUMS) total[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][h], ones, total[i], 0, 0, 0);
      }
  }
  if constexpr (SUMS) {
    if (row == 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) part_sums[wave][32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)] = total[i][r];
    }
  }
#pragma unroll
  for (int t = 0; t < MT * NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][t][r][lane] = acc[t / NT][t % NT][r];
  __syncthreads();
  // values in row-major order over the threads, so that one atomic
  // instruction covers neighbouring addresses (a column of sums, N = 1, took
  // 48 us with a wavefront's registers stored one by one, 32 lines' worth of
  // atomics on one line)
  float* C = g.C + b * g.sCb;
  for (int v = threadIdx.x; v < g.M * g.N; v += 256) {
    const int i = v / g.N, j = v % g.N;
    const int t = (i >> 5) * NT + (j >> 5), r = 4 * ((i & 31) >> 3) + (i & 3), l = (j & 31) + 32 * ((i >> 2) & 1);
    const float sum = (part[0][t][r][l] + part[1][t][r][l]) + (part[2][t][r][l] + part[3][t][r][l]);
    atomicAdd(C + i * g.sCi + j * g.sCj, g.alpha * sum);
  }
  if constexpr (SUMS) {
    const int i = threadIdx.x;
    if (i < g.M) atomicAdd(sums + i, (part_sums[0][i] + part_sums[1][i]) + (part_sums[2][i] + part_sums[3][i]));
  }
}

// Pointwise layers of networks of other widths than the row and head kernels
// of training are compiled for: few rows and a short K (M <= 32 MT, K <= 16 KS)
// over a long unit-stride N, the pixels of a batch.  Bound by streaming B and C once
// (a tile staged through LDS wrote its bf16 operands two bytes at a time and
// had nothing in flight across its barriers).  A wavefront holds A in the MFMA
// layout and takes PB blocks of 32 columns, every read of B issued before the
// first product.  Reads and writes are buffer accesses: a scalar row offset
// and one lane offset (with pointers the 64-bit addresses took 250 registers),
// rows past K read 0 and rows past M are not written, being past the buffer's
// end (pointwise_fits: no offset wraps).  The products run
// over k in the order of the staged kernel.  Over 462,400 columns: 32
// x 32 with bias 47 -> 32 us, with beta 57 -> 31, 32 x 7 44 -> 16, 64 x 32 with
// GELU 109 -> 82 (296 MB).
constexpr int kRawBuffer = 0x00020000;  // gfx9 raw-buffer resource word 3

template <int MT, int KS, int PB, bool BIAS>
__global__ void __launch_bounds__(256) gemm_pointwise_kernel(GemmArgs g) {
  const int lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5;
  const int sB = static_cast<int>(g.sBk) * 4, sC = static_cast<int>(g.sCi) * 4;  // row pitches in bytes
  const auto rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(g.B), 0, (g.K - 1) * sB + g.N * 4, kRawBuffer);
  const auto rc = __builtin_amdgcn_make_buffer_rsrc(g.C, 0, (g.M - 1) * sC + g.N * 4, kRawBuffer);
  const auto rp = __builtin_amdgcn_make_buffer_rsrc(g.P, 0, g.P ? (g.M - 1) * sC + g.N * 4 : 0, kRawBuffer);
  const int j0 = 32 * PB * (blockIdx.x * 4 + (threadIdx.x >> 6)) + col;
  float x[PB][KS][8];
#pragma unroll
  for (int p = 0; p < PB; ++p)
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        x[p][s][e] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(rb, 8 * half * sB + 4 * (j0 + 32 * p), (16 * s + e) * sB, 0));
  bf16x8 a[MT][KS];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int row = 32 * i + col, k = 16 * s + 8 * half + e;
        const float w = g.A[min(row, g.M - 1) * g.sAi + min(k, g.K - 1) * g.sAk];
        a[i][s][e] = __bf16(row < g.M && k < g.K ? w : 0.0f);
      }
  float bias[BIAS ? MT : 1][16];  // read here: a read after the products would wait for all of x
  if constexpr (BIAS) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) bias[i][r] = g.bias[min(32 * i + 8 * (r >> 2) + 4 * half + (r & 3), g.M - 1)];
  }
#pragma unroll
  for (int p = 0; p < PB; ++p) {
    const int j = j0 + 32 * p;
    bf16x8 b[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) b[s][e] = __bf16(x[p][s][e]);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      f32x16 acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][s], b[s], acc, 0, 0, 0);
      if (j >= g.N) continue;
      const int at = 4 * half * sC + 4 * j;
      float old[16];
      if (g.beta != 0.0f) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          old[r] = __builtin_bit_cast(
              float, __builtin_amdgcn_raw_buffer_load_b32(rc, at, (32 * i + 8 * (r >> 2) + (r & 3)) * sC, 0));
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row0 = 32 * i + 8 * (r >> 2) + (r & 3);
        float v = g.alpha * acc[r];
        if (g.beta != 0.0f) v += g.beta * old[r];
        if constexpr (BIAS) v += bias[i][r];
        if (g.bias_mode == 2) v += g.bias[j];
        if (g.gelu) {
          __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rp, at, row0 * sC, 0);
          v = gelu_tanh(v);
        }
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rc, at, row0 * sC, 0);
      }
    }
  }
}

template <int MT, int KS>
int launch_pointwise(const GemmArgs& g, hipStream_t st) {
  // blocks per wavefront: 4 with a bias (its 16 reads per 32 rows are then
  // paid once per 128 columns) and for K = 32, else 2
  constexpr int PB = KS == 2 ? 4 : 2;
  static_assert(128 * 4 <= kPointwiseCols, "pointwise_fits counts the columns of a workgroup");
  const auto grid = [&](int pb) { return dim3((g.N + 128 * pb - 1) / (128 * pb)); };
  if (g.bias_mode == 1)
    hipLaunchKernelGGL((gemm_pointwise_kernel<MT, KS, 4, true>), grid(4), dim3(256), 0, st, g);
  else
    hipLaunchKernelGGL((gemm_pointwise_kernel<MT, KS, PB, false>), grid(PB), dim3(256), 0, st, g);
  return check_hip(hipGetLastError(), "gemm_pointwise_kernel launch");
}

template <int MT, int NT, bool SUMS = false>
int launch_split(const GemmArgs& g, hipStream_t st, float* sums = nullptr) {
  const SplitPlan plan = split_plan(g.K, g.batch, device_cu_count());
  hipLaunchKernelGGL((gemm_split_kernel<MT, NT, SUMS>), dim3(plan.groups, g.batch), dim3(256), 0, st, g, plan.k_per,
                     sums);
  return check_hip(hipGetLastError(), "gemm_split_kernel launch");
}

template <int WM, int WN>
int launch_gemm(const GemmArgs& g, hipStream_t st) {
  constexpr int TM = 32 * WM, TN = 32 * WN;
  const long long tiles = static_cast<long long>((g.M + TM - 1) / TM) * ((g.N + TN - 1) / TN);
  if (tiles > 0x7fffffffLL) return fail(kErrArg, "namsa_gemm_bf16: too many tiles");
  hipLaunchKernelGGL((gemm_bf16_kernel<WM, WN>), dim3(static_cast<unsigned>(tiles), g.batch, g.split_k), dim3(256), 0,
                     st, g);
  return check_hip(hipGetLastError(), "gemm_bf16_kernel launch");
}

}  // namespace namsa

using namespace namsa;

extern "C" {

int namsa_gemm_bf16(const float* A, long long sAb, long long sAi, long long sAk, const float* B,
                    long long sBb, long long sBk, long long sBj, float* C, long long sCb,
                    long long sCi, long long sCj, int M, int N, int K, int batch, int split_k,
                    float alpha, float beta, const float* bias, int bias_mode, int gelu, float* P,
                    void* stream) {
  if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0 || batch <= 0 || split_k <= 0 || batch > 65535 ||
      split_k > 65535)
    return fail(kErrArg, "namsa_gemm_bf16: bad shape M=%d N=%d K=%d batch=%d split=%d", M, N, K,
                batch, split_k);
  if (split_k > 1 && (bias_mode || gelu))
    return fail(kErrArg, "namsa_gemm_bf16: split-K cannot apply bias or GELU");
  if ((bias_mode && !bias) || (gelu && !P) || bias_mode < 0 || bias_mode > 2)
    return fail(kErrArg, "namsa_gemm_bf16: missing bias or pre-activation buffer");
  GemmArgs g{A, sAb, sAi, sAk, B, sBb, sBk, sBj, C, sCb, sCi, sCj, M, N, K, batch, split_k,
             alpha, beta, bias, bias_mode, gelu, P};
  hipStream_t st = as_stream(stream);
  if (M <= 32 && N <= 32 && split_k == 1 && batch >= 64) {
    hipLaunchKernelGGL(gemm_small_kernel, dim3(static_cast<unsigned>(batch)), dim3(256), 0, st, g);
    return check_hip(hipGetLastError(), "gemm_small_kernel launch");
  }
  if (split_k > 1 && sAk == 1 && sBk == 1 && M <= 64 && N <= 64 && K <= kSplitMaxK) {
    if (M <= 32) return N <= 32 ? launch_split<1, 1>(g, st) : launch_split<1, 2>(g, st);
    return N <= 32 ? launch_split<2, 1>(g, st) : launch_split<2, 2>(g, st);
  }
  if (batch == 1 && split_k == 1 && sBj == 1 && sCj == 1 && N >= 8192 && pointwise_fits(M, N, K, sBk, sCi)) {
    const bool one = pointwise_mt(M) == 1;
    switch (pointwise_ks(K)) {
      case 1: return one ? launch_pointwise<1, 1>(g, st) : launch_pointwise<2, 1>(g, st);
      case 2: return one ? launch_pointwise<1, 2>(g, st) : launch_pointwise<2, 2>(g, st);
      default: return one ? launch_pointwise<1, 4>(g, st) : launch_pointwise<2, 4>(g, st);
    }
  }
  if (N <= 32) return launch_gemm<4, 1>(g, st);
  if (M <= 32) return launch_gemm<1, 4>(g, st);
  return launch_gemm<2, 2>(g, st);
}

int namsa_weight_grad(const float* gy, const float* x, long long n, int M, int N, float* gW, float* gb, void* stream) {
  if (!gy || !x || !gW || !gb || n <= 0 || n > kSplitMaxK || M < 1 || M > 32 || N < 1 || N > 32)
    return fail(kErrArg, "namsa_weight_grad: null argument, n=%lld or M=%d N=%d outside 1..32", n, M, N);
  const GemmArgs g{gy, 0, n, 1, x, 0, 1, n, gW, 0, N, 1, M, N, static_cast<int>(n), 1, 2, 1.0f, 0.0f, nullptr, 0, 0,
                   nullptr};
  return launch_split<1, 1, true>(g, as_stream(stream), gb);
}

}  // extern "C"
