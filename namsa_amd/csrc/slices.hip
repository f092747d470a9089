// Projected-potential slice builder for gfx950.
//
// namsa_atomic_tables: Kirkland projected potential per element on the
// reference's oversampled table grid (namsa/msa.py:137-146, :180-196), 2x2 block
// mean (namsa/utils.py:101-108), shifted to a zero minimum, stored as float32.
// K0 is evaluated from its integral form K0(x) = int_0^inf exp(-x cosh t) dt
// (Abramowitz & Stegun 9.6.24) with the trapezoid rule, whose error for this
// doubly-exponentially decaying analytic integrand falls geometrically with
// the step (step <= 0.7/sqrt(x) keeps the relative error near 1e-14).
//
// namsa_build_slices: the reference kernel (namsa/potential_kernels.cu:5-60)
// lets every pixel thread scan every site of its slice, O(N^2 S A).  Here a
// workgroup owns a tile of one slice (64 x 64 pixels, or 16 x 16 for small
// launches), streams that slice's sites through LDS, keeps (in site order, by
// ballot compaction) only those whose clipped footprint overlaps the tile, and accumulates table
// values for its pixels in float32 in site order; exp(i sigma V) with the NaN
// guard of potential_kernels.cu:48-57 is fused into the store.
#include <climits>

#include "common.hpp"
#include "namsa_hip.h"

namespace namsa {

__device__ double k0_integral(double x) {
  const double h = fmin(0.25, 0.7 / sqrt(x));
  double s = 0.5;
  for (int k = 1; k < 4096; ++k) {
    const double sh = sinh(0.5 * k * h);
    const double a = 2.0 * x * sh * sh;  // x (cosh(kh) - 1)
    if (a > 40.0) break;
    s += exp(-a);
  }
  return exp(-x) * h * s;
}

// Kirkland projected potential (msa.py:181-193), eps = 0.1 A, a0 = 0.529 A, e = 14.4 V A.
__device__ double kirkland_v(const double* p, double r) {
  const double pi = 3.141592653589793;
  const double pref = 4.0 * pi * pi * 0.529 * 14.4;
  double v = 0.0;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const double a = p[i], b = p[3 + i], c = p[6 + i], d = p[9 + i];
    v += pref * a * k0_integral(2.0 * pi * r * sqrt(b) + 0.1);
    v += pref / 2.0 * (c / d) * exp(-pi * pi * r * r / d);
  }
  return v;
}

// Subsample (dy, dx) of table pixel i; the subsample axes are
// linspace(-range/2, range/2, os*P) (the mgrid of msa.py:141-143).
__device__ double table_sample(const double* p, int i, int dy, int dx, int Py, int Px, int os, double range) {
  const int r = i / Px, c = i % Px;
  const double half = range / 2.0;
  const double s0 = range / double(os * Py - 1), s1 = range / double(os * Px - 1);
  const double gy = -half + double(os * r + dy) * s0;
  const double gx = -half + double(os * c + dx) * s1;
  return kirkland_v(p, sqrt(gy * gy + gx * gx));
}

// Mean of a pixel's os x os subsamples, sample(dy, dx).
template <class Sample>
__device__ double table_mean(int os, Sample sample) {
  double acc = 0.0;
  for (int dy = 0; dy < os; ++dy) {
    double row = 0.0;
    for (int dx = 0; dx < os; ++dx) row += sample(dy, dx);
    acc += row / os;
  }
  return acc / os;
}

constexpr int kTableThreads = 256;

// A table from its pixels alone, minimum first: one workgroup per element.
__device__ void table_by_one_workgroup(const double* p, int Py, int Px, int os, double range, float* out) {
  __shared__ double red[kTableThreads / 64];
  const int n = Py * Px;
  const auto mean = [&](int i) {
    return table_mean(os, [&](int dy, int dx) { return table_sample(p, i, dy, dx, Py, Px, os, range); });
  };
  double vmin = 1.0e300;
  for (int i = threadIdx.x; i < n; i += kTableThreads) vmin = fmin(vmin, mean(i));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) vmin = fmin(vmin, __shfl_xor(vmin, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = vmin;
  __syncthreads();
  double m = red[0];
  for (int w = 1; w < kTableThreads / 64; ++w) m = fmin(m, red[w]);
  for (int i = threadIdx.x; i < n; i += kTableThreads) out[i] = float(mean(i) - m);
}

// Tables shifted by the lowest of their corner pixels, which is the minimum
// of any table that falls off outwards; table_check_kernel redoes the others.
// Bound by the chain of FP64 instructions of one Bessel integral (about 7000
// per subsample), so every subsample has its own thread and the workgroups
// cover kTableThreads / os^2 pixels each; kCornerThreads more threads take
// the corners' subsamples meanwhile, in every workgroup.  Four elements of 64
// x 64 pixels, os = 2: 1960 us with a workgroup per element and every pixel
// evaluated twice, 42 us now, both kernels.
constexpr int kCornerThreads = 64;
constexpr int kMaxSplitOs = 4;  // 4 corners of os^2 subsamples in kCornerThreads

__global__ void __launch_bounds__(kTableThreads + kCornerThreads)
atomic_tables_kernel(const double* __restrict__ params, int Py, int Px, int os, double range,
                     float* __restrict__ tables) {
  __shared__ double val[kTableThreads + kCornerThreads];
  __shared__ double corner[4];
  const double* p = params + blockIdx.y * 12;
  const int n = Py * Px, os2 = os * os, per = kTableThreads / os2;
  const int tid = threadIdx.x;
  const bool edge = tid >= kTableThreads;
  const int slot = (edge ? tid - kTableThreads : tid) / os2, sub = (edge ? tid - kTableThreads : tid) % os2;
  const auto corner_pixel = [&](int k) { return (k >> 1) * (Py - 1) * Px + (k & 1) * (Px - 1); };
  const int i = edge ? (slot < 4 ? corner_pixel(slot) : n) : static_cast<int>(blockIdx.x) * per + slot;
  if (i < n && (edge || slot < per)) val[tid] = table_sample(p, i, sub / os, sub % os, Py, Px, os, range);
  __syncthreads();
  const int first = edge ? kTableThreads + slot * os2 : slot * os2;
  const bool lead = sub == 0 && i < n && (edge || slot < per);
  double mean = 0.0;
  if (lead) mean = table_mean(os, [&](int dy, int dx) { return val[first + dy * os + dx]; });
  if (lead && edge) corner[slot] = mean;
  __syncthreads();
  if (lead && !edge)
    tables[static_cast<long long>(blockIdx.y) * n + i] =
        float(mean - fmin(fmin(corner[0], corner[1]), fmin(corner[2], corner[3])));
}

// A table with a value below its corners' (or a NaN) is made again from its
// own minimum.
__global__ void __launch_bounds__(kTableThreads)
table_check_kernel(const double* __restrict__ params, int Py, int Px, int os, double range, int force,
                   float* __restrict__ tables) {
  const int n = Py * Px;
  float* out = tables + static_cast<long long>(blockIdx.x) * n;
  int bad = force;
  if (!force)
    for (int i = threadIdx.x; i < n; i += kTableThreads) bad |= !(out[i] >= 0.0f);
  if (__syncthreads_or(bad)) table_by_one_workgroup(params + blockIdx.x * 12, Py, Px, os, range, out);
}

// ------------------------------------------------------------------ slice builder
constexpr int kSliceThreads = 256;
constexpr int kWaves = kSliceThreads / 64;

// A site as the accumulation reads it: its table value at pixel (row, col) is
// tables[base + row * Px + col], for rows [r_lo, r_lo + rows) and columns
// [c_lo, c_lo + cols).
struct SiteBox {
  long long base;
  int r_lo, rows, c_lo, cols;
  __device__ __forceinline__ void set(long long b, int r, int nr, int c, int nc) {
    base = b;
    r_lo = r;
    rows = nr;
    c_lo = c;
    cols = nc;
  }
};

// The sites of one slice in order, K per thread at a time: scan() keeps those
// whose clipped footprint overlaps the tile, in site order, in list[0, total).
// The next chunk's sites are loaded before the current one is used.
template <int K>
struct SiteScan {
  static constexpr int kChunk = K * kSliceThreads;
  const int* __restrict__ sites;
  int nZ, Py, Px, Ny, Nx, end, next;
  int z[K], yc[K], xc[K];

  __device__ __forceinline__ void fetch() {
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const int i = next + j * kSliceThreads + static_cast<int>(threadIdx.x);
      z[j] = -1;
      if (i < end) {
        z[j] = sites[3LL * i];
        yc[j] = sites[3LL * i + 1];
        xc[j] = sites[3LL * i + 2];
      }
    }
    next += kChunk;
  }

  // Workgroup-wide: returns the number of boxes in list, which `pad` empty ones
  // follow (barriers inside).
  template <class Box>
  __device__ __forceinline__ int scan(Box* list, int pad, int (*wave_count)[kWaves], int ty0, int th, int tx0, int tw) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    bool hit[K];
    Box bx[K];
    int rank[K];
    __syncthreads();  // the previous chunk's list has been read
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const int y0 = static_cast<int>(rintf(float(yc[j]) - Py * 0.5f));
      const int y1 = static_cast<int>(rintf(float(yc[j]) + Py * 0.5f));
      const int x0 = static_cast<int>(rintf(float(xc[j]) - Px * 0.5f));
      const int x1 = static_cast<int>(rintf(float(xc[j]) + Px * 0.5f));
      const int r_lo = max(y0, 0), r_hi = min(min(y1, Ny), y0 + Py);
      const int c_lo = max(x0, 0), c_hi = min(min(x1, Nx), x0 + Px);
      bx[j].set((static_cast<long long>(z[j]) * Py - y0) * Px - x0, r_lo, r_hi - r_lo, c_lo, c_hi - c_lo);
      hit[j] = z[j] >= 0 && z[j] < nZ && r_lo < r_hi && c_lo < c_hi && r_lo < ty0 + th && r_hi > ty0 &&
               c_lo < tx0 + tw && c_hi > tx0;
      // order-preserving compaction: rank = hits in lower lanes, then in lower waves and rounds
      const unsigned long long ballot = __ballot(hit[j]);
      rank[j] = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(ballot >> 32),
                                          __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(ballot), 0));
      if (lane == 0) wave_count[j][wave] = __popcll(ballot);
    }
    __syncthreads();
    int total = 0;
#pragma unroll
    for (int j = 0; j < K; ++j)
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        if (w == wave && hit[j]) list[total + rank[j]] = bx[j];
        total += wave_count[j][w];
      }
    total = __builtin_amdgcn_readfirstlane(total);
    if (static_cast<int>(threadIdx.x) < pad) list[total + threadIdx.x] = Box{};
    if (next < end) fetch();
    __syncthreads();
    return total;
  }
};

// V or t = exp(i sigma V) of one pixel, NaN components of t replaced by 1.
template <bool POT>
__device__ __forceinline__ void put_pixel(float acc, float sigma, long long o, float2* t_out, float* v_out) {
  if constexpr (POT) {
    v_out[o] = acc;
  } else {
    float sn, cs;
    sincosf(acc * sigma, &sn, &cs);
    if (isnan(cs)) cs = 1.0f;
    if (isnan(sn)) sn = 1.0f;
    t_out[o] = make_float2(cs, sn);
  }
}

// Tile of 64 x 64 pixels, 16 rows of 64 columns per wavefront, for launches
// with enough tiles.  The sums are bound by instructions and address
// generation, so a site's box is decoded once per 16 rows, into scalar
// registers: inside the columns of the box a row is then one read (scalar row
// address, one lane offset) and one add, and all 16 reads are issued before
// the first sum.  Sums run in site order in float32, as in the narrow kernel,
// so both give the same bits.  Against 16 x 64 tiles of 4 rows per wavefront
// that took one site at a time, t of 512^2 x 150 slices (491 sites each):
// 321 -> 162 us, 1.9 TB/s written; 2048^2 x 60 (3930 sites): 2.10 -> 1.02 ms.
// POT: write the projected potential V (float) instead of t = exp(i sigma V).
constexpr int kWideRows = 16;

template <bool POT>
__global__ void __launch_bounds__(kSliceThreads)
build_slices_wide_kernel(const float* __restrict__ tables, int nZ, int Py, int Px, const int* __restrict__ sites,
                         const int* __restrict__ offsets, int Ny, int Nx, float sigma, float2* __restrict__ t_out,
                         float* __restrict__ v_out) {
  using Scan = SiteScan<1>;
  __shared__ SiteBox list[Scan::kChunk];
  __shared__ int wave_count[1][kWaves];
  const auto uni = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const int s = blockIdx.z;
  const int ty0 = blockIdx.y * kWaves * kWideRows, tx0 = blockIdx.x * 64;
  const int row0 = ty0 + uni(threadIdx.x >> 6) * kWideRows;
  const int col = tx0 + (threadIdx.x & 63);
  float acc[kWideRows];
#pragma unroll
  for (int k = 0; k < kWideRows; ++k) acc[k] = 0.0f;

  Scan scan{sites, nZ, Py, Px, Ny, Nx, offsets[s + 1], offsets[s]};
  if (scan.next < scan.end) {
    scan.fetch();
    for (int base = offsets[s]; base < scan.end; base += Scan::kChunk) {
      const int total = scan.scan(list, 0, wave_count, ty0, kWaves * kWideRows, tx0, 64);
      for (int e = 0; e < total; ++e) {
        const SiteBox& b = list[e];
        const int dr = row0 - uni(b.r_lo), rows = uni(b.rows);
        if (dr <= -kWideRows || dr >= rows) continue;
        if (static_cast<unsigned>(col - b.c_lo) >= static_cast<unsigned>(b.cols)) continue;
        const long long at = (static_cast<long long>(uni(static_cast<int>(b.base >> 32))) << 32) |
                             static_cast<unsigned>(uni(static_cast<int>(b.base)));
        const float* line = tables + at + static_cast<long long>(row0) * Px;
        float v[kWideRows];
        if (dr >= 0 && dr + kWideRows <= rows) {
#pragma unroll
          for (int k = 0; k < kWideRows; ++k) v[k] = (line + static_cast<long long>(k) * Px)[static_cast<unsigned>(col)];
        } else {  // rows outside the box add +0 to a sum that is never -0
#pragma unroll
          for (int k = 0; k < kWideRows; ++k) {
            v[k] = 0.0f;
            if (static_cast<unsigned>(dr + k) < static_cast<unsigned>(rows)) v[k] = (line + static_cast<long long>(k) * Px)[static_cast<unsigned>(col)];
          }
        }
#pragma unroll
        for (int k = 0; k < kWideRows; ++k) acc[k] += v[k];
      }
    }
  }
  const long long plane = static_cast<long long>(Ny) * Nx;
  // one copy of the sine and cosine: unrolled over the rows they take 89
  // registers (5 wavefronts per SIMD)
#pragma unroll 1
  for (int k = 0; k < kWideRows; ++k) {
    if (row0 + k < Ny && col < Nx)
      put_pixel<POT>(acc[0], sigma, s * plane + static_cast<long long>(row0 + k) * Nx + col, t_out, v_out);
#pragma unroll
    for (int j = 0; j + 1 < kWideRows; ++j) acc[j] = acc[j + 1];
  }
}

// Tile of 16 x 16 pixels, one per thread, for launches too small for the wide
// one (a single projected plane, short stacks of small grids).  There the
// chain of reads of a pixel is what takes the time: boxes and table values
// are read kNarrowBatch sites ahead of the sums, without conditions: a pixel
// outside a site's box reads past the end of the tables' buffer, which gives
// +0, and adds it to a sum that is never -0.  The list ends in empty boxes, so
// batches need no remainder.  Offsets into the tables are 32-bit and box sides
// 16-bit (the launcher checks).  One 256^2 plane of 24,573 sites: 2010 us in
// 16 x 64 tiles one site at a time, 175 us now.
// K: sites per thread and scan; 4 for one long list (a scan's barriers are
// then paid once per 1024 sites), 1 for many short ones.
constexpr int kNarrow = 16, kNarrowBatch = 8;

struct alignas(16) NarrowBox {  // one LDS read
  unsigned base;
  int r_lo, c_lo;
  unsigned size;  // columns << 16 | rows
  __device__ __forceinline__ void set(long long b, int r, int nr, int c, int nc) {
    base = static_cast<unsigned>(b);
    r_lo = r;
    c_lo = c;
    size = static_cast<unsigned>(nc) << 16 | static_cast<unsigned>(nr);
  }
};

template <bool POT, int K>
__global__ void __launch_bounds__(kSliceThreads)
build_slices_narrow_kernel(const float* __restrict__ tables, int nZ, int Py, int Px, const int* __restrict__ sites,
                           const int* __restrict__ offsets, int Ny, int Nx, float sigma, float2* __restrict__ t_out,
                           float* __restrict__ v_out) {
  using Scan = SiteScan<K>;
  __shared__ NarrowBox list[Scan::kChunk + 2 * kNarrowBatch];
  __shared__ int wave_count[K][kWaves];
  const int s = blockIdx.z;
  const int ty0 = blockIdx.y * kNarrow, tx0 = blockIdx.x * kNarrow;
  const int row = ty0 + static_cast<int>(threadIdx.x / kNarrow), col = tx0 + static_cast<int>(threadIdx.x % kNarrow);
  const unsigned pixel = static_cast<unsigned>(row) * static_cast<unsigned>(Px) + static_cast<unsigned>(col);
  const unsigned table_bytes = static_cast<unsigned>(nZ) * Py * Px * 4u;
  const auto buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(tables), 0, static_cast<int>(table_bytes),
                                                     0x00020000);
  float acc = 0.0f;
  Scan scan{sites, nZ, Py, Px, Ny, Nx, offsets[s + 1], offsets[s]};
  if (scan.next < scan.end) {
    scan.fetch();
    for (int base = offsets[s]; base < scan.end; base += Scan::kChunk) {
      const int total = scan.scan(list, 2 * kNarrowBatch, wave_count, ty0, kNarrow, tx0, kNarrow);
      float v[kNarrowBatch], w[kNarrowBatch];
      const auto read = [&](int e, float(&out)[kNarrowBatch]) {
        NarrowBox b[kNarrowBatch];
#pragma unroll
        for (int u = 0; u < kNarrowBatch; ++u) b[u] = list[e + u];
        // no short-circuit: a branch per site would wait for its LDS read
#pragma unroll
        for (int u = 0; u < kNarrowBatch; ++u) {
          const bool in = (static_cast<unsigned>(row - b[u].r_lo) < (b[u].size & 0xffffu)) &
                          (static_cast<unsigned>(col - b[u].c_lo) < (b[u].size >> 16));
          const unsigned at = (b[u].base + pixel) * 4u;
          out[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buf, in ? at : table_bytes, 0, 0));
        }
      };
      read(0, v);
      for (int e = 0; e < total; e += kNarrowBatch) {
        read(e + kNarrowBatch, w);
#pragma unroll
        for (int u = 0; u < kNarrowBatch; ++u) {
          acc += v[u];
          v[u] = w[u];
        }
      }
    }
  }
  if (row < Ny && col < Nx)
    put_pixel<POT>(acc, sigma, s * (static_cast<long long>(Ny) * Nx) + static_cast<long long>(row) * Nx + col, t_out,
                   v_out);
}

template <bool POT>
int launch_build(const float* tables, int nZ, int Py, int Px, const int* sites, const int* offsets, int S, int Ny,
                 int Nx, float sigma, float2* t_out, float* v_out, hipStream_t st) {
  const auto tiles = [](int n, int t) { return static_cast<unsigned>((n + t - 1) / t); };
  const dim3 wide(tiles(Nx, 64), tiles(Ny, kWaves * kWideRows), S);
  const dim3 narrow(tiles(Nx, kNarrow), tiles(Ny, kNarrow), S);
  // Wide from 4 workgroups per CU up (256^2 x 50 slices, 3.1 per CU: equal;
  // 128^2 x 60, 0.9 per CU: 14 us wide, 10 narrow; one 256^2 plane, 16
  // workgroups: 1014 and 95), or where narrow's offsets or grid end.
  if (static_cast<long long>(wide.x) * wide.y * S >= 4LL * device_cu_count() || narrow.y > 65535 ||
      static_cast<long long>(nZ) * Py * Px >= (1LL << 29) || Py > 65535 || Px > 65535)
    hipLaunchKernelGGL(build_slices_wide_kernel<POT>, wide, dim3(kSliceThreads), 0, st, tables, nZ, Py, Px, sites,
                       offsets, Ny, Nx, sigma, t_out, v_out);
  else if (S > 1)
    hipLaunchKernelGGL((build_slices_narrow_kernel<POT, 1>), narrow, dim3(kSliceThreads), 0, st, tables, nZ, Py, Px, sites,
                       offsets, Ny, Nx, sigma, t_out, v_out);
  else
    hipLaunchKernelGGL((build_slices_narrow_kernel<POT, 4>), narrow, dim3(kSliceThreads), 0, st, tables, nZ, Py, Px, sites,
                       offsets, Ny, Nx, sigma, t_out, v_out);
  return check_hip(hipGetLastError(), "build_slices_kernel launch");
}

// ------------------------------------------------- sampled 3D potentials
// Slice s of a potential sampled at z[0..Z) integrates samples [s d, (s+1) d)
// with the trapezoid rule on their own coordinates and negates the result
// (MSA.integrate_potential_slices, namsa/msa.py:390-407: np.split into S
// chunks, trapz over each, V = -integral; no interval spans two chunks), and
// t = exp(i sigma V) (MSAGPU.integrate_potential_slices, msa.py:568-571).
// Each term is (z1 - z0) * (p0 + p1) / 2, summed in z order without
// contraction, as numpy's trapz evaluates it.
__global__ void __launch_bounds__(256) integrate_slices_kernel(const double* pot, const double* z, int d,
                                                               long long plane, double sigma, float2* t_out,
                                                               double* v_out) {
#pragma clang fp contract(off)
  const long long p = blockIdx.x * 256LL + threadIdx.x;
  if (p >= plane) return;
  const long long s = blockIdx.y;
  const double* c = pot + s * d * plane + p;
  const double* zs = z + s * d;
  double acc = 0.0;
  double prev = c[0];
  for (int j = 1; j < d; ++j) {
    const double cur = c[j * plane];
    acc += (zs[j] - zs[j - 1]) * (prev + cur) / 2.0;
    prev = cur;
  }
  const double v = -acc;
  const long long o = s * plane + p;
  if (v_out) v_out[o] = v;
  if (t_out) {
    double sn, cs;
    sincos(sigma * v, &sn, &cs);
    t_out[o] = make_float2(static_cast<float>(cs), static_cast<float>(sn));
  }
}

// Sites of one slice per workgroup, in input order: every workgroup reads all
// depths (64 bytes a thread, from the L2 caches after the first), first to
// count the sites before its slice, then to place its own, ranked by ballot
// within a wavefront and by a running sum over wavefronts.  The reads grow with
// S times A, but a workgroup's chain of steps only with A, and no list of a
// site per step and slice has to be kept: 73,000 sites in 150 slices take
// 30 us, 2.4 million in 310 1.4 ms, where the host's sorted lookup, stable
// sort and three gathers took 7.3 and 350 ms.
constexpr int kBinThreads = 1024;
constexpr int kBinEach = 16;  // consecutive sites of a thread: 4 loads in flight a step (one took 73 us and 3.6 ms)

// truncation as the host's conversion has it: INT_MIN for what an int cannot hold
__device__ __forceinline__ int to_int(double v) {
  return v > -2147483649.0 && v < 2147483648.0 ? static_cast<int>(v) : INT_MIN;
}

__global__ void __launch_bounds__(kBinThreads)
bin_sites_kernel(const float* __restrict__ xyz, const float* __restrict__ z, const long long* __restrict__ Z, int A,
                 const long long* __restrict__ unique_Z, int nZ, const float* __restrict__ bounds, int S, double py,
                 double px, int* __restrict__ sites, int* __restrict__ offsets) {
  __shared__ int part[2][kBinThreads / 64];
  const int s = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float first = bounds[0], lo = bounds[s], hi = bounds[s + 1];
  const int steps = (A + kBinEach * kBinThreads - 1) / (kBinEach * kBinThreads);
  auto load = [&](int step, float (&v)[kBinEach]) {  // NaN past the end: in no slice
    const int i = kBinEach * (step * kBinThreads + static_cast<int>(threadIdx.x));
    if (i + kBinEach <= A) {
#pragma unroll
      for (int k = 0; k < kBinEach / 4; ++k) {
        const float4 f = *reinterpret_cast<const float4*>(z + i + 4 * k);
        v[4 * k] = f.x;
        v[4 * k + 1] = f.y;
        v[4 * k + 2] = f.z;
        v[4 * k + 3] = f.w;
      }
    } else {
#pragma unroll
      for (int e = 0; e < kBinEach; ++e) v[e] = i + e < A ? z[i + e] : __builtin_nanf("");
    }
  };
  int before = 0;
  for (int step = 0; step < steps; ++step) {
    float v[kBinEach];
    load(step, v);
#pragma unroll
    for (int e = 0; e < kBinEach; ++e) before += (v[e] >= first) & (v[e] < lo);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
  if (lane == 0) part[0][wave] = before;
  __syncthreads();
  int base = 0;
  for (int w = 0; w < kBinThreads / 64; ++w) base += part[0][w];
  if (threadIdx.x == 0) offsets[s] = base;
  for (int step = 0; step < steps; ++step) {
    float v[kBinEach];
    load(step, v);
    int mine = 0, rank = 0, all = 0;
    const unsigned long long below = (1ull << lane) - 1;
#pragma unroll
    for (int e = 0; e < kBinEach; ++e) {
      const bool in = (v[e] >= lo) & (v[e] < hi);
      const unsigned long long m = __ballot(in);
      mine |= in << e;
      rank += __popcll(m & below);
      all += __popcll(m);
    }
    int* sums = part[(step & 1) ^ 1];  // the other half may still be read
    if (lane == 0) sums[wave] = all;
    __syncthreads();
    int total = 0;
    for (int w = 0; w < kBinThreads / 64; ++w) {
      if (w == wave) rank += total;
      total += sums[w];
    }
    for (; mine; mine &= mine - 1) {
      const long long i = static_cast<long long>(kBinEach) * (step * kBinThreads + threadIdx.x) + __ffs(mine) - 1;
      int a = 0, b = nZ;  // the first element not below this site's
      const long long own = Z[i];
      while (a < b) {
        const int mid = (a + b) >> 1;
        if (unique_Z[mid] < own) a = mid + 1;
        else b = mid;
      }
      int* out = sites + 3ll * (base + rank++);
      out[0] = a;
      out[1] = to_int(static_cast<double>(xyz[3 * i + 1]) / py);
      out[2] = to_int(static_cast<double>(xyz[3 * i]) / px);
    }
    base += total;
  }
  if (s == S - 1 && threadIdx.x == 0) offsets[S] = base;
}

}  // namespace namsa

using namespace namsa;

extern "C" {

int namsa_integrate_slices(const double* pot, const double* z, int S, int d, int Ny, int Nx, double sigma,
                           void* t_out, double* v_out, void* stream) {
  if (!pot || !z || (!t_out && !v_out) || S < 0 || d < 1 || Ny <= 0 || Nx <= 0)
    return fail(kErrArg, "namsa_integrate_slices: bad arguments (S=%d d=%d Ny=%d Nx=%d)", S, d, Ny, Nx);
  if (S == 0) return kOk;
  if (S > 65535) return fail(kErrArg, "namsa_integrate_slices: S=%d exceeds the grid y limit", S);
  const long long plane = static_cast<long long>(Ny) * Nx;
  const long long blocks = (plane + 255) / 256;
  if (blocks > 0x7fffffffLL) return fail(kErrArg, "namsa_integrate_slices: plane too large");
  hipLaunchKernelGGL(integrate_slices_kernel, dim3(static_cast<unsigned>(blocks), S), dim3(256), 0,
                     as_stream(stream), pot, z, d, plane, sigma, static_cast<float2*>(t_out), v_out);
  return check_hip(hipGetLastError(), "integrate_slices_kernel launch");
}

}  // extern "C"

extern "C" {

int namsa_atomic_tables(const double* params, int nZ, int Py, int Px, double range, int oversample,
                        float* tables, void* stream) {
  if (!params || !tables || nZ <= 0 || Py <= 0 || Px <= 0 || !(range > 0) || oversample < 1 ||
      oversample * static_cast<long long>(Py) < 2 || oversample * static_cast<long long>(Px) < 2)
    return fail(kErrArg, "namsa_atomic_tables: bad arguments (nZ=%d Py=%d Px=%d os=%d)", nZ, Py,
                Px, oversample);
  hipStream_t st = as_stream(stream);
  // one thread per subsample while the corners' fit their wavefront (os <= 4)
  const bool split = oversample <= kMaxSplitOs && nZ <= 65535;
  if (split) {
    const int per = kTableThreads / (oversample * oversample);
    const long long n = static_cast<long long>(Py) * Px;
    hipLaunchKernelGGL(atomic_tables_kernel, dim3(static_cast<unsigned>((n + per - 1) / per), nZ),
                       dim3(kTableThreads + kCornerThreads), 0, st, params, Py, Px, oversample, range, tables);
  }
  hipLaunchKernelGGL(table_check_kernel, dim3(nZ), dim3(kTableThreads), 0, st, params, Py, Px, oversample, range,
                     split ? 0 : 1, tables);
  return check_hip(hipGetLastError(), "atomic_tables_kernel launch");
}

int namsa_bin_sites(const float* xyz, const float* z, const long long* Z, int A, const long long* unique_Z, int nZ,
                    const float* bounds, int S, double py, double px, int* sites, int* offsets, void* stream) {
  if (!xyz || !z || !Z || !unique_Z || !bounds || !sites || !offsets || A <= 0 || A > (1 << 30) || nZ <= 0 || S <= 0)
    return fail(kErrArg, "namsa_bin_sites: null argument or A=%d nZ=%d S=%d out of range", A, nZ, S);
  hipLaunchKernelGGL(bin_sites_kernel, dim3(S), dim3(kBinThreads), 0, as_stream(stream), xyz, z, Z, A, unique_Z, nZ,
                     bounds, S, py, px, sites, offsets);
  return check_hip(hipGetLastError(), "bin_sites_kernel launch");
}

int namsa_build_slices(const float* tables, int nZ, int Py, int Px, const int* sites,
                       const int* slice_offsets, int S, int Ny, int Nx, float sigma, void* t_out,
                       void* stream) {
  if (!tables || !slice_offsets || !t_out || nZ <= 0 || Py <= 0 || Px <= 0 || S < 0 || Ny <= 0 ||
      Nx <= 0)
    return fail(kErrArg, "namsa_build_slices: bad arguments");
  if (S == 0) return kOk;
  if (S > 65535) return fail(kErrArg, "namsa_build_slices: S=%d exceeds the grid z limit", S);
  return launch_build<false>(tables, nZ, Py, Px, sites, slice_offsets, S, Ny, Nx, sigma, static_cast<float2*>(t_out),
                             nullptr, as_stream(stream));
}

int namsa_build_potential(const float* tables, int nZ, int Py, int Px, const int* sites,
                          const int* slice_offsets, int S, int Ny, int Nx, float* v_out, void* stream) {
  if (!tables || !slice_offsets || !v_out || nZ <= 0 || Py <= 0 || Px <= 0 || S < 0 || Ny <= 0 ||
      Nx <= 0)
    return fail(kErrArg, "namsa_build_potential: bad arguments");
  if (S == 0) return kOk;
  if (S > 65535) return fail(kErrArg, "namsa_build_potential: S=%d exceeds the grid z limit", S);
  return launch_build<true>(tables, nZ, Py, Px, sites, slice_offsets, S, Ny, Nx, 0.0f, nullptr, v_out,
                            as_stream(stream));
}

}  // extern "C"
