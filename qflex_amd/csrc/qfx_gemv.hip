// Complex64 matrix-vector products and dot products of the contraction path
// (gfx950): the closings cblas_cgemv / cblas_cdotu_sub of the reference
// (src/tensor.cpp:982-1042).
//
// All of them read the matrix once and are bound by HBM (8 flop per 8
// bytes), so the kernels only have to keep enough loads in flight on all
// 256 CUs, for every aspect ratio: tall and narrow, short and wide.
// Reductions run in a fixed order (no atomics): results are deterministic.
// Measured against one wave per row (N) and against blocks that walked all
// columns of 4 to 16 rows, 64 at a time (T), in recorded sequences over inputs
// that no cache holds (a 1 GiB copy runs at 5.2 TB/s):
//   T 4096 x 4096 (134 MB)   145 -> 28.9 us     N 4096 x 4096    38.2 -> 26.1 us
//   T 227 x 37463 (68 MB)    1220 -> 21.0 us    N 81 x 12430     89 -> 7.0 us
//   T 16384 x 256 (34 MB)    78 -> 13.3 us      N 1000000 x 4    130 -> 10.1 us
//   T 1000000 x 4 (32 MB)    172 -> 14.3 us     N 20000 x 2048   73.8 -> 63.0 us
// The figures below are of the same kind where they name no other.
#include <algorithm>

#include "qfx_internal.h"

namespace {

__device__ __forceinline__ float2 cfma(float2 a, float2 b, float2 c) {
  c.x = fmaf(a.x, b.x, c.x);
  c.x = fmaf(-a.y, b.y, c.x);
  c.y = fmaf(a.x, b.y, c.y);
  c.y = fmaf(a.y, b.x, c.y);
  return c;
}

__device__ __forceinline__ float2 cadd(float2 a, float2 b) {
  return make_float2(a.x + b.x, a.y + b.y);
}

// V complex values from p: one 16-byte load (V = 2) or one 8-byte load.
template <int V>
struct Vec {
  float2 e[V];
};
template <int V>
__device__ __forceinline__ Vec<V> load_vec(const float2* p) {
  Vec<V> r;
  if constexpr (V == 2) {
    const float4 f = *reinterpret_cast<const float4*>(p);
    r.e[0] = make_float2(f.x, f.y);
    r.e[1] = make_float2(f.z, f.w);
  } else {
    r.e[0] = *p;
  }
  return r;
}

// y[m] = A[m x k] . x[k], many rows: groups of L = 2^llog lanes (L <= 64),
// each R rows at a time, so that a load of x serves R rows and every lane
// has R loads of A in flight.  WAVE: L is 64 and the loads' strides are
// immediates (worked out from llog, at the start of each block, they cost 0.4
// us: 1753 x 453 3.8 -> 3.5, 1535 x 829 4.0 -> 3.7).
template <int V, int R, bool WAVE>
__global__ __launch_bounds__(256) void gemv_n_rows_kernel(const float2* __restrict__ A,
                                                          const float2* __restrict__ x,
                                                          float2* __restrict__ y, uint64_t M,
                                                          uint64_t K, int llog) {
  if (WAVE) llog = 6;
  const int L = 1 << llog;
  const int lane = threadIdx.x & (L - 1);
  const uint64_t groups = uint64_t(256 >> llog) * gridDim.x;
  const uint64_t units = K / V;  // loads per row (V divides K)
  for (uint64_t g = (uint64_t(blockIdx.x) << (8 - llog)) + (threadIdx.x >> llog); g * R < M;
       g += groups) {
    const uint64_t r0 = g * R;
    const float2* a[R];
    float2 acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      a[r] = A + (r0 + r < M ? r0 + r : M - 1) * K;  // past the end: the last row again
      acc[r] = make_float2(0.f, 0.f);
    }
    // U loads of x and U * R of A in flight per lane
    constexpr int U = R == 1 ? 4 : 2;
    uint64_t u = lane;
    for (; u + (U - 1) * L < units; u += U * L) {
      Vec<V> xv[U], av[U][R];
#pragma unroll
      for (int j = 0; j < U; ++j) {
        xv[j] = load_vec<V>(x + (u + j * L) * V);
#pragma unroll
        for (int r = 0; r < R; ++r) av[j][r] = load_vec<V>(a[r] + (u + j * L) * V);
      }
#pragma unroll
      for (int j = 0; j < U; ++j)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int v = 0; v < V; ++v) acc[r] = cfma(av[j][r].e[v], xv[j].e[v], acc[r]);
    }
    for (; u < units; u += L) {
      const Vec<V> xv = load_vec<V>(x + u * V);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const Vec<V> av = load_vec<V>(a[r] + u * V);
#pragma unroll
        for (int v = 0; v < V; ++v) acc[r] = cfma(av.e[v], xv.e[v], acc[r]);
      }
    }
    for (int off = L >> 1; off > 0; off >>= 1)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        acc[r].x += __shfl_xor(acc[r].x, off);
        acc[r].y += __shfl_xor(acc[r].y, off);
      }
    if (lane == 0)
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (r0 + r < M) y[r0 + r] = acc[r];
  }
}

// y = A . x with few rows: one block per row, four loads in flight per
// thread (the row is split over up to 16 waves instead of one).
template <int V>
__global__ __launch_bounds__(1024) void gemv_n_block_kernel(const float2* __restrict__ A,
                                                            const float2* __restrict__ x,
                                                            float2* __restrict__ y, uint64_t M,
                                                            uint64_t K) {
  __shared__ float2 red[16];
  const uint64_t units = K / V, T = blockDim.x;
  for (uint64_t row = blockIdx.x; row < M; row += gridDim.x) {
    const float2* a = A + row * K;
    float2 acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = make_float2(0.f, 0.f);
    uint64_t u = threadIdx.x;
    for (; u + 3 * T < units; u += 4 * T) {
      Vec<V> av[4], xv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        av[j] = load_vec<V>(a + (u + j * T) * V);
        xv[j] = load_vec<V>(x + (u + j * T) * V);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int v = 0; v < V; ++v) acc[j] = cfma(av[j].e[v], xv[j].e[v], acc[j]);
    }
    for (; u < units; u += T) {
      const Vec<V> av = load_vec<V>(a + u * V), xv = load_vec<V>(x + u * V);
#pragma unroll
      for (int v = 0; v < V; ++v) acc[0] = cfma(av.e[v], xv.e[v], acc[0]);
    }
    float2 t = cadd(cadd(acc[0], acc[1]), cadd(acc[2], acc[3]));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      t.x += __shfl_xor(t.x, off);
      t.y += __shfl_xor(t.y, off);
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (unsigned w = 1; w < blockDim.x / 64; ++w) t = cadd(t, red[w]);
      y[row] = t;
    }
    __syncthreads();
  }
}

// Sums over the groups of a block of V values per thread, in a fixed tree:
// thread t belongs to group t / CL (CL threads each, G = T / CL groups of the
// block's T; the threads past G * CL take no part).  The sums are in group 0.
// Eight groups become one per step: halving them, for one value after the
// other, took ten barriers of 16 waves (100 x 100 5.5 us, now 4.2; 256 x 64 6.1
// and 4.8).
template <int T, int V>
__device__ __forceinline__ void group_sums(float2 (&v)[V], float2* red, int CL, int G) {
  const int t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < V; ++i) red[i * T + t] = v[i];
  __syncthreads();
  while (G > 1) {
    const int left = (G + 7) / 8;  // group g < left takes over g + left, g + 2 left, ...
    if (t < left * CL) {
      float2 x[V][8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int i = 0; i < V; ++i)
          x[i][j] = t + j * left * CL < G * CL ? red[i * T + t + j * left * CL] : make_float2(0.f, 0.f);
#pragma unroll
      for (int i = 0; i < V; ++i)
        v[i] = cadd(cadd(cadd(x[i][0], x[i][1]), cadd(x[i][2], x[i][3])),
                    cadd(cadd(x[i][4], x[i][5]), cadd(x[i][6], x[i][7])));
    }
    G = left;
    if (G == 1) break;
    __syncthreads();
    if (t < left * CL)
#pragma unroll
      for (int i = 0; i < V; ++i) red[i * T + t] = v[i];
    __syncthreads();
  }
}

// y[c] = sum_r x[r] A[r][c] (A is m x k, row-major).  Block (x, y, z): column
// tile t = x + z gridDim.x, the columns V * (CL t + lane), of the rows
// [rows_per * y, ...); its T threads
// are G = T / CL row groups of CL column lanes, four rows in flight each.
// A narrow matrix takes all its columns as the lanes (CL = k / V), so that
// the block reads whole rows one after the other.  One split over the rows
// writes y itself, several write part[split][c].
template <int V, int T>
__global__ __launch_bounds__(T) void gemv_t_kernel(const float2* __restrict__ A,
                                                     const float2* __restrict__ x,
                                                     float2* __restrict__ out, uint64_t M,
                                                     uint64_t K, uint64_t rows_per, int CL) {
  __shared__ float2 red[V * T];
  const int G = T / CL;
  const int rg = threadIdx.x / CL, cl = threadIdx.x - rg * CL;
  const uint64_t c = ((uint64_t(blockIdx.z) * gridDim.x + blockIdx.x) * CL + cl) * V;
  const uint64_t r0 = blockIdx.y * rows_per;
  const uint64_t r1 = r0 + rows_per < M ? r0 + rows_per : M;
  const bool in = rg < G && c < K;  // (V divides K)
  float2 acc[4][V];  // one chain per row in flight
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int v = 0; v < V; ++v) acc[j][v] = make_float2(0.f, 0.f);
  if (in) {
    uint64_t r = r0 + rg;
    for (; r + 3 * G < r1; r += 4 * G) {
      Vec<V> a[4];
      float2 xr[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        a[j] = load_vec<V>(A + (r + j * G) * K + c);
        xr[j] = x[r + j * G];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int v = 0; v < V; ++v) acc[j][v] = cfma(xr[j], a[j].e[v], acc[j][v]);
    }
    for (; r < r1; r += G) {
      const Vec<V> a = load_vec<V>(A + r * K + c);
#pragma unroll
      for (int v = 0; v < V; ++v) acc[0][v] = cfma(x[r], a.e[v], acc[0][v]);
    }
  }
  float2 sum[V];
#pragma unroll
  for (int v = 0; v < V; ++v)
    sum[v] = cadd(cadd(acc[0][v], acc[1][v]), cadd(acc[2][v], acc[3][v]));
  group_sums<T, V>(sum, red, CL, G);
  if (rg == 0 && in)
#pragma unroll
    for (int v = 0; v < V; ++v) out[blockIdx.y * K + c + v] = sum[v];
}

// The same for 256 threads and CL a power of two up to 64: in registers
// within a wave, then over the four waves.  (With a barrier per halving a dot
// product of 100 values, two launches, took 4.5 us, 3.8 so.)
__device__ __forceinline__ float2 lane_group_sum(float2 v, float2 (*red)[64], int CL) {
  const int lane = threadIdx.x & 63;
  for (int off = 32; off >= CL; off >>= 1) {
    v.x += __shfl_xor(v.x, off);
    v.y += __shfl_xor(v.y, off);
  }
  if (lane < CL) red[threadIdx.x >> 6][lane] = v;
  __syncthreads();
  if (threadIdx.x < CL) v = cadd(cadd(red[0][lane], red[1][lane]), cadd(red[2][lane], red[3][lane]));
  return v;
}

// y[c] = sum_s part[s][c]: CL columns per block, the splits shared by the
// 256 / CL groups (CL a power of two).
__global__ __launch_bounds__(256) void gemv_sum_kernel(const float2* __restrict__ part,
                                                       float2* __restrict__ y, uint64_t nsplit,
                                                       uint64_t K, int CL) {
  __shared__ float2 red[4][64];
  const int G = 256 / CL;
  const int g = threadIdx.x / CL, cl = threadIdx.x - g * CL;
  const uint64_t c = uint64_t(blockIdx.x) * CL + cl;
  float2 acc = make_float2(0.f, 0.f);
  if (c < K)
    for (uint64_t s = g; s < nsplit; s += G) acc = cadd(acc, part[s * K + c]);
  acc = lane_group_sum(acc, red, CL);
  if (g == 0 && c < K) y[c] = acc;
}

// Block partial sums of x[i]*y[i] in a fixed per-lane order, then a tree.
__global__ __launch_bounds__(256) void dot_partial_kernel(const float2* __restrict__ x,
                                                          const float2* __restrict__ y,
                                                          float2* __restrict__ part,
                                                          uint64_t n) {
  __shared__ float2 red[4][64];
  float2 acc = make_float2(0.f, 0.f);
#pragma unroll 4
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += uint64_t(gridDim.x) * blockDim.x)
    acc = cfma(x[i], y[i], acc);
  acc = lane_group_sum(acc, red, 1);
  if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// Smallest b with 2^b >= v (v >= 1), at most cap.
int log2_ceil(uint64_t v, int cap) {
  int b = 0;
  while (b < cap && (uint64_t(1) << b) < v) ++b;
  return b;
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

void launch_sum(hipStream_t s, const float2* part, float2* y, uint64_t nsplit, uint64_t k) {
  // Up to 16 columns per block (64 once k alone fills the chip), fewer where
  // a thread would otherwise add up more than 8 partials one after the other.
  int clog = k >= 65536 ? 6 : log2_ceil(k, 4);
  while (clog > 1 && (nsplit << clog) > 8 * 256) --clog;
  const int CL = 1 << clog;
  gemv_sum_kernel<<<unsigned((k + CL - 1) / CL), 256, 0, s>>>(part, y, nsplit, k, CL);
}

template <int V>
void launch_n(hipStream_t s, uint64_t m, uint64_t k, const float2* A, const float2* x, float2* y) {
  const uint64_t units = k / V;
  // Few rows: a block per row, if the row has enough loads to fill it (four
  // per thread; below 512 rows one).  Otherwise groups of lanes.
  if ((m < 4096 && units >= 1024) || (m < 512 && units >= 256)) {
    const unsigned threads = units >= 4096 && m <= 1024 ? 1024 : 256;
    gemv_n_block_kernel<V><<<unsigned(m), threads, 0, s>>>(A, x, y, m, k);
    return;
  }
  // Many rows: the largest group that a row keeps four fifths busy (33
  // columns: 8 lanes, 5 loads each).  Up to 3072 rows (three waves per SIMD,
  // were each row a wave's) idle lanes cost nothing and rounds of loads do: a
  // lane per load, up to a wave (1000 x 100: 2.9 us with 8 lanes, 2.5 so; 8000
  // x 100 3.0 and 3.3).
  int llog = 6;
  if (m <= 3072)
    llog = log2_ceil(units, 6);
  else
    while (llog > 0 && 5 * units < 4 * ((((units - 1) >> llog) + 1) << llog)) --llog;
  // rows per lane group: four share each load of x where there are enough rows
  const uint64_t per_block = 256 >> llog;
  const bool four = m >= 4 * per_block * 512;
  const uint64_t groups = four ? (m + 3) / 4 : m;
  const unsigned blocks =
      unsigned(std::min<uint64_t>((groups + per_block - 1) / per_block, 65535));
  // (four rows gain nothing from fixed strides: 20000 x 2048 61.6 and 66.6 us)
  (four        ? gemv_n_rows_kernel<V, 4, false>
   : llog == 6 ? gemv_n_rows_kernel<V, 1, true>
               : gemv_n_rows_kernel<V, 1, false>)<<<blocks, 256, 0, s>>>(A, x, y, m, k, llog);
}

}  // namespace

int qfx_launch_gemv_n(qfx_context* ctx, uint64_t m, uint64_t k, const float2* A, const float2* x,
                      float2* y) {
  if (k % 2 == 0 && aligned16(A) && aligned16(x))
    launch_n<2>(ctx->stream, m, k, A, x, y);
  else
    launch_n<1>(ctx->stream, m, k, A, x, y);
  QFX_HIP(hipGetLastError());
  return QFX_OK;
}

int qfx_launch_gemv_t(qfx_context* ctx, uint64_t m, uint64_t k, const float2* A, const float2* x,
                      float2* y) {
  const int V = k % 2 == 0 && aligned16(A) ? 2 : 1;
  // column lanes: the whole row up to 128 loads (300000 x 33: 27 to 29 us,
  // 36.6 with 64 lanes, 31 of them idle), else tiles of 64
  const uint64_t units = (k + V - 1) / V;
  const int CL = units <= 128 ? int(units) : 64;
  const uint64_t tile = uint64_t(V) * CL, tiles = (k + tile - 1) / tile;
  // Row splits: about 2048 blocks in all (8 per CU), each row group of a
  // block with at least 16 rows (four rounds of the four in flight; with 8,
  // 16384 x 256 takes the same 13.3 us and twice the scratch), at most 1024
  // splits of at least 16 rows (the scratch is then never more than 1024 x k
  // values).
  const uint64_t G = 256 / CL;
  const uint64_t want = (2048 + tiles - 1) / tiles;
  uint64_t nsplit = std::min<uint64_t>({want, uint64_t(1024), (m + 16 * G - 1) / (16 * G),
                                        (m + 15) / 16, uint64_t(65535)});
  nsplit = std::max<uint64_t>(nsplit, 1);
  const uint64_t rows_per = (m + nsplit - 1) / nsplit;
  nsplit = (m + rows_per - 1) / rows_per;
  // 2^23 tiles along x (2^31 threads of the 2^32 that a grid dimension can
  // hold), from 2^29 columns on several of those along z
  const uint64_t tiles_x = std::min(tiles, uint64_t(1) << 23);
  if (tiles > tiles_x * 65535) return qfx_set_error(QFX_ERR_UNSUPPORTED, "gemv: too many columns");
  // Blocks of 1024 threads that take all rows of fewer columns save the
  // partials and their launch.  Taken with at most 32 rows per thread in at
  // least 128 blocks (4096 x 4096: 33.0 -> 28.9 us, 4.6 TB/s; 1024 x 65536 100 ->
  // 90; 227 x 37463 22.2 -> 21.0; with 63 blocks 1000 x 4000 took 17.2 instead
  // of 11.1) and otherwise with at most 8 (100 x 100: 5.0 -> 4.2; 1000 x 4000
  // 11.1 -> 10.4; with 23, 1409 x 17 took 8.5 instead of 5.8).  8-byte loads of
  // many rows want the widest blocks (2047 x 8191: 39.7 with 16 columns, 35.7
  // split).
  for (uint64_t cl = units <= 64 ? units : 64; nsplit > 1 && cl > 0; cl /= 2) {
    const uint64_t cols = (units + cl - 1) / cl, rows = (m * cl + 1023) / 1024;
    const bool few = rows <= 8 && (cl == units || cl * V >= 16);
    const bool many = rows <= 32 && cols >= 128 && cl >= (V == 2 ? 8 : 64);
    if (m > 65536 || (!few && !many)) continue;
    if (V == 2)
      gemv_t_kernel<2, 1024><<<unsigned(cols), 1024, 0, ctx->stream>>>(A, x, y, m, k, m, int(cl));
    else
      gemv_t_kernel<1, 1024><<<unsigned(cols), 1024, 0, ctx->stream>>>(A, x, y, m, k, m, int(cl));
    QFX_HIP(hipGetLastError());
    return QFX_OK;
  }
  float2* out = y;
  if (nsplit > 1) {
    void* ws = nullptr;
    const int st = qfx_workspace(ctx, nsplit * k * sizeof(float2), &ws);
    if (st != QFX_OK) return st;
    out = static_cast<float2*>(ws);
  }
  const dim3 g{unsigned(tiles_x), unsigned(nsplit), unsigned((tiles + tiles_x - 1) / tiles_x)};
  if (V == 2)
    gemv_t_kernel<2, 256><<<g, 256, 0, ctx->stream>>>(A, x, out, m, k, rows_per, CL);
  else
    gemv_t_kernel<1, 256><<<g, 256, 0, ctx->stream>>>(A, x, out, m, k, rows_per, CL);
  if (nsplit > 1) launch_sum(ctx->stream, out, y, nsplit, k);
  QFX_HIP(hipGetLastError());
  return QFX_OK;
}

extern "C" int qfx_cgemv_c64(qfx_context* ctx, int trans, uint64_t m, uint64_t k,
                             const qfx_c64* A, const qfx_c64* x, qfx_c64* y) {
  QFX_CHECK_CTX(ctx);
  uint64_t ny = trans ? k : m;
  if (ny == 0) return QFX_OK;
  if (!A || !x || !y) return qfx_set_error(QFX_ERR_INVALID, "qfx_cgemv_c64: null pointer");
  if ((trans ? m : k) == 0) return qfx_zero(ctx, y, ny * sizeof(qfx_c64));
  QFX_EXTENT(ctx, A, 8.0 * double(m) * double(k), "qfx_cgemv_c64: A");
  QFX_EXTENT(ctx, x, 8.0 * double(trans ? m : k), "qfx_cgemv_c64: x");
  QFX_EXTENT(ctx, y, 8.0 * double(ny), "qfx_cgemv_c64: y");
  QfxLaunchScope scope(ctx, QFX_K_GEMV, 8.0 * (m * k + m + k), 8.0 * m * k);
  const float2* A2 = reinterpret_cast<const float2*>(A);
  const float2* x2 = reinterpret_cast<const float2*>(x);
  float2* y2 = reinterpret_cast<float2*>(y);
  return trans ? qfx_launch_gemv_t(ctx, m, k, A2, x2, y2) : qfx_launch_gemv_n(ctx, m, k, A2, x2, y2);
}

extern "C" int qfx_cdotu_c64(qfx_context* ctx, uint64_t n, const qfx_c64* x, const qfx_c64* y,
                             qfx_c64* out) {
  QFX_CHECK_CTX(ctx);
  if (!out) return qfx_set_error(QFX_ERR_INVALID, "qfx_cdotu_c64: null output");
  if (n == 0) return qfx_zero(ctx, out, sizeof(qfx_c64));
  if (!x || !y) return qfx_set_error(QFX_ERR_INVALID, "qfx_cdotu_c64: null pointer");
  QFX_EXTENT(ctx, x, 8.0 * double(n), "qfx_cdotu_c64: x");
  QFX_EXTENT(ctx, y, 8.0 * double(n), "qfx_cdotu_c64: y");
  QFX_EXTENT(ctx, out, 8.0, "qfx_cdotu_c64: out");
  QfxLaunchScope scope(ctx, QFX_K_DOT, 16.0 * n, 8.0 * n);
  // up to 1024 values one block without partial sums (1000: 4.3 -> 2.7 us)
  const uint64_t blocks = n <= 1024 ? 1 : std::min<uint64_t>((n + 255) / 256, 1024);
  float2* part = reinterpret_cast<float2*>(out);
  if (blocks > 1) {
    void* ws = nullptr;
    const int st = qfx_workspace(ctx, blocks * sizeof(float2), &ws);
    if (st != QFX_OK) return st;
    part = static_cast<float2*>(ws);
  }
  dot_partial_kernel<<<unsigned(blocks), 256, 0, ctx->stream>>>(
      reinterpret_cast<const float2*>(x), reinterpret_cast<const float2*>(y), part, n);
  if (blocks > 1) launch_sum(ctx->stream, part, reinterpret_cast<float2*>(out), blocks, 1);
  QFX_HIP(hipGetLastError());
  return QFX_OK;
}
