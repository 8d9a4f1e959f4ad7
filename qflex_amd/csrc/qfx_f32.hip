// FP32 complex GEMM on the matrix cores (gfx950): every FP32 product with
// k > 16, and the products of the split precisions that are too small for
// their tiles.
//
// v_mfma_f32_32x32x2_f32 multiplies 32 real rows by 32 real columns, two k at
// a time, at 64 flops per cycle and SIMD (157 TFLOP/s on the chip at 2.4 GHz).
// A complex A[m x k] is its real [m x 2k]; B goes into LDS as the 2 x 2 blocks
// [[Br, Bi], [-Bi, Br]], one row per real output column with k along it, so
// that 16 bytes of LDS feed four MFMAs of a lane and nothing is selected or
// negated between them.  Lanes 0-31 hold the first two k of a group of four,
// lanes 32-63 the other two.
//
// What bounds it: the MFMAs for large products (2048^3 ran at 119 TFLOP/s on
// a card at 2.1 GHz, where they could do 139), the chain of stages (1 us each, load
// to use) for small ones, which is why those take smaller tiles, deeper stages
// and splits of k.  Measured against one 128 x 64 tile with selects between
// the MFMAs, vector-ALU partial sums over 16 k each for up to 2^16 outputs,
// and one thread per output for n < 16 or m < 64 (us, in recorded sequences
// over inputs that no cache holds):
//   2048^3                    593 -> 556     300 x 300 x 300       53.2 -> 8.8
//   65536 x 256 x 256         312 -> 300     256 x 256 x 4096      65.5 -> 30.2
//   6145 x 515 x 333          106 ->  99     16 x 4096 x 4096       124 -> 55.6
//   3719 x 642 x 516          157 -> 119     65536 x 8 x 1024       541 -> 125
//   13066 x 36 x 948          163 ->  75     3000 x 2 x 900         253 -> 14.8
//   57 x 104 x 3384          1050 -> 11.3    86 x 169 x 470        80.8 -> 7.5
// Errors against complex128 are the same (128 x 64 tile) or lower (the other
// tiles add their sums up once per stage): 57 x 104 x 3384 1e-6 -> 1e-7.
#include <algorithm>
#include <type_traits>
#include <vector>

#include "qfx_internal.h"

namespace {

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// A block of four waves, WM x WN x WK of them along m, n and k; each wave owns
// I x J MFMA tiles of 32 rows x 16 complex columns, KB complex k per stage.
template <int WM_, int WN_, int WK_, int I_, int J_, int KB_>
struct Tile {
  static constexpr int WM = WM_, WN = WN_, WK = WK_, I = I_, J = J_, KB = KB_;
  static constexpr int TM = 32 * I * WM, TN = 16 * J * WN;
  static constexpr int SR = KB + 2;  // complex per LDS row: 16-byte reads of 8 rows hit all banks
  static constexpr int NA = TM * KB / 256, NB = TN * KB / 256;  // loads per thread and stage
  static constexpr int kLds = 2 * (TM + 2 * TN) * SR;           // complex
  static_assert(WM * WN * WK == 4 && (WK == 1 || I * J == 1), "four waves");
};
typedef Tile<2, 2, 1, 2, 2, 16> TileA;  // 128 x 64
typedef Tile<2, 2, 1, 1, 1, 32> TileF;  // 64 x 32
typedef Tile<4, 1, 1, 1, 1, 16> TileD;  // 128 x 16
typedef Tile<1, 4, 1, 1, 1, 16> TileE;  // 32 x 64
typedef Tile<1, 1, 4, 1, 1, 64> TileC;  // 32 x 16, the waves split each stage's k

struct Maps {
  qfx_index_map ar, ac, br, bc;
  uint64_t a_span, b_span;  // elements from the operand's start to its last one
};

// map_offset with the digits unrolled: they stay in scalar registers.
__device__ __forceinline__ unsigned map_bytes(const qfx_index_map& d, uint64_t idx) {
  unsigned off = 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    if (j >= d.ndigits) break;
    off += unsigned(idx & ((uint64_t(1) << d.bits[j]) - 1)) << d.shift[j];
    idx >>= d.bits[j];
  }
  return off * 8u;
}

// How a block reads its operands: row-major through buffer resources (32-bit
// offsets from the block's first row or column and the stage's first k, zeros
// past the end), digit maps through them (32-bit offsets from the operand's
// start, up to kMapStages stages), or either through 64-bit addresses where
// the offsets don't reach.
enum { kRowMajor, kMapped, kWide };
constexpr int kMapStages = 256;

// C[m0.., n0..] over the stages [s0, s1) of KB k each.  a_mfast: consecutive
// threads take consecutive rows of A, else consecutive k; b_kfast likewise.
template <class T, int LOAD>
__device__ __forceinline__ void f32_tile(const float2* __restrict__ A,
                                         const float2* __restrict__ B, float2* __restrict__ C,
                                         int M, int N, int64_t K, const Maps& maps, bool mapped,
                                         bool a_mfast, bool b_kfast, int m0, int n0, int s0,
                                         int s1, float2* lds) {
  constexpr int KB = T::KB, SR = T::SR, NA = T::NA, NB = T::NB, I = T::I, J = T::J;
  constexpr int kStage = (T::TM + 2 * T::TN) * SR, kB0 = T::TM * SR;  // LDS of a stage, of its B
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wk = wave % T::WK, wn = (wave / T::WK) % T::WN, wm = wave / (T::WK * T::WN);
  const int col = lane & 31, half = lane >> 5;

  // The thread's elements of a stage: A (row ar0 + h ars, k ak0 + h aks), the
  // same for B with columns.
  const int ar0 = a_mfast ? tid % T::TM : tid / KB, ak0 = a_mfast ? tid / T::TM : tid % KB;
  const int ars = a_mfast ? 0 : 256 / KB, aks = a_mfast ? 256 / T::TM : 0;
  const int bc0 = b_kfast ? tid / KB : tid % T::TN, bk0 = b_kfast ? tid % KB : tid / T::TN;
  const int bcs = b_kfast ? 256 / KB : 0, bks = b_kfast ? 0 : 256 / T::TN;

  // Byte offsets of the thread's loads from the stage's base.  Digit maps: the
  // block's threads work the offsets of its rows, columns and stages out
  // together (each thread by itself took longer than a small product).
  unsigned ao[NA], bo[NB];
  int64_t a_rec = 0, b_rec = 0;  // bytes from the stage base to the operand's end
  __shared__ unsigned rows[LOAD == kMapped ? T::TM : 1], cols[LOAD == kMapped ? T::TN : 1];
  __shared__ unsigned ka[LOAD == kMapped ? KB : 1], kb[LOAD == kMapped ? KB : 1];
  __shared__ unsigned sa[LOAD == kMapped ? kMapStages : 1], sb[LOAD == kMapped ? kMapStages : 1];
  if constexpr (LOAD == kRowMajor) {
#pragma unroll
    for (int h = 0; h < NA; ++h) ao[h] = unsigned((ar0 + h * ars) * K + ak0 + h * aks) * 8u;
#pragma unroll
    for (int h = 0; h < NB; ++h)
      bo[h] = unsigned((bk0 + h * bks) * int64_t(N) + bc0 + h * bcs) * 8u;
    a_rec = int64_t(M - m0) * K * 8;
    b_rec = (K * int64_t(N) - n0) * 8;
    A += int64_t(m0) * K;
    B += n0;
  } else if constexpr (LOAD == kMapped) {
    if (tid < T::TM) rows[tid] = map_bytes(maps.ar, uint64_t(m0 + tid));
    if (tid < T::TN) cols[tid] = map_bytes(maps.bc, uint64_t(n0 + tid));
    if (tid < KB) ka[tid] = map_bytes(maps.ac, uint64_t(tid));
    if (tid < KB) kb[tid] = map_bytes(maps.br, uint64_t(tid));
    if (tid < s1 - s0) sa[tid] = map_bytes(maps.ac, uint64_t(s0 + tid) * KB);
    if (tid < s1 - s0) sb[tid] = map_bytes(maps.br, uint64_t(s0 + tid) * KB);
    __syncthreads();
#pragma unroll
    for (int h = 0; h < NA; ++h) ao[h] = rows[ar0 + h * ars] + ka[ak0 + h * aks];
#pragma unroll
    for (int h = 0; h < NB; ++h) bo[h] = cols[bc0 + h * bcs] + kb[bk0 + h * bks];
    a_rec = int64_t(maps.a_span) * 8;
    b_rec = int64_t(maps.b_span) * 8;
  }

  float2 ra[NA], rb[NB];
  auto fetch = [](__amdgpu_buffer_rsrc_t r, unsigned off, bool in) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, int(in ? off : 0xfffffff0u), 0, 0);
    return make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
  };
  auto records = [](int64_t bytes) {
    return __builtin_amdgcn_readfirstlane(int(unsigned(bytes < 0x80000000LL ? bytes : 0x80000000LL)));
  };
  // Elements past the end of k are zero in both operands; rows and columns
  // past the end are zero or another one's, and are not stored.
  auto load = [&](int s) {
    const int64_t k0 = int64_t(s) * KB;
    const int krem = int(K - k0 < KB ? K - k0 : KB);
    if constexpr (LOAD == kWide) {
#pragma unroll
      for (int h = 0; h < NA; ++h) {
        const int r = min(m0 + ar0 + h * ars, M - 1), kk = ak0 + h * aks;
        const uint64_t k = uint64_t(k0 + kk);
        ra[h] = make_float2(0.f, 0.f);
        if (kk < krem)
          ra[h] = A[mapped ? map_offset(maps.ar, uint64_t(r)) + map_offset(maps.ac, k)
                           : uint64_t(r) * uint64_t(K) + k];
      }
#pragma unroll
      for (int h = 0; h < NB; ++h) {
        const int c = min(n0 + bc0 + h * bcs, N - 1), kk = bk0 + h * bks;
        const uint64_t k = uint64_t(k0 + kk);
        rb[h] = make_float2(0.f, 0.f);
        if (kk < krem)
          rb[h] = B[mapped ? map_offset(maps.bc, uint64_t(c)) + map_offset(maps.br, k)
                           : k * uint64_t(N) + uint64_t(c)];
      }
    } else {
      const int64_t a_at = LOAD == kRowMajor ? k0 : 0, b_at = LOAD == kRowMajor ? k0 * N : 0;
      const unsigned a_add = LOAD == kMapped ? sa[s - s0] : 0, b_add = LOAD == kMapped ? sb[s - s0] : 0;
      const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float2*>(A + a_at), 0, records(a_rec - a_at * 8), 0x00020000);
      const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float2*>(B + b_at), 0, records(b_rec - b_at * 8), 0x00020000);
#pragma unroll
      for (int h = 0; h < NA; ++h) ra[h] = fetch(rsrc_a, ao[h] + a_add, ak0 + h * aks < krem);
#pragma unroll
      for (int h = 0; h < NB; ++h) rb[h] = fetch(rsrc_b, bo[h] + b_add, bk0 + h * bks < krem);
    }
    __builtin_amdgcn_sched_barrier(0);  // in flight during the stage's MFMAs
  };
  // Into LDS: A as it is, B as the rows (Br, -Bi) and (Bi, Br) of its real and
  // imaginary output column.
  auto store = [&](int buf) {
    float2* as = lds + buf * kStage + ar0 * SR + ak0;
    float2* bs = lds + buf * kStage + kB0 + 2 * bc0 * SR + bk0;
#pragma unroll
    for (int h = 0; h < NA; ++h) as[h * (ars * SR + aks)] = ra[h];
#pragma unroll
    for (int h = 0; h < NB; ++h) {
      float2* p = bs + h * (2 * bcs * SR + bks);
      p[0] = make_float2(rb[h].x, -rb[h].y);
      p[SR] = make_float2(rb[h].y, rb[h].x);
    }
  };

  constexpr bool kFlush = I * J == 1;  // one level of partial sums per stage
  floatx16 acc[I][J], sum;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    sum[r] = 0.f;
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) acc[i][j][r] = 0.f;
  }
  load(s0);
  store(0);
  __syncthreads();
  for (int s = s0; s < s1; ++s) {
    const int buf = (s - s0) & 1;
    if (s + 1 < s1) load(s + 1);
    constexpr int G = KB / 4 / T::WK;  // groups of four k per wave
    const float2* as = lds + buf * kStage + (wm * 32 * I + col) * SR + wk * 4 * G + 2 * half;
    const float2* bs = lds + buf * kStage + kB0 + (wn * 32 * J + col) * SR + wk * 4 * G + 2 * half;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      // lanes 0..31 hold k = 4g, 4g + 1, lanes 32..63 k = 4g + 2, 4g + 3
      float4 a[I], b[J];
#pragma unroll
      for (int i = 0; i < I; ++i) a[i] = *reinterpret_cast<const float4*>(as + 32 * i * SR + 4 * g);
#pragma unroll
      for (int j = 0; j < J; ++j) b[j] = *reinterpret_cast<const float4*>(bs + 32 * j * SR + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
          for (int j = 0; j < J; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32((&a[i].x)[e], (&b[j].x)[e],
                                                             acc[i][j], 0, 0, 0);
    }
    if constexpr (kFlush) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        sum[r] += acc[0][0][r];
        acc[0][0][r] = 0.f;
      }
    }
    if (s + 1 < s1) store(buf ^ 1);
    __syncthreads();
  }

  // Register r of lane l holds row 8 (r / 4) + 4 (l / 32) + r % 4, real column
  // l % 32 of its tile.
  float* Cf = reinterpret_cast<float*>(C);
  if constexpr (T::WK > 1) {
    float* red = reinterpret_cast<float*>(lds);  // (the last barrier freed the stages)
#pragma unroll
    for (int r = 0; r < 16; ++r) red[(wave * 16 + r) * 64 + lane] = sum[r];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = wave * 4 + q;
      float v = red[r * 64 + lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) v += red[(w * 16 + r) * 64 + lane];
      const int row = m0 + 8 * wave + 4 * half + q, cn = n0 + (col >> 1);
      if (row < M && cn < N) Cf[(uint64_t(row) * N + cn) * 2 + (col & 1)] = v;
    }
  } else {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = m0 + (wm * I + i) * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
          const int cn = n0 + (wn * J + j) * 16 + (col >> 1);
          if (row < M && cn < N)
            Cf[(uint64_t(row) * N + cn) * 2 + (col & 1)] = kFlush ? sum[r] : acc[i][j][r];
        }
  }
}

template <class T, int LOAD>
__global__ __launch_bounds__(256, 2) void cgemm_f32_kernel(
    const float2* __restrict__ A, const float2* __restrict__ B, float2* __restrict__ C, int M,
    int N, int64_t K, Maps maps, bool mapped, bool a_mfast, bool b_kfast, int tiles_n, int stages,
    int stages_per) {
  __shared__ __align__(16) float2 lds[T::kLds];
  const uint64_t t = xcd_tile(blockIdx.x, gridDim.x);
  const int tm = __builtin_amdgcn_readfirstlane(int(t / tiles_n));
  const int s0 = int(blockIdx.y) * stages_per;
  f32_tile<T, LOAD>(A, B, C + uint64_t(blockIdx.y) * uint64_t(M) * uint64_t(N), M, N, K, maps,
                    mapped, a_mfast, b_kfast, tm * T::TM, (int(t) - tm * tiles_n) * T::TN, s0,
                    min(s0 + stages_per, stages), lds);
}

// One problem of a grouped launch (row-major operands).
struct F32Prob {
  const float2* A;
  const float2* B;
  float2* C;
  int64_t K;
  int M, N, tiles_n, stages;
  uint64_t first_tile;  // index of its first tile in the launch
};

// A block per tile of all problems that take this tile; one launch each took
// 5 to 10 us (100 products of 512 x 64 x 64: 1045 -> 38 us, 250 of 64 x 5 x 100
// 6534 -> 41, most of the last the caller's list).
template <class T>
__device__ __forceinline__ void f32_grouped_block(const F32Prob* probs, int count, float2* lds) {
  const uint64_t t = xcd_tile(blockIdx.x, gridDim.x);
  const F32Prob p = probs[group_entry(&probs[0].first_tile, sizeof(F32Prob), count, t)];
  const int local = int(t - p.first_tile);
  const int tm = __builtin_amdgcn_readfirstlane(local / p.tiles_n);
  f32_tile<T, kRowMajor>(p.A, p.B, p.C, p.M, p.N, p.K, Maps{}, false, false, false, tm * T::TM,
                         (local - tm * p.tiles_n) * T::TN, 0, p.stages, lds);
}
template <class T>
__global__ __launch_bounds__(256, 2) void cgemm_f32_grouped_kernel(
    const F32Prob* __restrict__ probs, int count) {
  __shared__ __align__(16) float2 lds[T::kLds];
  f32_grouped_block<T>(probs, count, lds);
}
template <class T>
__global__ __launch_bounds__(256, 2) void cgemm_f32_grouped_args_kernel(ArgList<F32Prob> list,
                                                                        int count) {
  __shared__ __align__(16) float2 lds[T::kLds];
  f32_grouped_block<T>(list.p, count, lds);
}

// C[c] = sum_s part[s][c]: four groups of 64 lanes, eight loads in flight.
__global__ __launch_bounds__(256) void f32_sum_kernel(const float2* __restrict__ part,
                                                      float2* __restrict__ C, int nsplit,
                                                      uint64_t size) {
  __shared__ float2 red[4][64];
  const int cl = threadIdx.x & 63, sg = threadIdx.x >> 6;
  const uint64_t c = uint64_t(blockIdx.x) * 64 + cl;
  float2 acc = make_float2(0.f, 0.f);
  if (c < size) {
#pragma unroll 8
    for (int s = sg; s < nsplit; s += 4) {
      const float2 v = part[uint64_t(s) * size + c];
      acc.x += v.x;
      acc.y += v.y;
    }
  }
  red[sg][cl] = acc;
  __syncthreads();
  if (sg == 0 && c < size) {
#pragma unroll
    for (int g = 1; g < 4; ++g) {
      acc.x += red[g][cl].x;
      acc.y += red[g][cl].y;
    }
    C[c] = acc;
  }
}

enum F32Tile { kTileA, kTileF, kTileD, kTileE, kTileC };
struct F32Plan {
  F32Tile tile;
  int splits;
  double us;  // estimated time
};

uint64_t tiles_of(F32Tile t, uint64_t m, uint64_t n) {
  static const uint64_t tm[] = {128, 64, 128, 32, 32}, tn[] = {64, 32, 16, 64, 16};
  return ((m + tm[t] - 1) / tm[t]) * ((n + tn[t] - 1) / tn[t]);
}

int stage_of(F32Tile t) {
  static const int kb[] = {16, 32, 16, 16, 64};
  return kb[t];
}

// The tile and the splits over k with the least estimated time: `us` per stage
// of a tile, as measured with every CU busy (a CU with a single block, whose
// waits nothing hides, takes 1.35 of that), times the blocks of the busiest
// CU, and for splits the sum's launch and its traffic.  Within 10% of the best
// measured choice on 30 shapes but for 12-20% on three below 13 us.  Only
// products of up to 2^16 outputs are split (16 MiB of partial sums at most).
constexpr double kStageUs[] = {2.0, 1.2, 0.6, 0.6, 0.9};  // per tile, every CU busy
constexpr double kAlone = 1.35;                           // of a CU with one block
F32Plan f32_plan(uint64_t m, uint64_t n, uint64_t k) {
  F32Plan best{kTileC, 1, 1e30};
  for (int t = kTileA; t <= kTileC; ++t) {
    const uint64_t tiles = tiles_of(F32Tile(t), m, n), kb = stage_of(F32Tile(t));
    const uint64_t stages = (k + kb - 1) / kb;
    for (uint64_t s = 1; s <= 64 && s <= stages; s *= 2) {
      if (s > 1 && (m * n > 65536 || stages < 4 || tiles * s > 1024 ||
                    s * m * n * sizeof(float2) > kFixedScratchBytes))
        break;
      const uint64_t per = (stages + s - 1) / s, splits = (stages + per - 1) / per;
      const uint64_t rounds = (tiles * splits + 255) / 256;
      double time = kStageUs[t] * double(per) * (rounds == 1 ? kAlone : double(rounds));
      if (splits > 1) time += 2.5 + double(splits * m * n) * 4e-6;
      if (time < best.us) best = F32Plan{F32Tile(t), int(splits), time};
    }
  }
  return best;
}

// Offset of the map's index idx, as the kernels compute it.
uint64_t map_at(const qfx_index_map& d, uint64_t idx) {
  uint64_t off = 0;
  for (int j = 0; j < d.ndigits; ++j) {
    off += (idx & ((uint64_t(1) << d.bits[j]) - 1)) << d.shift[j];
    idx >>= d.bits[j];
  }
  return off;
}

template <class T>
hipError_t launch_tile(qfx_context* ctx, const float2* A, const float2* B, float2* C, uint64_t m,
                       uint64_t n, uint64_t k, const qfx_index_map* maps, bool a_mfast,
                       bool b_kfast, int splits) {
  const uint64_t tiles_n = (n + T::TN - 1) / T::TN, tiles = tiles_n * ((m + T::TM - 1) / T::TM);
  const int stages = int((k + T::KB - 1) / T::KB), per = (stages + splits - 1) / splits;
  const dim3 grid{unsigned(tiles), unsigned(splits), 1};
  // what the 32-bit offsets have to reach, in elements, against 2 GiB
  const uint64_t a_span = maps ? map_at(maps[0], m - 1) + map_at(maps[1], k - 1) + 1
                               : T::TM * k + T::KB;
  const uint64_t b_span = maps ? map_at(maps[3], n - 1) + map_at(maps[2], k - 1) + 1
                               : T::KB * n + T::TN;
  const bool wide = std::max(a_span, b_span) >= (uint64_t(1) << 28) || (maps && per > kMapStages);
  const Maps mp = maps ? Maps{maps[0], maps[1], maps[2], maps[3], a_span, b_span} : Maps{};
  auto go = [&](auto load) {
    cgemm_f32_kernel<T, decltype(load)::value><<<grid, 256, 0, ctx->stream>>>(
        A, B, C, int(m), int(n), int64_t(k), mp, maps != nullptr, a_mfast, b_kfast, int(tiles_n),
        stages, per);
  };
  if (wide) go(std::integral_constant<int, kWide>{});
  else if (maps) go(std::integral_constant<int, kMapped>{});
  else go(std::integral_constant<int, kRowMajor>{});
  return hipGetLastError();
}

}  // namespace

double qfx_f32_time(uint64_t m, uint64_t n, uint64_t k) { return f32_plan(m, n, k).us; }

bool qfx_f32_fits(uint64_t m, uint64_t n, uint64_t k) {
  return m <= 0x7fffff00ULL && n <= 0x7fffff00ULL && k <= (1ULL << 34) &&
         (tiles_of(kTileC, m, n) <= kMaxBlocks ||  // (the smallest tile)
          tiles_of(f32_plan(m, n, k).tile, m, n) <= kMaxBlocks);
}

int qfx_launch_f32(qfx_context* ctx, const float2* A, const float2* B, float2* C, uint64_t m,
                   uint64_t n, uint64_t k, const qfx_index_map* maps, bool a_mfast,
                   bool b_kfast, bool needs_reservation) {
  const F32Plan p = f32_plan(m, n, k);
  float2* out = C;
  if (p.splits > 1) {
    const size_t bytes = size_t(p.splits) * m * n * sizeof(float2);  // <= kFixedScratchBytes
    void* ws = nullptr;
    // A sequence being recorded cannot grow the workspace: the partial sums
    // go into the context's own scratch for it, or the product is refused.
    if (ctx->capturing && !ctx->use_fixed_scratch && bytes > ctx->work_bytes && !needs_reservation) {
      ws = ctx->record_scratch;
    } else {
      const int st = qfx_workspace(ctx, bytes, &ws);
      if (st != QFX_OK) return st;
    }
    out = static_cast<float2*>(ws);
  }
  auto go = [&](auto tile) {
    return launch_tile<decltype(tile)>(ctx, A, B, out, m, n, k, maps, a_mfast, b_kfast, p.splits);
  };
  QFX_HIP(p.tile == kTileA   ? go(TileA{})
          : p.tile == kTileF ? go(TileF{})
          : p.tile == kTileD ? go(TileD{})
          : p.tile == kTileE ? go(TileE{})
                             : go(TileC{}));
  if (p.splits > 1)
    f32_sum_kernel<<<unsigned((m * n + 63) / 64), 256, 0, ctx->stream>>>(out, C, p.splits, m * n);
  QFX_HIP(hipGetLastError());
  return QFX_OK;
}

int qfx_launch_f32_grouped(qfx_context* ctx, const qfx_gemm_desc* descs,
                           const std::vector<int>& which) {
  // Each product takes the tile that would be the fastest if all were like it.
  // Those that fill the chip alone run as qfx_cgemm_c64 runs them, and so do
  // all of a few where that is estimated faster (long k, split alone) and
  // what is beyond one grid.
  std::vector<std::vector<int>> by_tile(kTileC + 1);
  double alone_us = 0, group_us = 6, longest = 0;
  auto alone = [&](const qfx_gemm_desc& d) {
    QfxLaunchScope scope(ctx, QFX_K_CGEMM,
                         8.0 * (double(d.m) * d.k + double(d.k) * d.n + double(d.m) * d.n),
                         8.0 * double(d.m) * double(d.n) * double(d.k));
    return qfx_launch_f32(ctx, reinterpret_cast<const float2*>(d.A),
                          reinterpret_cast<const float2*>(d.B), reinterpret_cast<float2*>(d.C),
                          d.m, d.n, d.k, nullptr, false, false, false);
  };
  for (int i : which) {
    const qfx_gemm_desc& d = descs[i];
    const bool reach = 128 * d.k + 64 < (1ULL << 28) && 64 * d.n + 64 < (1ULL << 28) &&
                       tiles_of(kTileC, d.m, d.n) < (1ULL << 24);
    if (!reach || tiles_of(kTileA, d.m, d.n) >= 512) {
      const int st = alone(d);
      if (st != QFX_OK) return st;
      continue;
    }
    int best = -1;
    double best_us = 1e30, best_work = 0, best_chain = 0;
    for (int t = kTileA; t <= kTileC; ++t) {
      const uint64_t kb = stage_of(F32Tile(t));
      const double chain = kStageUs[t] * double((d.k + kb - 1) / kb);
      const double work = chain * double(tiles_of(F32Tile(t), d.m, d.n)) / 256;
      const double us = work * double(which.size()) + kAlone * chain;
      if (us < best_us) best = t, best_us = us, best_work = work, best_chain = chain;
    }
    by_tile[best].push_back(i);
    alone_us += which.size() > 16 ? 1e9 : f32_plan(d.m, d.n, d.k).us + 4;
    group_us += best_work;
    longest = std::max(longest, kAlone * best_chain);
  }
  std::vector<F32Prob> probs;
  uint64_t tiles[kTileC + 1] = {};
  int counts[kTileC + 1] = {};
  for (int t = kTileA; t <= kTileC; ++t)
    for (int i : by_tile[t]) {
      const qfx_gemm_desc& d = descs[i];
      const uint64_t more = tiles_of(F32Tile(t), d.m, d.n);
      if (alone_us < group_us + longest || tiles[t] + more > kMaxBlocks) {
        const int st = alone(d);
        if (st != QFX_OK) return st;
        continue;
      }
      static const int tn[] = {64, 32, 16, 64, 16};
      probs.push_back(F32Prob{reinterpret_cast<const float2*>(d.A),
                              reinterpret_cast<const float2*>(d.B), reinterpret_cast<float2*>(d.C),
                              int64_t(d.k), int(d.m), int(d.n), int((d.n + tn[t] - 1) / tn[t]),
                              int((d.k + stage_of(F32Tile(t)) - 1) / stage_of(F32Tile(t))),
                              tiles[t]});
      tiles[t] += more;
      ++counts[t];
    }
  if (probs.empty()) return QFX_OK;
  const bool args = probs.size() <= size_t(kArgProblems);
  void* ws = nullptr;
  if (!args) {
    int st = qfx_workspace(ctx, probs.size() * sizeof(F32Prob), &ws);
    if (st != QFX_OK) return st;
    st = qfx_upload_problems(ctx, ws, probs.data(), probs.size() * sizeof(F32Prob));
    if (st != QFX_OK) return st;
  }
  double flops = 0, bytes = 0;
  for (const F32Prob& p : probs) {
    flops += 8.0 * p.M * p.N * double(p.K);
    bytes += 8.0 * (double(p.M) * p.K + double(p.K) * p.N + double(p.M) * p.N);
  }
  QfxLaunchScope scope(ctx, QFX_K_CGEMM, bytes, flops);
  const F32Prob* dev = static_cast<const F32Prob*>(ws);
  const F32Prob* host = probs.data();
  auto go = [&](auto tile, int t) {
    const int n = counts[t];
    if (n == 0) return;
    if (args) {
      ArgList<F32Prob> list{};
      std::copy(host, host + n, list.p);
      cgemm_f32_grouped_args_kernel<decltype(tile)>
          <<<unsigned(tiles[t]), 256, 0, ctx->stream>>>(list, n);
    } else {
      cgemm_f32_grouped_kernel<decltype(tile)><<<unsigned(tiles[t]), 256, 0, ctx->stream>>>(dev, n);
      dev += n;
    }
    host += n;
  };
  go(TileA{}, kTileA);
  go(TileF{}, kTileF);
  go(TileD{}, kTileD);
  go(TileE{}, kTileE);
  go(TileC{}, kTileC);
  QFX_HIP(hipGetLastError());
  return QFX_OK;
}
