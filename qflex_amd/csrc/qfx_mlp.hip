// The cost model's network: an MLP 64 -> 256 -> 256 -> 1 (ReLU) in BF16
// with FP32 accumulation, trained with MSE and Adam, all on the GPU.
// (No counterpart in the reference: it scores candidate contraction
// orderings; amplitudes always come from exact contraction.)
//
// Parameters live in one FP32 buffer (layout in include/qfx.h); every GEMM
// rounds its operands to BF16 (round to nearest even) and accumulates in
// FP32 on v_mfma_f32_32x32x16_bf16.  Activations are kept as BF16, the
// values the next GEMM consumes, so the backward pass differentiates
// exactly the function the forward pass computed.
#include <algorithm>

#include "qfx_internal.h"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kIn = QFX_MLP_IN, kHid = QFX_MLP_HIDDEN;
constexpr int kW1 = 0, kB1 = kW1 + kIn * kHid, kW2 = kB1 + kHid, kB2 = kW2 + kHid * kHid,
              kW3 = kB2 + kHid, kB3 = kW3 + kHid, kParams = kB3 + 1;
static_assert(kParams == QFX_MLP_PARAMS, "parameter layout");

// One training step's forward and backward pass is two launches.  As one
// launch per GEMM, conversion, ReLU gradient and column sum it was about 20
// of them, each a few us of launch and drain for well under 1 us of work (512
// rows: 218 us a step, 17 us now; 4096 rows: 1097 and 27).
//
// mlp_rows_kernel takes 32 rows of the batch at a time through the whole
// network: forward, and for training the error and the two hidden layers'
// gradients.  8 waves; wave w owns 32 columns of both hidden layers and
// keeps its columns of W1 and W2 as MFMA fragments in 80 registers (W2 by
// rows, for dH1 = dZ2 W2^T, is in LDS), so the weights are read once per
// block however many row tiles it walks; only activations of 32 rows pass
// through LDS.  A small batch has one block per tile; what bounds it there is
// reading the weights (320 KiB per block, from L2).
//
// mlp_grad_kernel forms the weight gradients, contractions over the batch:
// one 32 x 32 output tile per block, 8 waves taking the batch's k-steps in
// turn, summed in LDS.  The first kernel leaves both operands in fragment
// order (frag_offset): the MFMA result holds 4 rows of one column per lane,
// half of what a lane of the next product's fragment takes, so the stores are
// 8 bytes side by side and a fragment is one contiguous 1 KiB load.
constexpr int kRows = 32;             // batch rows per tile
constexpr int kXPitch = kIn + 8;      // BF16 per LDS row: 16-byte reads of 8 rows hit distinct banks
constexpr int kHPitch = kHid + 8;
constexpr int kPartCols = 3 * kHid + 2;  // db1, db2, dw3, db3, loss

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ floatx16 zero16() {
  floatx16 v;
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = 0.f;
  return v;
}

// What the row tiles leave for the weight gradients: BF16 activations and
// gradients as fragments of 32 units by 16 rows, `steps` of them along the
// batch (two per row tile, the rows past the batch zero), and kPartCols sums
// per block.
struct MlpWork {
  __bf16 *xT, *h1T, *dz1T, *dz2T;
  float* part;
  int64_t steps;
  int blocks;
};

// Offset of four rows (from `row`, a multiple of 4) of `unit` in fragment
// order: [unit / 32][row / 16][lane = 32 (row / 8 % 2) + unit % 32][row % 8].
__device__ __forceinline__ int64_t frag_offset(const MlpWork& w, int unit, int64_t row) {
  return (((unit >> 5) * w.steps + (row >> 4)) * 64 + ((row >> 3) & 1) * 32 + (unit & 31)) * 8 +
         (row & 7);
}

// Sum of v[r] over the 32 lanes of each half wave: lane c ends with the sum
// of element c & 15 (a reduce-scatter: 8 + 4 + 2 + 1 exchanges, and one more
// across the two lanes that then hold the same element).
template <int S>
__device__ __forceinline__ void fold_lanes(float (&v)[16], int col) {
  const bool upper = (col & S) != 0;
#pragma unroll
  for (int i = 0; i < S; ++i) {
    const float lo = v[i], hi = v[i + S];
    const float other = __shfl_xor(upper ? lo : hi, S);
    v[i] = (upper ? hi : lo) + other;
  }
}

__device__ __forceinline__ float half_wave_sums(float (&v)[16], int col) {
  fold_lanes<8>(v, col);
  fold_lanes<4>(v, col);
  fold_lanes<2>(v, col);
  fold_lanes<1>(v, col);
  return v[0] + __shfl_xor(v[0], 16);
}

// TRAIN false: y[b] for the batch.  TRAIN true: the work of `w`.
template <bool TRAIN>
__global__ __launch_bounds__(512) void mlp_rows_kernel(const float* __restrict__ X,
                                                       const float* __restrict__ P,
                                                       const float* __restrict__ target,
                                                       float* __restrict__ y, MlpWork w, int B) {
  __shared__ __align__(16) __bf16 Xs[kRows * kXPitch];
  __shared__ __align__(16) __bf16 H1s[kRows * kHPitch];
  __bf16* const Zs = H1s;  // dZ2 takes H1's place once layer 2 has read it
  __shared__ float ysum[8][kRows];
  __shared__ float dys[kRows];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int j = wave * 32 + col;  // this lane's hidden unit

  bf16x8 w1[kIn / 16], w2[kHid / 16];
#pragma unroll
  for (int ks = 0; ks < kIn / 16; ++ks)
#pragma unroll
    for (int e = 0; e < 8; ++e)
      w1[ks][e] = static_cast<__bf16>(P[kW1 + (ks * 16 + 8 * half + e) * kHid + j]);
#pragma unroll
  for (int ks = 0; ks < kHid / 16; ++ks)
#pragma unroll
    for (int e = 0; e < 8; ++e)
      w2[ks][e] = static_cast<__bf16>(P[kW2 + (ks * 16 + 8 * half + e) * kHid + j]);
  // W2 by rows in LDS (TRAIN), for dH1 = dZ2 W2^T: out of the columns the
  // waves hold, as reading it from memory a lane per row makes every 16 bytes
  // an access of their own (a step of 32 rows took 17 us that way).  Lanes of
  // adjacent columns exchange halves, so that each stores two columns of one row.
  extern __shared__ __align__(16) __bf16 Ws[];
  if constexpr (TRAIN) {
#pragma unroll
    for (int ks = 0; ks < kHid / 16; ++ks)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const bf16x2 own = {w2[ks][e], w2[ks][e + 1]};
        const bf16x2 next =
            __builtin_bit_cast(bf16x2, __builtin_amdgcn_mov_dpp(  // quad_perm [1, 0, 3, 2]
                                           __builtin_bit_cast(int, own), 0xb1, 0xf, 0xf, true));
        const bool odd = col & 1;
        const bf16x2 v = odd ? bf16x2{next[1], own[1]} : bf16x2{own[0], next[0]};
        const int row = ks * 16 + 8 * half + e + (odd ? 1 : 0);
        *reinterpret_cast<bf16x2*>(Ws + row * kHPitch + (j & ~1)) = v;
      }
  }
  const float b1 = P[kB1 + j], b2 = P[kB2 + j], b3 = P[kB3];
  const float w3 = static_cast<float>(static_cast<__bf16>(P[kW3 + j]));
  float db1 = 0.f, db2 = 0.f, dw3 = 0.f, db3 = 0.f, loss = 0.f;

  const int tiles = (B + kRows - 1) / kRows;
  for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
    const int64_t r0 = int64_t(t) * kRows;
#pragma unroll
    for (int h = 0; h < kRows * kIn / 512; ++h) {
      const int e = tid + 512 * h, r = e / kIn, i = e % kIn;
      const float x = r0 + r < B ? X[(r0 + r) * kIn + i] : 0.f;
      Xs[r * kXPitch + i] = static_cast<__bf16>(x);
    }
    __syncthreads();
    // register r of a result: row 8*(r/4) + 4*half + r%4 of the tile
    auto row_of = [&](int r) { return 8 * (r >> 2) + 4 * half + (r & 3); };
    // H1 = relu(X W1 + b1)
    floatx16 acc = zero16();
#pragma unroll
    for (int ks = 0; ks < kIn / 16; ++ks) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(Xs + col * kXPitch + ks * 16 + 8 * half);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w1[ks], acc, 0, 0, 0);
    }
    unsigned live1 = 0;  // bit r: H1 > 0
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * g + e;
        v[e] = static_cast<__bf16>(fmaxf(acc[r] + b1, 0.f));
        if (static_cast<float>(v[e]) > 0.f) live1 |= 1u << r;
        H1s[row_of(r) * kHPitch + j] = v[e];
      }
      if constexpr (TRAIN) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (r0 + row_of(4 * g + e) >= B) v[e] = static_cast<__bf16>(0.f);
        *reinterpret_cast<bf16x4*>(w.h1T + frag_offset(w, j, r0 + row_of(4 * g))) = v;
      }
    }
    if constexpr (TRAIN) {
      const int i = tid & (kIn - 1), b = 4 * (tid / kIn);
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = Xs[(b + e) * kXPitch + i];
      *reinterpret_cast<bf16x4*>(w.xT + frag_offset(w, i, r0 + b)) = v;
    }
    __syncthreads();
    // H2 = relu(H1 W2 + b2), rounded to BF16; y = H2 w3 + b3
    acc = zero16();
#pragma unroll
    for (int ks = 0; ks < kHid / 16; ++ks) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(H1s + col * kHPitch + ks * 16 + 8 * half);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w2[ks], acc, 0, 0, 0);
    }
    float prod[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[r] = static_cast<float>(static_cast<__bf16>(fmaxf(acc[r] + b2, 0.f)));
      prod[r] = acc[r] * w3;
    }
    const float s = half_wave_sums(prod, col);
    if (col < 16) ysum[wave][row_of(col)] = s;
    __syncthreads();
    if (tid < kRows) {
      float v = ysum[0][tid];
#pragma unroll
      for (int q = 1; q < 8; ++q) v += ysum[q][tid];
      v += b3;
      if constexpr (TRAIN) {
        float dy = 0.f;
        if (r0 + tid < B) {
          const float d = v - target[r0 + tid];
          dy = 2.f * d / float(B);
          loss += d * d / float(B);
        }
        dys[tid] = dy;
        db3 += dy;
      } else if (r0 + tid < B) {
        y[r0 + tid] = v;
      }
    }
    if constexpr (TRAIN) {
      __syncthreads();
      // dZ2 = relu'(H2) dy w3^T
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 4 * g + e;
          const float dy = dys[row_of(r)];
          const float dz = acc[r] > 0.f ? dy * w3 : 0.f;
          db2 += dz;
          // (the layer-3 gradient's operands are BF16 like every product's)
          if (r0 + row_of(r) < B) dw3 += acc[r] * static_cast<float>(static_cast<__bf16>(dy));
          v[e] = static_cast<__bf16>(dz);
          Zs[row_of(r) * kHPitch + j] = v[e];
        }
        *reinterpret_cast<bf16x4*>(w.dz2T + frag_offset(w, j, r0 + row_of(4 * g))) = v;
      }
      __syncthreads();
      // dZ1 = relu'(H1) (dZ2 W2^T)
      acc = zero16();
#pragma unroll
      for (int ks = 0; ks < kHid / 16; ++ks) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(Zs + col * kHPitch + ks * 16 + 8 * half);
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(Ws + j * kHPitch + ks * 16 + 8 * half);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        bf16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 4 * g + e;
          const float dz = (live1 >> r) & 1u && r0 + row_of(r) < B ? acc[r] : 0.f;
          db1 += dz;
          v[e] = static_cast<__bf16>(dz);
        }
        *reinterpret_cast<bf16x4*>(w.dz1T + frag_offset(w, j, r0 + row_of(4 * g))) = v;
      }
    }
    // The next tile's first writes (Xs, H1s, ysum) are all separated from
    // this tile's last reads of them by a barrier above.
  }
  if constexpr (TRAIN) {
    db1 += __shfl_xor(db1, 32);
    db2 += __shfl_xor(db2, 32);
    dw3 += __shfl_xor(dw3, 32);
    float* part = w.part + int64_t(blockIdx.x) * kPartCols;
    if (half == 0) {
      part[j] = db1;
      part[kHid + j] = db2;
      part[2 * kHid + j] = dw3;
    }
    if (wave == 0) {
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) {
        db3 += __shfl_xor(db3, o);
        loss += __shfl_xor(loss, o);
      }
      if (lane == 0) {
        part[3 * kHid] = db3;
        part[3 * kHid + 1] = loss;
      }
    }
  }
}

// Blocks [0, 64): dW2 = H1^T dZ2 in 8 x 8 tiles; [64, 80): dW1 = X^T dZ1 in
// 2 x 8 tiles; the rest: 64 columns each of the row blocks' sums, added in
// block order within 8 interleaved groups.
constexpr int kGradTiles = (kHid / 32 + kIn / 32) * (kHid / 32);
constexpr int kGradBlocks = kGradTiles + (kPartCols + 63) / 64;

__global__ __launch_bounds__(512) void mlp_grad_kernel(MlpWork w, float* __restrict__ grads,
                                                       float* __restrict__ loss) {
  __shared__ float red[8][64 * 17];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (int(blockIdx.x) >= kGradTiles) {
    const int c = (int(blockIdx.x) - kGradTiles) * 64 + lane;
    float s = 0.f;
    if (c < kPartCols)
      for (int b = wave; b < w.blocks; b += 8) s += w.part[int64_t(b) * kPartCols + c];
    red[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && c < kPartCols) {
#pragma unroll
      for (int q = 1; q < 8; ++q) s += red[q][lane];
      if (c < kHid) grads[kB1 + c] = s;
      else if (c < 2 * kHid) grads[kB2 + c - kHid] = s;
      else if (c < 3 * kHid) grads[kW3 + c - 2 * kHid] = s;
      else if (c == 3 * kHid) grads[kB3] = s;
      else *loss = s;
    }
    return;
  }
  const bool second = blockIdx.x < (kHid / 32) * (kHid / 32);
  const int tile = second ? int(blockIdx.x) : int(blockIdx.x) - (kHid / 32) * (kHid / 32);
  const int m0 = tile / (kHid / 32) * 32, n0 = tile % (kHid / 32) * 32;
  const __bf16* a = (second ? w.h1T : w.xT) + (m0 / 32 * w.steps * 64 + lane) * 8;
  const __bf16* b = (second ? w.dz2T : w.dz1T) + (n0 / 32 * w.steps * 64 + lane) * 8;
  floatx16 acc = zero16();
  for (int64_t k = wave; k < w.steps; k += 4 * 8) {
    bf16x8 fa[4], fb[4];  // four k-steps of loads in flight
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t ku = k + 8 * u;
      const bool in = ku < w.steps;
      fa[u] = in ? *reinterpret_cast<const bf16x8*>(a + ku * 512) : bf16x8{};
      fb[u] = in ? *reinterpret_cast<const bf16x8*>(b + ku * 512) : bf16x8{};
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[u], fb[u], acc, 0, 0, 0);
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) red[wave][lane * 17 + r] = acc[r];
  __syncthreads();
  float* out = grads + (second ? kW2 : kW1);
#pragma unroll
  for (int h = 0; h < 2; ++h) {  // element (row e / 32, column e % 32) of the tile
    const int e = tid + 512 * h, i = e >> 5, jj = e & 31;
    const int l = jj + 32 * ((i >> 2) & 1), r = 4 * (i >> 3) + (i & 3);
    float s = red[0][l * 17 + r];
#pragma unroll
    for (int q = 1; q < 8; ++q) s += red[q][l * 17 + r];
    out[(m0 + i) * kHid + n0 + jj] = s;
  }
}

__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ g,
                            float* __restrict__ m, float* __restrict__ v, int64_t n, float lr,
                            float b1, float b2, float eps, float c1, float c2) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

unsigned grid_for(int64_t n) { return unsigned(std::min<int64_t>((n + 255) / 256, 4096)); }

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// Blocks of the row kernel for a batch of B: one per tile up to what the
// compute units hold at once (W2 in LDS when training: one each; forward
// only: two).
int row_blocks(qfx_context* ctx, int B, bool train) {
  if (ctx->cus <= 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) !=
        hipSuccess)
      cus = 0;
    ctx->cus = cus > 0 ? cus : 256;
  }
  return std::min((B + kRows - 1) / kRows, (train ? 1 : 2) * ctx->cus);
}

int mlp_work(qfx_context* ctx, int B, MlpWork* w) {
  const int64_t rows = (int64_t(B) + kRows - 1) / kRows * kRows;
  w->steps = rows / 16;
  w->blocks = row_blocks(ctx, B, true);
  const size_t hb = align256(size_t(kHid) * rows * 2), xb = align256(size_t(kIn) * rows * 2);
  void* base = nullptr;
  int st = qfx_workspace(ctx, 3 * hb + xb + size_t(w->blocks) * kPartCols * sizeof(float), &base);
  if (st != QFX_OK) return st;
  char* p = static_cast<char*>(base);
  w->h1T = reinterpret_cast<__bf16*>(p);
  w->dz1T = reinterpret_cast<__bf16*>(p + hb);
  w->dz2T = reinterpret_cast<__bf16*>(p + 2 * hb);
  w->xT = reinterpret_cast<__bf16*>(p + 3 * hb);
  w->part = reinterpret_cast<float*>(p + 3 * hb + xb);
  return QFX_OK;
}

}  // namespace

extern "C" int qfx_mlp_forward(qfx_context* ctx, uint64_t batch, const float* X,
                               const float* params, float* y) {
  QFX_CHECK_CTX(ctx);
  if (batch == 0) return QFX_OK;
  if (!X || !params || !y) return qfx_set_error(QFX_ERR_INVALID, "qfx_mlp_forward: null pointer");
  if (batch > (uint64_t(1) << 20))
    return qfx_set_error(QFX_ERR_INVALID, "qfx_mlp_forward: batch above 2^20");
  const int B = int(batch);
  mlp_rows_kernel<false><<<row_blocks(ctx, B, false), 512, 0, ctx->stream>>>(X, params, nullptr, y,
                                                                      MlpWork{}, B);
  QFX_HIP(hipGetLastError());
  return QFX_OK;
}

extern "C" int qfx_mlp_backward(qfx_context* ctx, uint64_t batch, const float* X,
                                const float* target, const float* params, float* grads,
                                float* loss) {
  QFX_CHECK_CTX(ctx);
  if (batch == 0) return qfx_set_error(QFX_ERR_INVALID, "qfx_mlp_backward: empty batch");
  if (!X || !target || !params || !grads || !loss)
    return qfx_set_error(QFX_ERR_INVALID, "qfx_mlp_backward: null pointer");
  if (batch > (uint64_t(1) << 20))
    return qfx_set_error(QFX_ERR_INVALID, "qfx_mlp_backward: batch above 2^20");
  const int B = int(batch);
  MlpWork w;
  int st = mlp_work(ctx, B, &w);
  if (st != QFX_OK) return st;
  constexpr int kWsBytes = kHid * kHPitch * 2;
  static const hipError_t lds = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&mlp_rows_kernel<true>),
      hipFuncAttributeMaxDynamicSharedMemorySize, kWsBytes);
  QFX_HIP(lds);
  mlp_rows_kernel<true><<<w.blocks, 512, kWsBytes, ctx->stream>>>(X, params, target, nullptr, w, B);
  mlp_grad_kernel<<<kGradBlocks, 512, 0, ctx->stream>>>(w, grads, loss);
  QFX_HIP(hipGetLastError());
  return QFX_OK;
}

extern "C" int qfx_mlp_adam(qfx_context* ctx, float* params, const float* grads, float* m,
                            float* v, int step, float lr, float beta1, float beta2, float eps) {
  QFX_CHECK_CTX(ctx);
  if (!params || !grads || !m || !v)
    return qfx_set_error(QFX_ERR_INVALID, "qfx_mlp_adam: null pointer");
  if (step < 1) return qfx_set_error(QFX_ERR_INVALID, "qfx_mlp_adam: step counts from 1");
  const float c1 = 1.f - powf(beta1, float(step)), c2 = 1.f - powf(beta2, float(step));
  adam_kernel<<<grid_for(kParams), 256, 0, ctx->stream>>>(params, grads, m, v, kParams, lr, beta1,
                                                          beta2, eps, c1, c2);
  QFX_HIP(hipGetLastError());
  return QFX_OK;
}
