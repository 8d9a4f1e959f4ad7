// Index permutation ("reorder") of complex64 tensors.
//
// Tensor::reorder (reference src/tensor.cpp:866-911) moves data with up to
// five left/right block passes over the tensor (_fast_reorder,
// src/tensor.cpp:494-710).  Here a permutation is one pass:
//
//  * axes of size 1 are dropped and axes that stay adjacent are fused;
//  * if every fused dimension is a power of two the permutation is a
//    permutation of the bits of the linear index.  A tile is the set of
//    elements that differ only in a chosen set T of index bits:
//    T = the lowest input bits (so a tile's loads are contiguous runs)
//    plus the lowest output bits not already in T (so its stores are too).
//    Each workgroup stages tiles through LDS: load in input order, store in
//    output order.  The bits outside T select the tile.
//  * otherwise a tile is a box: the innermost input axes up to a run of some
//    32 elements (so loads are contiguous runs) and the innermost output axes
//    likewise (so stores are), long axes cut into near-equal blocks; staged
//    through LDS the same way;
//  * small tensors, and those of 2^31 elements and more, with other dimensions
//    take a kernel that computes each element's source offset.
#include <algorithm>
#include <numeric>

#include "qfx_internal.h"

namespace {

constexpr int kMaxBits = 48;
constexpr int kMaxRank = 24;

struct BitPermParams {
  int tbits;   // bits inside a tile
  int nfree;   // bits selecting the tile
  uint64_t ntiles;
  uint8_t tin[16];   // tile bit k (input order) -> input bit position
  uint8_t trank[16]; // tile bit k (input order) -> LDS position bit
  uint8_t tout[16];  // tile bit k (output order) -> output bit position
  uint8_t fin[kMaxBits];
  uint8_t fout[kMaxBits];
};

__device__ __forceinline__ uint32_t lds_slot(uint32_t s) { return s + (s >> 5); }

// Offsets of tile element e: the input offset, output offset and LDS
// position are OR-sums over e's set bits.  Elements e = t + e_j with t
// (this thread's bits) and e_j (the unrolled iteration's bits, the same in
// every lane) disjoint split each offset into a per-lane term computed once
// and a per-iteration term that lives in scalar registers.  lds_slot is
// additive over such a split: the low five bits of the two terms are disjoint,
// so their sum carries nothing past bit 4.
struct TileOffsets {
  uint64_t in, out;
  uint32_t slot;
};

template <int TBITS>
__device__ __forceinline__ TileOffsets tile_offsets(const BitPermParams& p, uint32_t e, int k0) {
  TileOffsets r{0, 0, 0};
  for (int k = k0; k < TBITS; ++k)
    if ((e >> k) & 1u) {
      r.in |= uint64_t(1) << p.tin[k];
      r.out |= uint64_t(1) << p.tout[k];
      r.slot |= 1u << p.trank[k];
    }
  return r;
}

__device__ __forceinline__ void tile_base(const BitPermParams& p, uint64_t t, uint64_t& bin,
                                          uint64_t& bout) {
  bin = 0;
  bout = 0;
  for (int k = 0; k < p.nfree; ++k)
    if ((t >> k) & 1u) {
      bin |= uint64_t(1) << p.fin[k];
      bout |= uint64_t(1) << p.fout[k];
    }
}

template <int TBITS, int BLOCK>
__global__ __launch_bounds__(BLOCK) void permute_bits_kernel(const float2* __restrict__ src,
                                                             float2* __restrict__ dst,
                                                             BitPermParams p) {
  constexpr int TILE = 1 << TBITS;
  constexpr int PER = TILE / BLOCK;
  static_assert(PER >= 1, "tile smaller than block");
  __shared__ float2 lds[TILE + TILE / 32];

  // Tile-local element e = tid + j*BLOCK.
  const uint32_t tid = threadIdx.x;
  const TileOffsets lane = tile_offsets<TBITS>(p, tid, 0);
  const uint32_t lane_slot = lds_slot(lane.slot);

  for (uint64_t t = blockIdx.x; t < p.ntiles; t += gridDim.x) {
    uint64_t bin, bout;
    tile_base(p, t, bin, bout);
    float2 v[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j)
      v[j] = src[bin + (tile_offsets<TBITS>(p, uint32_t(j) * BLOCK, 0).in | lane.in)];
#pragma unroll
    for (int j = 0; j < PER; ++j)
      lds[lds_slot(tile_offsets<TBITS>(p, uint32_t(j) * BLOCK, 0).slot) + lane_slot] = v[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t ej = uint32_t(j) * BLOCK;
      dst[bout + (tile_offsets<TBITS>(p, ej, 0).out | lane.out)] = lds[lds_slot(ej) + lds_slot(tid)];
    }
    __syncthreads();
  }
}

// Pair variant: each thread moves element pairs, 16 bytes per global access.
// Input bit 0 is tile bit 0, so tile elements e, e+1 (input order) are
// adjacent in memory; output bit 0 is the lowest output bit of the tile, so
// output-order positions o, o+1 are adjacent too.  Needs TBITS >= 2.
template <int TBITS, int BLOCK>
__global__ __launch_bounds__(BLOCK) void permute_pairs_kernel(const float2* __restrict__ src,
                                                              float2* __restrict__ dst,
                                                              BitPermParams p) {
  constexpr int TILE = 1 << TBITS;
  constexpr int PER = TILE / (2 * BLOCK);  // pairs per thread
  static_assert(PER >= 1, "tile smaller than two elements per thread");
  __shared__ float2 lds[TILE + TILE / 32];

  // Pair tid + j*BLOCK covers tile elements e = 2*(tid + j*BLOCK) and e + 1.
  const uint32_t tid = threadIdx.x;
  const TileOffsets lane = tile_offsets<TBITS>(p, 2u * tid, 1);
  const uint32_t slot0 = lds_slot(lane.slot), slot1 = lds_slot(lane.slot | (1u << p.trank[0]));
  const uint32_t rslot = lds_slot(2u * tid);

  for (uint64_t t = blockIdx.x; t < p.ntiles; t += gridDim.x) {
    uint64_t bin, bout;
    tile_base(p, t, bin, bout);
    float4 v[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint64_t off = tile_offsets<TBITS>(p, 2u * uint32_t(j) * BLOCK, 1).in | lane.in;
      v[j] = *reinterpret_cast<const float4*>(src + bin + off);
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t sj = lds_slot(tile_offsets<TBITS>(p, 2u * uint32_t(j) * BLOCK, 1).slot);
      lds[sj + slot0] = make_float2(v[j].x, v[j].y);
      lds[sj + slot1] = make_float2(v[j].z, v[j].w);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const uint32_t ej = 2u * uint32_t(j) * BLOCK;
      const uint32_t r = lds_slot(ej) + rslot;
      const float2 x = lds[r];
      const float2 y = lds[r + 1];
      const uint64_t off = tile_offsets<TBITS>(p, ej, 1).out | lane.out;
      *reinterpret_cast<float4*>(dst + bout + off) = make_float4(x.x, x.y, y.x, y.y);
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------ boxes
// Any dimensions, fewer than 2^31 elements.  Bound by HBM.  A box holds whole
// runs of `run_in` contiguous input and `run_out` contiguous output elements;
// only the runs' starts need mixed-radix digits, from small LDS tables made
// once per block (digits for every element were most of the time), and a
// thread keeps the offsets of its PER elements, the same in every box, in
// registers.  The next box's loads are in flight while a box is stored.
// One thread per element, its loads gathered, 64-bit divisions: 10.8 M
// elements of 16 x 11 x 16 x 3 x 16 x 16 x 5 took 68 us, now 41 (4.2 TB/s);
// 29 M of 5 x 7 x 16 x 3 x 7 x 2 x 11 x 7 x 16 282, now 153.
constexpr int kBoxAxes = 24;
constexpr int kBoxMax = 2048;  // elements of a box
// Below kBoxesFrom, two elements per thread without boxes is faster, it has more
// to run at once.  From there to kSmallUpTo it is where a wave's 64 gathered loads
// share lines: of 40 tensors of 1.1 to 1.9 M elements, the ones that touch 6 to 18
// lines were 1.0 to 1.6 times faster without boxes (8 x 7 x 16 x 4 x 7 x 7 x 8:
// 10.7 -> 6.9 us), two with 28 lines 1.65 and 0.73 times, those with 32 to 64
// lines 0.47 to 0.97 times.
constexpr uint64_t kBoxesFrom = uint64_t(1) << 20, kSmallUpTo = uint64_t(1) << 21;
constexpr int kSmallLines = 20;
struct BoxParams {
  int size;
  int naxes;  // axes with more than one coordinate in a box
  int nfree;  // axes with more than one box
  int run_in, run_out;
  float inv_run_in, inv_run_out;
  uint32_t nboxes;
  // box axes, from the innermost input axis on / from the innermost output axis on
  uint16_t in_dim[kBoxAxes], out_dim[kBoxAxes];
  uint32_t in_step[kBoxAxes], out_step[kBoxAxes];  // input / output stride
  uint16_t slot[kBoxAxes];                         // of in_dim's axis: LDS stride
  // free axes, fastest first: boxes, coordinates per box, start of the last
  // box (flush with the axis's end, so that every box is whole: elements two
  // boxes share are written twice, with the same value), strides
  uint32_t free_n[kBoxAxes], free_block[kBoxAxes], free_last[kBoxAxes];
  uint32_t free_in[kBoxAxes], free_out[kBoxAxes];
};

// Blocks per compute unit: what the registers allow without spilling.
constexpr int box_blocks(int per) { return per <= 5 ? 8 : 5; }

// e / d for e, d <= 2^12 and inv = 1 / d: e + 1/2 is at least 1/2 from a
// multiple of d, far more than the product's rounding moves it.
__device__ __forceinline__ uint32_t box_div(uint32_t e, float inv) {
  return uint32_t((float(e) + 0.5f) * inv);
}

template <int PER>
__global__ __launch_bounds__(256, box_blocks(PER)) void permute_boxes_kernel(const float2* __restrict__ src,
                                                            float2* __restrict__ dst,
                                                            BoxParams p) {
  constexpr int kSize = PER * 256;
  __shared__ float2 lds[kSize + kSize / 32];
  uint2* tab = reinterpret_cast<uint2*>(lds);  // before the first box is staged
  const uint32_t tid = threadIdx.x;
  uint32_t in_off[PER], out_off[PER], slots[PER];
  // input offset and slot of element e
  auto digits_in = [&](uint32_t e) {
    uint2 r{0, 0};
    for (int a = 0; a < p.naxes && e > 0; ++a) {
      const uint32_t d = p.in_dim[a], q = e / d, x = e - q * d;
      e = q;
      r.x += x * p.in_step[a];
      r.y += x * p.slot[a];
    }
    return r;
  };
  const uint32_t runs_in = uint32_t(p.size / p.run_in), runs_out = uint32_t(p.size / p.run_out);
  for (uint32_t i = tid; i < runs_in; i += 256) tab[i] = digits_in(i * p.run_in);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t e = min(tid + j * 256, uint32_t(p.size - 1));
    const uint32_t hi = box_div(e, p.inv_run_in);
    const uint2 start = tab[hi];
    in_off[j] = start.x + (e - hi * p.run_in);
    slots[j] = start.y;
  }
  __syncthreads();
  for (uint32_t i = tid; i < uint32_t(p.run_in); i += 256) tab[i] = digits_in(i);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t e = min(tid + j * 256, uint32_t(p.size - 1));
    slots[j] = lds_slot(slots[j] + tab[e - box_div(e, p.inv_run_in) * p.run_in].y);
  }
  __syncthreads();
  for (uint32_t i = tid; i < runs_out; i += 256) {
    uint32_t e = i * p.run_out, off = 0;
    for (int a = 0; a < p.naxes && e > 0; ++a) {
      const uint32_t d = p.out_dim[a], q = e / d;
      off += (e - q * d) * p.out_step[a];
      e = q;
    }
    tab[i].x = off;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t e = min(tid + j * 256, uint32_t(p.size - 1));
    const uint32_t hi = box_div(e, p.inv_run_out);
    out_off[j] = tab[hi].x + (e - hi * p.run_out);
  }
  __syncthreads();

  auto starts = [&](uint32_t t, uint32_t& bin, uint32_t& bout) {
    bin = bout = 0;
    for (int f = 0; f < p.nfree; ++f) {
      const uint32_t n = p.free_n[f], q = t / n;
      const uint32_t x = min((t - q * n) * p.free_block[f], p.free_last[f]);
      t = q;
      bin += x * p.free_in[f];
      bout += x * p.free_out[f];
    }
  };
  float2 v[PER];
  uint32_t bin, bout;
  auto load = [&]() {
    const float2* s = src + bin;
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (int(tid) + j * 256 < p.size) v[j] = s[in_off[j]];
  };
  uint32_t t = blockIdx.x;
  starts(t, bin, bout);
  load();
  for (;;) {
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (int(tid) + j * 256 < p.size) lds[slots[j]] = v[j];
    __syncthreads();
    float2* d = dst + bout;
    t += gridDim.x;
    const bool more = t < p.nboxes;
    if (more) {
      starts(t, bin, bout);
      load();
    }
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (int(tid) + j * 256 < p.size) d[out_off[j]] = lds[lds_slot(tid + j * 256)];
    if (!more) break;
    __syncthreads();
  }
}

struct GenericParams {
  int rank;
  uint64_t total;
  uint64_t out_dims[kMaxRank];
  uint64_t in_stride_of_out[kMaxRank];  // input stride of output axis k
};

// 2^31 elements and more.
__global__ void permute_generic_kernel(const float2* __restrict__ src, float2* __restrict__ dst,
                                       GenericParams p) {
  uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
  for (; i < p.total; i += stride) {
    uint64_t rem = i, off = 0;
    for (int k = p.rank - 1; k >= 0; --k) {
      const uint64_t d = p.out_dims[k], q = rem / d;
      off += (rem - q * d) * p.in_stride_of_out[k];
      rem = q;
    }
    dst[i] = src[off];
  }
}

// At most kSmallUpTo = 2^21 elements, whose digits single precision
// divides exactly: e + 1/2 is exact, 1 / d and the product are off by 2^-24 each,
// together by less than 1 / (4 d), and (e + 1/2) / d is at least 1 / (2 d) from a
// whole number.  Two elements per thread.  The integer divisions bounded it:
// 0.74 M elements of 16 x 2 x 4 x 11 x 3 x 5 x 7 x 5 11.0 -> 8.5 us, 0.79 M of
// 8 x 16 x 7 x 11 x 5 x 4 x 4 9.2 -> 7.3; below 2^19 a call is bound by its launch.
struct SmallParams {
  int rank;
  uint32_t total;
  uint32_t dim[kMaxRank], step[kMaxRank];  // from the innermost output axis; input strides
  float inv[kMaxRank];
};
__global__ __launch_bounds__(256) void permute_small_kernel(const float2* __restrict__ src,
                                                            float2* __restrict__ dst,
                                                            SmallParams p) {
  const uint32_t i = blockIdx.x * 512 + threadIdx.x;
  uint32_t rem[2] = {i, i + 256}, off[2] = {0, 0};
  for (int k = 0; k + 1 < p.rank; ++k) {
    const uint32_t d = p.dim[k], step = p.step[k];
    const float inv = p.inv[k];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint32_t q = uint32_t((float(rem[u]) + 0.5f) * inv);
      off[u] += (rem[u] - q * d) * step;
      rem[u] = q;
    }
  }
  float2 v[2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
    if (i + 256 * u < p.total) v[u] = src[off[u] + rem[u] * p.step[p.rank - 1]];
#pragma unroll
  for (int u = 0; u < 2; ++u)
    if (i + 256 * u < p.total) dst[i + 256 * u] = v[u];
}

// The box of a permutation of fused axes: dims in input order, perm[k] the
// axis of output position k.  block[a] coordinates of axis a lie in a box.
// Runs of at least `want` elements on either side (or whole tensors), boxes
// of at most kBoxMax elements; `want` starts at 16 (128 bytes) and doubles
// while the box is small: below 1024 elements, or, in tensors of less than
// 2^21, below what leaves 2048 boxes (the blocks the chip holds).
void choose_box(const std::vector<uint64_t>& dims, const std::vector<int>& perm, uint64_t total,
                std::vector<uint64_t>& block) {
  const int r = int(dims.size());
  const uint64_t enough = std::min<uint64_t>(1024, std::max<uint64_t>(256, total / 2048));
  for (uint64_t want = 16; want <= kBoxMax; want *= 2) {
    std::vector<uint64_t> b(r, 1);
    auto grow = [&](auto axis_at) {  // axis_at(i): the i-th axis from the inside
      uint64_t run = 1;
      for (int i = 0; i < r && run < want; ++i) {
        const int a = axis_at(i);
        const uint64_t need = (want + run - 1) / run;
        if (b[a] < dims[a] && b[a] < need) {
          const uint64_t parts = dims[a] < 2 * need ? 1 : dims[a] / need;
          b[a] = (dims[a] + parts - 1) / parts;
        }
        run *= b[a];
        if (b[a] < dims[a]) break;  // the run ends inside this axis
      }
    };
    grow([&](int i) { return r - 1 - i; });
    grow([&](int i) { return perm[r - 1 - i]; });
    uint64_t size = 1;
    for (uint64_t x : b) size *= x;
    if (size > kBoxMax) break;
    block = b;
    if (size >= enough) break;
  }
}

// Lines of 128 bytes that 64 consecutive output elements, from the middle of
// the tensor on, are read from.
int lines_of_a_wave(const std::vector<uint64_t>& dims, const std::vector<int>& perm,
                    uint64_t total) {
  const int r = int(dims.size());
  std::vector<uint64_t> stride(r);
  uint64_t st = 1;
  for (int a = r - 1; a >= 0; st *= dims[a], --a) stride[a] = st;
  uint64_t line[64];
  for (int i = 0; i < 64; ++i) {
    uint64_t e = total / 2 / 64 * 64 + i, off = 0;
    for (int k = r - 1; k >= 0 && e > 0; --k) {
      off += e % dims[perm[k]] * stride[perm[k]];
      e /= dims[perm[k]];
    }
    line[i] = off / 16;
  }
  std::sort(line, line + 64);
  return int(std::unique(line, line + 64) - line);
}

template <int PER>
void launch_boxes(const BoxParams& p, const float2* src, float2* dst, hipStream_t s) {
  const unsigned g = std::min<uint32_t>(p.nboxes, 256 * box_blocks(PER));
  permute_boxes_kernel<PER><<<g, 256, 0, s>>>(src, dst, p);
}

bool is_pow2(uint64_t x) { return x && !(x & (x - 1)); }
int log2u(uint64_t x) { return 63 - __builtin_clzll(x); }

template <int TBITS, int BLOCK>
void launch_bits(const BitPermParams& p, const float2* src, float2* dst, hipStream_t s) {
  uint64_t g = std::min<uint64_t>(p.ntiles, 256 * 16);
  permute_bits_kernel<TBITS, BLOCK><<<unsigned(g), BLOCK, 0, s>>>(src, dst, p);
}

template <int TBITS, int BLOCK>
void launch_pairs(const BitPermParams& p, const float2* src, float2* dst, hipStream_t s) {
  uint64_t g = std::min<uint64_t>(p.ntiles, 256 * 8);
  permute_pairs_kernel<TBITS, BLOCK><<<unsigned(g), BLOCK, 0, s>>>(src, dst, p);
}

}  // namespace

extern "C" int qfx_reorder_c64(qfx_context* ctx, const qfx_c64* src, qfx_c64* dst, int rank,
                               const uint64_t* dims, const int* perm) {
  QFX_CHECK_CTX(ctx);
  if (rank < 0 || rank > 64) return qfx_set_error(QFX_ERR_INVALID, "qfx_reorder_c64: bad rank");
  if (rank > 0 && (!dims || !perm))
    return qfx_set_error(QFX_ERR_INVALID, "qfx_reorder_c64: null dims/perm");
  std::vector<int> seen(rank, 0);
  uint64_t total = 1;
  for (int k = 0; k < rank; ++k) {
    if (perm[k] < 0 || perm[k] >= rank || seen[perm[k]]++)
      return qfx_set_error(QFX_ERR_INVALID, "qfx_reorder_c64: perm is not a permutation");
    if (dims[k] == 0) return QFX_OK;
    total *= dims[k];
  }
  if (!src || !dst) return qfx_set_error(QFX_ERR_INVALID, "qfx_reorder_c64: null data pointer");
  if (src == dst) return qfx_set_error(QFX_ERR_INVALID, "qfx_reorder_c64: src and dst alias");
  QFX_EXTENT(ctx, src, 8.0 * double(total), "qfx_reorder_c64: src");
  QFX_EXTENT(ctx, dst, 8.0 * double(total), "qfx_reorder_c64: dst");

  // Drop unit axes, then fuse axes that remain adjacent in the output.
  std::vector<int> keep_map(rank, -1);
  std::vector<uint64_t> d1;
  for (int a = 0; a < rank; ++a)
    if (dims[a] != 1) {
      keep_map[a] = int(d1.size());
      d1.push_back(dims[a]);
    }
  std::vector<int> p1;
  for (int k = 0; k < rank; ++k)
    if (keep_map[perm[k]] >= 0) p1.push_back(keep_map[perm[k]]);
  // runs of consecutive input axes in output order
  std::vector<std::pair<int, int>> runs;  // (first input axis, length)
  for (size_t k = 0; k < p1.size(); ++k) {
    if (!runs.empty() && runs.back().first + runs.back().second == p1[k])
      runs.back().second++;
    else
      runs.push_back({p1[k], 1});
  }
  const int r = int(runs.size());
  if (r <= 1) return qfx_copy_d2d(ctx, dst, src, total * sizeof(qfx_c64));
  // fused input axes sorted by first input axis
  std::vector<int> order(r);
  std::iota(order.begin(), order.end(), 0);
  std::sort(order.begin(), order.end(),
            [&](int x, int y) { return runs[x].first < runs[y].first; });
  std::vector<int> run_to_in(r);
  for (int i = 0; i < r; ++i) run_to_in[order[i]] = i;
  std::vector<uint64_t> fdims(r);  // fused input dims (input order)
  for (int i = 0; i < r; ++i) {
    uint64_t d = 1;
    for (int a = runs[order[i]].first; a < runs[order[i]].first + runs[order[i]].second; ++a)
      d *= d1[a];
    fdims[i] = d;
  }
  std::vector<int> fperm(r);  // output axis k -> fused input axis
  for (int k = 0; k < r; ++k) fperm[k] = run_to_in[k];

  QfxLaunchScope scope(ctx, QFX_K_PERMUTE, 16.0 * double(total), 0);
  const float2* s2 = reinterpret_cast<const float2*>(src);
  float2* d2 = reinterpret_cast<float2*>(dst);

  bool pow2 = std::all_of(fdims.begin(), fdims.end(), is_pow2);
  if (pow2) {
    // bit positions: input axis a occupies bits [s_a, s_a + b_a)
    std::vector<int> bits(r), in_start(r), out_start(r);
    int nbits = 0;
    for (int a = r - 1; a >= 0; --a) {
      bits[a] = log2u(fdims[a]);
      in_start[a] = nbits;
      nbits += bits[a];
    }
    if (nbits > kMaxBits) return qfx_set_error(QFX_ERR_UNSUPPORTED, "tensor too large");
    int ob_acc = 0;
    for (int k = r - 1; k >= 0; --k) {
      out_start[fperm[k]] = ob_acc;
      ob_acc += bits[fperm[k]];
    }
    std::vector<int> ob(nbits), ib_of_ob(nbits);
    for (int a = 0; a < r; ++a)
      for (int j = 0; j < bits[a]; ++j) ob[in_start[a] + j] = out_start[a] + j;
    for (int i = 0; i < nbits; ++i) ib_of_ob[ob[i]] = i;

    // Tiles of 2^12 elements (6 lowest input bits + 6 lowest output bits)
    // moved as 16-byte pairs for tensors of >= 2^16 elements; 2^10-element
    // tiles of single elements below that.
    const bool pairs = nbits >= 16 && (reinterpret_cast<uintptr_t>(src) % 16 == 0) &&
                       (reinterpret_cast<uintptr_t>(dst) % 16 == 0);
    const int tile_target = pairs ? 12 : 10;
    int tbits = std::min(nbits, tile_target);
    int abits = std::min(tbits, pairs ? 6 : 5);
    std::vector<char> in_t(nbits, 0);
    for (int i = 0; i < abits; ++i) in_t[i] = 1;
    int have = abits;
    for (int o = 0; o < nbits && have < tbits; ++o) {
      int ib = ib_of_ob[o];
      if (!in_t[ib]) {
        in_t[ib] = 1;
        ++have;
      }
    }
    // tbits may still exceed have only if nbits < tbits (not possible)
    BitPermParams p{};
    p.tbits = tbits;
    std::vector<int> tin, touts;
    for (int i = 0; i < nbits; ++i)
      if (in_t[i]) tin.push_back(i);
    for (int i = 0; i < nbits; ++i)
      if (in_t[i]) touts.push_back(ob[i]);
    std::sort(touts.begin(), touts.end());
    for (int k = 0; k < tbits; ++k) {
      p.tin[k] = uint8_t(tin[k]);
      p.trank[k] = uint8_t(std::lower_bound(touts.begin(), touts.end(), ob[tin[k]]) - touts.begin());
      p.tout[k] = uint8_t(touts[k]);
    }
    int nf = 0;
    for (int i = 0; i < nbits; ++i)
      if (!in_t[i]) {
        p.fin[nf] = uint8_t(i);
        p.fout[nf] = uint8_t(ob[i]);
        ++nf;
      }
    p.nfree = nf;
    p.ntiles = uint64_t(1) << nf;
    if (pairs) {
      launch_pairs<12, 256>(p, s2, d2, ctx->stream);
    } else switch (tbits) {
      case 10: launch_bits<10, 256>(p, s2, d2, ctx->stream); break;
      case 9: launch_bits<9, 256>(p, s2, d2, ctx->stream); break;
      case 8: launch_bits<8, 256>(p, s2, d2, ctx->stream); break;
      case 7: launch_bits<7, 128>(p, s2, d2, ctx->stream); break;
      case 6: launch_bits<6, 64>(p, s2, d2, ctx->stream); break;
      case 5: launch_bits<5, 32>(p, s2, d2, ctx->stream); break;
      case 4: launch_bits<4, 16>(p, s2, d2, ctx->stream); break;
      case 3: launch_bits<3, 8>(p, s2, d2, ctx->stream); break;
      case 2: launch_bits<2, 4>(p, s2, d2, ctx->stream); break;
      default: launch_bits<1, 2>(p, s2, d2, ctx->stream); break;
    }
  } else if (total >= kBoxesFrom && total < (uint64_t(1) << 31) && r <= kBoxAxes &&
             (total > kSmallUpTo || lines_of_a_wave(fdims, fperm, total) > kSmallLines)) {
    std::vector<uint64_t> block(r, 1), in_stride(r), out_stride(r);
    choose_box(fdims, fperm, total, block);
    uint64_t st = 1;
    for (int a = r - 1; a >= 0; st *= fdims[a], --a) in_stride[a] = st;
    st = 1;
    for (int k = r - 1; k >= 0; st *= fdims[fperm[k]], --k) out_stride[fperm[k]] = st;
    BoxParams p{};
    p.size = 1;
    p.nboxes = 1;
    std::vector<int> slot(r, 0);
    for (int k = r - 1; k >= 0; --k) {  // output order, innermost first
      const int a = fperm[k];
      const uint64_t boxes = (fdims[a] + block[a] - 1) / block[a];
      if (boxes > 1) {
        p.free_n[p.nfree] = uint32_t(boxes);
        p.free_block[p.nfree] = uint32_t(block[a]);
        p.free_last[p.nfree] = uint32_t(fdims[a] - block[a]);
        p.free_in[p.nfree] = uint32_t(in_stride[a]);
        p.free_out[p.nfree] = uint32_t(out_stride[a]);
        ++p.nfree;
        p.nboxes *= uint32_t(boxes);
      }
      if (block[a] > 1) {
        p.out_dim[p.naxes] = uint16_t(block[a]);
        p.out_step[p.naxes] = uint32_t(out_stride[a]);
        slot[a] = p.size;
        p.size *= int(block[a]);
        ++p.naxes;
      }
    }
    int i = 0;
    for (int a = r - 1; a >= 0; --a) {
      if (block[a] == 1) continue;
      p.in_dim[i] = uint16_t(block[a]);
      p.in_step[i] = uint32_t(in_stride[a]);
      p.slot[i] = uint16_t(slot[a]);
      ++i;
    }
    // contiguous runs: the innermost axes up to the first that is not whole
    auto run = [&](auto axis_at) {
      uint64_t n = 1;
      for (int j = 0; j < r; ++j) {
        n *= block[axis_at(j)];
        if (block[axis_at(j)] < fdims[axis_at(j)]) break;
      }
      return int(n);
    };
    p.run_in = run([&](int j) { return r - 1 - j; });
    p.run_out = run([&](int j) { return fperm[r - 1 - j]; });
    p.inv_run_in = 1.f / float(p.run_in);
    p.inv_run_out = 1.f / float(p.run_out);
    switch ((p.size + 255) / 256) {
      case 1: launch_boxes<1>(p, s2, d2, ctx->stream); break;
      case 2: launch_boxes<2>(p, s2, d2, ctx->stream); break;
      case 3: launch_boxes<3>(p, s2, d2, ctx->stream); break;
      case 4: launch_boxes<4>(p, s2, d2, ctx->stream); break;
      case 5: launch_boxes<5>(p, s2, d2, ctx->stream); break;
      case 6: launch_boxes<6>(p, s2, d2, ctx->stream); break;
      case 7: launch_boxes<7>(p, s2, d2, ctx->stream); break;
      default: launch_boxes<8>(p, s2, d2, ctx->stream); break;
    }
  } else if (total <= kSmallUpTo && r <= kMaxRank) {
    SmallParams p{};
    p.rank = r;
    p.total = uint32_t(total);
    std::vector<uint32_t> in_stride(r);
    uint32_t st = 1;
    for (int a = r - 1; a >= 0; st *= uint32_t(fdims[a]), --a) in_stride[a] = st;
    for (int k = 0; k < r; ++k) {
      const int a = fperm[r - 1 - k];
      p.dim[k] = uint32_t(fdims[a]);
      p.step[k] = in_stride[a];
      p.inv[k] = 1.f / float(fdims[a]);
    }
    permute_small_kernel<<<unsigned((total + 511) / 512), 256, 0, ctx->stream>>>(s2, d2, p);
  } else {
    if (r > kMaxRank) return qfx_set_error(QFX_ERR_UNSUPPORTED, "rank too large");
    GenericParams p{};
    p.rank = r;
    p.total = total;
    std::vector<uint64_t> in_stride(r);
    uint64_t st = 1;
    for (int a = r - 1; a >= 0; --a) {
      in_stride[a] = st;
      st *= fdims[a];
    }
    for (int k = 0; k < r; ++k) {
      p.out_dims[k] = fdims[fperm[k]];
      p.in_stride_of_out[k] = in_stride[fperm[k]];
    }
    uint64_t g = std::min<uint64_t>((total + 255) / 256, 65536);
    permute_generic_kernel<<<unsigned(g), 256, 0, ctx->stream>>>(s2, d2, p);
  }
  QFX_HIP(hipGetLastError());
  return QFX_OK;
}
