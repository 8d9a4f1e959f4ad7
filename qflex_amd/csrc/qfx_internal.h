// Internal declarations shared by the qfx HIP translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <array>
#include <cstdint>
#include <map>
#include <string>
#include <vector>

#include "qfx.h"

struct QfxProfRec {
  int cls;
  hipEvent_t start, stop;
  double bytes, flops;
};

struct qfx_context {
  int device = 0;
  hipStream_t stream = nullptr;
  // Arena: chunks from hipMalloc, bump-allocated; freed blocks are kept in
  // per-size free lists (sizes rounded to the arena's size classes).
  struct Chunk {
    char* base;
    size_t size, used;
  };
  std::vector<Chunk> chunks;
  size_t chunk_bytes = size_t(1) << 30;
  std::map<size_t, std::vector<void*>> free_lists;
  std::map<void*, size_t> live;  // pointer -> rounded size
  // Some of `live` by address, for operands that start their block (nearly
  // all): the map's search took 50 ns of every check, 30 of the 865 us of a
  // 4 x 4 circuit of depth 16 once its grouped products were checked.
  struct LiveBlock {
    const void* p;
    size_t size;
  };
  std::array<LiveBlock, 1024> live_at{};
  LiveBlock& live_slot(const void* p) {
    return live_at[(reinterpret_cast<uintptr_t>(p) >> 8) % live_at.size()];
  }
  size_t in_use = 0;
  // Device workspace for split reductions (grows on demand).
  void* work = nullptr;
  size_t work_bytes = 0;
  // Recorded graphs replay with the workspace's address: one that a recorded
  // call took stays out of the arena when it is outgrown, until no graph of
  // the context is left.
  int graphs = 0;                  // recorded and not destroyed
  bool work_recorded = false;      // a recorded call took `work`
  std::vector<void*> kept_works;   // outgrown ones
  // Partial sums of recorded FP32 products that the reserved workspace does
  // not hold: kFixedScratchBytes of the arena, from the first qfx_graph_begin
  // on (a replay may come at any time after it).
  void* record_scratch = nullptr;
  // Profiling.
  bool profiling = false;
  std::vector<QfxProfRec> pending;
  std::vector<hipEvent_t> event_pool;
  uint64_t launches[QFX_K_NUM_CLASSES] = {};
  double ms[QFX_K_NUM_CLASSES] = {};
  double bytes[QFX_K_NUM_CLASSES] = {};
  double flops[QFX_K_NUM_CLASSES] = {};
  hipEvent_t timer_start = nullptr, timer_stop = nullptr;
  // Autotuner of the large-tile GEMM layouts: (precision, operand form, m,
  // n, k) -> layout, measured on first use while enabled.
  bool capturing = false;  // between qfx_graph_begin and qfx_graph_end
  // Pinned staging area of qfx_copy_h2d_async: filled from offset
  // stage_off on, rewound only after the stream has been synchronized.
  // The copies are batched: `uploads` lists the staged copies not yet
  // launched (destination, offset in the staging area, bytes), `upload_at`
  // their destination ranges (start -> end); one scatter launch moves them
  // all before the next call that puts work on the stream.
  unsigned char* stage = nullptr;
  void* stage_dev = nullptr;  // the staging area's device address
  size_t stage_off = 0;
  struct Upload {
    uint64_t dst, src_off, bytes;
  };
  std::vector<Upload> uploads;
  std::map<uintptr_t, uintptr_t> upload_at;
  int cus = 0;  // compute units of the device (0: not yet read)
  bool autotune = false;
  std::map<std::array<uint64_t, 5>, int> tuned;
  hipEvent_t tune_ev[2] = {nullptr, nullptr};
  // This device's copy of the library's fixed scratch array (the device
  // address hipGetSymbolAddress returned at context creation), and whether
  // the call in progress must take its workspace from it instead of the
  // growable workspace above (qfx_cgemm_noalloc_c64).
  void* fixed_scratch = nullptr;
  bool use_fixed_scratch = false;
};

// Size of the fixed scratch array (one copy per GPU, held until the process
// ends) that the entry point allocating nothing uses as its workspace.
constexpr size_t kFixedScratchBytes = QFX_NOALLOC_SCRATCH_BYTES;

// Error plumbing: every entry point returns a status and records a message.
int qfx_set_error(int status, const std::string& msg);
int qfx_hip_error(hipError_t e, const char* what);

#define QFX_HIP(call)                                      \
  do {                                                     \
    hipError_t e_ = (call);                                \
    if (e_ != hipSuccess) return qfx_hip_error(e_, #call); \
  } while (0)

// Launches the batched staged uploads (qfx_copy_h2d_async) on the stream.
int qfx_flush_uploads(qfx_context* ctx);

// Start of every entry point that puts work on the stream, reads device
// memory from the host or waits for the stream: staged uploads go first.
#define QFX_CHECK_CTX(ctx)                                                \
  do {                                                                    \
    if (!(ctx)) return qfx_set_error(QFX_ERR_INVALID, "null context");    \
    if (!(ctx)->uploads.empty()) {                                        \
      const int flush_status_ = qfx_flush_uploads(ctx);                   \
      if (flush_status_ != QFX_OK) return flush_status_;                  \
    }                                                                     \
  } while (0)

// Entry points that only keep books (arena, profiling records, tables).
#define QFX_CHECK_CTX_NO_FLUSH(ctx)                                       \
  do {                                                                    \
    if (!(ctx)) return qfx_set_error(QFX_ERR_INVALID, "null context");    \
  } while (0)

// Bracket a launch with profiling events (no-op unless profiling is on).
struct QfxLaunchScope {
  qfx_context* ctx;
  QfxProfRec rec;
  bool active;
  QfxLaunchScope(qfx_context* c, int cls, double bytes, double flops);
  ~QfxLaunchScope();
};

// A recorded sequence of stream work (qfx_graph_begin / qfx_graph_end).
struct qfx_graph {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  qfx_context* ctx = nullptr;
};

#define QFX_NOT_CAPTURING(ctx, what)                                                        \
  if ((ctx)->capturing)                                                                     \
  return qfx_set_error(QFX_ERR_INVALID, std::string(what) +                                 \
                                            ": not allowed while a graph is being recorded")

// Device workspace of at least `bytes` (reused across calls on the stream).
int qfx_workspace(qfx_context* ctx, size_t bytes, void** out);

// Host-side guard before a launch: when p lies in one of the context's arena
// chunks, [p, p + bytes) must lie inside one live (allocated, not freed)
// block; otherwise QFX_ERR_INVALID with a message naming `what`.  Memory
// outside the arena (allocated by the caller) is not checked.
int qfx_check_extent(qfx_context* ctx, const void* p, double bytes, const char* what);
#define QFX_EXTENT(ctx, p, bytes, what)                        \
  do {                                                         \
    const int extent_status_ = qfx_check_extent(ctx, p, bytes, what); \
    if (extent_status_ != QFX_OK) return extent_status_;       \
  } while (0)

// Offset of matrix index idx under a digit map (see qfx_index_map).  The
// map is a bit permutation, so for i0 a multiple of 2^b and d < 2^b,
// offset(i0 + d) = offset(i0) + offset(d).
__device__ __forceinline__ uint64_t map_offset(const qfx_index_map& d, uint64_t idx) {
  uint64_t off = 0;
  for (int j = 0; j < d.ndigits; ++j) {
    const int b = d.bits[j];
    off += (idx & ((uint64_t(1) << b) - 1)) << d.shift[j];
    idx >>= b;
  }
  return off;
}

// The last of `count` > 0 entries of a grouped launch whose first index (at
// `first`, stride `bytes`, increasing, 0 at entry 0) is <= t.  Called by whole
// waves: 64 entries are probed at a time, so 192 entries take two dependent
// loads, where a binary search takes eight (4 us of each block's life).
__device__ __forceinline__ int group_entry(const uint64_t* first, size_t bytes, int count,
                                           uint64_t t) {
  const int lane = threadIdx.x & 63;
  int lo = 0, n = count;
  while (n > 1) {
    const int step = (n + 63) / 64;
    const int i = lane * step;
    const bool le = i < n && *reinterpret_cast<const uint64_t*>(
                                 reinterpret_cast<const char*>(first) + size_t(lo + i) * bytes) <= t;
    const int c = __popcll(__ballot(le)) - 1;  // the last probed entry <= t
    lo += c * step;
    n = min(step, n - c * step);
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

// Tile of block b of `tiles`: each of the 8 XCDs (which take blocks in turn)
// gets a contiguous range of them, so that the column tiles that share rows
// of A read them through one L2.
__device__ __forceinline__ uint64_t xcd_tile(uint64_t b, uint64_t tiles) {
  const uint64_t q = tiles / 8, r = tiles % 8, x = b % 8;
  return x * q + (x < r ? x : r) + b / 8;
}

// Blocks of 256 threads along one dimension of a launch: a grid dimension
// holds less than 2^32 threads, and a launch of more is cut without an error.
constexpr uint64_t kMaxBlocks = (uint64_t(1) << 24) - 1;

// A short problem list as a kernel argument: no workspace and no upload launch
// before the grouped one (5 us of a call).
constexpr int kArgProblems = 32;
template <class P>
struct ArgList {
  P p[kArgProblems];
};

// Matrix-vector products of qfx_gemv.hip (pointers checked by the caller,
// m, k > 0): y[m] = A[m x k] . x, without device scratch, and y[k] =
// sum_r x[r] A[r][.].
int qfx_launch_gemv_n(qfx_context* ctx, uint64_t m, uint64_t k, const float2* A, const float2* x,
                      float2* y);
int qfx_launch_gemv_t(qfx_context* ctx, uint64_t m, uint64_t k, const float2* A, const float2* x,
                      float2* y);

// FP32 MFMA products of qfx_f32.hip, any m, n, k that fit (pointers checked by
// the caller); maps = {a_rows, a_cols, b_rows, b_cols} or null for row-major,
// a_mfast / b_kfast the operands' contiguous direction.  Products of few
// outputs are split over k through the workspace, at most kFixedScratchBytes
// of it.  Where a sequence being recorded has reserved too little they take
// the context's record_scratch, or are refused with needs_reservation.  The
// splits depend on m, n and k alone, so recorded and eager bits are equal.
bool qfx_f32_fits(uint64_t m, uint64_t n, uint64_t k);
// The products of a grouped call that would run there, `which` of them, in one
// launch per tile (row-major operands, pointers checked).
int qfx_launch_f32_grouped(qfx_context* ctx, const qfx_gemm_desc* descs,
                           const std::vector<int>& which);
// A grouped launch's problem list to the device, through the staged uploads.
int qfx_upload_problems(qfx_context* ctx, void* dev, const void* host, size_t bytes);
double qfx_f32_time(uint64_t m, uint64_t n, uint64_t k);  // estimate of its kernels, in us
int qfx_launch_f32(qfx_context* ctx, const float2* A, const float2* B, float2* C, uint64_t m,
                   uint64_t n, uint64_t k, const qfx_index_map* maps, bool a_mfast,
                   bool b_kfast, bool needs_reservation);

// FP8 (E4M3, per-128x128-tile power-of-two scales) complex GEMM of
// qfx_fp8.hip: whether the shape is large enough for its tiles, and the
// launch (maps = {a_rows, a_cols, b_rows, b_cols} or null for row-major).
bool qfx_fp8_applies(uint64_t m, uint64_t n, uint64_t k);
int qfx_cgemm_fp8(qfx_context* ctx, const float2* A, const float2* B, float2* C, uint64_t m,
                  uint64_t n, uint64_t k, const qfx_index_map* maps);
