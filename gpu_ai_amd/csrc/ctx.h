// ctx.h -- the context object behind mi_ctx (internal to the library).
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <string>
#include <vector>

#include "gpuai/mi_playout.h"

namespace gpuai {
struct DevBuf {
  void *ptr = nullptr;
  size_t bytes = 0;
};
// Pinned host memory (hipHostMalloc): copies from and to it run asynchronously on the copy
// engines, where copies of pageable memory are staged through the runtime's own buffers.
struct HostBuf {
  void *ptr = nullptr;
  size_t bytes = 0;
};
}  // namespace gpuai

// Default launch shape: 64-thread blocks, 12 per CU (3 waves per SIMD), queue refill, defer_min
// 16.  A small batch spreads over many CUs this way instead of sharing a few SIMDs; larger ones take
// batch_shape's.
constexpr mi_tuning kDefaultTuning = {64u, 12u, MI_REFILL_QUEUE, 16u};

// Whether a tuning asks for the defaults: a program that saves a context's tuning and sets it again
// later gets its routes by size back.
constexpr bool is_default(const mi_tuning &t) {
  return t.block_size == kDefaultTuning.block_size &&
         t.blocks_per_cu == kDefaultTuning.blocks_per_cu && t.refill == kDefaultTuning.refill &&
         t.defer_min == kDefaultTuning.defer_min;
}

// Launch-shape table: the fastest shape the autotuner measured for a policy, a batch-size bucket
// (floor(log2(playouts))) and a refill policy; kernel_ms < 0 marks an empty entry.
constexpr uint32_t kTuneBuckets = 32;
struct TuneEntry {
  mi_tuning tuning = {0u, 0u, 0u, 0u};  // of one lane per game
  float kernel_ms = -1.f;
  float wave_ms = -1.f;   // the same batch with one wave per game; < 0: not measured (too large)
  uint32_t playouts = 0;  // size of the batch it was measured on
};

struct mi_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev_start = nullptr, ev_stop = nullptr;
  mi_tuning tuning = kDefaultTuning;  // as given, or the fastest of mi_autotune's batch
  bool shaped = false;  // `tuning` was given: batches of every size take it unless the table has theirs
  TuneEntry tune_table[3][kTuneBuckets][2];  // [policy][bucket][refill]
  uint32_t cus = 0, wave = 64, clock_khz = 0;
  gpuai::DevBuf pos, offs, winners, plies, hashes, work, tallies, moves, counts, keys;
  // longest-first order of the uploaded batch (see upload_batch): positions permuted into it,
  // the original index of each, and (uneven counts) prefix offsets in that order
  gpuai::DevBuf ord_pos, order, ord_offs;
  bool ordered = false;
  std::vector<uint32_t> host_order, host_ord_offs;
  std::vector<mi_pos> host_ord_pos;
  // pinned staging of mi_stage and of batches too large for the packed route: positions |
  // offsets on the way in, work words | winners on the way back.  Rewritten only while the
  // stream is idle.
  gpuai::HostBuf h_in, h_back;
  // the packed batch of mi_run_playouts (inputs | work words | winners in one device block and
  // its pinned mirror, one copy each way), and the work words and results of start positions; both
  // wait for the stream before they return
  gpuai::DevBuf batch;
  gpuai::HostBuf h_batch;
  // staged batch
  uint32_t staged_npos = 0, staged_per_pos = 0, staged_total = 0;
  bool staged = false, staged_offs = false;
  std::vector<uint32_t> host_offs;
  std::string last_error;
  std::mutex mu;
};

namespace gpuai {
namespace ctxutil {
// Records `msg` as the context's last error and returns `code`.
int fail(mi_ctx *ctx, int code, const std::string &msg);
// Records a HIP failure and returns MI_ERR_DEVICE or MI_ERR_OUT_OF_MEMORY.
int hip_fail(mi_ctx *ctx, hipError_t e, const char *what);
// Grows a device buffer to at least `bytes`.
int ensure(mi_ctx *ctx, DevBuf &b, size_t bytes);
// Grows a pinned host buffer to at least `bytes` (the caller's stream must be idle).
int ensure_host(mi_ctx *ctx, HostBuf &b, size_t bytes);
// Batch-size bucket of the launch-shape table: floor(log2(total)).
uint32_t tune_bucket(uint64_t total);
// The launch shape of a batch of `total` playouts that the table has none for: the context's, when
// one was given.  Otherwise a workgroup per CU with the waves that the batch fills, up to 12 (3 a
// SIMD), and 16 from two games a lane on: waves of a workgroup hand their last games over to each
// other (playout_kernels.hip), and 16 hide each other's latencies better but have more last games.
// Against 64x12, in ms: 1024x1024 0.546 -> 0.480 with 16 waves (0.499 with 12), 64x4096 0.243 ->
// 0.210 with 12 (0.216 with 16), 65536x256 4.76 -> 4.45 with 16 (4.77 with 12).  Up to four waves a CU
// there is nothing to hand over, and 64-thread blocks it is.  The noisy heuristic waits for 24 plies:
// its walk phases cost much the same for any number of them (noisy-1024x1024 0.582, 0.564, 0.552,
// 0.539 and 0.546 ms at 12, 16, 20, 24 and 32; the other policies are level from 16 on).  What
// mi_autotune measured on one batch holds for that batch's bucket: at 65,536 random playouts the shape
// of 1,048,576 takes 0.203 ms, the size's own 0.139.  total 0: the size is not known here, and the
// context's tuning it is.
mi_tuning batch_shape(const mi_ctx *ctx, uint32_t policy, uint64_t total);
// The launch shape of a batch with one lane per game: the table's entry for its policy and bucket
// (the faster refill, or refill `only` when it is 0 or 1), else batch_shape's.
mi_tuning shape_for(const mi_ctx *ctx, uint32_t policy, uint64_t total, int only = -1);
// Whether a batch runs with one wave per game instead (`only` as for shape_for).
bool wave_batch(const mi_ctx *ctx, uint32_t policy, uint64_t total, int only = -1);
}  // namespace ctxutil
// Looks up the device address of the allocation-free entry point's scratch array for the
// context's device (once per device; the device must be current).
int noalloc_setup(mi_ctx *ctx);
}  // namespace gpuai

#define MI_HIP(ctx, call)                                                 \
  do {                                                                    \
    hipError_t e_ = (call);                                               \
    if (e_ != hipSuccess) return gpuai::ctxutil::hip_fail(ctx, e_, #call); \
  } while (0)
