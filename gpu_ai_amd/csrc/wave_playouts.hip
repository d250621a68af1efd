// wave_playouts.hip -- gfx950 kernel for small playout batches: one wave64 plays one game.
//
// A batch of a few thousand playouts leaves most lanes of the chip idle whatever the layout, and
// with a game per lane (k_playouts) it lasts as long as its longest game, some 150 plies at the
// latency of one wave: about 300 vector instructions, nine cycles each, for any number of games in
// the wave.  Here a ply is spread over the wave's lanes (wave_play.h), so the longest game ends
// several times sooner; per game its instructions are spent by a whole wave, so large batches stay
// with k_playouts (ctxutil::wave_batch).
#include <hip/hip_runtime.h>

#include "checkers.h"
#include "kernels.h"
#include "wave_play.h"

namespace gpuai {

namespace {

using namespace wave;

// Index of the last of n >= 1 ascending values that is <= g (values[0] <= g), by the whole wave:
// each round looks at 64 evenly spaced values of what is left.
__device__ __forceinline__ uint32_t last_not_above(const uint32_t *values, uint32_t n, uint32_t g,
                                                   uint32_t lane) {
  uint32_t lo = 0;
  while (n > 1u) {
    const uint32_t step = (n + 63u) / 64u;
    const uint32_t i = lane * step;
    const uint64_t below = __ballot(i < n && values[lo + i] <= g);
    const uint32_t at = ((uint32_t)__popcll(below) - 1u) * step;
    lo += at;
    n = n - at < step ? n - at : step;
  }
  return lo;
}

template <uint32_t POLICY>
__global__ void __launch_bounds__(kWaveBlock) k_playouts_wave(PlayoutArgs a) {
  if (a.desc) {  // graph replays and allocation-free launches: the batch lives in device memory
    const LaunchDesc *d = a.desc;
    a.npos = d->npos;
    a.total = d->total;
    a.seed = d->seed;
    a.epoch = d->epoch;
    const char *base = (const char *)d;
    if (d->pos_at) a.pos = (const mi_pos *)(base + d->pos_at);
    if (d->offs_at) a.offs = (const uint32_t *)(base + d->offs_at);
    a.keys = d->keys_at ? (const uint32_t *)(base + d->keys_at) : nullptr;
  }
  const uint32_t game = blockIdx.x;
  if (game >= a.total) return;
  const uint32_t lane = threadIdx.x;
  // position p and playout j of this game
  uint32_t p, j;
  if (a.offs) {
    p = last_not_above(a.offs, a.npos, game, lane);
    j = game - uniform(a.offs[p]);
  } else if (a.per_pos_shift < 32u) {
    p = game >> a.per_pos_shift;
    j = game & (a.per_pos - 1u);
  } else {
    p = game / a.per_pos;
    j = game % a.per_pos;
  }
  const mi_pos q = a.pos[p];
  const uint32_t key = a.keys ? uniform(a.keys[p]) : p;
  ck::Lane L = ck::lane_from_abs(uniform(q.p1), uniform(q.p2), uniform(q.kings),
                                 uniform(q.turn), uniform(q.counter));
  uint32_t ply = 0, maxn = 0;
  play<POLICY>(L, geometry(lane), {j, ck::TAG_PLAYOUT, a.epoch, a.seed, key}, ply, maxn);
  if (lane == 0u) {
    a.winners[game] = (int8_t)(L.counter < 50u ? (int32_t)(L.turn ^ 1u) : -1);
    WorkWords::QueueLine &line = a.work->queue[game % kSlabs];
    atomicAdd(&line.plies, (unsigned long long)ply);
    atomicMax(&line.max_moves, maxn);
  }
}

}  // namespace

hipError_t launch_playouts_wave(const PlayoutArgs &args, uint32_t policy, uint32_t games,
                                hipStream_t stream) {
  const dim3 grid(games), block(kWaveBlock);
  if (policy == MI_POLICY_RANDOM)
    hipLaunchKernelGGL(k_playouts_wave<MI_POLICY_RANDOM>, grid, block, 0, stream, args);
  else if (policy == MI_POLICY_HEURISTIC)
    hipLaunchKernelGGL(k_playouts_wave<MI_POLICY_HEURISTIC>, grid, block, 0, stream, args);
  else
    hipLaunchKernelGGL(k_playouts_wave<MI_POLICY_HEURISTIC_NOISY>, grid, block, 0, stream, args);
  return hipGetLastError();
}

}  // namespace gpuai
