// playout_kernels.hip -- gfx950 kernels of the playout engine.
//
// k_playouts is a persistent kernel: each lane of a wave64 runs one playout at a time with the
// position in VGPRs (ck::Lane) and, when its game ends, takes the next playout index.  New
// playouts start only on wave iterations that are multiples of four, where the Philox4x32-10 call
// that yields the next four words runs for the whole wave (one call per four plies instead of a
// divergent call on almost every iteration).  The kernel is bound by the issue of vector
// instructions (every integer instruction, multiplications included, takes four cycles of a SIMD;
// only reciprocals take longer), so what a ply would compute from small operands -- the factor of
// r mod n, the j-th slot of a square, a move's masks -- and its Philox words are read from LDS,
// one issue slot each, flags of the lanes are wave masks in scalar registers (355 -> 269 vector
// instructions per wave iteration on random-1024x1024, 0.778 -> 0.629 ms), a walk phase takes
// every origin's capture tree at once (ck::capture_trees; 0.577 ms), and all lanes look at their
// position, whatever they hold, so that which of them wait, play or are done are comparisons
// straight into wave masks instead of flags carried out of branches (0.525 ms).  Refill policy
// MI_REFILL_QUEUE claims playout indices for the whole wave in multiples of kChunk from its slab's
// device counter (one atomic per claim, broadcast with a lane read; slabs are described in
// kernels.h), MI_REFILL_STATIC strides lanes over the index space without atomics.
#include <hip/hip_runtime.h>

#include "checkers.h"
#include "kernels.h"
#include "wave_play.h"

namespace gpuai {

namespace {

// Queue claims are made in multiples of kChunk playouts (a wave holds at most one partly used
// claim).  With one counter per slab in a line of its own, claims of 16 beat 32 by about 1%
// (less unplayed work held when a slab runs dry); on a single shared counter, 16 had lost 9% to
// the contention of twice as many atomics on one line.  Each claim is a device atomic, which
// travels to memory as a 32-byte request (random-1024x1024: about 65,500 per launch, twice the
// winners' bytes in the write-request counters).  Workgroup pools in LDS, refilled by guided
// claims from the slab counter, cut that to about 5,000 but cost 5-9% of the launch in
// instructions on the refill path, which this VALU-bound loop cannot hide; claims stay per wave.
constexpr uint32_t kChunk = 16;

__device__ __forceinline__ uint32_t lane_rank(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Whether this lane is in a wave mask.
__device__ __forceinline__ bool lane_in(uint64_t mask) {
  return __builtin_amdgcn_inverse_ballot_w64(mask);
}

// The lanes of the wave in the lane logic that it shares with the host (ck::OneLane).
struct WaveLanes {
  typedef uint64_t Mask;
  static __device__ __forceinline__ Mask where(bool x) { return __ballot(x); }
  static __device__ __forceinline__ bool in(Mask m) { return lane_in(m); }
};

__device__ __forceinline__ uint32_t uniform(uint32_t x) {
  return __builtin_amdgcn_readfirstlane(x);
}

__device__ __forceinline__ uint64_t uniform64(uint64_t x) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
  return (uint64_t)hi << 32 | lo;
}

__device__ __forceinline__ uint64_t rotate_right(uint64_t x, uint32_t n) {
  return x >> n | x << ((64u - n) & 63u);
}

__device__ __forceinline__ void clear_work(WorkWords *work) {
  if (threadIdx.x < kSlabs) {
    work->queue[threadIdx.x].next = 0;
    work->queue[threadIdx.x].max_moves = 0;
    work->queue[threadIdx.x].plies = 0ull;
  }
  if (threadIdx.x == 0) {
    work->max_moves = 0;
    work->overflow = 0;
    work->plies = 0ull;
  }
}

__global__ void k_reset(WorkWords *work) { clear_work(work); }

// Uploads a packed batch (LaunchDesc and its sections, 16-byte words) from pinned host memory and
// clears the work words, in one launch.  A copy command before the graph and a launch to clear the
// words took 42 us until the playouts began (504 KB: 15 of them the copy); with this kernel in the
// graph a replay of 21000x3 takes 213 us instead of 231.
__global__ void __launch_bounds__(kStageBlock) k_stage(const LaunchDesc *from, LaunchDesc *to,
                                                       WorkWords *work) {
  if (blockIdx.x == 0) clear_work(work);
  const uint32_t words = from->words;
  for (uint32_t i = blockIdx.x * kStageBlock + threadIdx.x; i < words; i += kStageGrid * kStageBlock)
    ((uint4 *)to)[i] = ((const uint4 *)from)[i];
}

// Queue index of slab-local index c of slab s of ns (blocks of kSlabBlock dealt round-robin).
__device__ __forceinline__ uint32_t slab_index(uint32_t c, uint32_t s, uint32_t ns) {
  return (((c / kSlabBlock) * ns + s) * kSlabBlock) | (c % kSlabBlock);
}

// Position p, playout j and result slot `out` of the playout with queue index g, and the
// position itself.
__device__ __forceinline__ void locate(const PlayoutArgs &a, uint32_t g, uint32_t &p, uint32_t &j,
                                       uint32_t &out, mi_pos &q) {
  const uint32_t *offs = a.order ? a.ord_offs : a.offs;
  uint32_t r;
  if (offs) {
    uint32_t lo = 0, hi = a.npos;
    while (hi - lo > 1u) {
      uint32_t mid = (lo + hi) >> 1;
      if (offs[mid] <= g) lo = mid; else hi = mid;
    }
    r = lo;
    j = g - offs[lo];
  } else if (a.per_pos_shift < 32u) {
    r = g >> a.per_pos_shift;
    j = g & (a.per_pos - 1u);
  } else {
    ck::divmod_u32(g, a.per_pos, r, j);
  }
  if (a.order) {  // two independent loads
    p = a.order[r];
    q = a.ord_pos[r];
    out = a.offs ? a.offs[p] + j : p * a.per_pos + j;
  } else {
    p = r;
    q = a.pos[r];
    out = g;
  }
}

// The lane logic's lookups (ck::Direct's functions) from LDS, filled once per workgroup.
struct LdsTables {
  uint32_t factor[ck::kModMax + 1];
  uint16_t nth8[64];  // a slot << 8
  uint8_t nth[64];
  uint32_t path[32];
  uint2 move[512];

  __device__ void fill() {
    for (uint32_t i = threadIdx.x; i < 512u; i += blockDim.x) {
      uint2 m;
      ck::move_masks(i, m.x, m.y);
      move[i] = m;
    }
    for (uint32_t i = threadIdx.x; i <= ck::kModMax; i += blockDim.x) factor[i] = ck::mod_factor(i);
    if (threadIdx.x < 32u) path[threadIdx.x] = ck::path_word(threadIdx.x);
    if (threadIdx.x < 64u) {
      const uint32_t sl = ck::nth_slot(threadIdx.x >> 2, threadIdx.x & 3u);
      nth[threadIdx.x] = (uint8_t)sl;
      nth8[threadIdx.x] = (uint16_t)(sl << 8);
    }
  }
};

struct Lookup {
  const LdsTables &t;
  __device__ uint32_t mod(uint32_t r, uint32_t n) const { return ck::mod_by(r, n, t.factor[n]); }
  __device__ uint32_t kth(uint32_t m, uint32_t j) const { return t.nth[m * 4u + j]; }
  __device__ uint32_t path(uint32_t i) const { return t.path[i]; }
  __device__ uint32_t slot8(uint32_t y, uint32_t j) const {  // bytes weigh 4, 8, 16 and 32
    return t.nth8[__builtin_amdgcn_udot4(y, 0x20100804u, j, false)];
  }
  __device__ void move(uint32_t i, uint32_t &flip, uint32_t &removed) const {
    const uint2 m = *(const uint2 *)((const char *)t.move + i);
    flip = m.x;
    removed = m.y;
  }
};

// Philox words of a wave's lanes, two blocks of four per lane: word w of a lane's stream sits in
// row w & 7 (64 lanes wide, so that the lanes' reads fall on different banks whatever rows they
// are at).  Blocks are generated on wave iterations that are multiples of four (wave-uniform
// work): the one that holds word ply + 3, so that with the words left from the block before it
// the lane has the next four -- it consumes at most one word per iteration.
constexpr uint32_t kWordRows = 8;

// The heuristics' walk phases work on all lanes of the wave, whichever wait: the moves of the
// deferred plies are numbered through and dealt to the lanes, whose best weight per ply is found in
// LDS.  Done by the waiting lanes for their own plies, the walk over a ply's captures (twice: for
// the best weight, then for the chosen move) and the draws of its moves (some ninety instructions a
// pair) cost a wave its longest lists.  noisy-1024x1024: 0.98 ms with both done so, 0.72 with the
// steps' draws shared, 0.67 with the captures too; heuristic-1024x1024: 0.52 -> 0.475 ms (0.486 by a
// single walk that keeps the best moves, which plays the long king sequences here).
constexpr uint32_t kSharedSteps = 32, kSharedCaptures = 16;  // plies a walk phase takes
union WalkShare {  // of a wave
  struct {
    struct Ply {
      uint32_t r;      // the ply's word
      uint32_t moves;  // n | base << 8 | turn << 16 (promoting_moves)
      uint32_t first;  // its first pair of moves
      uint32_t promote;
      float w0, w1;
    } ply[kSharedSteps];
    unsigned long long best[kSharedSteps];
    unsigned long long marks[kSharedSteps * 25u / 64u + 1u];  // at most 49 moves each
  } steps;
  struct {
    struct Ply {
      ck::CaptureTrees trees;  // (deep is not used)
      uint32_t r, first;
      uint32_t turn, sm, so;
    } ply[kSharedCaptures];
    unsigned long long best[kSharedCaptures];
    uint2 choice[kSharedCaptures];  // from | to << 8 | move << 16, removed pieces
    unsigned long long marks;
  } captures;
};

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Sum of `count` (below 32) over the lanes before this one, and over all.
__device__ __forceinline__ uint32_t lanes_before(uint32_t count, uint32_t &total) {
  uint32_t before = 0u;
  total = 0u;
#pragma unroll
  for (uint32_t b = 0; b < 5u; b++) {
    const uint64_t m = __ballot(count >> b & 1u);
    before += lane_rank(m) << b;
    total += (uint32_t)__popcll(m) << b;
  }
  return before;
}

// Deferred capture plies (the lanes `todo`, analyses g, words r), a move to a lane; plies with a
// king sequence past two jumps or more than 31 moves are left to their lane's walk.  Takes the
// plies that it has not played out of `todo`.
template <uint32_t POLICY, bool TRACE>
__device__ __forceinline__ void capture_plies(WalkShare &share, uint64_t &todo, ck::Lane &L,
                                              const ck::Gen &g, uint32_t r, ck::PlyResult &res,
                                              uint32_t &ld, const Lookup &tab) {
  auto &sh = share.captures;
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t n = 0u;  // moves to be dealt
  bool walk = false;
  ck::CaptureTrees t;
  if (lane_in(todo)) {
    ck::capture_trees(L, g, t);
    walk = t.deep || t.n > 31u;
    n = walk || L.counter >= 50u ? 0u : t.n;
  }
  uint32_t total;
  const uint32_t first = lanes_before(n, total);
  const uint64_t dealt = __ballot(n != 0u && first + n <= 64u);
  const uint32_t rank = lane_rank(dealt);
  const uint64_t mine = __ballot(lane_in(dealt) && rank < kSharedCaptures);
  todo &= ~__ballot(n != 0u) | mine;
  if (lane == 0u) sh.marks = 0ull;
  wave_lds_fence();
  if (lane_in(mine)) {
    atomicOr(&sh.marks, 1ull << first);
    auto &p = sh.ply[rank];
    p.trees = t;
    p.r = r;
    p.first = first;
    p.turn = L.turn;
    p.sm = ck::material(L.own, L.kings);
    p.so = ck::material(L.opp, L.kings);
    sh.best[rank] = 0ull;
  }
  total = mine ? __builtin_amdgcn_readlane(first + n, 63u - (uint32_t)__builtin_clzll(mine)) : 0u;
  wave_lds_fence();
  if (total) {
    const unsigned long long marks = sh.marks;
    const bool on = lane < total;
    const uint32_t at = lane_rank(marks) + (uint32_t)(marks >> lane & 1ull) - 1u;
    ck::Choice c = {0u, 0u, 0u};
    uint32_t k = 0u, begin = 0u, moves = 0u, turn = 0u, word = 0u;
    float w = 0.0f;
    unsigned long long key = 0ull;
    if (on) {
      const auto p = sh.ply[at];
      begin = p.first;
      moves = p.trees.n;
      turn = p.turn;
      word = p.r;
      k = lane - begin;
      uint64_t order;
      c = ck::weigh_capture<POLICY>(p.trees, k, p.sm, p.so, turn, word, tab, w, order);
      key = order;
      atomicMax(&sh.best[at], key);
    }
    wave_lds_fence();
    const unsigned long long best = on ? sh.best[at] : 1ull;
    // the ply's lanes that hold a move of largest weight (noisy: of the weight of its first move)
    const float w_first = __shfl(w, (int)begin);
    const uint64_t same =
        __ballot(on && (POLICY == MI_POLICY_HEURISTIC ? key == best : w == w_first));
    const uint32_t set = (uint32_t)(same >> begin) & ((1u << moves) - 1u);
    bool chosen = false;
    if (on)
      chosen = ck::plays_capture<POLICY>(k, moves, key == best, set, w_first, turn, word, tab);
    if (chosen) sh.choice[at] = make_uint2(c.from | c.to << 8 | k << 16, c.removed);
    wave_lds_fence();
  }
  if (lane_in(todo)) {
    if (walk) {
      res = POLICY == MI_POLICY_HEURISTIC ? ck::ply_heuristic_given<TRACE>(L, g, r, &ld)
                                          : ck::ply_noisy_given<TRACE>(L, g, r, &ld);
    } else {
      res.n = t.n;
      if (TRACE) ld = ck::list_digest(L, g, t.n);
      if (n == 0u) {  // the draw count has run out
        res.over = 1u;
        res.chosen = 0xFFFFu;
        res.winner = -1;
      } else {
        const uint2 c = sh.choice[rank];
        res.chosen = TRACE ? (L.turn ? n - 1u - (c.x >> 16) : c.x >> 16) : 0u;
        ck::apply(L, c.x & 31u, c.x >> 8 & 31u, c.y);
      }
    }
  }
  wave_lds_fence();
}

// Deferred noisy steps of two weights (the lanes `todo`, at most kSharedSteps), a pair of moves to
// a lane: it draws for both and enters the better one.
template <bool TRACE>
__device__ __forceinline__ void noisy_steps(WalkShare &share, uint64_t todo, ck::Lane &L,
                                            const ck::Gen &g, uint32_t r, ck::PlyResult &res,
                                            uint32_t &ld, const Lookup &tab) {
  auto &sh = share.steps;
  const uint32_t lane = threadIdx.x & 63u;
  const bool on = lane_in(todo);
  const uint32_t rank = lane_rank(todo);
  ck::SlotWords w = {0u, 0u, 0u, 0u, 0u, 0u, 0u};
  if (on) w = ck::slot_words(g.slot);
  uint32_t total;
  const uint32_t first = lanes_before((w.n + 1u) >> 1, total);
  if (lane < sizeof(sh.marks) / 8u) sh.marks[lane] = 0ull;
  wave_lds_fence();
  if (on) {
    atomicOr(&sh.marks[first >> 6], 1ull << (first & 63u));
    auto &p = sh.ply[rank];
    uint32_t base;
    p.promote = ck::promoting_moves(w, ck::promoting(L, g), base);
    p.moves = w.n | base << 8 | L.turn << 16;
    p.r = r;
    p.first = first;
    const uint32_t sm = ck::material(L.own, L.kings);
    const float so = (float)ck::material(L.opp, L.kings);
    p.w0 = (float)sm / so;
    p.w1 = (float)(sm + 3u) / so;
    sh.best[rank] = 0ull;
  }
  wave_lds_fence();
  uint32_t before = 0u;  // plies that begin in earlier rounds
  for (uint32_t q0 = 0u; q0 < total; q0 += 64u) {
    const unsigned long long mk = sh.marks[q0 >> 6];
    const uint32_t at = before + lane_rank(mk) + (uint32_t)(mk >> lane & 1ull) - 1u;
    before += __builtin_amdgcn_readfirstlane((uint32_t)__popcll(mk));
    if (q0 + lane < total) {
      const auto p = sh.ply[at];
      const unsigned long long key =
          ck::steps_key(p.r, q0 + lane - p.first, p.moves & 255u, p.moves >> 8 & 255u, p.promote,
                        p.w0, p.w1, p.moves >> 16);
      atomicMax(&sh.best[at], key);
    }
  }
  wave_lds_fence();
  if (on) {
    const uint32_t n = w.n;
    res.n = n;
    if (TRACE) ld = ck::list_digest(L, g, n);
    if (L.counter >= 50u) {  // (a step of two weights is not the only move)
      res.over = 1u;
      res.chosen = 0xFFFFu;
      res.winner = -1;
    } else {
      const uint32_t m = ck::noisy_key_move(sh.best[rank], L.turn);
      res.chosen = TRACE ? (L.turn ? n - 1u - m : m) : 0u;
      uint32_t sq, sl8;
      ck::select_move(w, m, sq, sl8, tab);
      ck::play_slot(L, 0u, sq, sl8, tab);
    }
  }
  wave_lds_fence();
}

// A wave's last game is played by the whole wave (wave_play.h), at 0.33 us a ply instead of 0.85:
// 21000x3 0.137 -> 0.129 ms, random-64x4096 0.213 -> 0.203.  With two such games the second one
// waits for the first and nothing is gained over playing both in their lanes (0.133, 0.210).
struct LastGame {
  int32_t winner;
  uint32_t plies, longest;
};
template <uint32_t POLICY>
__device__ __forceinline__ LastGame last_game(ck::Lane L, uint32_t ply, uint32_t lane,
                                              const wave::Stream &stream) {
  LastGame end = {0, ply, 0u};
  wave::play<POLICY>(L, wave::geometry(lane), stream, end.plies, end.longest);
  end.winner = L.counter < 50u ? (int32_t)(L.turn ^ 1u) : -1;
  return end;
}

// The waves of a workgroup hand their last games over.  Once no playout is left to claim, a wave's
// games end one after the other while an iteration costs the same to its last one: on
// random-64x4096 72% of all wave iterations had 18 of 64 lanes playing.  A wave with at most half of
// its lanes playing therefore asks for games (its bit in `asking`) or, where another wave asks,
// leaves it its own and ends.  The giver takes the other's bit back, writes the games over its own
// Philox words, which it needs no more, and then sets the other's entry in `given`; a wave whose bit
// was taken so does not end before it has its games, and the giver writes them without waiting for
// anything.  Games leave a SIMD that has several waves for one with no more (wave w of a workgroup
// runs on SIMD w & 3): what is saved is the turns that waves of a SIMD wait for each other.  Up to
// four waves have a SIMD each and nothing to save (there the checks alone took 21000x3 from 133 to
// 150 us).  random-1024x1024 0.525 -> 0.48 ms, random-64x4096 0.232 -> 0.21 ms with 16 and 12 waves
// in a workgroup per CU against as many workgroups of one wave.
struct Handover {
  uint32_t asking;     // a bit per wave
  uint32_t alive;      // waves that play
  uint32_t given[16];  // games handed to a wave << 8 | giver + 1
};

__device__ __forceinline__ uint32_t lds_value(const uint32_t &x) {
  return __builtin_amdgcn_readfirstlane(
      __hip_atomic_load(&x, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
}
// Clears the bits in a word; returns what it held.
__device__ __forceinline__ uint32_t lds_take(uint32_t &x, uint32_t bits) {
  uint32_t old = 0u;
  if ((threadIdx.x & 63u) == 0u)
    old = __hip_atomic_fetch_and(&x, ~bits, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
  return __builtin_amdgcn_readfirstlane(old);
}
__device__ __forceinline__ void lds_set(uint32_t &x, uint32_t bits) {
  if ((threadIdx.x & 63u) == 0u)
    __hip_atomic_fetch_or(&x, bits, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// FEW: for launches of single-wave workgroups whose number of games the host does not know: a batch
// with at most a game for each wave is played as such (300 positions, 1191 random games by counts in
// device memory 182 -> 104 us; as a branch of the other launches' kernel it cost those 1%).
template <uint32_t POLICY, bool TRACE, uint32_t REFILL, bool FEW = false>
__global__ void __launch_bounds__(1024) k_playouts(PlayoutArgs a) {
  if (a.desc) {  // graph replays and allocation-free launches: the batch lives in device memory
    const LaunchDesc *d = a.desc;
    a.npos = d->npos;
    a.total = d->total;
    a.seed = d->seed;
    a.epoch = d->epoch;
    if (!d->ordered) a.order = nullptr;
    const char *base = (const char *)d;
    if (d->pos_at) a.pos = (const mi_pos *)(base + d->pos_at);
    if (d->offs_at) a.offs = (const uint32_t *)(base + d->offs_at);
    a.keys = d->keys_at ? (const uint32_t *)(base + d->keys_at) : nullptr;
  }
  __shared__ LdsTables tables;
  // kWordRows x 64 words per wave, then the heuristics' WalkShare per wave
  extern __shared__ __align__(8) uint32_t wave_words[];
  __shared__ Handover handover;
  tables.fill();
  if (threadIdx.x < 16u) handover.given[threadIdx.x] = 0u;
  if (threadIdx.x == 0u) {
    handover.asking = 0u;
    handover.alive = (1u << (blockDim.x >> 6)) - 1u;
  }
  __syncthreads();
  const Lookup tab = {tables};
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t *const words = wave_words + (threadIdx.x >> 6) * (kWordRows * 64u) + lane;
  WalkShare &share =
      ((WalkShare *)(wave_words + (blockDim.x >> 6) * (kWordRows * 64u)))[threadIdx.x >> 6];
  const uint32_t nthreads = gridDim.x * blockDim.x;
  // Lanes that hold a game.  A wave mask (in scalar registers) rather than a per-lane flag: flags
  // changed on divergent paths are kept in vector registers, a dozen instructions per ply.
  uint64_t active = 0;
  // ply counts in units of kPly, the row stride of `words`: a word's row offset is one mask away
  constexpr uint32_t kPly = 64u;
  uint32_t g = 0, p = 0, j = 0, ply = 0, h = 0, maxn = 0;
  uint32_t plies_acc = 0;  // a lane's plies of a launch stay far below 2^32 (2^31 playouts in all)
  ck::Lane L = {0u, 0u, 0u, 0u, 0u};
  // wave-uniform refill and deferral state: the reservation [res_next, res_end) is slab-local in
  // slab `slab`
  uint32_t res_next = 0, res_end = 0, since_walk = 0;
  const uint32_t nslabs = gridDim.x < kSlabs ? gridDim.x : kSlabs;
  const uint32_t slab = blockIdx.x % nslabs;
  bool exhausted = false;
  uint32_t static_next = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t defer_min = a.defer_min;

  // A game on its way to another wave: word w of the game in place i is games[w * 32 + i].
  auto give = [&](uint32_t *games, uint32_t i) {
    games[i] = L.own;
    games[32u + i] = L.opp;
    games[64u + i] = L.kings;
    games[96u + i] = L.turn | L.counter << 1;
    games[128u + i] = g;
    games[160u + i] = p;
    games[192u + i] = j;
    games[224u + i] = ply;
    if (TRACE) games[256u + i] = h;
  };
  auto receive = [&](const uint32_t *games, uint32_t i) {
    L.own = games[i];
    L.opp = games[32u + i];
    L.kings = games[64u + i];
    L.turn = games[96u + i] & 1u;
    L.counter = games[96u + i] >> 1;
    g = games[128u + i];
    p = games[160u + i];
    j = games[192u + i];
    ply = games[224u + i];
    if (TRACE) h = games[256u + i];
  };
  // The next four words' block b of the lanes' streams.
  auto generate = [&](uint32_t b) {
    uint32_t o[4], seed = a.seed;
    // (the rounds' keys are ten additions; kept for the whole loop they do not fit the scalar
    // registers and come back by lane reads)
    asm volatile("" : "+s"(seed));
    ck::philox(b, j, ck::TAG_PLAYOUT, a.epoch, seed, p, o);
    uint32_t *const row = words + (b & 1u) * (4u * 64u);
#pragma unroll
    for (uint32_t w = 0; w < 4u; w++) row[w * 64u] = o[w];
  };
  uint32_t asks = 0u;  // this wave's bit in handover.asking was set and no games came yet

  // Games that are over on the lanes `over`.
  auto ended = [&](uint64_t over, int32_t winner) {
    if (lane_in(over)) {
      a.winners[g] = (int8_t)winner;
      if (TRACE) {
        if (a.plies) a.plies[g] = ply / kPly;
        if (a.hashes) a.hashes[g] = h;
      }
      plies_acc += ply / kPly;
    }
    active &= ~over;
  };
  // The game in g from its start.
  auto begin = [&]() {
    mi_pos q;
    locate(a, g, p, j, g, q);  // from here on g is the playout's result slot
    if (a.keys) p = a.keys[p];  // from here on p is the stream key
    L = ck::lane_from_abs(q.p1, q.p2, q.kings, q.turn, q.counter);
    ply = 0;
    h = 0;
  };

  if (FEW && a.total <= gridDim.x) {  // each game is its wave's last one from the start
    exhausted = true;
    if (blockIdx.x < a.total) {
      g = blockIdx.x;
      if (lane == 0u) begin();
      active = 1u;
    }
  }
  for (;;) {
    bool start = false;
    if (REFILL == MI_REFILL_STATIC) {
      if (!lane_in(active) && static_next < a.total) {
        g = static_next;
        static_next += nthreads;
        start = true;
      }
    } else if (!exhausted && ~active) {
      const uint64_t idle = ~active;
      const uint32_t cnt = (uint32_t)__popcll(idle);
      const uint32_t rank = lane_rank(idle);  // of an idle lane among the idle lanes
      const uint32_t avail = res_end - res_next;
      uint32_t c = 0;
      // the new claim covers every idle lane that the old one cannot
      const uint32_t want = avail < cnt ? ((cnt - avail + kChunk - 1u) / kChunk) * kChunk : 0u;
      if (avail < cnt) {
        if (lane == 0u) c = atomicAdd(&a.work->queue[slab].next, want);
        c = __builtin_amdgcn_readfirstlane(c);
      }
      if (lane_in(idle)) {
        const uint32_t idx =
            slab_index(rank < avail ? res_next + rank : c + (rank - avail), slab, nslabs);
        if (idx < a.total) {
          g = idx;
          start = true;
        }
      }
      if (avail < cnt) {
        res_next = c + (cnt - avail);
        res_end = c + want;
      } else {
        res_next += cnt;
      }
      if (slab_index(res_next, slab, nslabs) >= a.total) exhausted = true;  // slab dry
    }
    if (start) begin();
    active |= __ballot(start);
    const bool dry = REFILL == MI_REFILL_STATIC ? !__ballot(static_next < a.total) : exhausted;
    uint32_t leaves = 0u;  // this wave's games, if any, go to another one
    if (blockDim.x > 256u && dry && (uint32_t)__popcll(active) <= 32u) {
      const uint32_t me = 1u << wave;
      uint32_t games = 0u;
      if (asks) games = lds_value(handover.given[wave]);
      if (asks && !games && !active && !(lds_take(handover.asking, me) & me)) {
        // a giver took the bit: it writes its games now
        while (!(games = lds_value(handover.given[wave]))) __builtin_amdgcn_s_sleep(1);
      }
      if (games) {
        asks = 0u;
        if (lane == 0u) handover.given[wave] = 0u;
        const uint32_t *from = wave_words + ((games & 255u) - 1u) * (kWordRows * 64u);
        const uint32_t rank = lane_rank(~active);
        const bool take = !lane_in(active) && rank < games >> 8;
        if (take) {
          receive(from, rank);
          generate(ply / kPly >> 2);
        }
        active |= __ballot(take);
      } else if (active) {
        // another wave that asks, on a SIMD that is no busier than this one's
        const uint32_t alive = lds_value(handover.alive);
        auto load = [alive](uint32_t w) { return __builtin_popcount(alive >> (w & 3u) & 0x1111u); };
        uint32_t others = load(wave) < 2u ? 0u : lds_value(handover.asking) & ~me, to = 0u;
        for (; others; others &= others - 1u) {
          to = (uint32_t)__builtin_ctz(others);
          if (load(to) <= load(wave)) break;
        }
        if (others && (!asks || (lds_take(handover.asking, me) & me))) {
          asks = 0u;
          if (lds_take(handover.asking, 1u << to) >> to & 1u) {
            if (lane_in(active)) give(words - lane, lane_rank(active));
            if (lane == 0u)
              __hip_atomic_store(&handover.given[to], (uint32_t)__popcll(active) << 8 | (wave + 1u),
                                 __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
            leaves = 1u;
          }
        } else if (!others && !asks) {
          asks = 1u;
          lds_set(handover.asking, me);
        }
      }
      if (leaves || !active) lds_take(handover.alive, me);
    }
    // (uniform, but not to the compiler: the branches above hold divergent ones)
    active = uniform64(active);
    asks = __builtin_amdgcn_readfirstlane(asks);
    if (__builtin_amdgcn_readfirstlane(leaves)) active = 0;
    if (!active) break;
    // the last game of a wave that nobody will give any is played below
    if (!TRACE && !(active & (active - 1ull)) && uniform(dry) &&
        (!asks || (lds_take(handover.asking, 1u << wave) >> wave & 1u)))
      break;
    if (lane_in(active)) generate((ply / kPly + 3u) >> 2);
#pragma unroll 1
    for (uint32_t step = 0; step < 4u; step++) {
      // The common part of the ply: every lane looks at its position (an idle lane's or a waiting
      // one's yields what it did before), and those that can play do.  The others wait for the walk
      // phase, where they take the same word.
      ck::Gen gen;
      ck::analyse(L, gen);
      uint32_t from;
      const uint64_t deferred = ck::waiting<POLICY, WaveLanes>(L, gen, active, from);
      {
        uint32_t n;
        const ck::SlotWords w = ck::common_moves<POLICY>(gen, from, n);
        const uint64_t can = active & ~deferred;
        const uint64_t go = can & __ballot(w.n != 0u) & __ballot(L.counter < 50u);
        // (a waiting ply has no fewer moves than first jumps, an idle lane's last game had these)
        maxn = n > maxn ? n : maxn;
        uint32_t ld = 0u, chosen = 0xFFFFu;
        if (TRACE && lane_in(can)) ld = ck::list_digest(L, gen, n);
        if (lane_in(go)) {
          const uint32_t r = words[ply & ((kWordRows - 1u) * kPly)];
          chosen = ck::play_common<POLICY, TRACE>(L, gen, w, n, r, tab);
          ply += kPly;
        }
        if (TRACE && lane_in(can)) h = ck::hash_step(h, ck::ply_record(ld, n, chosen));
        if (can & ~go) ended(can & ~go, L.counter < 50u ? (int32_t)(L.turn ^ 1u) : -1);
      }
      if (deferred) {
        const uint32_t nd = (uint32_t)__popcll(deferred);
        if (nd >= defer_min || deferred == active || since_walk >= 8u) {
          since_walk = 0;
          uint64_t todo = deferred;
          const uint32_t r = words[ply & ((kWordRows - 1u) * kPly)];
          ck::PlyResult res = {0u, 0u, 0u, 0};
          uint32_t ld = 0;
          if (POLICY == MI_POLICY_RANDOM) {
            if (lane_in(todo)) {
              // capture trees in closed form; the walk only for king trees past two jumps
              bool deep = false;
              res = ck::ply_random_captures<TRACE>(L, gen, r, &ld, deep, tab);
              if (deep) res = ck::ply_random_given<TRACE>(L, gen, r, &ld);
            }
          } else {
            uint64_t captures = deferred;
            if (POLICY == MI_POLICY_HEURISTIC_NOISY) captures &= __ballot(gen.capture != 0u);
            uint64_t steps = deferred & ~captures;
            if (captures) capture_plies<POLICY, TRACE>(share, captures, L, gen, r, res, ld, tab);
            if (POLICY == MI_POLICY_HEURISTIC_NOISY && steps) {
              if (__popcll(steps) > kSharedSteps)
                steps = __ballot(lane_in(steps) && lane_rank(steps) < kSharedSteps);
              noisy_steps<TRACE>(share, steps, L, gen, r, res, ld, tab);
            }
            todo = captures | steps;
          }
          if (lane_in(todo)) {
            if (TRACE) h = ck::hash_step(h, ck::ply_record(ld, res.n, res.chosen));
            maxn = res.n > maxn ? res.n : maxn;
          }
          const uint64_t over = todo & __ballot(res.over != 0u);
          if (over) ended(over, res.winner);
          if (lane_in(todo)) ply += kPly;
        } else {
          since_walk++;
        }
      }
    }
  }
  if (!TRACE && active) {
    const uint32_t from = (uint32_t)__builtin_ctzll(active);
    auto of = [from](uint32_t x) { return wave::lane_value(x, from); };
    const LastGame end = last_game<POLICY>(
        {of(L.own), of(L.opp), of(L.kings), of(L.turn), of(L.counter)}, of(ply) / kPly, lane,
        {of(j), ck::TAG_PLAYOUT, a.epoch, a.seed, of(p)});
    maxn = end.longest > maxn ? end.longest : maxn;
    if (lane == from) {
      a.winners[g] = (int8_t)end.winner;
      plies_acc += end.plies;
    }
  }
  // statistics: per wave, then per workgroup in LDS, then one device atomic each (device atomics
  // travel to memory as 32-byte requests)
  unsigned long long wave_plies = plies_acc;
  for (int off = 32; off >= 1; off >>= 1) {
    wave_plies += __shfl_xor(wave_plies, off);
    uint32_t m = __shfl_xor(maxn, off);
    maxn = m > maxn ? m : maxn;
  }
  __shared__ unsigned long long wg_plies;
  __shared__ uint32_t wg_maxn;
  if (threadIdx.x == 0) {
    wg_plies = 0ull;
    wg_maxn = 0u;
  }
  __syncthreads();
  if (lane == 0u) {
    atomicAdd(&wg_plies, wave_plies);
    atomicMax(&wg_maxn, maxn);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicAdd(&a.work->plies, wg_plies);
    atomicMax(&a.work->max_moves, wg_maxn);
  }
}

// One lane per position: the whole move list in reference order, absolute squares.
__global__ void __launch_bounds__(256) k_gen_moves(const mi_pos *__restrict__ pos, uint32_t npos,
                                                   mi_move *__restrict__ out, uint32_t cap,
                                                   uint32_t *__restrict__ counts,
                                                   WorkWords *work) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npos) return;
  const mi_pos q = pos[i];
  const ck::Lane L = ck::lane_from_abs(q.p1, q.p2, q.kings, q.turn, q.counter);
  ck::Gen gen;
  ck::analyse(L, gen);
  const uint32_t n = gen.capture ? ck::count_walks(L, gen) : ck::slot_count(gen.slot);
  counts[i] = n;
  if (n > cap) {
    atomicOr(&work->overflow, 1u);
    return;
  }
  mi_move *dst = out + (size_t)i * cap;
  auto v = [&](uint32_t idx, uint32_t from, uint32_t to, uint32_t, uint32_t jumps, uint32_t dirs,
               uint32_t king) {
    const uint32_t ref = L.turn ? n - 1u - idx : idx;
    mi_move m;
    m.from = (uint8_t)ck::abs_sq(L, from);
    m.to = (uint8_t)ck::abs_sq(L, to);
    m.jumps = (uint8_t)jumps;
    m.promoted = (uint8_t)((!king && to >= ck::FAR_ROW_FIRST) ? 1 : 0);
    uint32_t x = from;
#pragma unroll
    for (uint32_t t = 0; t < 8u; t++) {
      m.inter[t] = 0;
      m.removed[t] = 0;
    }
    for (uint32_t t = 0; t < jumps; t++) {
      const uint32_t d = (dirs >> (2u * t)) & 3u;
      const uint32_t land = (uint32_t)((int)x + ck::jump_off(d));
      m.inter[t] = (uint8_t)ck::abs_sq(L, land);
      m.removed[t] = (uint8_t)ck::abs_sq(L, ck::mid_sq(x, land));
      x = land;
    }
    dst[ref] = m;
  };
  ck::enumerate(L, gen, v);
}

// One wave per position: tallies of draws, player-1 wins and player-2 wins.
__global__ void __launch_bounds__(256) k_tally(const int8_t *__restrict__ winners,
                                               const uint32_t *__restrict__ offs, uint32_t npos,
                                               uint32_t per_pos, uint32_t *__restrict__ tallies) {
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t lane = threadIdx.x & 63u;
  if (wave >= npos) return;
  const uint64_t begin = offs ? offs[wave] : (uint64_t)wave * per_pos;
  const uint64_t end = offs ? offs[wave + 1] : begin + per_pos;
  uint32_t c[3] = {0u, 0u, 0u};
  for (uint64_t g = begin + lane; g < end; g += 64u) {
    const int w = winners[g];
    c[0] += w < 0;
    c[1] += w == 0;
    c[2] += w == 1;
  }
  for (int off = 32; off >= 1; off >>= 1) {
    c[0] += __shfl_xor(c[0], off);
    c[1] += __shfl_xor(c[1], off);
    c[2] += __shfl_xor(c[2], off);
  }
  if (lane == 0u) {
    tallies[3u * wave + 0u] = c[0];
    tallies[3u * wave + 1u] = c[1];
    tallies[3u * wave + 2u] = c[2];
  }
}

// Start positions (the stream layout of mi_gen_start_positions): lanes play attempts, with
// k_playouts' word rows and walk phase.  A position takes the first attempt that does not end
// before its plies are played, and with kmax = 150 more than half of the attempts end: one lane per
// position would run up to twenty in turn (a call for 262,144 positions took 1.7 ms that way).  So
// each wave keeps up to a.slots positions open, and lanes that no position needs play the next
// attempts of the open ones ahead; a position is decided when an attempt is accepted and all
// before it have ended (1.05 ms, 0.72 of it the kernel; 64 positions 0.27 -> 0.16).
// Slot q's position is kept by lane q: its attempts before `lo` have ended, those from `hi` on have
// not begun; bit (attempt mod 64) of marks[q] tells which of those between (at most 64) ended, of
// marks[64 + q] which were accepted.
__global__ void __launch_bounds__(64) k_start_positions(StartArgs a) {
  __shared__ LdsTables tables;
  __shared__ uint32_t rows[kWordRows * 64u];
  __shared__ unsigned long long marks[128];  // fails, accepts
  __shared__ uint32_t decided[64], index[64], next[64], limits[64], list[64];
  constexpr uint32_t kOpen = 0xFFFFFFFFu;  // in decided[]: no attempt yet
  const uint32_t lane = threadIdx.x;
  tables.fill();
  marks[lane] = marks[64u + lane] = 0ull;
  decided[lane] = kOpen;
  __syncthreads();
  const Lookup tab = {tables};
  uint32_t *const words = rows + lane;
  constexpr uint32_t kPly = 64u;  // as in k_playouts
  // lanes that play an attempt, and lanes that hold an accepted attempt's position
  uint64_t active = 0, held = 0;
  uint64_t open = 0;           // slots with a position
  uint32_t lo = 0, hi = 0;     // of this lane's slot
  uint32_t slot = 0, i = 0, attempt = 0, ply = 0, limit = 0;
  ck::Lane L = {0u, 0u, 0u, 0u, 0u};
  uint32_t since_walk = 0;
  // Where the slots hold all positions a wave takes its own at once: claims on one counter go one by
  // one, some 20 ns each (3,000 positions of no ply by as many waves: 90 -> 29 us a call).
  const bool dealt = (uint64_t)gridDim.x * a.slots >= a.n;
  const uint32_t nslabs = min(gridDim.x, kSlabs);
  const uint32_t slab = blockIdx.x % nslabs;
  bool exhausted = false;
  for (;;) {
    __syncthreads();  // (one wave: orders the LDS accesses)
    if (lane_in(open)) {
      const uint32_t turn = lo & 63u;
      const uint64_t f = rotate_right(marks[lane], turn);
      const uint32_t ended = f == ~0ull ? 64u : (uint32_t)__builtin_ctzll(~f);
      if (ended < 64u && (rotate_right(marks[64u + lane], turn) >> ended & 1u)) {
        decided[lane] = lo + ended;
      } else if (ended) {
        const uint64_t gone = ended == 64u ? ~0ull : (1ull << ended) - 1ull;
        marks[lane] &= ~rotate_right(gone, (64u - turn) & 63u);
        lo += ended;
      }
    }
    __syncthreads();
    {  // a decided position: its attempt's lane writes it, the lanes of later attempts are free
      const uint32_t by = lane_in(active | held) ? decided[slot] : kOpen;
      if (by != kOpen && by == attempt) a.out[i] = packed_position(L);
      const uint64_t gone = __ballot(by != kOpen);
      active &= ~gone;
      held &= ~gone;
    }
    {  // close decided slots (a position all of whose attempts ended is reported)
      const bool lost = lane_in(open) && lo == kStartAttempts;
      if (lost) atomicOr(&a.work->overflow, 1u);
      const bool close = lane_in(open) && (lost || decided[lane] != kOpen);
      if (close) {
        decided[lane] = kOpen;
        marks[lane] = marks[64u + lane] = 0ull;
      }
      open &= ~__ballot(close);
    }
    // Idle lanes go to the open positions without an attempt, then to new positions, then to
    // further attempts of the open ones: list[] names the slots in that order.
    const uint64_t idle = ~(active | held);
    const uint32_t cnt = (uint32_t)__popcll(idle);
    const uint64_t bare = __ballot(lane_in(open) && lo == hi);
    uint32_t named = (uint32_t)__popcll(bare);
    if (lane_in(bare)) {
      list[lane_rank(bare)] = lane;
      next[lane] = hi++;
    }
    const uint32_t room = a.slots - min(a.slots, (uint32_t)__popcll(open));
    const uint32_t want = min(cnt - named, room);
    if (!exhausted && want) {
      const uint32_t rank = lane_rank(~open);
      uint32_t at;
      if (dealt) {  // want == a.slots
        at = blockIdx.x * a.slots + rank;
        exhausted = true;
      } else {
        uint32_t c = 0;
        if (lane == 0u) c = atomicAdd(&a.work->queue[slab].next, want);
        c = __builtin_amdgcn_readfirstlane(c);
        at = slab_index(c + rank, slab, nslabs);
        exhausted = slab_index(c + want, slab, nslabs) >= a.n;
      }
      const bool taken = !lane_in(open) && rank < want && at < a.n;
      if (taken) {
        list[named + rank] = lane;
        index[lane] = at;
        next[lane] = lo = 0u;
        hi = 1u;
      }
      const uint64_t fresh = __ballot(taken);
      open |= fresh;
      named += (uint32_t)__popcll(fresh);
    }
    if (!open) {
      if (exhausted) break;
      continue;
    }
    const uint32_t spare = cnt - named, nopen = (uint32_t)__popcll(open);
    const uint32_t ahead = hi;  // the first attempt that a spare lane may take here
    __syncthreads();
    const uint32_t rank = lane_rank(idle);
    bool start = false;
    if (lane_in(idle) && rank < named) {
      slot = list[rank];
      attempt = next[slot];
      start = true;
    }
    if (spare && a.reject) {
      __syncthreads();
      const float per = 1.0f / (float)nopen;
      if (lane_in(open)) {
        const uint32_t r = lane_rank(open);
        list[r] = lane;
        next[lane] = ahead;
        // spare lanes x = r, r + nopen, ... take attempts ahead, ahead + 1, ...
        const uint32_t share = r < spare ? (uint32_t)(((float)(spare - 1u - r) + 0.5f) * per) + 1u : 0u;
        const uint32_t top = min(lo + 64u, kStartAttempts);
        hi = max(ahead, min(ahead + share, top));
        limits[lane] = hi;
      }
      __syncthreads();
      if (lane_in(idle) && rank >= named) {
        const uint32_t x = rank - named;
        const uint32_t q = (uint32_t)(((float)x + 0.5f) * per);
        slot = list[x - q * nopen];
        attempt = next[slot] + q;
        start = attempt < limits[slot];
      }
    }
    if (start) {
      i = index[slot];
      L = ck::start_position();
      limit = ck::start_plies(a.seed, a.base + i, attempt, a.kmin, a.span) * kPly;
      ply = 0;
    }
    active |= __ballot(start);
    if (lane_in(active)) {
      const uint32_t b = (ply / kPly + 3u) >> 2;
      uint32_t o[4];
      ck::philox(b, attempt, ck::TAG_START, 0u, a.seed, a.base + i, o);
      uint32_t *const row = words + (b & 1u) * (4u * 64u);
#pragma unroll
      for (uint32_t w = 0; w < 4u; w++) row[w * 64u] = o[w];
    }
#pragma unroll 1
    for (uint32_t step = 0; step < 4u; step++) {
      // The common part of the ply, as in k_playouts; a position at its limit is left as it is.
      ck::Gen gen;
      ck::analyse(L, gen);
      const ck::SlotWords w = ck::slot_words(gen.slot);
      const uint64_t stop = __ballot(ply == limit);
      // (an origin of longer captures has its slot's bit too)
      const uint64_t over = ~(__ballot(w.n != 0u) & __ballot(L.counter < 50u));
      const uint64_t done = active & (stop | over);
      const uint64_t deferred = active & ~done & __ballot(gen.multi != 0u);
      const uint64_t go = active & ~done & ~deferred;
      const uint32_t r = words[ply & ((kWordRows - 1u) * kPly)];
      if (lane_in(go)) {
        const uint32_t k = tab.mod(r, w.n);
        uint32_t sq, sl8;
        ck::select_move(w, L.turn ? w.n - 1u - k : k, sq, sl8, tab);
        ck::play_slot(L, gen.capture, sq, sl8, tab);
        ply += kPly;
      }
      if (done) {
        const uint64_t accepted = a.reject ? done & ~over : done;
        if (lane_in(done))
          atomicOr(&marks[lane_in(accepted) ? 64u + slot : slot], 1ull << (attempt & 63u));
        active &= ~done;
        held |= accepted;
      }
      if (deferred) {
        const uint32_t nd = (uint32_t)__popcll(deferred);
        if (nd >= 16u || deferred == active || since_walk >= 8u) {
          since_walk = 0;
          if (lane_in(deferred)) {
            uint32_t unused = 0;
            bool deep = false;  // (the game is not over: captures, and the draw count below 50)
            ck::ply_random_captures<false>(L, gen, r, &unused, deep, tab);
            if (deep) ck::ply_random_given<false>(L, gen, r, &unused);
            ply += kPly;
          }
        } else {
          since_walk++;
        }
      }
    }
  }
}

__global__ void __launch_bounds__(256) k_divmod(const uint32_t *__restrict__ r,
                                                const uint32_t *__restrict__ n, uint32_t count,
                                                uint32_t *__restrict__ q, uint32_t *__restrict__ rem) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  uint32_t qq, rr;
  ck::divmod_u32(r[i], n[i], qq, rr);
  q[i] = qq;
  // the remainder, or all ones when the general or (below 2^18) the per-ply remainder differs
  const bool small_ok = n[i] >= (1u << 18) || ck::mod_small(r[i], n[i]) == rr;
  rem[i] = ck::mod_u32(r[i], n[i]) == rr && small_ok ? rr : 0xFFFFFFFFu;
}

// Plain grid-stride copy of 16-byte words (traffic-counter calibration).
__global__ void __launch_bounds__(256) k_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst,
                                              uint64_t n16) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride)
    dst[i] = src[i];
}

// Integer VALU issue-rate probe (the roofline's peak, measured).  Every lane runs eight
// independent chains of v_add_u32 / v_xor_b32 with uniform (SGPR) operands, written as asm so
// that the compiler can neither fuse them (v_xad_u32, v_bitop3_b32) nor fold them: one loop trip
// is exactly 32 VALU instructions, so lane-ops per launch = threads x iters x 32.
#define VALU_STEP(a)                                                                     \
  asm volatile("v_add_u32 %0, %1, %0\n\tv_xor_b32 %0, %2, %0" : "+v"(a) : "s"(k0), "s"(k1))

__global__ void __launch_bounds__(256) k_valu_rate(uint32_t iters, uint32_t salt, uint32_t *out) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t k0 = salt | 1u, k1 = salt * 0x9E3779B9u;
  uint32_t a0 = t ^ salt, a1 = a0 + 1u, a2 = a0 + 2u, a3 = a0 + 3u;
  uint32_t a4 = a0 + 4u, a5 = a0 + 5u, a6 = a0 + 6u, a7 = a0 + 7u;
  for (uint32_t i = 0; i < iters; i++) {
    VALU_STEP(a0); VALU_STEP(a1); VALU_STEP(a2); VALU_STEP(a3);
    VALU_STEP(a4); VALU_STEP(a5); VALU_STEP(a6); VALU_STEP(a7);
    VALU_STEP(a0); VALU_STEP(a1); VALU_STEP(a2); VALU_STEP(a3);
    VALU_STEP(a4); VALU_STEP(a5); VALU_STEP(a6); VALU_STEP(a7);
  }
  out[t] = a0 ^ a1 ^ a2 ^ a3 ^ a4 ^ a5 ^ a6 ^ a7;
}
#undef VALU_STEP

}  // namespace

uint32_t playout_lds(uint32_t policy, uint32_t block) {
  return block / 64u * (uint32_t)(kWordRows * 64u * sizeof(uint32_t) +
                                  (policy == MI_POLICY_RANDOM ? 0u : sizeof(WalkShare)));
}

namespace {

template <uint32_t POLICY, bool TRACE>
hipError_t launch_refill(const PlayoutArgs &args, uint32_t refill, uint32_t grid, uint32_t block,
                         hipStream_t stream) {
  if (refill == MI_REFILL_STATIC)
    hipLaunchKernelGGL((k_playouts<POLICY, TRACE, MI_REFILL_STATIC>), dim3(grid), dim3(block),
                       playout_lds(POLICY, block), stream, args);
  else if (!TRACE && args.desc && args.offs && block == 64u)
    hipLaunchKernelGGL((k_playouts<POLICY, false, MI_REFILL_QUEUE, !TRACE>), dim3(grid), dim3(block),
                       playout_lds(POLICY, block), stream, args);
  else
    hipLaunchKernelGGL((k_playouts<POLICY, TRACE, MI_REFILL_QUEUE>), dim3(grid), dim3(block),
                       playout_lds(POLICY, block), stream, args);
  return hipGetLastError();
}

}  // namespace

const void *playout_kernel(uint32_t policy, uint32_t refill) {
  if (policy == MI_POLICY_RANDOM)
    return refill == MI_REFILL_STATIC
               ? (const void *)k_playouts<MI_POLICY_RANDOM, false, MI_REFILL_STATIC>
               : (const void *)k_playouts<MI_POLICY_RANDOM, false, MI_REFILL_QUEUE>;
  if (policy == MI_POLICY_HEURISTIC)
    return refill == MI_REFILL_STATIC
               ? (const void *)k_playouts<MI_POLICY_HEURISTIC, false, MI_REFILL_STATIC>
               : (const void *)k_playouts<MI_POLICY_HEURISTIC, false, MI_REFILL_QUEUE>;
  return refill == MI_REFILL_STATIC
             ? (const void *)k_playouts<MI_POLICY_HEURISTIC_NOISY, false, MI_REFILL_STATIC>
             : (const void *)k_playouts<MI_POLICY_HEURISTIC_NOISY, false, MI_REFILL_QUEUE>;
}

const void *stage_kernel() { return (const void *)k_stage; }

hipError_t launch_stage(const LaunchDesc *from, LaunchDesc *to, WorkWords *work, hipStream_t stream) {
  hipLaunchKernelGGL(k_stage, dim3(kStageGrid), dim3(kStageBlock), 0, stream, from, to, work);
  return hipGetLastError();
}

hipError_t launch_reset(WorkWords *work, hipStream_t stream) {
  hipLaunchKernelGGL(k_reset, dim3(1), dim3(64), 0, stream, work);
  return hipGetLastError();
}

hipError_t launch_playouts(const PlayoutArgs &args, uint32_t policy, bool trace, uint32_t refill,
                           uint32_t grid, uint32_t block, hipStream_t stream) {
  if (policy == MI_POLICY_RANDOM)
    return trace ? launch_refill<MI_POLICY_RANDOM, true>(args, refill, grid, block, stream)
                 : launch_refill<MI_POLICY_RANDOM, false>(args, refill, grid, block, stream);
  if (policy == MI_POLICY_HEURISTIC)
    return trace ? launch_refill<MI_POLICY_HEURISTIC, true>(args, refill, grid, block, stream)
                 : launch_refill<MI_POLICY_HEURISTIC, false>(args, refill, grid, block, stream);
  return trace ? launch_refill<MI_POLICY_HEURISTIC_NOISY, true>(args, refill, grid, block, stream)
               : launch_refill<MI_POLICY_HEURISTIC_NOISY, false>(args, refill, grid, block, stream);
}

hipError_t launch_gen_moves(const mi_pos *pos, uint32_t npos, mi_move *moves, uint32_t cap,
                            uint32_t *counts, WorkWords *work, hipStream_t stream) {
  const uint32_t block = 256;
  const uint32_t grid = (npos + block - 1) / block;
  hipLaunchKernelGGL(k_gen_moves, dim3(grid), dim3(block), 0, stream, pos, npos, moves, cap,
                     counts, work);
  return hipGetLastError();
}

hipError_t launch_start_positions(const StartArgs &args, uint32_t grid, hipStream_t stream) {
  hipLaunchKernelGGL(k_start_positions, dim3(grid), dim3(kStartBlock), 0, stream, args);
  return hipGetLastError();
}

hipError_t launch_divmod(const uint32_t *r, const uint32_t *n, uint32_t count, uint32_t *q,
                         uint32_t *rem, hipStream_t stream) {
  const uint32_t block = 256;
  const uint32_t grid = (count + block - 1) / block;
  hipLaunchKernelGGL(k_divmod, dim3(grid), dim3(block), 0, stream, r, n, count, q, rem);
  return hipGetLastError();
}

hipError_t launch_copy(const uint4 *src, uint4 *dst, uint64_t n16, hipStream_t stream) {
  const uint32_t block = 256;
  const uint64_t want = (n16 + block - 1) / block;
  const uint32_t grid = (uint32_t)(want < 16384u ? want : 16384u);
  hipLaunchKernelGGL(k_copy, dim3(grid ? grid : 1u), dim3(block), 0, stream, src, dst, n16);
  return hipGetLastError();
}

hipError_t launch_valu_rate(uint32_t iters, uint32_t salt, uint32_t *out, uint32_t threads,
                            hipStream_t stream) {
  const uint32_t block = 256;
  hipLaunchKernelGGL(k_valu_rate, dim3(threads / block), dim3(block), 0, stream, iters, salt, out);
  return hipGetLastError();
}

hipError_t launch_tally(const int8_t *winners, const uint32_t *offs, uint32_t npos,
                        uint32_t per_pos, uint32_t *tallies, hipStream_t stream) {
  const uint32_t block = 256;
  const uint64_t threads = (uint64_t)npos * 64u;
  const uint32_t grid = (uint32_t)((threads + block - 1) / block);
  hipLaunchKernelGGL(k_tally, dim3(grid), dim3(block), 0, stream, winners, offs, npos, per_pos,
                     tallies);
  return hipGetLastError();
}

}  // namespace gpuai
