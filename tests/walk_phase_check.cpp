// walk_phase_check.cpp -- the plies that wait for k_playouts' walk phase, played on the host by the
// lane logic that the phase's lanes take by turns (gpu_ai_amd/csrc/checkers.h: ply_random_captures;
// weigh_capture and plays_capture, a move to a lane; promoting_moves and steps_key, a pair of noisy
// steps to a lane) and checked against the oracle's traces, with the common plies by ply_common.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "checkers.h"
#include "oracle.h"

using namespace ck;

namespace {

long captures = 0, steps = 0, walks = 0, bad = 0;

PlyResult draw_count_ran_out(uint32_t n) { return {n, 0xFFFFu, 1u, -1}; }

template <uint32_t POLICY>
PlyResult capture_ply(Lane &L, const Gen &g, uint32_t r, uint32_t *ld) {
  CaptureTrees t;
  capture_trees(L, g, t);
  if (t.deep || t.n > 31u) {  // these are walked
    walks++;
    return POLICY == HEURISTIC ? ply_heuristic_given<true>(L, g, r, ld) : ply_noisy_given<true>(L, g, r, ld);
  }
  captures++;
  *ld = list_digest(L, g, t.n);
  if (L.counter >= 50u) return draw_count_ran_out(t.n);
  const uint32_t sm = material(L.own, L.kings), so = material(L.opp, L.kings);
  Choice c[31];
  float w[31];
  uint64_t key[31], best = 0;
  for (uint32_t k = 0; k < t.n; k++) {
    c[k] = weigh_capture<POLICY>(t, k, sm, so, L.turn, r, Direct(), w[k], key[k]);
    best = key[k] > best ? key[k] : best;
  }
  uint32_t set = 0, played = 0, at = 0;
  for (uint32_t k = 0; k < t.n; k++)
    set |= (POLICY == HEURISTIC ? key[k] == best : w[k] == w[0]) ? 1u << k : 0u;
  for (uint32_t k = 0; k < t.n; k++)
    if (plays_capture<POLICY>(k, t.n, key[k] == best, set, w[0], L.turn, r, Direct())) {
      played++;
      at = k;
    }
  bad += played != 1u;
  apply(L, c[at].from, c[at].to, c[at].removed);
  return {t.n, L.turn ? at : t.n - 1u - at, 0u, 0};  // (the turn has passed)
}

PlyResult noisy_steps(Lane &L, const Gen &g, uint32_t r, uint32_t *ld) {
  steps++;
  const SlotWords w = slot_words(g.slot);
  *ld = list_digest(L, g, w.n);
  if (L.counter >= 50u) return draw_count_ran_out(w.n);
  uint32_t base;
  const uint32_t promote = promoting_moves(w, promoting(L, g), base);
  const uint32_t sm = material(L.own, L.kings);
  const float so = (float)material(L.opp, L.kings), w0 = (float)sm / so, w1 = (float)(sm + 3u) / so;
  uint64_t best = 0;
  for (uint32_t j = 0; 2u * j < w.n; j++) {
    const uint64_t key = steps_key(r, j, w.n, base, promote, w0, w1, L.turn);
    best = key > best ? key : best;
  }
  const uint32_t m = noisy_key_move(best, L.turn);
  uint32_t sq, sl8;
  select_move(w, m, sq, sl8, Direct());
  play_slot(L, 0u, sq, sl8, Direct());
  return {w.n, L.turn ? m : w.n - 1u - m, 0u, 0};
}

template <uint32_t POLICY>
or_trace play(const or_pos &p, uint32_t seed, uint32_t key, uint32_t j, uint32_t epoch) {
  Lane L = lane_from_abs(p.p1, p.p2, p.kings, p.turn, p.counter);
  uint32_t h = 0, maxn = 0, w[4] = {0, 0, 0, 0};
  for (uint32_t ply = 0;; ply++) {
    if ((ply & 3u) == 0u) philox(ply >> 2, j, TAG_PLAYOUT, epoch, seed, key, w);
    const uint32_t r = w[ply & 3u];
    uint32_t ld = 0;
    bool waits = false, deep = false;
    Gen g;
    PlyResult res = ply_common<POLICY, true>(L, r, &ld, waits, g, Direct());
    if (waits && POLICY == RANDOM) {
      captures++;
      res = ply_random_captures<true>(L, g, r, &ld, deep);
      if (deep) res = ply_random_given<true>(L, g, r, &ld);
    } else if (waits) {
      res = g.capture ? capture_ply<POLICY>(L, g, r, &ld) : noisy_steps(L, g, r, &ld);
    }
    h = hash_step(h, ply_record(ld, res.n, res.chosen));
    maxn = res.n > maxn ? res.n : maxn;
    if (res.over) {
      or_trace tr = {};
      tr.winner = (int8_t)res.winner;
      tr.plies = ply;
      tr.hash = h;
      tr.max_n = (uint8_t)(maxn > 255u ? 255u : maxn);
      return tr;
    }
  }
}

// Placements of men and kings: crowded capture boards, and steps of two weights (men before the far
// row, kings behind them).
std::vector<or_pos> placements(int n) {
  std::vector<or_pos> v((size_t)n);
  uint64_t x = 31;
  auto next = [&]() {
    x = x * 6364136223846793005ull + 1442695040888963407ull;
    return (uint32_t)(x >> 32);
  };
  for (int i = 0; i < n; i++) {
    const uint32_t occ = i % 2 ? next() & (next() | next()) : (next() & next() & 0x00FFFFFFu) | (ROW6 & next());
    const uint32_t side = i % 2 ? next() : ~(next() & next() & next());
    v[i].p1 = occ & side;
    v[i].p2 = occ & ~side;
    v[i].kings = i % 2 ? occ & next() & next() : occ & ~ROW6;
    v[i].turn = (uint8_t)(i % 2 ? next() & 1u : 0u);
    v[i].counter = (uint8_t)(i % 8 == 0 ? 49 : i % 8 == 1 ? 50 : 0);
  }
  return v;
}

}  // namespace

int main(int argc, char **argv) {
  const int N = argc > 1 ? std::atoi(argv[1]) : 1024, P = 6;
  long playouts = 0;
  for (int set = 0; set < 3; set++) {
    std::vector<or_pos> pos(N);
    if (set == 0) or_gen_start_positions(5, N, 0, 60, 0, pos.data());
    else if (set == 1) or_gen_start_positions(6, N, 40, 120, 1, pos.data());
    else pos = placements(N);
    for (uint32_t policy : {RANDOM, HEURISTIC, NOISY}) {
      std::vector<or_trace> ot((size_t)N * P);
      or_run_playouts(pos.data(), N, nullptr, P, 77, 4, (int)policy, nullptr, ot.data(), 0);
      for (int i = 0; i < N * P; i++) {
        const or_pos &p = pos[i / P];
        const or_trace t = policy == RANDOM      ? play<RANDOM>(p, 77, i / P, i % P, 4)
                           : policy == HEURISTIC ? play<HEURISTIC>(p, 77, i / P, i % P, 4)
                                                 : play<NOISY>(p, 77, i / P, i % P, 4);
        playouts++;
        if (t.winner != ot[i].winner || t.plies != ot[i].plies || t.hash != ot[i].hash ||
            t.max_n != ot[i].max_n) {
          if (bad++ < 5) std::printf("set %d policy %u position %d playout %d\n", set, policy, i / P, i % P);
        }
      }
    }
  }
  std::printf("playouts %ld, captures %ld, steps %ld, walks %ld, mismatches %ld\n", playouts, captures,
              steps, walks, bad);
  return bad != 0;
}
