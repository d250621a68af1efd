// Host check of the capture plies' closed forms (checkers.h): capture_trees and capture_choice
// against the depth-first walk's enumeration, for every move of random boards from a few pieces to
// crowded ones, with few kings and with many; and, where the draw counter or a long king sequence
// ends or refuses the ply, ply_random_captures against ply_random_given.
#include <cstdio>
#include <cstring>

#include "checkers.h"

using namespace ck;

int main() {
  uint64_t x = 99;
  auto next = [&]() {
    x = x * 6364136223846793005ull + 1442695040888963407ull;
    return (uint32_t)(x >> 32);
  };
  long bad = 0, plies = 0, moves = 0, deep_plies = 0, most = 0;
  for (int i = 0; i < 3000000; i++) {
    const uint32_t a = next(), b = next(), c = next(), side = next();
    uint32_t occ = i % 4 == 0 ? a & b : i % 4 == 1 ? a & (b | c) : i % 4 == 2 ? a & b & c : a;
    uint32_t kings = next();
    if (i % 3) kings &= next();
    if (i % 3 == 2) kings &= next();
    const uint32_t counter = i % 16 == 0 ? 50u : i % 16 == 1 ? 49u : next() % 49u;
    const Lane L = lane_from_abs(occ & side, occ & ~side, kings & occ, next() & 1u, counter);
    Gen g;
    analyse(L, g);
    if (!g.capture || !g.multi) continue;
    plies++;
    CaptureTrees t;
    capture_trees(L, g, t);
    uint32_t longest = 0;
    Choice list[1024];
    uint32_t n = 0;
    auto visit = [&](uint32_t, uint32_t from, uint32_t to, uint32_t removed, uint32_t jumps,
                     uint32_t, uint32_t king) {
      if (king && jumps > longest) longest = jumps;
      if (n < 1024u) list[n] = Choice{from, to, removed};
      n++;
    };
    enumerate(L, g, visit);
    bad += (t.deep != 0u) != (longest >= 3u);
    if (t.deep) {
      deep_plies++;
      continue;
    }
    most = (long)n > most ? (long)n : most;
    bad += t.n != n;
    for (uint32_t k = 0; k < n && k < t.n && k < 1024u; k++) {
      const Choice m = capture_choice(t, k, Direct());
      moves++;
      bad += m.from != list[k].from || m.to != list[k].to || m.removed != list[k].removed;
    }
    const uint32_t r = next();
    Lane A = L, B = L;
    uint32_t da = 0, db = 0;
    bool deep = false;
    const PlyResult ra = ply_random_captures<true>(A, g, r, &da, deep);
    const PlyResult rb = ply_random_given<true>(B, g, r, &db);
    bad += deep != (n > kModMax);
    if (!deep)
      bad += std::memcmp(&A, &B, sizeof A) || std::memcmp(&ra, &rb, sizeof ra) || da != db;
  }
  std::printf("plies %ld (deep %ld), moves %ld (longest list %ld), mismatches %ld\n", plies,
              deep_plies, moves, most, bad);
  return bad != 0;
}
