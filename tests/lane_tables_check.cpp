// Host check of the lane logic's lookups (checkers.h): the table remainder against %, the j-th slot
// of a square against a scan, and the move masks against the geometry functions.
#include <cstdio>

#include "checkers.h"

using namespace ck;

int main() {
  long bad = 0, checked = 0;
  uint64_t x = 7;
  auto next = [&]() {
    x = x * 6364136223846793005ull + 1442695040888963407ull;
    return (uint32_t)(x >> 32);
  };
  for (uint32_t n = 1; n <= kModMax; n++) {
    const uint32_t m = mod_factor(n);
    auto check = [&](uint32_t r) {
      checked++;
      bad += mod_by(r, n, m) != r % n;
    };
    for (uint32_t d = 0; d < 3u * n; d++) {  // both ends of the range and around multiples of n
      check(d);
      check(0xFFFFFFFFu - d);
      check(0x80000000u / n * n + d);
    }
    for (int i = 0; i < 20000; i++) check(next());
  }
  for (uint32_t nib = 1; nib < 16u; nib++) {
    const uint32_t y = (nib & 1u) | (nib & 2u) << 7 | (nib & 4u) << 14 | (nib & 8u) << 21;
    bad += gather4(y) != nib << 2;
    uint32_t j = 0;
    for (uint32_t t = 0; t < 4u; t++)
      if (nib >> t & 1u) {
        checked++;
        bad += Direct().nth(y, j++) != t;
      }
  }
  for (uint32_t i = 0; i < 512u; i++) {  // moves that stay on the board
    const uint32_t sq = i & 31u, sl = i >> 5 & 3u, king = i >> 7 & 1u, cap = i >> 8;
    const uint32_t d = cap && !king && sl < 2u ? sl ^ 1u : sl;
    auto step = [](uint32_t b, uint32_t dir) {
      return dir == 0u ? step0(b) : dir == 1u ? step1(b) : dir == 2u ? step2(b) : step3(b);
    };
    const uint32_t one = step(bit(sq), d), two = step(one, d);
    if (!(cap ? two : one)) continue;
    uint32_t flip, removed;
    move_masks(i, flip, removed);
    checked++;
    bad += flip != (bit(sq) | (cap ? two : one)) || removed != (cap ? one : 0u);
  }
  std::printf("lookups %ld, mismatches %ld\n", checked, bad);
  return bad != 0;
}
