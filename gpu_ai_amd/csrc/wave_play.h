// wave_play.h -- one game by a whole wave64, on the device: k_playouts_wave (wave_playouts.hip)
// plays small batches this way, k_playouts (playout_kernels.hip) a wave's last games.
//
// The position is wave-uniform (scalar registers) and a ply is spread over the lanes: lane (s, h)
// looks at square s in directions 2h and 2h + 1, comparisons collect each direction's squares as
// wave masks, and ranks of moves are counts of mask bits below a lane.  A ply takes about a hundred
// instructions.  Plies with capture sequences longer than one jump (3%) go through the capture trees
// of checkers.h (random: on the uniform position; the heuristics: a move to a lane).
//
// The position stays in scalar registers only where no branch on a lane's own value joins the loop
// that carries it, and the loop that plays has one exit: with a select chain over the Philox words
// (a branch to the compiler) and three exits a ply took 465 ns in a wave alone on its SIMD, with
// neither 336, and 256 playouts 56 us instead of 77.
#pragma once

#include "checkers.h"
#include "gpuai/mi_playout.h"

namespace gpuai {
namespace wave {

__device__ __forceinline__ uint32_t uniform(uint32_t x) {
  return __builtin_amdgcn_readfirstlane(x);
}
__device__ __forceinline__ uint32_t lane_value(uint32_t x, uint32_t lane) {
  return __builtin_amdgcn_readlane(x, lane);
}
__device__ __forceinline__ uint32_t lo32(uint64_t x) { return (uint32_t)x; }
__device__ __forceinline__ uint32_t hi32(uint64_t x) { return (uint32_t)(x >> 32); }
__device__ __forceinline__ uint64_t pair(uint32_t lo, uint32_t hi) { return (uint64_t)hi << 32 | lo; }

// The lane logic's analysis from the wave masks (ck::Gen).
__device__ __forceinline__ ck::Gen analysis(uint64_t jA, uint64_t jB, uint64_t m0, uint64_t m1,
                                            uint64_t longer, uint32_t capture) {
  ck::Gen g;
  g.cap[0] = lo32(jA);
  g.cap[1] = lo32(jB);
  g.cap[2] = hi32(jA);
  g.cap[3] = hi32(jB);
  g.slot[0] = lo32(m0);
  g.slot[1] = lo32(m1);
  g.slot[2] = hi32(m0);
  g.slot[3] = hi32(m1);
  g.multi = lo32(longer) | hi32(longer);
  g.capture = capture;
  g.origins = capture ? g.slot[0] | g.slot[1] | g.slot[2] | g.slot[3] : 0u;
  return g;
}

// A float's place in the order of floats, as an integer.
__device__ __forceinline__ int32_t ordered(float x) {
  const int32_t b = (int32_t)ck::f32_bits(x);
  return b ^ (b >> 31 & 0x7FFFFFFF);
}

// Largest value over the wave: rotations within the rows of 16 lanes, then a lane of each row.
template <int ROTATE>
__device__ __forceinline__ int32_t row_max(int32_t x) {
  return max(x, __builtin_amdgcn_update_dpp(x, x, 0x120 + ROTATE, 0xF, 0xF, false));
}
__device__ __forceinline__ int32_t wave_max(int32_t x) {
  x = row_max<1>(row_max<2>(row_max<4>(row_max<8>(x))));
  const int32_t a = (int32_t)lane_value((uint32_t)x, 0u), b = (int32_t)lane_value((uint32_t)x, 16u);
  const int32_t c = (int32_t)lane_value((uint32_t)x, 32u), d = (int32_t)lane_value((uint32_t)x, 48u);
  return max(max(a, b), max(c, d));
}

// A capture ply of the heuristics, a move to a lane: it decodes its move from the ply's capture
// trees and weighs it (noisy: draws for it).  Leaves the position as it is and returns false where a
// king has three jumps or more, or there are more than 64 moves.  Against the walk, which goes through
// them one after the other: 421 -> 389 ns a ply over all of 256 heuristic games.
template <uint32_t POLICY>
__device__ __forceinline__ bool capture_ply(ck::Lane &L, const ck::Gen &g, uint32_t r, uint32_t lane,
                                            ck::PlyResult &res) {
  ck::CaptureTrees t;
  ck::capture_trees(L, g, t);
  if (t.deep || t.n > 64u) return false;
  res = {t.n, 0u, 0u, 0};
  if (L.counter >= 50u) {
    res.over = 1u;
    res.winner = -1;
    return true;
  }
  const uint32_t sm = ck::material(L.own, L.kings), so = ck::material(L.opp, L.kings);
  const bool on = lane < t.n;
  ck::Choice c = {0u, 0u, 0u};
  float w = 0.0f;
  int32_t v = (int32_t)0x80000000;
  if (on) {
    c = ck::capture_choice(t, lane, ck::Direct());
    const bool promotes = !ck::getbit(L.kings, c.from) && c.to >= ck::FAR_ROW_FIRST;
    // (as whole numbers these quotients are equal or differ by more than their rounding)
    w = (float)(sm + (promotes ? 3u : 0u)) / (float)(so - ck::material(c.removed, L.kings));
    v = ordered(w);
    if (POLICY == MI_POLICY_HEURISTIC_NOISY) {
#pragma clang fp contract(off)
      float e0, e1;
      ck::noise_pair(r, lane >> 1, e0, e1);
      v = ordered(w + ((lane & 1u) ? e1 : e0));
    }
  }
  // lanes whose moves the word chooses among; none: the best draw, the first in reference order
  const int32_t best = wave_max(v);
  uint64_t among = __ballot(on && v == best);
  uint32_t pick = 0u;
  bool word = true;
  if (POLICY == MI_POLICY_HEURISTIC_NOISY) {
    const float w0 = ck::f32_from_bits(lane_value(ck::f32_bits(w), 0u));
    const uint64_t all = __ballot(on);
    word = __ballot(on && w == w0) == all;
    if (word) among = all;
    else pick = L.turn ? 63u - (uint32_t)__builtin_clzll(among) : (uint32_t)__builtin_ctzll(among);
    if (word && w0 == __builtin_inff()) {  // every weight is +inf: the first move
      pick = L.turn ? t.n - 1u : 0u;
      word = false;
    }
  }
  if (word) {
    const uint32_t ties = (uint32_t)__popcll(among);
    const uint32_t i = ck::mod_small(r, ties);
    const uint32_t km = L.turn ? ties - 1u - i : i;
    const uint32_t rank = __builtin_amdgcn_mbcnt_hi(hi32(among),
                                                    __builtin_amdgcn_mbcnt_lo(lo32(among), 0u));
    // the last lane with at most km of them below it that is one of them
    pick = 63u - (uint32_t)__builtin_clzll(__ballot(rank <= km) & among);
  }
  ck::apply(L, lane_value(c.from, pick), lane_value(c.to, pick), lane_value(c.removed, pick));
  return true;
}

// What a lane looks at: its square s and the square's neighbours in directions A = 2h and
// B = 2h + 1.
struct Geometry {
  uint32_t s, h, self;
  uint32_t stepA, stepB, jumpA, jumpB;  // one step away, where a jump lands (0 off the board)
  uint32_t wantA, wantB;                // what a valid jump's test yields
  uint32_t squares;                     // the four squares' numbers (step A, B, jump A, B) in bytes
  // The factor of r mod n for n = lane: n <= 49, since a step uses one of the board's 49 pairs of
  // adjacent squares, a single jump one of 36 lines of three, and no two moves of a position share
  // theirs.
  uint32_t factor;
};

__device__ __forceinline__ Geometry geometry(uint32_t lane) {
  Geometry q;
  q.s = lane & 31u;
  q.h = lane >> 5;
  q.self = ck::bit(q.s);
  q.stepA = q.h ? ck::step2(q.self) : ck::step0(q.self);
  q.stepB = q.h ? ck::step3(q.self) : ck::step1(q.self);
  q.jumpA = q.h ? ck::step2(q.stepA) : ck::step0(q.stepA);
  q.jumpB = q.h ? ck::step3(q.stepB) : ck::step1(q.stepB);
  q.wantA = q.jumpA ? q.stepA | q.jumpA : 0xFFFFFFFFu;
  q.wantB = q.jumpB ? q.stepB | q.jumpB : 0xFFFFFFFFu;
  q.squares = (31u - __clz(q.stepA | 1u)) | (31u - __clz(q.stepB | 1u)) << 8 |
              (31u - __clz(q.jumpA | 1u)) << 16 | (31u - __clz(q.jumpB | 1u)) << 24;
  q.factor = ck::mod_factor(lane);
  return q;
}

// Slot of the j-th set bit of a nibble, at bit 8 * (nibble & 7) + 2 j: nibbles below 8, and the rest.
constexpr uint64_t nth_table(uint32_t from) {
  uint64_t t = 0;
  for (uint32_t n = 0; n < 8u; n++) {
    uint32_t j = 0;
    for (uint32_t s = 0; s < 4u; s++)
      if ((n + from) >> s & 1u) t |= (uint64_t)s << (8u * n + 2u * j++);
  }
  return t;
}
constexpr uint64_t kNthLow = nth_table(0u), kNthHigh = nth_table(8u);

// A stream of Philox words: that of ply t is word t & 3 of counter (t >> 2, c1, c2, c3).
struct Stream {
  uint32_t c1, c2, c3, seed, key;
};

// Plays a game from L, its ply `ply`, to its end and counts its plies.  The scalar code works with masks (all ones
// or zero) rather than flags: a flag becomes a pair of scalar registers and back at two or three
// instructions each, nine cycles apiece where nothing else runs on the SIMD.
template <uint32_t POLICY>
__device__ __forceinline__ void play(ck::Lane &L, const Geometry &geo, const Stream &st,
                                     uint32_t &ply, uint32_t &maxn) {
  const uint32_t lane = geo.h << 5 | geo.s, s = geo.s, h = geo.h, self = geo.self;
  const uint32_t stepA = geo.stepA, stepB = geo.stepB, jumpA = geo.jumpA, jumpB = geo.jumpB;
  const uint32_t wantA = geo.wantA, wantB = geo.wantB, squares = geo.squares, factor = geo.factor;
  uint32_t words = 0;  // this lane's Philox word: that of ply (ply & ~63) + lane
  auto refresh = [&](bool first = false) {
    if (first || (ply & 63u) == 0u) {
      uint32_t o[4];
      ck::philox((ply >> 6 << 4) + (lane >> 2), st.c1, st.c2, st.c3, st.seed, st.key, o);
      // (by masks: a chain of selects becomes a branch on the lane, and what the loop carries past
      // it is no longer known to be uniform)
      const uint32_t odd = 0u - (lane & 1u), high = 0u - (lane >> 1 & 1u);
      words = (((o[0] & ~odd) | (o[1] & odd)) & ~high) | (((o[2] & ~odd) | (o[3] & odd)) & high);
    }
  };
  refresh(true);
  // The inner loop plays plies until the game is over or one has longer capture sequences, which
  // the outer loop plays (a loop of its own keeps the common plies' registers in place: 20% of the
  // instructions were copies without it; it has one exit, since each further one costs every ply
  // the flags that tell them apart).
  for (;;) {
    uint64_t jA, jB, m0, m1, longer;
    uint32_t r;
    bool walk;  // the ply is the walk's
    for (;;) {
      longer = 0;
      walk = false;
      r = lane_value(words, ply & 63u);
      // squares with a valid jump in A and B, whatever stands on them
      const uint32_t empty = ~(L.own | L.opp);
      const uint32_t kng = L.own & L.kings;
      jA = __ballot(((L.opp & stepA) | (empty & jumpA)) == wantA);
      jB = __ballot(((L.opp & stepB) | (empty & jumpB)) == wantB);
      const uint64_t movers = pair(L.own, kng);  // pieces that move in the lanes' directions
      // the moves' slots in reference order: slots 0 and 2 in m0, 1 and 3 in m1
      uint32_t cap;  // all ones: captures are mandatory
      if ((jA | jB) & movers) {
        cap = 0xFFFFFFFFu;
        const uint64_t men = L.own & ~L.kings, kings = pair(kng, kng);
        m0 = (jA & kings) | (jB & men);  // a man's jump in direction 1 comes first
        m1 = (jB & kings) | (jA & men);
        // origins of longer sequences: a jump lands where the piece can jump on
        const uint32_t fwd = lo32(jA) | lo32(jB), any = fwd | hi32(jA) | hi32(jB);
        const uint64_t fA = __ballot((jumpA & fwd) != 0u), fB = __ballot((jumpB & fwd) != 0u);
        const uint64_t aA = __ballot((jumpA & any) != 0u), aB = __ballot((jumpB & any) != 0u);
        longer = (((jA & fA) | (jB & fB)) & men) | (((jA & aA) | (jB & aB)) & kings);
        if (POLICY != MI_POLICY_RANDOM) {
          // jumps of several kinds (as in ck::waiting) are the walk's as well
          const uint64_t prom = men & ck::ROW5;
          const uint64_t kinds = m0 | m1;
          bool mixed = (kinds & prom) && (kinds & ~prom);
          if (const uint32_t okings = L.opp & L.kings) {
            const uint64_t kA = __ballot((okings & stepA) != 0u), kB = __ballot((okings & stepB) != 0u);
            const uint64_t k0 = (kA & kings) | (kB & men), k1 = (kB & kings) | (kA & men);
            mixed |= ((m0 & k0) | (m1 & k1)) && ((m0 & ~k0) | (m1 & ~k1));
          }
          walk = mixed;
        }
        walk |= longer != 0;
      } else {
        cap = 0u;
        m0 = __ballot((empty & stepA) != 0u) & movers;
        m1 = __ballot((empty & stepB) != 0u) & movers;
      }
      const uint32_t n = (uint32_t)__popcll(m0) + (uint32_t)__popcll(m1);
      maxn = n > maxn ? n : maxn;  // (a ply of the walk's has no fewer moves than first jumps)
      if (walk || n == 0u || L.counter >= 50u) break;
      uint32_t sq = 0, sl = 0, pick = 1u;  // pick: the word chooses among the moves in m0 and m1
      uint32_t ties = n, first = 0u;       // first: every weight is +inf, index 0 wins
      uint64_t prom = 0;  // promoting steps' men, where only some of the steps promote
      if (POLICY != MI_POLICY_RANDOM) {
        const uint64_t kinds = m0 | m1, p = L.own & ~L.kings & ck::ROW6 & ~cap;
        if ((kinds & p) && (kinds & ~p) && L.opp) prom = p;
      }
      if (POLICY == MI_POLICY_HEURISTIC && prom) {
        m0 &= prom;
        m1 &= prom;
        ties = (uint32_t)__popcll(m0) + (uint32_t)__popcll(m1);
      }
      if (POLICY == MI_POLICY_HEURISTIC_NOISY) {
        if (!prom) {
          first = !(cap ? L.opp & (L.opp - 1u) : L.opp) ? 1u : 0u;
        } else {
          const uint32_t t0 = lo32(m0), t1 = lo32(m1), t2 = hi32(m0), t3 = hi32(m1);
          // lane m draws for move m (n <= 49); lane (s, h) then takes the draws of its square's
          // slots 2h and 2h + 1
          float e0, e1;
          ck::noise_pair(r, lane >> 1, e0, e1);
          const float e = (lane & 1u) ? e1 : e0;
          const uint32_t below = self - 1u;
          uint32_t at = ck::popc(t0 & below) + ck::popc(t1 & below) + ck::popc(t2 & below) +
                        ck::popc(t3 & below);
          const uint32_t a0 = h ? t2 : t0, a1 = h ? t3 : t1;
          at += h ? ck::getbit(t0, s) + ck::getbit(t1, s) : 0u;
          const bool on0 = (a0 & self) != 0u, on1 = (a1 & self) != 0u;
          float v0 = __shfl(e, at & 63u), v1 = __shfl(e, (at + (on0 ? 1u : 0u)) & 63u);
          {
#pragma clang fp contract(off)
            const uint32_t sm = ck::material(L.own, L.kings), so = ck::material(L.opp, L.kings);
            const float w0 = (float)sm / (float)so, w1 = (float)(sm + 3u) / (float)so;
            const float w = (lo32(prom) & self) && h == 0u ? w1 : w0;
            v0 = w + v0;
            v1 = w + v1;
          }
          const int32_t i0 = on0 ? ordered(v0) : (int32_t)0x80000000;
          const int32_t i1 = on1 ? ordered(v1) : (int32_t)0x80000000;
          const int32_t best = wave_max(max(i0, i1));
          const uint64_t b0 = __ballot(i0 == best), b1 = __ballot(i1 == best);
          // the first in reference order: player 2's is the reverse of the order here
          const uint32_t hit = lo32(b0) | lo32(b1) | hi32(b0) | hi32(b1);
          sq = L.turn ? 31u - (uint32_t)__builtin_clz(hit) : ck::ctz(hit);
          const uint32_t on = ck::getbit(lo32(b0), sq) | ck::getbit(lo32(b1), sq) << 1 |
                              ck::getbit(hi32(b0), sq) << 2 | ck::getbit(hi32(b1), sq) << 3;
          sl = L.turn ? 31u - (uint32_t)__builtin_clz(on) : ck::ctz(on);
          pick = 0u;
        }
      }
      uint32_t king;  // all ones: the piece is a king
      if (pick) {
        const uint32_t k = first ? 0u : ck::mod_by(r, ties, lane_value(factor, ties));
        const uint32_t tm = 0u - L.turn;
        const uint32_t km = (k ^ tm) + (ties & tm);  // player 2: ties - 1 - k
        // moves on lower squares, per lane of the first half; the last square where they are at most
        // km holds the move
        const uint32_t rank = __builtin_amdgcn_mbcnt_lo(
            lo32(m0), __builtin_amdgcn_mbcnt_lo(
                          lo32(m1), __builtin_amdgcn_mbcnt_lo(
                                        hi32(m0), __builtin_amdgcn_mbcnt_lo(hi32(m1), 0u))));
        sq = 31u - (uint32_t)__builtin_clz(lo32(__ballot(rank <= km)));
        const uint32_t left = km - lane_value(rank, sq);
        king = 0u - ck::getbit(L.kings, sq);
        const uint32_t n0 = ck::getbit(lo32(m0), sq);
        if (king) {
          // slots 0 and 2 are bits 0 and 32 of m0 >> sq, 1 and 3 of m1 >> sq
          const uint64_t two = (m0 >> sq & 0x100000001ull) | (m1 >> sq & 0x100000001ull) << 1;
          const uint32_t nibble = lo32(two) | hi32(two) << 2;
          // entry (nibble, left) of a table of the left-th set bits, two bits each
          sl = (uint32_t)((nibble & 8u ? kNthHigh : kNthLow) >> ((nibble * 8u + left * 2u) & 63u)) & 3u;
        } else {
          sl = left + 1u - n0;  // slots 0 and 1 alone: slot 1 if it is the second or the only one
        }
      } else {
        king = 0u - ck::getbit(L.kings, sq);
      }
      const uint32_t d = sl ^ (cap & ~king & 1u);  // a man's capture slots name directions 1 and 0
      const uint32_t near = lane_value(squares, sq | (d & 2u) << 4) >> ((d & 1u) * 8u);
      const uint32_t one = ck::bit(near & 31u);
      const uint32_t removed = one & cap;
      const uint32_t flip = ck::bit(sq) | ck::bit((near >> (cap & 16u)) & 31u);
      const uint32_t own = L.own ^ flip, opp = L.opp & ~removed;
      const uint32_t kings = (L.kings & ~removed) ^ (flip & (king | ck::ROW7));
      L.counter = (L.counter + 1u) & ~cap;
      L.own = ck::brev(opp);
      L.opp = ck::brev(own);
      L.kings = ck::brev(kings);
      L.turn ^= 1u;
      ply++;
      refresh();
    }
    if (!walk) return;  // the game is over
    const ck::Gen g = analysis(jA, jB, m0, m1, longer, 1u);
    uint32_t unused = 0;
    ck::PlyResult res;
    if (POLICY == MI_POLICY_RANDOM) {
      bool deep = false;
      res = ck::ply_random_trees<false>(L, g, r, &unused, deep);
      if (deep) res = ck::ply_random_given<false>(L, g, r, &unused);
    } else if (!capture_ply<POLICY>(L, g, r, lane, res)) {
      res = POLICY == MI_POLICY_HEURISTIC ? ck::ply_heuristic_given<false>(L, g, r, &unused)
                                          : ck::ply_noisy_given<false>(L, g, r, &unused);
    }
    maxn = res.n > maxn ? res.n : maxn;
    if (res.over) return;
    ply++;
    refresh();
  }
}

}  // namespace wave
}  // namespace gpuai
