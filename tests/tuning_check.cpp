// Host check of the routes that playout batches take (capi.cpp over hip_stub.hpp): by their size on
// a context without a shape of its own, with the shape that a context was given, and by size again
// once the defaults are set; after a tuning run, whatever it measured fastest for the batch's size,
// one wave per game among the rest, and by size where it measured nothing.
#include "hip_stub.hpp"

#include <cstdio>

namespace {

long bad = 0, checked = 0;

// One call of n playouts: whether it ran with a wave per game, and its workgroups' threads.
void expect(mi_ctx *ctx, uint32_t n, bool wave, uint32_t block, int line,
            uint32_t policy = MI_POLICY_RANDOM) {
  const uint32_t per = n < 4096u ? 1u : 64u;
  std::vector<mi_pos> pos(n / per);
  std::vector<int8_t> winners(n);
  for (auto &p : pos) p = mi_pos{0xFFFu, 0xFFF00000u, 0u, 0, 0, {0, 0}};
  mi_stats st;
  const int rc = mi_run_playouts(ctx, pos.data(), n / per, nullptr, per, 1, 1, policy,
                                 winners.data(), &st);
  checked++;
  if (rc == MI_OK && stub::wave == wave && stub::block == block && st.block_size == block) return;
  std::printf("line %d: %u playouts returned %d: wave %d, %u threads (expected %d, %u)\n", line, n,
              rc, (int)stub::wave, stub::block, (int)wave, block);
  bad++;
}
#define EXPECT(ctx, n, wave, block) expect(ctx, n, wave, block, __LINE__)

void by_size(mi_ctx *ctx, int line) {
  expect(ctx, 256, true, 64, line);
  expect(ctx, 8192, true, 64, line);
  expect(ctx, 16384, false, 64, line);
  expect(ctx, 131072, false, 512, line);
  expect(ctx, 1048576, false, 1024, line);
}

mi_ctx *context(const mi_tuning *t = nullptr) {
  mi_ctx *ctx = nullptr;
  bad += mi_create(&ctx, 0, t) != MI_OK;
  return ctx;
}

void defaults() {
  const mi_tuning zero = {0u, 0u, MI_REFILL_QUEUE, 0u}, given = {128u, 4u, MI_REFILL_QUEUE, 16u};
  const mi_tuning still = {0u, 0u, MI_REFILL_STATIC, 0u};
  mi_ctx *ctx = context();
  by_size(ctx, __LINE__);
  mi_tuning kept;
  bad += mi_get_tuning(ctx, &kept) != MI_OK;
  for (const mi_tuning *back : {&zero, (const mi_tuning *)&kept}) {  // the defaults, or what they read as
    bad += mi_set_tuning(ctx, &given) != MI_OK;
    EXPECT(ctx, 256, false, 128);
    EXPECT(ctx, 1048576, false, 128);
    bad += mi_set_tuning(ctx, back) != MI_OK;
    by_size(ctx, __LINE__);
  }
  bad += mi_set_tuning(ctx, &still) != MI_OK;  // a refill policy is a shape
  EXPECT(ctx, 256, false, 64);
  mi_destroy(ctx);
  ctx = context(&zero);
  by_size(ctx, __LINE__);
  mi_destroy(ctx);
  ctx = context(&given);
  EXPECT(ctx, 256, false, 128);
  bad += mi_set_tuning(ctx, &zero) != MI_OK;
  by_size(ctx, __LINE__);
  mi_destroy(ctx);
}

// Kernel times that a tuning run sees: 256 threads are the fastest of the lanes' shapes, and a wave
// per game is faster than all of them or slower.
float wave_time = 0.05f;
float times(uint32_t block, uint32_t, bool wave) {
  return wave ? wave_time : 0.1f + 0.001f * (block > 256u ? block - 256u : 256u - block);
}

// One replay of a graph for 4096 playouts.
void expect_replay(mi_graph *g, uint32_t n, bool wave, uint32_t block, uint32_t refill, int line) {
  std::vector<mi_pos> pos(n, mi_pos{0xFFFu, 0xFFF00000u, 0u, 0, 0, {0, 0}});
  std::vector<uint32_t> counts(n, 1u);
  std::vector<int8_t> winners(n);
  mi_stats st;
  const int rc = mi_graph_run(g, pos.data(), n, counts.data(), nullptr, 1, 1, winners.data(), &st);
  checked++;
  if (rc == MI_OK && stub::wave == wave && stub::block == block && st.block_size == block &&
      st.refill == refill)
    return;
  std::printf("line %d: replay of %u returned %d: wave %d, %u threads, refill %u (expected %d, %u)\n",
              line, n, rc, (int)stub::wave, stub::block, st.refill, (int)wave, block);
  bad++;
}

void tuned(bool fast) {
  stub::kernel_ms = times;
  wave_time = fast ? 0.05f : 0.5f;
  const uint32_t few = fast ? 64 : 256;  // threads of a small measured batch
  std::vector<mi_pos> pos(1024, mi_pos{0xFFFu, 0xFFF00000u, 0u, 0, 0, {0, 0}});
  mi_ctx *ctx = context();
  mi_tuning best;
  mi_tune_result rows[256];
  uint32_t n = 0;
  // one large batch: its bucket takes what was measured, every other size its own shape
  bad += mi_autotune(ctx, pos.data(), 1024, nullptr, 1024, MI_POLICY_RANDOM, 1, rows, 256, &n, &best);
  bad += best.block_size != 256u || best.blocks_per_cu == 0u;
  EXPECT(ctx, 1048576, false, 256);
  EXPECT(ctx, 131072, false, 512);
  EXPECT(ctx, 16384, false, 64);
  EXPECT(ctx, 256, true, 64);
  const uint32_t many = n;
  // one small batch: one wave per game is among the candidates
  bad += mi_autotune(ctx, pos.data(), 1024, nullptr, 4, MI_POLICY_RANDOM, 1, rows, 256, &n, &best);
  bad += n != many + 2u || best.block_size != few || (best.blocks_per_cu == 0u) != fast;
  for (uint32_t i = 0; i < n; i++) bad += (rows[i].tuning.blocks_per_cu == 0u) != (i >= many);
  mi_tuning t;
  bad += mi_get_tuning(ctx, &t) != MI_OK || t.block_size != 256u || t.blocks_per_cu == 0u;
  EXPECT(ctx, 4096, fast, few);
  EXPECT(ctx, 256, true, 64);
  expect(ctx, 4096, true, 64, __LINE__, MI_POLICY_HEURISTIC_NOISY);  // (not measured)
  // the sizes of a table, under a shape that was given: measured ones take what was measured
  const mi_tuning given = {128u, 4u, MI_REFILL_QUEUE, 16u};
  bad += mi_set_tuning(ctx, &given) != MI_OK;
  const uint32_t sizes[] = {64, 1024, 8192, 65536};
  mi_tune_entry e[4];
  bad += mi_autotune_sizes(ctx, pos.data(), 1024, MI_POLICY_RANDOM, sizes, 4, 1, e) != MI_OK;
  for (const auto &x : e)
    bad += x.tuning.block_size != (x.playouts <= 8192u ? few : 256u) ||
           (x.tuning.blocks_per_cu == 0u) != (fast && x.playouts <= 8192u);
  EXPECT(ctx, 64, fast, few);
  EXPECT(ctx, 1500, fast, few);
  EXPECT(ctx, 8192, fast, few);
  EXPECT(ctx, 8256, false, 256);  // the bucket's, past the sizes of a wave per game
  EXPECT(ctx, 65536, false, 256);
  EXPECT(ctx, 256, false, 128);
  mi_tune_entry table[16];
  bad += mi_get_tuning_table(ctx, table, 16, &n) != MI_OK || n != 8u;
  for (uint32_t i = 0; i < n && i < 16u; i++)
    bad += table[i].tuning.refill != i % 2u ||
           (table[i].tuning.blocks_per_cu == 0u) != (fast && table[i].bucket <= 13u);
  for (uint32_t refill = 0; refill < 2u; refill++) {  // a graph keeps its refill policy
    const mi_tuning as = {128u, 4u, refill, 16u};
    bad += mi_set_tuning(ctx, &as) != MI_OK;
    mi_graph *g = nullptr;
    bad += mi_graph_create(ctx, 8192, 8192, MI_POLICY_RANDOM, &g) != MI_OK;
    expect_replay(g, 1024, false, 128, refill, __LINE__);
    bad += mi_autotune_sizes(ctx, pos.data(), 1024, MI_POLICY_RANDOM, sizes, 4, 1, e) != MI_OK;
    expect_replay(g, 1024, fast, few, refill, __LINE__);
    expect_replay(g, 256, false, 128, refill, __LINE__);
    mi_graph_destroy(g);
  }
  mi_destroy(ctx);
  stub::kernel_ms = nullptr;
}

}  // namespace

int main() {
  defaults();
  tuned(true);
  tuned(false);
  std::printf("calls %ld, mismatches %ld\n", checked, bad);
  return bad != 0;
}
