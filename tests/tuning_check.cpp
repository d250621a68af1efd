// Host check of the routes that playout batches take (capi.cpp over hip_stub.hpp): by their size on
// a context without a shape of its own, with the shape that a context was given, and by size again
// once the defaults are set.
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

}  // namespace

int main() {
  defaults();
  std::printf("calls %ld, mismatches %ld\n", checked, bad);
  return bad != 0;
}
