// Host check of what mi_mlp_train_epoch times (mlp.cpp over hip_stub.hpp): every launch of the epoch
// lies between its two events, for a set whose order is drawn on the host and for one drawn on the
// device.
#include "hip_stub.hpp"

#include <algorithm>
#include <cstdio>

#include "gpuai/mi_mlp.h"

int main() {
  long bad = 0;
  std::vector<mi_pos> pos(8192);
  std::vector<float> t(8192);
  mi_ctx *ctx = nullptr;
  mi_mlp *net = nullptr;
  bad += mi_create(&ctx, 0, nullptr) != MI_OK || mi_mlp_create(ctx, 256, 1, &net) != MI_OK;
  for (uint32_t n : {600u, 4096u, 4097u, 8192u}) {
    bad += mi_mlp_set_dataset(net, pos.data(), t.data(), n) != MI_OK;
    stub::calls.clear();
    float loss = 0.f, ms = 0.f;
    bad += mi_mlp_train_epoch(net, 256, 1e-3f, 1, 1, &loss, &ms) != MI_OK || ms != 1.0f;
    const auto &c = stub::calls;
    const auto first = std::find(c.begin(), c.end(), "event");
    long launches = 0, outside = 0;
    for (auto i = c.begin(); i != c.end(); ++i)
      if (*i == "shuffle" || *i == "take" || *i == "train_rows" || *i == "update") {
        launches++;
        outside += i < first || std::find(i, c.end(), "event") == c.end();
      }
    if (outside || launches != 1 + 2 * (long)(n / 256u) || std::count(c.begin(), c.end(), "event") != 2) {
      std::printf("%u positions: %ld of %ld launches outside the events\n", n, outside, launches);
      bad++;
    }
  }
  mi_mlp_destroy(net);
  mi_destroy(ctx);
  std::printf("mismatches %ld\n", bad);
  return bad != 0;
}
