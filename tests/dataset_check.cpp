// Host check of a training set's lifetime (mlp.cpp over hip_stub.hpp): each of the allocations of
// mi_mlp_set_dataset fails in turn, for a set that replaces a smaller one, and an epoch is asked for
// afterwards.  It must be refused, and no launch or copy may be given a null pointer.
#include "hip_stub.hpp"

#include <cstdio>

#include "gpuai/mi_mlp.h"

int main() {
  long bad = 0, failed = 0;
  const uint32_t small = 8192, large = 65536;
  std::vector<mi_pos> pos(large);
  std::vector<float> t(large);
  for (int left = 0;; left++) {
    mi_ctx *ctx = nullptr;
    mi_mlp *net = nullptr;
    bad += mi_create(&ctx, 0, nullptr) != MI_OK || mi_mlp_create(ctx, 256, 1, &net) != MI_OK;
    bad += mi_mlp_set_dataset(net, pos.data(), t.data(), small) != MI_OK;
    bad += mi_mlp_train_epoch(net, 256, 1e-3f, 1, 1, nullptr, nullptr) != MI_OK;
    stub::allocations_left = left;
    const int rc = mi_mlp_set_dataset(net, pos.data(), t.data(), large);
    stub::allocations_left = -1;
    const int epoch = mi_mlp_train_epoch(net, 256, 1e-3f, 1, 2, nullptr, nullptr);
    if (rc != MI_OK) {
      failed++;
      if (rc != MI_ERR_OUT_OF_MEMORY || epoch != MI_ERR_INVALID_ARGUMENT) {
        std::printf("allocation %d failed: set_dataset %d, the epoch after it %d\n", left + 1, rc, epoch);
        bad++;
      }
      // a set that fits is taken again
      bad += mi_mlp_set_dataset(net, pos.data(), t.data(), small) != MI_OK;
      bad += mi_mlp_train_epoch(net, 256, 1e-3f, 1, 3, nullptr, nullptr) != MI_OK;
    }
    mi_mlp_destroy(net);
    mi_destroy(ctx);
    if (rc == MI_OK) break;
  }
  bad += stub::null_arguments;
  std::printf("failed allocations %ld, null arguments %d, mismatches %ld\n", failed,
              stub::null_arguments, bad);
  return bad != 0;
}
