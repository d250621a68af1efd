// mlp_kernels.h -- launch interface of the value-network kernels (internal to the library).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gpuai/mi_mlp.h"
#include "gpuai/mi_playout.h"

namespace gpuai {
namespace mlp {

// Rows per workgroup of k_train_rows (a multiple of 16, dividing 64): the training batch is a
// multiple of 64 rows.
constexpr uint32_t kTrainRows = 32;

// Rows per split of the weight-gradient products (split-K over the batch; a multiple of 32).
constexpr uint32_t kWSplitRows = 128;

// Partial slots per row block of k_train_rows: b1 at 0-255, b2 256-511, w3 512-767, b3 768,
// loss 769.
constexpr uint32_t kVecSlots = 1024;

// One training step's row pass (k_train_rows), kTrainRows rows per workgroup: row r < n is pos[r]
// with target targets[r]; rows n and up (to the multiple of kTrainRows) are padding.  Writes the activations and their gradients in operand order
// (mlp_kernels.hip) and block b's vector partials at pV + b * kVecSlots.
struct TrainArgs {
  const mi_pos *pos;
  const float *targets;
  uint32_t n;
  uint32_t slices;  // 32-row slices per 16 features of the operands (>= rows / 32)
  const uint16_t *W1f, *W2f, *W2rf;
  const float *b1, *b2, *w3, *b3;
  uint16_t *Xf, *H1f, *dH2f, *dH1f;
  float *pV;
};

// Weight gradients over the step's rows in splits of kWSplitRows, vector gradients from the row
// pass's partials, and Adam (k_update).  rows = 0 takes every gradient as 0.
struct AdamArgs {
  float *w, *m, *v;
  float *grads;      // when set, receives every gradient
  const uint16_t *Xf, *H1f, *dH2f, *dH1f;  // as the row pass wrote them
  uint32_t rows, slices;
  uint32_t splits;   // ceil(rows / kWSplitRows)
  const float *pV;   // the row pass's vector partials, `blocks` of them (rows / kTrainRows)
  uint32_t blocks;
  uint16_t *W1f, *W2f, *W2rf;
  float lr, beta1, beta2, eps, c1, c2;  // c1 = 1/(1-beta1^t), c2 = 1/(1-beta2^t)
  float omb1, omb2;        // 1 - beta1, 1 - beta2 (formed in double precision on the host)
  int update;              // 0: only sum the gradients and refresh the BF16 copies
  float *loss_out;         // when set, receives the sum of the loss partials (slot 769)
};

// Inference in one launch (k_forward): y[r] = network(pos[r]) for r < n, 16 rows per workgroup.
hipError_t forward(const mi_pos *pos, uint32_t n, const uint16_t *W1f, const float *b1,
                   const uint16_t *W2f, const float *b2, const float *w3, const float *b3, float *y,
                   hipStream_t stream);
hipError_t train_rows(const TrainArgs &a, uint32_t rows, hipStream_t stream);
hipError_t update(const AdamArgs &a, hipStream_t stream);

// The order of an epoch over n >= 1 positions: a Fisher-Yates shuffle drawn from Philox key (seed,
// epoch), counter (c >> 2, 0, 3, 1).  head, next, target, chain: n words of scratch each.
struct ShuffleArgs {
  uint32_t n, seed, epoch;
  uint32_t *head, *next, *target, *chain;
  const mi_pos *pos;      // the dataset
  const float *targets;
  mi_pos *rows;           // receive it in the epoch's order
  float *row_targets;
};
hipError_t shuffle(const ShuffleArgs &a, hipStream_t stream);
// The epoch's order given (device memory).
hipError_t shuffle_take(const ShuffleArgs &a, const uint32_t *order, hipStream_t stream);
hipError_t zero(float *p, uint32_t n, hipStream_t stream);

}  // namespace mlp
}  // namespace gpuai
