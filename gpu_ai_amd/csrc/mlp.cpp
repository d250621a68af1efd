// mlp.cpp -- the value network's C ABI (include/gpuai/mi_mlp.h): buffers, the sequence of
// kernels of a forward pass, of a backward pass and of an Adam step, device-resident epochs and
// checkpoints.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <numeric>
#include <vector>

#include "checkers.h"
#include "ctx.h"
#include "gpuai/mi_mlp.h"
#include "mlp_kernels.h"

using gpuai::DevBuf;
using gpuai::ctxutil::ensure;
using gpuai::ctxutil::fail;
using gpuai::ctxutil::hip_fail;
namespace K = gpuai::mlp;

struct mi_mlp {
  mi_ctx *ctx = nullptr;
  uint32_t max_rows = 0;
  uint32_t step = 0;
  double beta1 = 0.9, beta2 = 0.999, eps = 1e-8;  // rounded to float where a kernel takes them
  // parameters, Adam moments (FP32) and BF16 operand copies
  float *w = nullptr, *m = nullptr, *v = nullptr;
  uint16_t *W1f = nullptr, *W2f = nullptr, *W2rf = nullptr;
  // a training step's activations in operand order (max_rows rows) and its per 32-row block
  // partials of the vector gradients
  uint16_t *Xf = nullptr, *H1f = nullptr, *dH2f = nullptr, *dH1f = nullptr;
  float *pV = nullptr;
  // Pinned host staging of one batch: positions (max_rows), then values and targets (max_rows
  // floats each), the batch's loss, and two sets of parameters (gradients; parameters and moments
  // on their way to the caller). The kernels read a batch from here and write its results here,
  // each once: a copy before and one after cost 9 us of a forward pass of 4096 (29 -> 20 us per
  // call) and 3 us of one position (22 -> 18), and still 23 us of 65536 (114 -> 91), so no size is
  // copied. The gradients of 4096 with the copies of the batch, the gradients and the loss took
  // 86 us, without 54.
  void *h_stage = nullptr;
  // device-resident training set; ds_shuffle: the epoch shuffle's scratch, ds_rows: the set in the
  // epoch's order (positions, then targets)
  DevBuf ds_pos, ds_t, ds_rows, ds_loss, ds_shuffle;
  uint32_t ds_n = 0;
  std::vector<uint32_t> host_perm;  // of small sets
  hipEvent_t e0 = nullptr, e1 = nullptr;
  std::vector<void *> allocs;
};

namespace {

uint32_t round64(uint32_t n) { return (n + 63u) & ~63u; }

// Makes the network's device current on the calling thread (as every playout entry point does).
int use_device(mi_mlp *n) {
  if (hipSetDevice(n->ctx->device) != hipSuccess)
    return fail(n->ctx, MI_ERR_DEVICE, "hipSetDevice failed");
  return MI_OK;
}

mi_pos *stage_pos(mi_mlp *n) { return (mi_pos *)n->h_stage; }
float *stage_values(mi_mlp *n) { return (float *)((char *)n->h_stage + sizeof(mi_pos) * n->max_rows); }
float *stage_targets(mi_mlp *n) { return stage_values(n) + n->max_rows; }
float *stage_loss(mi_mlp *n) { return stage_targets(n) + n->max_rows; }
float *stage_params(mi_mlp *n, uint32_t set) { return stage_loss(n) + 4 + set * (size_t)MI_MLP_PARAMS; }
size_t stage_bytes(size_t rows) {
  return rows * (sizeof(mi_pos) + 2 * sizeof(float)) + (4 + 2 * (size_t)MI_MLP_PARAMS) * sizeof(float);
}

K::AdamArgs adam_args(mi_mlp *n, uint32_t rows, float lr, float c1, float c2, int update,
                      float *loss_out = nullptr, float *grads = nullptr) {
  K::AdamArgs a = {};
  a.loss_out = loss_out;
  a.w = n->w;
  a.m = n->m;
  a.v = n->v;
  a.grads = grads;
  a.Xf = n->Xf;
  a.H1f = n->H1f;
  a.dH2f = n->dH2f;
  a.dH1f = n->dH1f;
  a.rows = rows;
  a.slices = n->max_rows / 32u;
  a.splits = (rows + K::kWSplitRows - 1) / K::kWSplitRows;
  a.pV = n->pV;
  a.blocks = rows / K::kTrainRows;
  a.W1f = n->W1f;
  a.W2f = n->W2f;
  a.W2rf = n->W2rf;
  a.lr = lr;
  a.beta1 = (float)n->beta1;
  a.beta2 = (float)n->beta2;
  a.eps = (float)n->eps;
  a.c1 = c1;
  a.c2 = c2;
  a.omb1 = (float)(1.0 - n->beta1);  // formed in double precision, as Adam's usual
  a.omb2 = (float)(1.0 - n->beta2);  // implementations do
  a.update = update;
  return a;
}

template <class T>
hipError_t dev_alloc(mi_mlp *n, T **p, size_t count) {
  void *q = nullptr;
  hipError_t e = hipMalloc(&q, count * sizeof(T));
  if (e == hipSuccess) {
    n->allocs.push_back(q);
    *p = (T *)q;
  }
  return e;
}

// He-uniform initialisation: U(-a, a), a = sqrt(6 / fan_in), from Philox key (seed, tensor),
// counter (i >> 2, 0, 3, 0), word i & 3, mapped to [0, 1) by its top 24 bits.
void init_params(uint32_t seed, std::vector<float> &w) {
  w.assign(MI_MLP_PARAMS, 0.f);
  struct T { uint32_t off, count, fan_in; } tensors[] = {
      {MI_MLP_OFF_W1, 128 * 256, 128}, {MI_MLP_OFF_W2, 256 * 256, 256}, {MI_MLP_OFF_W3, 256, 256}};
  for (uint32_t t = 0; t < 3; t++) {
    const float a = std::sqrt(6.f / (float)tensors[t].fan_in);
    uint32_t words[4];
    for (uint32_t i = 0; i < tensors[t].count; i++) {
      if ((i & 3) == 0) ck::philox(i >> 2, 0u, ck::TAG_MLP, 0u, seed, t, words);
      const float u = (float)(words[i & 3] >> 8) * (1.f / 16777216.f);
      w[tensors[t].off + i] = (2.f * u - 1.f) * a;
    }
  }
}

int upload_params(mi_mlp *n, const float *w) {
  mi_ctx *ctx = n->ctx;
  MI_HIP(ctx, hipMemcpyAsync(n->w, w, sizeof(float) * MI_MLP_PARAMS, hipMemcpyHostToDevice, ctx->stream));
  MI_HIP(ctx, K::zero(n->m, MI_MLP_PARAMS, ctx->stream));
  MI_HIP(ctx, K::zero(n->v, MI_MLP_PARAMS, ctx->stream));
  // refresh the BF16 copies without updating (no partials: every gradient reads as 0)
  MI_HIP(ctx, K::update(adam_args(n, 0, 0.f, 1.f, 1.f, 0), ctx->stream));
  MI_HIP(ctx, hipStreamSynchronize(ctx->stream));
  n->step = 0;
  return MI_OK;
}

// One training step over `rows` rows (count valid): k_train_rows' forward and backward pass to
// the activations and vector partials, then the weight gradients and Adam (k_update; when
// update == 0, only the gradient sums).  loss_out receives the batch loss and
// `grads` every gradient (either may be null; device or pinned host memory).
int train_rows(mi_mlp *n, const mi_pos *pos, const float *targets, uint32_t count, uint32_t rows,
               float lr, int update, float *loss_out, float *grads = nullptr) {
  mi_ctx *ctx = n->ctx;
  K::TrainArgs ta = {};
  ta.pos = pos;
  ta.targets = targets;
  ta.n = count;
  ta.slices = n->max_rows / 32u;
  ta.W1f = n->W1f;
  ta.W2f = n->W2f;
  ta.W2rf = n->W2rf;
  ta.b1 = n->w + MI_MLP_OFF_B1;
  ta.b2 = n->w + MI_MLP_OFF_B2;
  ta.w3 = n->w + MI_MLP_OFF_W3;
  ta.b3 = n->w + MI_MLP_OFF_B3;
  ta.Xf = n->Xf;
  ta.H1f = n->H1f;
  ta.dH2f = n->dH2f;
  ta.dH1f = n->dH1f;
  ta.pV = n->pV;
  MI_HIP(ctx, K::train_rows(ta, rows, ctx->stream));
  // the bias corrections are formed in double precision, as Adam's usual implementations do
  float c1 = 1.f, c2 = 1.f;
  if (update) {
    n->step++;
    c1 = (float)(1.0 / (1.0 - std::pow(n->beta1, (double)n->step)));
    c2 = (float)(1.0 / (1.0 - std::pow(n->beta2, (double)n->step)));
  }
  MI_HIP(ctx, K::update(adam_args(n, rows, lr, c1, c2, update, loss_out, grads), ctx->stream));
  return MI_OK;
}

// The order of an epoch over at most this many positions is drawn on the host: four launches take
// longer than 2 ns a position and one copy (64 positions: 50 against 70 us an epoch; 4099: alike).
constexpr uint32_t kHostShuffle = 4096;

// Fisher-Yates with Philox key (seed, epoch), counter (c >> 2, 0, 3, 1) (as K::shuffle).
void host_shuffle(std::vector<uint32_t> &perm, uint32_t seed, uint32_t epoch) {
  std::iota(perm.begin(), perm.end(), 0u);
  uint32_t words[4];
  for (uint32_t i = (uint32_t)perm.size() - 1, c = 0; i > 0; i--, c++) {
    if ((c & 3) == 0) ck::philox(c >> 2, 0u, ck::TAG_MLP, 1u, seed, epoch, words);
    std::swap(perm[i], perm[words[c & 3] % (i + 1)]);
  }
}

int check_batch(mi_mlp *n, uint32_t count, const void *pos) {
  if (count == 0) return MI_OK;
  if (!pos) return fail(n->ctx, MI_ERR_INVALID_ARGUMENT, "null positions");
  if (round64(count) > n->max_rows)
    return fail(n->ctx, MI_ERR_INVALID_ARGUMENT, "batch larger than the network's max_batch");
  return MI_OK;
}

// Copies one or two device arrays of MI_MLP_PARAMS floats to the caller's memory (either target may
// be null) through the pinned staging memory: one wait for both.
int download_params(mi_mlp *n, const float *src0, float *dst0, const float *src1, float *dst1) {
  mi_ctx *ctx = n->ctx;
  constexpr size_t bytes = sizeof(float) * MI_MLP_PARAMS;
  float *h0 = stage_params(n, 0), *h1 = stage_params(n, 1);
  if (dst0) MI_HIP(ctx, hipMemcpyAsync(h0, src0, bytes, hipMemcpyDeviceToHost, ctx->stream));
  if (dst1) MI_HIP(ctx, hipMemcpyAsync(h1, src1, bytes, hipMemcpyDeviceToHost, ctx->stream));
  MI_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (dst0) std::memcpy(dst0, h0, bytes);
  if (dst1) std::memcpy(dst1, h1, bytes);
  return MI_OK;
}

}  // namespace

extern "C" {

int mi_mlp_create(mi_ctx *ctx, uint32_t max_batch, uint32_t seed, mi_mlp **out) {
  if (!ctx || !out || max_batch == 0) return MI_ERR_INVALID_ARGUMENT;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->last_error.clear();
  *out = nullptr;
  if (hipSetDevice(ctx->device) != hipSuccess) return fail(ctx, MI_ERR_DEVICE, "hipSetDevice failed");
  mi_mlp *n = new mi_mlp();
  n->ctx = ctx;
  n->max_rows = round64(max_batch);
  const size_t R = n->max_rows, P = MI_MLP_PARAMS;
  hipError_t e = hipSuccess;
  if (e == hipSuccess) e = dev_alloc(n, &n->w, P);
  if (e == hipSuccess) e = dev_alloc(n, &n->m, P);
  if (e == hipSuccess) e = dev_alloc(n, &n->v, P);
  if (e == hipSuccess) e = dev_alloc(n, &n->W1f, (size_t)128 * 256);
  if (e == hipSuccess) e = dev_alloc(n, &n->W2f, (size_t)256 * 256);
  if (e == hipSuccess) e = dev_alloc(n, &n->W2rf, (size_t)256 * 256);
  if (e == hipSuccess) e = dev_alloc(n, &n->Xf, 128 * R);
  if (e == hipSuccess) e = dev_alloc(n, &n->H1f, 256 * R);
  if (e == hipSuccess) e = dev_alloc(n, &n->dH2f, 256 * R);
  if (e == hipSuccess) e = dev_alloc(n, &n->dH1f, 256 * R);
  if (e == hipSuccess) e = dev_alloc(n, &n->pV, (R / K::kTrainRows) * K::kVecSlots);
  if (e == hipSuccess)
    e = hipHostMalloc(&n->h_stage, stage_bytes(R), hipHostMallocDefault);
  if (e == hipSuccess) e = hipEventCreate(&n->e0);
  if (e == hipSuccess) e = hipEventCreate(&n->e1);
  int rc = MI_OK;
  if (e != hipSuccess) rc = hip_fail(ctx, e, "mi_mlp_create");
  std::vector<float> w;
  init_params(seed, w);
  if (!rc) rc = upload_params(n, w.data());
  if (rc) {
    for (void *p : n->allocs) (void)hipFree(p);
    if (n->h_stage) (void)hipHostFree(n->h_stage);
    if (n->e0) (void)hipEventDestroy(n->e0);
    if (n->e1) (void)hipEventDestroy(n->e1);
    delete n;
    return rc;
  }
  *out = n;
  return MI_OK;
}

int mi_mlp_destroy(mi_mlp *n) {
  if (!n) return MI_OK;
  std::lock_guard<std::mutex> lock(n->ctx->mu);
  (void)hipSetDevice(n->ctx->device);
  (void)hipStreamSynchronize(n->ctx->stream);
  for (void *p : n->allocs) (void)hipFree(p);
  if (n->h_stage) (void)hipHostFree(n->h_stage);
  gpuai::DevBuf *bufs[] = {&n->ds_pos, &n->ds_t, &n->ds_rows, &n->ds_loss,
                         &n->ds_shuffle};
  for (auto *b : bufs)
    if (b->ptr) (void)hipFree(b->ptr);
  if (n->e0) (void)hipEventDestroy(n->e0);
  if (n->e1) (void)hipEventDestroy(n->e1);
  delete n;
  return MI_OK;
}

int mi_mlp_get_params(mi_mlp *n, float *params) {
  if (!n || !params) return MI_ERR_INVALID_ARGUMENT;
  mi_ctx *ctx = n->ctx;
  std::lock_guard<std::mutex> lock(ctx->mu);
  if (int rc = use_device(n)) return rc;
  return download_params(n, n->w, params, nullptr, nullptr);
}

int mi_mlp_set_params(mi_mlp *n, const float *params) {
  if (!n || !params) return MI_ERR_INVALID_ARGUMENT;
  std::lock_guard<std::mutex> lock(n->ctx->mu);
  n->ctx->last_error.clear();
  if (int rc = use_device(n)) return rc;
  return upload_params(n, params);
}

int mi_mlp_forward(mi_mlp *n, const mi_pos *pos, uint32_t count, float *values) {
  if (!n) return MI_ERR_INVALID_ARGUMENT;
  mi_ctx *ctx = n->ctx;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->last_error.clear();
  int rc;
  if ((rc = check_batch(n, count, pos))) return rc;
  if (count == 0) return MI_OK;
  if (!values) return fail(ctx, MI_ERR_INVALID_ARGUMENT, "null values");
  if ((rc = use_device(n))) return rc;
  // one launch: encoding, both hidden layers and the output layer (k_forward)
  float *hv = stage_values(n);
  std::memcpy(stage_pos(n), pos, sizeof(mi_pos) * count);
  MI_HIP(ctx, K::forward(stage_pos(n), count, n->W1f, n->w + MI_MLP_OFF_B1, n->W2f,
                         n->w + MI_MLP_OFF_B2, n->w + MI_MLP_OFF_W3, n->w + MI_MLP_OFF_B3, hv,
                         ctx->stream));
  MI_HIP(ctx, hipStreamSynchronize(ctx->stream));
  std::memcpy(values, hv, sizeof(float) * count);
  return MI_OK;
}

static int grad_common(mi_mlp *n, const mi_pos *pos, const float *targets, uint32_t count,
                       float lr, int update, float *grads, float *loss) {
  mi_ctx *ctx = n->ctx;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->last_error.clear();
  int rc;
  if ((rc = check_batch(n, count, pos))) return rc;
  if (count == 0 || !targets) return fail(ctx, MI_ERR_INVALID_ARGUMENT, "empty batch or null targets");
  if ((rc = use_device(n))) return rc;
  std::memcpy(stage_pos(n), pos, sizeof(mi_pos) * count);
  std::memcpy(stage_targets(n), targets, sizeof(float) * count);
  float *hg = stage_params(n, 0);
  if ((rc = train_rows(n, stage_pos(n), stage_targets(n), count, round64(count), lr, update,
                       stage_loss(n), grads ? hg : nullptr)))
    return rc;
  MI_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (grads) std::memcpy(grads, hg, sizeof(float) * MI_MLP_PARAMS);
  if (loss) *loss = *stage_loss(n);
  return MI_OK;
}

int mi_mlp_gradients(mi_mlp *n, const mi_pos *pos, const float *targets, uint32_t count,
                     float *grads, float *loss) {
  if (!n || !grads) return MI_ERR_INVALID_ARGUMENT;
  return grad_common(n, pos, targets, count, 0.f, 0, grads, loss);
}

int mi_mlp_train_step(mi_mlp *n, const mi_pos *pos, const float *targets, uint32_t count,
                      float lr, float *loss) {
  if (!n) return MI_ERR_INVALID_ARGUMENT;
  return grad_common(n, pos, targets, count, lr, 1, nullptr, loss);
}

int mi_mlp_adam_state(mi_mlp *n, float *m, float *v, uint32_t *step) {
  if (!n) return MI_ERR_INVALID_ARGUMENT;
  mi_ctx *ctx = n->ctx;
  std::lock_guard<std::mutex> lock(ctx->mu);
  if (int rc = use_device(n)) return rc;
  if (int rc = download_params(n, n->m, m, n->v, v)) return rc;
  if (step) *step = n->step;
  return MI_OK;
}

int mi_mlp_set_dataset(mi_mlp *n, const mi_pos *pos, const float *targets, uint32_t count) {
  if (!n || (count && (!pos || !targets))) return MI_ERR_INVALID_ARGUMENT;
  mi_ctx *ctx = n->ctx;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->last_error.clear();
  int rc;
  if ((rc = use_device(n))) return rc;
  n->ds_n = 0;  // the buffers go one by one: a call that fails leaves no set
  if ((rc = ensure(ctx, n->ds_pos, sizeof(mi_pos) * (size_t)std::max<uint32_t>(count, 1)))) return rc;
  if ((rc = ensure(ctx, n->ds_t, sizeof(float) * (size_t)std::max<uint32_t>(count, 1)))) return rc;
  if ((rc = ensure(ctx, n->ds_rows,
                   (sizeof(mi_pos) + sizeof(float)) * (size_t)std::max<uint32_t>(count, 1))))
    return rc;
  if ((rc = ensure(ctx, n->ds_shuffle, 4 * sizeof(uint32_t) * (size_t)std::max<uint32_t>(count, 1))))
    return rc;
  MI_HIP(ctx, hipMemcpyAsync(n->ds_pos.ptr, pos, sizeof(mi_pos) * count, hipMemcpyHostToDevice, ctx->stream));
  MI_HIP(ctx, hipMemcpyAsync(n->ds_t.ptr, targets, sizeof(float) * count, hipMemcpyHostToDevice, ctx->stream));
  MI_HIP(ctx, hipStreamSynchronize(ctx->stream));
  n->ds_n = count;
  return MI_OK;
}

int mi_mlp_train_epoch(mi_mlp *n, uint32_t batch, float lr, uint32_t shuffle_seed, uint32_t epoch,
                       float *mean_loss, float *ms) {
  if (!n) return MI_ERR_INVALID_ARGUMENT;
  mi_ctx *ctx = n->ctx;
  std::lock_guard<std::mutex> lock(ctx->mu);
  ctx->last_error.clear();
  if (batch == 0 || batch % 64 || batch > n->max_rows)
    return fail(ctx, MI_ERR_INVALID_ARGUMENT, "batch must be a multiple of 64 within max_batch");
  const uint32_t nb = n->ds_n / batch;
  if (nb == 0) return fail(ctx, MI_ERR_INVALID_ARGUMENT, "the dataset holds less than one batch");
  if (int rc0 = use_device(n)) return rc0;
  int rc;
  if ((rc = ensure(ctx, n->ds_loss, sizeof(float) * nb))) return rc;
  K::ShuffleArgs sh;
  sh.n = n->ds_n;
  sh.seed = shuffle_seed;
  sh.epoch = epoch;
  sh.head = (uint32_t *)n->ds_shuffle.ptr;
  sh.next = sh.head + (size_t)n->ds_n;
  sh.target = sh.next + (size_t)n->ds_n;
  sh.chain = sh.target + (size_t)n->ds_n;
  sh.pos = (const mi_pos *)n->ds_pos.ptr;
  sh.targets = (const float *)n->ds_t.ptr;
  sh.rows = (mi_pos *)n->ds_rows.ptr;
  sh.row_targets = (float *)(sh.rows + (size_t)n->ds_n);
  if (n->ds_n <= kHostShuffle) {
    std::vector<uint32_t> &perm = n->host_perm;
    perm.resize(n->ds_n);
    host_shuffle(perm, shuffle_seed, epoch);
    MI_HIP(ctx, hipMemcpyAsync(sh.head, perm.data(), sizeof(uint32_t) * n->ds_n,
                               hipMemcpyHostToDevice, ctx->stream));
    MI_HIP(ctx, hipEventRecord(n->e0, ctx->stream));
    MI_HIP(ctx, K::shuffle_take(sh, sh.head, ctx->stream));
  } else {
    MI_HIP(ctx, hipEventRecord(n->e0, ctx->stream));
    MI_HIP(ctx, K::shuffle(sh, ctx->stream));
  }
  float *losses = (float *)n->ds_loss.ptr;
  for (uint32_t b = 0; b < nb; b++) {
    const size_t at = (size_t)b * batch;
    if ((rc = train_rows(n, sh.rows + at, sh.row_targets + at, batch, batch, lr, 1, losses + b)))
      return rc;
  }
  MI_HIP(ctx, hipEventRecord(n->e1, ctx->stream));
  std::vector<float> l(nb);
  MI_HIP(ctx, hipMemcpyAsync(l.data(), losses, sizeof(float) * nb, hipMemcpyDeviceToHost, ctx->stream));
  MI_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (mean_loss) *mean_loss = std::accumulate(l.begin(), l.end(), 0.f) / (float)nb;
  if (ms) MI_HIP(ctx, hipEventElapsedTime(ms, n->e0, n->e1));
  return MI_OK;
}

int mi_mlp_save(mi_mlp *n, const char *path) {
  if (!n || !path) return MI_ERR_INVALID_ARGUMENT;
  std::vector<float> w(MI_MLP_PARAMS), m(MI_MLP_PARAMS), v(MI_MLP_PARAMS);
  uint32_t step = 0;
  int rc;
  if ((rc = mi_mlp_get_params(n, w.data()))) return rc;
  if ((rc = mi_mlp_adam_state(n, m.data(), v.data(), &step))) return rc;
  FILE *f = std::fopen(path, "wb");
  if (!f) return fail(n->ctx, MI_ERR_INVALID_ARGUMENT, std::string("cannot write ") + path);
  const char magic[8] = {'G', 'P', 'U', 'A', 'I', 'M', 'L', 'P'};
  const uint32_t head[3] = {1u, step, (uint32_t)MI_MLP_PARAMS};
  bool ok = std::fwrite(magic, 1, 8, f) == 8 && std::fwrite(head, 4, 3, f) == 3 &&
            std::fwrite(w.data(), 4, MI_MLP_PARAMS, f) == MI_MLP_PARAMS &&
            std::fwrite(m.data(), 4, MI_MLP_PARAMS, f) == MI_MLP_PARAMS &&
            std::fwrite(v.data(), 4, MI_MLP_PARAMS, f) == MI_MLP_PARAMS;
  ok = (std::fclose(f) == 0) && ok;
  return ok ? MI_OK : fail(n->ctx, MI_ERR_INVALID_ARGUMENT, std::string("short write to ") + path);
}

int mi_mlp_load(mi_mlp *n, const char *path) {
  if (!n || !path) return MI_ERR_INVALID_ARGUMENT;
  FILE *f = std::fopen(path, "rb");
  if (!f) return fail(n->ctx, MI_ERR_INVALID_ARGUMENT, std::string("cannot read ") + path);
  char magic[8];
  uint32_t head[3];
  std::vector<float> w(MI_MLP_PARAMS), m(MI_MLP_PARAMS), v(MI_MLP_PARAMS);
  bool ok = std::fread(magic, 1, 8, f) == 8 && std::memcmp(magic, "GPUAIMLP", 8) == 0 &&
            std::fread(head, 4, 3, f) == 3 && head[0] == 1u && head[2] == MI_MLP_PARAMS &&
            std::fread(w.data(), 4, MI_MLP_PARAMS, f) == MI_MLP_PARAMS &&
            std::fread(m.data(), 4, MI_MLP_PARAMS, f) == MI_MLP_PARAMS &&
            std::fread(v.data(), 4, MI_MLP_PARAMS, f) == MI_MLP_PARAMS;
  std::fclose(f);
  if (!ok) return fail(n->ctx, MI_ERR_INVALID_ARGUMENT, std::string("not a checkpoint: ") + path);
  mi_ctx *ctx = n->ctx;
  std::lock_guard<std::mutex> lock(ctx->mu);
  int rc = use_device(n);
  if (!rc) rc = upload_params(n, w.data());
  if (rc) return rc;
  MI_HIP(ctx, hipMemcpyAsync(n->m, m.data(), sizeof(float) * MI_MLP_PARAMS, hipMemcpyHostToDevice, ctx->stream));
  MI_HIP(ctx, hipMemcpyAsync(n->v, v.data(), sizeof(float) * MI_MLP_PARAMS, hipMemcpyHostToDevice, ctx->stream));
  MI_HIP(ctx, hipStreamSynchronize(ctx->stream));
  n->step = head[1];
  return MI_OK;
}

}  // extern "C"
