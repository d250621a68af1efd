// hip_stub.hpp -- stand-ins for the HIP runtime and the kernel launches, so that the library's host
// code (capi.cpp, mlp.cpp) runs without a device and without libamdhip64: device memory is host
// memory, a launch only records what it was given.  For one translation unit per program.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <set>
#include <string>
#include <vector>

#include "ctx.h"
#include "kernels.h"
#include "mlp_kernels.h"

namespace stub {

int allocations_left = -1;          // device allocations until one fails; < 0: none fails
std::set<void *> live;              // device allocations
hipError_t last = hipSuccess;       // what hipGetLastError returns next, a launch too
std::vector<std::string> calls;     // launches, event records and copies, in order
// the last playout launch: threads a workgroup, workgroups, one wave per game or not
uint32_t block = 0, grid = 0;
bool wave = false;
// kernel time in ms of a launch (default: alike for all)
float (*kernel_ms)(uint32_t block, uint32_t grid, bool wave) = nullptr;
// launches that were given a null pointer
int null_arguments = 0;

inline void need(std::initializer_list<const void *> ptrs) {
  for (const void *p : ptrs) null_arguments += p == nullptr;
}

}  // namespace stub

extern "C" {

hipError_t hipGetLastError(void) {
  const hipError_t e = stub::last;
  stub::last = hipSuccess;
  return e;
}
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  p->clockRate = 2400000;
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipMalloc(void **p, size_t bytes) {
  *p = nullptr;
  if (stub::allocations_left == 0) return stub::last = hipErrorOutOfMemory;
  if (stub::allocations_left > 0) stub::allocations_left--;
  *p = std::calloc(bytes, 1);
  stub::live.insert(*p);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!stub::live.erase(p)) std::abort();
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned int) {
  *p = std::calloc(bytes, 1);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int) {
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
  static uintptr_t next = 0;
  *e = (hipEvent_t)(++next);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) {
  stub::calls.push_back("event");
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = stub::kernel_ms ? stub::kernel_ms(stub::block, stub::grid, stub::wave) : 1.0f;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t) {
  stub::need({dst, src});
  stub::calls.push_back(kind == hipMemcpyHostToDevice ? "upload" : "copy");
  if (dst && src) std::memmove(dst, src, bytes);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int value, size_t bytes, hipStream_t) {
  std::memset(p, value, bytes);
  return hipSuccess;
}
// graphs: a replay stands for its playout node
static hipKernelNodeParams stub_node;
hipError_t hipGraphCreate(hipGraph_t *g, unsigned int) {
  *g = nullptr;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphAddKernelNode(hipGraphNode_t *n, hipGraph_t, const hipGraphNode_t *, size_t,
                                 const hipKernelNodeParams *p) {
  *n = nullptr;
  stub_node = *p;
  return hipSuccess;
}
hipError_t hipGraphAddMemcpyNode1D(hipGraphNode_t *n, hipGraph_t, const hipGraphNode_t *, size_t,
                                   void *, const void *, size_t, hipMemcpyKind) {
  *n = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  *x = nullptr;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphExecMemcpyNodeSetParams1D(hipGraphExec_t, hipGraphNode_t, void *, const void *,
                                             size_t, hipMemcpyKind) {
  return hipSuccess;
}
hipError_t hipGraphExecKernelNodeSetParams(hipGraphExec_t, hipGraphNode_t,
                                           const hipKernelNodeParams *p) {
  stub_node = *p;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
  stub::calls.push_back("graph");
  stub::block = stub_node.blockDim.x;
  stub::grid = stub_node.gridDim.x;
  stub::wave = false;
  return hipSuccess;
}

}  // extern "C"

namespace gpuai {

int noalloc_setup(mi_ctx *) { return MI_OK; }
uint32_t playout_lds(uint32_t, uint32_t) { return 0u; }
const void *stage_kernel() { return "stage"; }
const void *playout_kernel(uint32_t, uint32_t) { return "playouts"; }
hipError_t launch_reset(WorkWords *work, hipStream_t) {
  stub::need({work});
  return hipGetLastError();
}
hipError_t launch_stage(const LaunchDesc *from, LaunchDesc *to, WorkWords *work, hipStream_t) {
  stub::need({from, to, work});
  return hipGetLastError();
}
hipError_t launch_playouts(const PlayoutArgs &, uint32_t, bool, uint32_t, uint32_t grid,
                           uint32_t block, hipStream_t) {
  stub::calls.push_back("playouts");
  stub::block = block;
  stub::grid = grid;
  stub::wave = false;
  return hipGetLastError();
}
hipError_t launch_playouts_wave(const PlayoutArgs &, uint32_t, uint32_t games, hipStream_t) {
  stub::calls.push_back("playouts");
  stub::block = kWaveBlock;
  stub::grid = games;
  stub::wave = true;
  return hipGetLastError();
}
hipError_t launch_gen_moves(const mi_pos *, uint32_t, mi_move *, uint32_t, uint32_t *, WorkWords *,
                            hipStream_t) {
  return hipGetLastError();
}
hipError_t launch_start_positions(const StartArgs &, uint32_t, hipStream_t) { return hipGetLastError(); }
hipError_t launch_divmod(const uint32_t *, const uint32_t *, uint32_t, uint32_t *, uint32_t *,
                         hipStream_t) {
  return hipGetLastError();
}
hipError_t launch_copy(const uint4 *, uint4 *, uint64_t, hipStream_t) { return hipGetLastError(); }
hipError_t launch_valu_rate(uint32_t, uint32_t, uint32_t *, uint32_t, hipStream_t) {
  return hipGetLastError();
}
hipError_t launch_tally(const int8_t *, const uint32_t *, uint32_t, uint32_t, uint32_t *,
                        hipStream_t) {
  return hipGetLastError();
}

namespace mlp {
hipError_t forward(const mi_pos *, uint32_t, const uint16_t *, const float *, const uint16_t *,
                   const float *, const float *, const float *, float *, hipStream_t) {
  return hipGetLastError();
}
hipError_t train_rows(const TrainArgs &a, uint32_t, hipStream_t) {
  stub::need({a.pos, a.targets, a.Xf, a.H1f, a.dH2f, a.dH1f, a.pV});
  stub::calls.push_back("train_rows");
  return hipGetLastError();
}
hipError_t update(const AdamArgs &, hipStream_t) {
  stub::calls.push_back("update");
  return hipGetLastError();
}
hipError_t shuffle(const ShuffleArgs &a, hipStream_t) {
  stub::need({a.head, a.next, a.target, a.chain, a.pos, a.targets, a.rows, a.row_targets});
  stub::calls.push_back("shuffle");
  return hipGetLastError();
}
hipError_t shuffle_take(const ShuffleArgs &a, const uint32_t *order, hipStream_t) {
  stub::need({order, a.pos, a.targets, a.rows, a.row_targets});
  stub::calls.push_back("take");
  return hipGetLastError();
}
hipError_t zero(float *, uint32_t, hipStream_t) { return hipGetLastError(); }
}  // namespace mlp

}  // namespace gpuai
