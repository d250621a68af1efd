// mlp_kernels.hip -- gfx950 kernels of the 128-256-256-1 value network.
//
// MFMA v_mfma_f32_16x16x32_bf16 throughout: lane l supplies row l%16 of A and column l%16 of B
// for eight K values of its lane group l/16 (the same eight for A and B, which is all the dot
// product needs: every operand is stored with K contiguous, so each is one 16-byte read), and
// receives D[4*(l/16)+v][l%16], v = 0..3.
//
// What a matrix product reads from memory is kept in the order of its MFMA operands: fragment
// (16-wide tile, 32-deep slice) holds for lane l the eight K values of its group of row or column
// l%16 of the tile, 16 bytes per lane, so that a wave's load of one operand is 1 KB of consecutive
// memory.  As plain matrices a load touched sixteen lines, half of each: a workgroup's 320 KB of
// weights took 8.7 us of k_train_rows' 15.4.  That holds for the BF16 weight copies W1f, W2f
// (column = output, K = input) and W2rf (column = input, K = output) and for the activations and
// activation gradients of a training step Xf, H1f, dH2f, dH1f (K = row of the batch).
//
// A training step is two launches.  k_train_rows runs the forward and backward pass of kTrainRows
// (32) rows per workgroup up to the activation gradients, with the activations in LDS, and writes
// what the weight gradients need plus each block's partial sums of the vector gradients.  Every
// workgroup reads all of the BF16 weights (320 KB) from L2.  k_update forms a tile of dW1 or dW2 over
// the whole batch, or sums a vector gradient's partials, and applies Adam to it.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "checkers.h"
#include "mlp_kernels.h"

namespace gpuai {
namespace mlp {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Round to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint16_t to_bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ float from_bf(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// Workgroup barrier for exchanges through LDS only: this wave's LDS accesses complete, then
// s_barrier.  __syncthreads() also waits for the wave's global stores to complete, which costs a
// memory round trip after every store of activations or partial sums; nothing here reads back
// what the workgroup stored to global memory.  The memory clobber keeps the compiler from moving
// memory accesses across it.
__device__ __forceinline__ void lds_barrier() {
  __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// x plus the x of a lane of the same 16, by DPP (one instruction; a shuffle through LDS takes a
// round trip).  With equal values on the lanes that the earlier steps have joined, the sums are
// those of a butterfly: quad_perm 1032 and 2301 are the partners at distances 1 and 2, mirroring
// eight lanes then stands for distance 4 and mirroring sixteen for 8; rotations by 8, 4, 2 and 1
// stand for the distances in descending order.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
constexpr int kQuad1 = 0xB1, kQuad2 = 0x4E, kMirror8 = 0x141, kMirror16 = 0x140;
constexpr int kRotate = 0x120;  // + n: by n lanes

// Operand (column tile, slice) of a BF16 weight copy with `slices` 32-deep slices (see above).
__device__ __forceinline__ bf16x8 fragment(const uint16_t *W, int tile, int slices, int slice,
                                           int lane) {
  return *(const bf16x8 *)(W + ((tile * slices + slice) * 64 + lane) * 8);
}

// The four input planes of a position in the mover's frame (own men, own kings, opponent's men,
// opponent's kings), 32 squares each.
__device__ __forceinline__ uint32_t plane_bits(const mi_pos &p, int plane) {
  uint32_t own = p.turn ? __builtin_bitreverse32(p.p2) : p.p1;
  uint32_t opp = p.turn ? __builtin_bitreverse32(p.p1) : p.p2;
  uint32_t kings = p.turn ? __builtin_bitreverse32(p.kings) : p.kings;
  kings &= own | opp;
  return plane == 0 ? (own & ~kings) : plane == 1 ? (own & kings)
       : plane == 2 ? (opp & ~kings) : (opp & kings);
}

// Inference in one launch: encoding, both hidden layers and the output layer for FR rows per
// workgroup, with the activations in LDS: H1 = bf(relu(X W1 + b1)), H2 = bf(relu(H1 W2 + b2)),
// y = tanh(H2 . w3 + b3), the output layer summing four columns per lane and then over the wave
// with a butterfly.  Wave w computes output columns 32w..32w+31 of each layer as two 16x16 tiles.
// The pass is a chain of latencies (9 us for one row as for 4096 when each layer's weights were
// loaded where they are used), so every load is issued before the first value is needed (4.0 us).
constexpr int FR = 16, XP = 128 + 8, HP = 256 + 8;  // rows; LDS row pitches (BF16 elements)

__global__ void __launch_bounds__(512) k_forward(const mi_pos *pos, uint32_t n,
                                                const uint16_t *__restrict__ W1f,
                                                const float *__restrict__ b1,
                                                const uint16_t *__restrict__ W2f,
                                                const float *__restrict__ b2,
                                                const float *__restrict__ w3, const float *b3,
                                                float *y) {
  __shared__ __attribute__((aligned(16))) uint16_t X[FR][XP];
  __shared__ __attribute__((aligned(16))) uint16_t H[2][FR][HP];  // H1, H2
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, lr = lane & 15;
  const uint32_t r0 = blockIdx.x * FR;
  const int erow = t >> 4;  // encoding: threads 0..255, thread t -> row t/16, plane (t/4)%4, squares 8(t%4)..+7
  mi_pos q = {};
  if (t < FR * 16 && r0 + erow < n) q = pos[r0 + erow];
  bf16x8 w1p[4][2], w2p[8][2];  // this wave's weights: [slice][column tile]
#pragma unroll
  for (int s = 0; s < 4; s++)
#pragma unroll
    for (int c = 0; c < 2; c++) w1p[s][c] = fragment(W1f, wave * 2 + c, 4, s, lane);
#pragma unroll
  for (int s = 0; s < 8; s++)
#pragma unroll
    for (int c = 0; c < 2; c++) w2p[s][c] = fragment(W2f, wave * 2 + c, 8, s, lane);
  float b1c[2], b2c[2];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    b1c[c] = b1[wave * 32 + c * 16 + lr];
    b2c[c] = b2[wave * 32 + c * 16 + lr];
  }
  const float4 w3c = *(const float4 *)(w3 + lane * 4);
  const float b3c = b3[0];
  __asm__ volatile("" ::: "memory");  // the loads stay above the first wait
  if (t < FR * 16) {
    const int plane = (t >> 2) & 3, s0 = (t & 3) * 8;
    const uint32_t bits = plane_bits(q, plane) >> s0;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
      w[j] = ((bits >> (2 * j)) & 1u ? 0x3F80u : 0u) | ((bits >> (2 * j + 1)) & 1u ? 0x3F800000u : 0u);
    *(uint4 *)&X[erow][plane * 32 + s0] = uint4{w[0], w[1], w[2], w[3]};
  }
  lds_barrier();
  const int kg = (lane >> 4) * 8;  // this lane's eight K values within a slice
  f32x4 acc[2];
#pragma unroll
  for (int c = 0; c < 2; c++) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 4; s++) {  // layer 1: X[16][128] . W1
    const bf16x8 a = *(const bf16x8 *)&X[lr][s * 32 + kg];
#pragma unroll
    for (int c = 0; c < 2; c++)
      acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w1p[s][c], acc[c], 0, 0, 0);
  }
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      float x = acc[c][v] + b1c[c];
      x = x > 0.f ? x : 0.f;
      H[0][4 * (lane >> 4) + v][wave * 32 + c * 16 + lr] = to_bf(x);
      acc[c][v] = 0.f;
    }
  lds_barrier();
#pragma unroll
  for (int s = 0; s < 8; s++) {  // layer 2: H1[16][256] . W2
    const bf16x8 a = *(const bf16x8 *)&H[0][lr][s * 32 + kg];
#pragma unroll
    for (int c = 0; c < 2; c++)
      acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w2p[s][c], acc[c], 0, 0, 0);
  }
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      float x = acc[c][v] + b2c[c];
      x = x > 0.f ? x : 0.f;
      H[1][4 * (lane >> 4) + v][wave * 32 + c * 16 + lr] = to_bf(x);
    }
  lds_barrier();
  float part[FR / 8];
#pragma unroll
  for (int i = 0; i < FR / 8; i++) {  // output layer: wave w, rows 2w, 2w+1
    const uint16_t *h = &H[1][wave * (FR / 8) + i][lane * 4];
    float d = 0.f;
    d += from_bf(h[0]) * w3c.x;
    d += from_bf(h[1]) * w3c.y;
    d += from_bf(h[2]) * w3c.z;
    d += from_bf(h[3]) * w3c.w;
    d += __shfl_xor(d, 32);
    d += __shfl_xor(d, 16);
    part[i] = dpp_add<kRotate + 1>(
        dpp_add<kRotate + 2>(dpp_add<kRotate + 4>(dpp_add<kRotate + 8>(d))));
  }
  if (lane < FR / 8) {
    const uint32_t row = r0 + wave * (FR / 8) + lane;
    const float z = lane == 0 ? part[0] : part[1];
    if (row < n) y[row] = tanhf(z + b3c);
  }
}

// ---------------------------------------------------------------------------------------------
// Training.  Row r of the batch is pos[r] with target targets[r];
// rows n and up (to the multiple of kTrainRows) are padding: zero inputs and no loss.  The
// arithmetic: H1 = bf(relu(X W1 + b1)), H2 = bf(relu(H1 W2 + b2)), y = tanh(H2 . w3 + b3),
// dz = 2 (y - t)(1 - y^2) / n, dH2 = bf(dz w3) where H2 > 0, dH1 = bf(dH2 W2^T) where H1 > 0;
// dW1 = X^T dH1, dW2 = H1^T dH2, b1 and b2 the column sums of dH1 and dH2, w3 = sum of dz H2,
// b3 = sum of dz, loss = sum of (y - t)^2 / n.

constexpr int KR = (int)kTrainRows;  // rows per workgroup of k_train_rows
constexpr int RT = KR / 16;          // row tiles
static_assert(KR == 32, "the row pass assigns its threads for 32 rows");

// The forward and backward pass of KR rows: wave w (of eight) owns columns 32w..32w+31 of each
// 256-wide layer (two 16x16 column tiles, RT row tiles).  Each workgroup reads the whole of the
// BF16 weights (320 KB), so the rows per workgroup set the weight traffic through L2.  A operands
// come from LDS ([row][k]), B operands from the BF16 weight copies in operand order.  Every global
// load is issued at the start (a dependent load waits out the memory latency); the pass then only
// computes and stores.  A lane's four values of a tile are four consecutive rows of one column, half
// of an operand's 16 bytes, so what the weight gradients need goes to memory from registers.
// A wave's 15.4 us in it at 4096 rows became 7.1 (the loads 8.7 -> 3.0): operand-order weights, two
// waves instead of all fetching the positions, no staging of the transposed tiles through LDS
// (three barriers of nine), sums over 16 lanes by DPP, conversions by instruction, and the output
// layer computed by every wave for itself.
__global__ void __launch_bounds__(512) k_train_rows(TrainArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t Xs[KR][XP];
  __shared__ __attribute__((aligned(16))) uint16_t H1s[KR][HP];
  __shared__ __attribute__((aligned(16))) uint16_t dH2s[KR][HP];
  __shared__ uint32_t planes[4][KR];
  __shared__ float red[8][KR];
  __shared__ float tgts[KR];
  __shared__ __attribute__((aligned(16))) float dzs[8][KR];  // each wave's own
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int lr = lane & 15, kg = (lane >> 4) * 8;
  const uint32_t r0 = blockIdx.x * KR, nsl = a.slices;
  float *pv = a.pV + (size_t)blockIdx.x * kVecSlots;
  // the wave's columns, rotated by the block index: all workgroups read the same weights at the
  // same time, and the rotation spreads their requests over different lines of L2
  const int cw = ((wave + (int)blockIdx.x) & 7) * 32;
  // Loads, issued before any is used, in an order that lets each wait cover only what it needs --
  // loads complete in issue order as far as the wait counter goes: the position and target of this
  // thread's row (threads 0..127: row t/4, plane t%4), the wave's W1 operands, then the W2 operands
  // of both directions and the biases.  The empty asm statements keep the compiler from reordering
  // the groups.
  const int erow = t >> 2;
  const bool encodes = t < 4 * KR, evalid = r0 + erow < a.n;
  const uint32_t esrc = min(r0 + erow, a.n - 1u);
  mi_pos epos = {};
  float tgt = 0.f;
  if (encodes) {
    epos = a.pos[esrc];
    tgt = a.targets[esrc];
  }
  __asm__ volatile("" ::: "memory");
  bf16x8 w1p[4][2], w2p[8][2], w2rp[8][2];  // this wave's weights: [slice][column tile]
#pragma unroll
  for (int s = 0; s < 4; s++)
#pragma unroll
    for (int c = 0; c < 2; c++) w1p[s][c] = fragment(a.W1f, cw / 16 + c, 4, s, lane);
  __asm__ volatile("" ::: "memory");
#pragma unroll
  for (int s = 0; s < 8; s++)
#pragma unroll
    for (int c = 0; c < 2; c++) w2p[s][c] = fragment(a.W2f, cw / 16 + c, 8, s, lane);
  float b1c[2], b2c[2], w3c[2];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    b1c[c] = a.b1[cw + c * 16 + lr];
    b2c[c] = a.b2[cw + c * 16 + lr];
    w3c[c] = a.w3[cw + c * 16 + lr];
  }
  const float b3 = a.b3[0];
#pragma unroll
  for (int s = 0; s < 8; s++)
#pragma unroll
    for (int c = 0; c < 2; c++) w2rp[s][c] = fragment(a.W2rf, cw / 16 + c, 8, s, lane);
  __asm__ volatile("" ::: "memory");
  if (encodes) {
    planes[t & 3][erow] = evalid ? plane_bits(epos, t & 3) : 0u;
    if ((t & 3) == 0) tgts[erow] = tgt;
  }
  lds_barrier();
  {  // X in LDS (thread t: row t/16, plane (t/4)%4, squares 8(t%4)..+7) and Xf (input t/4, rows 8(t%4)..)
    const int row = t >> 4, plane = (t >> 2) & 3, s0 = (t & 3) * 8;
    const uint32_t bits = planes[plane][row] >> s0;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
      w[j] = ((bits >> (2 * j)) & 1u ? 0x3F80u : 0u) | ((bits >> (2 * j + 1)) & 1u ? 0x3F800000u : 0u);
    *(uint4 *)&Xs[row][plane * 32 + s0] = uint4{w[0], w[1], w[2], w[3]};
    const int f = t >> 2, rows0 = (t & 3) * 8;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t lo = planes[f >> 5][rows0 + 2 * j] >> (f & 31);
      const uint32_t hi = planes[f >> 5][rows0 + 2 * j + 1] >> (f & 31);
      w[j] = (lo & 1u ? 0x3F80u : 0u) | (hi & 1u ? 0x3F800000u : 0u);
    }
    *(uint4 *)(a.Xf + ((size_t)((f >> 4) * nsl + blockIdx.x) * 64 + (t & 3) * 16 + (f & 15)) * 8) =
        uint4{w[0], w[1], w[2], w[3]};
  }
  lds_barrier();
  // this lane's four rows of (column col, row tile r), from registers to the operands G: half of
  // the eight K values of K group 2r + lane/32 (the block's rows are slice blockIdx.x)
  auto store_rows = [&](uint16_t *G, int col, int r, const uint16_t h[4]) {
    *(uint2 *)(G + ((size_t)((col >> 4) * nsl + blockIdx.x) * 64 + (2 * r + (lane >> 5)) * 16 + lr) * 8 +
               (lane >> 4 & 1) * 4) =
        uint2{(uint32_t)h[0] | (uint32_t)h[1] << 16, (uint32_t)h[2] | (uint32_t)h[3] << 16};
  };
  f32x4 acc[RT][2];
  // ---- layer 1: X[KR][128] . W1 -> H1 (LDS and memory)
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int c = 0; c < 2; c++) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 4; s++) {
#pragma unroll
    for (int r = 0; r < RT; r++) {
      const bf16x8 x = *(const bf16x8 *)&Xs[r * 16 + lr][s * 32 + kg];
#pragma unroll
      for (int c = 0; c < 2; c++)
        acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, w1p[s][c], acc[r][c], 0, 0, 0);
    }
  }
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const int col = cw + c * 16 + lr;
    const float bias = b1c[c];
#pragma unroll
    for (int r = 0; r < RT; r++) {
      uint16_t h[4];
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const float x = acc[r][c][v] + bias;
        h[v] = to_bf(x > 0.f ? x : 0.f);
        H1s[r * 16 + 4 * (lane >> 4) + v][col] = h[v];
      }
      store_rows(a.H1f, col, r, h);
    }
  }
  lds_barrier();
  // ---- layer 2: H1[KR][256] . W2 -> H2 (registers), the output layer, dz
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int c = 0; c < 2; c++) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 8; s++) {
#pragma unroll
    for (int r = 0; r < RT; r++) {
      const bf16x8 h = *(const bf16x8 *)&H1s[r * 16 + lr][s * 32 + kg];
#pragma unroll
      for (int c = 0; c < 2; c++)
        acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h, w2p[s][c], acc[r][c], 0, 0, 0);
    }
  }
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const float bias = b2c[c];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const float x = acc[r][c][v] + bias;
        acc[r][c][v] = from_bf(to_bf(x > 0.f ? x : 0.f));  // H2
      }
  }
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int v = 0; v < 4; v++) {  // this wave's share of the row's dot product with w3
      float d = 0.f;
#pragma unroll
      for (int c = 0; c < 2; c++) d += acc[r][c][v] * w3c[c];
      d = dpp_add<kMirror16>(dpp_add<kMirror8>(dpp_add<kQuad2>(dpp_add<kQuad1>(d))));
      if (lr == 0) red[cw / 32][r * 16 + 4 * (lane >> 4) + v] = d;
    }
  lds_barrier();
  // output and dz per row (lane = row, both halves of the wave alike), by every wave for itself;
  // the shares are added in the order of their columns' waves in this workgroup
  float dz = 0.f, loss = 0.f;
  {
    float dot = 0.f;
#pragma unroll
    for (int w = 0; w < 8; w++) dot += red[(w + (int)blockIdx.x) & 7][lane % KR];
    const float y = tanhf(dot + b3);
    if (r0 + lane % KR < a.n) {
      const float e = y - tgts[lane % KR];
      dz = 2.f * e * (1.f - y * y) / (float)a.n;
      loss = e * e / (float)a.n;
    }
    if (lane < KR) dzs[wave][lane] = dz;
  }
  {  // dH2 = bf(dz w3) where H2 > 0 (LDS and memory); b2 and w3 partials
    f32x4 d4[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) d4[r] = *(const f32x4 *)&dzs[wave][r * 16 + 4 * (lane >> 4)];
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const int col = cw + c * 16 + lr;
      float sb2 = 0.f, sw3 = 0.f;
#pragma unroll
      for (int r = 0; r < RT; r++) {
        uint16_t g[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const float d = d4[r][v], h = acc[r][c][v];
          g[v] = to_bf(h > 0.f ? d * w3c[c] : 0.f);
          dH2s[r * 16 + 4 * (lane >> 4) + v][col] = g[v];
          sb2 += from_bf(g[v]);
          sw3 += d * h;
        }
        store_rows(a.dH2f, col, r, g);
      }
      sb2 += __shfl_xor(sb2, 16);
      sw3 += __shfl_xor(sw3, 16);
      sb2 += __shfl_xor(sb2, 32);
      sw3 += __shfl_xor(sw3, 32);
      if (lane < 16) {
        pv[256 + col] = sb2;
        pv[512 + col] = sw3;
      }
    }
  }
  lds_barrier();
  // ---- dH1 = bf(dH2 . W2^T) where H1 > 0; b1 partials
#pragma unroll
  for (int r = 0; r < RT; r++)
#pragma unroll
    for (int c = 0; c < 2; c++) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 8; s++) {
#pragma unroll
    for (int r = 0; r < RT; r++) {
      const bf16x8 g = *(const bf16x8 *)&dH2s[r * 16 + lr][s * 32 + kg];
#pragma unroll
      for (int c = 0; c < 2; c++)
        acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g, w2rp[s][c], acc[r][c], 0, 0, 0);
    }
  }
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const int col = cw + c * 16 + lr;
    float sb1 = 0.f;
#pragma unroll
    for (int r = 0; r < RT; r++) {
      uint16_t g[4];
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int row = r * 16 + 4 * (lane >> 4) + v;
        g[v] = to_bf(H1s[row][col] ? acc[r][c][v] : 0.f);  // H1 >= 0: nonzero is > 0
        sb1 += from_bf(g[v]);
      }
      store_rows(a.dH1f, col, r, g);
    }
    sb1 += __shfl_xor(sb1, 16);
    sb1 += __shfl_xor(sb1, 32);
    if (lane < 16) pv[col] = sb1;
  }
  if (wave == 7) {  // the b3 and loss partials: rows on lanes 0..31
    float d = lane < KR ? dz : 0.f, l = lane < KR ? loss : 0.f;
    for (int off = 32; off >= 1; off >>= 1) {
      d += __shfl_xor(d, off);
      l += __shfl_xor(l, off);
    }
    if (lane == 0) {
      pv[768] = d;
      pv[769] = l;
    }
  }
}

// One Adam step of parameter p with gradient g, from its values w, m, v (loaded by the caller
// beforehand, together with the gradient's partials); returns the new value.
__device__ __forceinline__ float adam_step(const AdamArgs &a, uint32_t p, float g, float w, float m,
                                           float v) {
  if (a.grads) a.grads[p] = g;
  if (a.update) {
    m = a.beta1 * m + a.omb1 * g;
    v = a.beta2 * v + a.omb2 * g * g;
    a.m[p] = m;
    a.v[p] = v;
    w -= a.lr * (m * a.c1) / (sqrtf(v * a.c2) + a.eps);
    a.w[p] = w;
  }
  return w;
}

// The sum of n partials at p, p + stride, ... in order, their loads issued 16 at a time.
__device__ __forceinline__ float sum_partials(const float *p, size_t stride, uint32_t n) {
  float g = 0.f;
  for (uint32_t s0 = 0; s0 < n; s0 += 16u) {
    float x[16];
#pragma unroll
    for (uint32_t j = 0; j < 16u; j++) x[j] = s0 + j < n ? p[(s0 + j) * stride] : 0.f;
#pragma unroll
    for (uint32_t j = 0; j < 16u; j++) g += x[j];
  }
  return g;
}

// Weight gradients and Adam in one launch.  A workgroup (eight waves) forms a 32x16 tile of dW1 =
// X^T dH1 ([128 in][256 out]) or dW2 = H1^T dH2 ([256][256]) over the whole batch, so that no
// partial product leaves it, and updates the tile's parameters and their BF16 copies.  The batch
// is summed as ever in splits of kWSplitRows rows: wave w forms the splits w, w + 8, ... (two MFMA
// row tiles, one operand load each per slice, half a load for the shared column tile), their sums
// meet in LDS and every gradient adds them in split order (training is deterministic).
// What bounds it is the operands' way to the compute units: 384 KB per workgroup at 4096 rows.
// The 192 tiles are dealt to the XCDs (workgroup b runs on XCD b % 8) by halves of the inputs and
// quarters of the outputs, so that one XCD's L2 fetches 2.5 MB of the 7.3.  The launches it
// replaces, 64x64 tiles per split with their partials (12.6 MB at 4096 rows) written and read
// back, took 12.4 us of kernel time a step; this one takes 6.5.
// The last workgroups take the vector parameters: b1, b2, w3 and b3 are sums over the row pass's
// row blocks (pV; slot 769 holds the loss), as eight sums over consecutive eighths of the blocks,
// added in order.
constexpr uint32_t UI = 32, UO = 16;  // tile: inputs x outputs
constexpr uint32_t kTilesW2 = (256 / UI) * (256 / UO), kTilesW1 = (128 / UI) * (256 / UO);
constexpr uint32_t kTiles = kTilesW1 + kTilesW2;
constexpr uint32_t kVecPerWg = 64, kVecWgs = (770 + kVecPerWg - 1) / kVecPerWg;
constexpr uint32_t kSplitsAtOnce = 32;        // splits whose sums LDS holds
constexpr uint32_t kValue = 64 + 16;          // pitch of one accumulator register's 64 lanes
constexpr uint32_t kSplitSlices = kWSplitRows / 32;
static_assert(kTiles % 8 == 0 && kWSplitRows % 32 == 0, "tiles per XCD, slices per split");

__global__ void __launch_bounds__(512) k_update(AdamArgs a) {
  __shared__ float sums[kSplitsAtOnce][8 * kValue];  // [split][row tile, register][lane]
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6, b = blockIdx.x;
  if (b < kTiles) {
    const uint32_t xcd = b & 7u, j = b >> 3;
    const bool w1 = j >= kTilesW2 / 8u;
    const uint32_t j1 = w1 ? j - kTilesW2 / 8u : j;
    const uint32_t it = (xcd >> 2) * (w1 ? 2u : 4u) + (j1 >> 2), ot = (xcd & 3u) * 4u + (j1 & 3u);
    const uint16_t *A = (w1 ? a.Xf : a.H1f) + (size_t)it * 2u * a.slices * 512u + lane * 8u;
    const uint16_t *B = (w1 ? a.dH1f : a.dH2f) + (size_t)ot * a.slices * 512u + lane * 8u;
    // this thread's parameter
    const uint32_t il = t / UO, ol = t % UO;
    const uint32_t p = (w1 ? MI_MLP_OFF_W1 : MI_MLP_OFF_W2) + (it * UI + il) * 256u + ot * UO + ol;
    const float w = a.w[p], m = a.m[p], v = a.v[p];
    const uint32_t used = a.rows / 32u;  // slices of the batch
    float g = 0.f;
    for (uint32_t s0 = 0; s0 < a.splits; s0 += kSplitsAtOnce) {
      if (s0) __syncthreads();  // the sums of the splits before have been read
      const uint32_t n = min(kSplitsAtOnce, a.splits - s0);
      // split q of these from its operands x, y
      auto form = [&](uint32_t q, const bf16x8 (&x)[kSplitSlices][2], const bf16x8 (&y)[kSplitSlices]) {
        f32x4 acc[2];
        acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (uint32_t k = 0; k < kSplitSlices; k++)
#pragma unroll
          for (uint32_t r = 0; r < 2u; r++)
            acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[k][r], y[k], acc[r], 0, 0, 0);
#pragma unroll
        for (uint32_t r = 0; r < 2u; r++)
#pragma unroll
          for (uint32_t u = 0; u < 4u; u++) sums[q][(r * 4u + u) * kValue + lane] = acc[r][u];
      };
      if ((s0 + kSplitsAtOnce) * kSplitSlices <= used) {
        // a full round: the wave's splits all in flight
        constexpr uint32_t W = kSplitsAtOnce / 8u;
        bf16x8 x[W][kSplitSlices][2], y[W][kSplitSlices];
#pragma unroll
        for (uint32_t i = 0; i < W; i++)
#pragma unroll
          for (uint32_t k = 0; k < kSplitSlices; k++) {
            const size_t at = (size_t)((s0 + wave + 8u * i) * kSplitSlices + k) * 512u;
#pragma unroll
            for (uint32_t r = 0; r < 2u; r++) x[i][k][r] = *(const bf16x8 *)(A + r * a.slices * 512u + at);
            y[i][k] = *(const bf16x8 *)(B + at);
          }
        __asm__ volatile("" ::: "memory");
#pragma unroll
        for (uint32_t i = 0; i < W; i++) form(wave + 8u * i, x[i], y[i]);
      } else {
        for (uint32_t q = wave; q < n; q += 8u) {
          bf16x8 x[kSplitSlices][2], y[kSplitSlices];
#pragma unroll
          for (uint32_t k = 0; k < kSplitSlices; k++) {
            const uint32_t sl = (s0 + q) * kSplitSlices + k;
            const bool in = sl < used;  // slices past the batch read as zero
#pragma unroll
            for (uint32_t r = 0; r < 2u; r++)
              x[k][r] = in ? *(const bf16x8 *)(A + (r * a.slices + (size_t)sl) * 512u) : bf16x8{};
            y[k] = in ? *(const bf16x8 *)(B + (size_t)sl * 512u) : bf16x8{};
          }
          form(q, x, y);
        }
      }
      __syncthreads();
      const float *mine = &sums[0][((il >> 4) * 4u + (il & 3u)) * kValue + (il & 15u) / 4u * 16u + ol];
      if (n == kSplitsAtOnce) {
#pragma unroll
        for (uint32_t q = 0; q < kSplitsAtOnce; q++) g += mine[q * 8u * kValue];
      } else {
        for (uint32_t q = 0; q < n; q++) g += mine[q * 8u * kValue];
      }
    }
    __shared__ uint16_t tile[UI][UO + 2];
    tile[il][ol] = to_bf(adam_step(a, p, g, w, m, v));
    lds_barrier();
    // the copies: a 16x16 tile of the matrix is 512 consecutive bytes of each; element e of its
    // 256 is K group e/128, column (e/8)%16, K value e%8
    const uint32_t e = t & 255u, i16 = (t >> 8) * 16u, kt = (e >> 7) * 8u + (e & 7u), ct = (e >> 3) & 15u;
    auto at = [&](uint32_t col0, uint32_t k0, uint32_t slices) {
      return ((col0 / 16u * slices + k0 / 32u) * 64u + k0 % 32u / 8u * 16u) * 8u + e;
    };
    const uint32_t i0 = it * UI + i16, o0 = ot * UO;
    if (w1) {
      a.W1f[at(o0, i0, 4u)] = tile[i16 + kt][ct];
    } else {
      a.W2f[at(o0, i0, 8u)] = tile[i16 + kt][ct];
      a.W2rf[at(i0, o0, 8u)] = tile[i16 + ct][kt];
    }
    return;
  }
  float(*eighth)[kVecPerWg] = (float(*)[kVecPerWg])&sums[0][0];
  const uint32_t sl = t % kVecPerWg, e = t / kVecPerWg;  // slot in the workgroup, eighth
  const uint32_t slot = (b - kTiles) * kVecPerWg + sl;   // b1 0-255, b2 256-511, w3 512-767,
  const uint32_t per = (a.blocks + 7u) / 8u;             // b3 768, loss 769
  const uint32_t lo = min(e * per, a.blocks), hi = min(lo + per, a.blocks);
  eighth[e][sl] = slot <= 769u ? sum_partials(a.pV + (size_t)lo * kVecSlots + slot, kVecSlots, hi - lo)
                               : 0.f;
  lds_barrier();
  if (e != 0u || slot > 769u) return;
  float g = 0.f;
#pragma unroll
  for (int k = 0; k < 8; k++) g += eighth[k][sl];
  if (slot == 769u) {
    if (a.loss_out) *a.loss_out = g;
    return;
  }
  const uint32_t p = slot < 256u ? MI_MLP_OFF_B1 + slot : MI_MLP_OFF_B2 + (slot - 256u);
  adam_step(a, p, g, a.w[p], a.m[p], a.v[p]);
}

// An epoch's order: the Fisher-Yates shuffle p = 0..n-1, for i = n-1 .. 1 swap(p[i], p[j(i)]) with
// j(i) = word (n-1-i) of the stream mod (i + 1), computed without running it.  Position i is last
// touched at its own step, when it takes what stands on j(i).  What stands on position x at step i
// <= x' was put there by the last step before i that targeted x, that is the smallest i' > i with
// j(i') = x, and is what stood on i' at that step; without such a step it is x itself.  So with
// chain(x) = the smallest i' > x with j(i') = x, the value comes from following chain() to its end.
// The steps that target a position are linked in a list per position (k_shuffle_link; one or two
// on average, ln n at most positions), chain() is read off the lists (k_shuffle_chain), and every
// position follows its own (k_shuffle_order), which copies what it finds into the epoch's order, so
// that the steps read consecutive rows.  262,144 positions: 26 us against 0.7 ms on the host with
// the upload of its result; 8M: 1.2 ms against 38.  A step of 4096 rows takes 19.7 us from
// consecutive rows, 20.2 when it looks the order up itself; the shuffle's share of a step, which it
// takes either way but for the copy, is 0.4 us of 262,144 positions and 0.6 to 0.8 of 2M and 8M.
constexpr uint32_t kNone = 0xFFFFFFFFu;

__global__ void __launch_bounds__(256) k_shuffle_clear(uint32_t *head, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) head[i] = kNone;
}

// Smallest i' > i in the list of position x, or kNone.
__device__ __forceinline__ uint32_t step_after(const uint32_t *head, const uint32_t *next, uint32_t x,
                                               uint32_t i) {
  uint32_t best = kNone;
  for (uint32_t k = head[x]; k != kNone; k = next[k])
    if (k > i && k < best) best = k;
  return best;
}

__global__ void __launch_bounds__(256) k_shuffle_link(ShuffleArgs a) {
  const uint32_t b = blockIdx.x * 256u + threadIdx.x;  // word block: steps n-1-4b .. n-4-4b
  if (b >= (a.n + 2u) / 4u) return;                    // n - 1 steps
  uint32_t w[4];
  ck::philox(b, 0u, ck::TAG_MLP, 1u, a.seed, a.epoch, w);
#pragma unroll
  for (uint32_t k = 0; k < 4u; k++) {
    const uint32_t c = 4u * b + k;
    if (c + 1u >= a.n) return;
    const uint32_t i = a.n - 1u - c, j = ck::mod_u32(w[k], i + 1u);
    a.target[i] = j;
    a.next[i] = atomicExch(&a.head[j], i);
  }
}

__global__ void __launch_bounds__(256) k_shuffle_chain(ShuffleArgs a) {
  const uint32_t x = blockIdx.x * 256u + threadIdx.x;
  if (x < a.n) a.chain[x] = step_after(a.head, a.next, x, x);
}

__global__ void __launch_bounds__(256) k_shuffle_order(ShuffleArgs a) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= a.n) return;
  uint32_t x = i ? a.target[i] : 0u;
  uint32_t k = step_after(a.head, a.next, x, i);
  while (k != kNone) {  // (strictly ascending)
    x = k;
    k = a.chain[x];
  }
  a.rows[i] = a.pos[x];
  a.row_targets[i] = a.targets[x];
}

// The same from an order made on the host.
__global__ void __launch_bounds__(256) k_shuffle_take(ShuffleArgs a, const uint32_t *order) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= a.n) return;
  a.rows[i] = a.pos[order[i]];
  a.row_targets[i] = a.targets[order[i]];
}

__global__ void k_zero(float *p, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

}  // namespace

hipError_t forward(const mi_pos *pos, uint32_t n, const uint16_t *W1f, const float *b1,
                   const uint16_t *W2f, const float *b2, const float *w3, const float *b3, float *y,
                   hipStream_t stream) {
  hipLaunchKernelGGL(k_forward, dim3((n + FR - 1) / FR), dim3(512), 0, stream, pos, n, W1f, b1,
                     W2f, b2, w3, b3, y);
  return hipGetLastError();
}

hipError_t train_rows(const TrainArgs &a, uint32_t rows, hipStream_t stream) {
  if (rows % KR || rows == 0 || rows / 32u > a.slices || a.n == 0 || a.n > rows)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_train_rows, dim3(rows / KR), dim3(512), 0, stream, a);
  return hipGetLastError();
}

hipError_t update(const AdamArgs &a, hipStream_t stream) {
  if (a.rows % KR || a.rows / 32u > a.slices || a.blocks * KR != a.rows ||
      a.splits != (a.rows + kWSplitRows - 1) / kWSplitRows)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_update, dim3(kTiles + kVecWgs), dim3(512), 0, stream, a);
  return hipGetLastError();
}

hipError_t shuffle(const ShuffleArgs &a, hipStream_t stream) {
  if (a.n == 0) return hipErrorInvalidValue;
  const dim3 block(256), all((a.n + 255u) / 256u), words(((a.n + 2u) / 4u + 255u) / 256u);
  hipLaunchKernelGGL(k_shuffle_clear, all, block, 0, stream, a.head, a.n);
  if (a.n > 1u) hipLaunchKernelGGL(k_shuffle_link, words, block, 0, stream, a);
  hipLaunchKernelGGL(k_shuffle_chain, all, block, 0, stream, a);
  hipLaunchKernelGGL(k_shuffle_order, all, block, 0, stream, a);
  return hipGetLastError();
}

hipError_t shuffle_take(const ShuffleArgs &a, const uint32_t *order, hipStream_t stream) {
  hipLaunchKernelGGL(k_shuffle_take, dim3((a.n + 255u) / 256u), dim3(256), 0, stream, a, order);
  return hipGetLastError();
}

hipError_t zero(float *p, uint32_t n, hipStream_t stream) {
  hipLaunchKernelGGL(k_zero, dim3((n + 255) / 256), dim3(256), 0, stream, p, n);
  return hipGetLastError();
}

}  // namespace mlp
}  // namespace gpuai
