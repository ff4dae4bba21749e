// Device side of the learned per-level scheduler: the network's layout and
// its inference, shared by the stand-alone decision kernel and the
// level-end kernel (which decides the next level in the same launch).
#pragma once
#include "bfsx_internal.hpp"

namespace bfsx {

constexpr int IN = 8, H1 = 32, H2 = 32, OUT = 4;
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + H1 * IN, OFF_W2 = OFF_B1 + H1,
              OFF_B2 = OFF_W2 + H2 * H1, OFF_W3 = OFF_B2 + H2, OFF_B3 = OFF_W3 + OUT * H2,
              NPARAM = OFF_B3 + OUT;
static_assert(NPARAM == BFSX_SCHED_PARAMS, "parameter count");
static_assert(NPARAM % 4 == 0, "weights load as float4");

// The weights in LDS: rows of the three matrices one word apart, so that the
// lanes of a layer, which read one column at a time, hit different banks (a
// row of 32 words is a bank cycle: the second layer's 32 reads were 32-way
// conflicts).
constexpr uint32_t LDS_W1 = 0, LDS_B1 = LDS_W1 + H1 * (IN + 1), LDS_W2 = LDS_B1 + H1,
                   LDS_B2 = LDS_W2 + H2 * (H1 + 1), LDS_W3 = LDS_B2 + H2,
                   LDS_B3 = LDS_W3 + OUT * (H2 + 1), LDS_PARAM = LDS_B3 + OUT;
static_assert(IN % 4 == 0 && H1 % 4 == 0 && H2 % 4 == 0, "a float4 lies in one row");
struct SchedLds {
  float w[LDS_PARAM];
};

// The j-th four weights into their places.
__device__ __forceinline__ void stage_weights(SchedLds &s, int j, float4 v) {
  const uint32_t i = 4u * j;
  const uint32_t p = i < OFF_B1   ? LDS_W1 + i / IN * (IN + 1) + i % IN
                     : i < OFF_W2 ? LDS_B1 + (i - OFF_B1)
                     : i < OFF_B2 ? LDS_W2 + (i - OFF_W2) / H1 * (H1 + 1) + (i - OFF_W2) % H1
                     : i < OFF_W3 ? LDS_B2 + (i - OFF_B2)
                     : i < OFF_B3 ? LDS_W3 + (i - OFF_W3) / H2 * (H2 + 1) + (i - OFF_W3) % H2
                                  : LDS_B3 + (i - OFF_B3);
  s.w[p] = v.x;
  s.w[p + 1] = v.y;
  s.w[p + 2] = v.z;
  s.w[p + 3] = v.w;
}

// Lane k's value of x, in every lane.
__device__ __forceinline__ float lane_value(float x, int k) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), k));
}

// Inference by the first wave of a work-group (the others only pass), with
// the weights staged before a barrier: the inputs of
// frontier buffer `idx` from the control block, the three layers, and
// ctl->choice = argmin over the allowed kinds (fixed LLB when an output is
// NaN); inputs and outputs are recorded in the control block.  Returns the
// choice in the first wave (0 in the others).
//   x0 = log2((1+F)/(1+n))/32          x1 = log2((1+EF)/(1+nnz))/32
//   x2 = log2((1+UV)/(1+n))/32         x3 = log2((1+UE)/(1+nnz))/32
//   x4 = log2(1+EF/F)/16               x5 = log2(1+nnz/n)/16
//   x6 = log2(1+n)/32                  x7 = 1 if the last step was bottom-up
// F/EF: frontier vertices/edges, UV/UE: unvisited vertices/edges (isolated
// vertices count as visited).
// The decision is a chain of dependent operations, so the chain is short:
// the two logarithms of an input are taken in two lanes, and a layer's values
// go to the next one through scalar registers (no LDS round trip or barrier
// between the layers).  Learned searches against one LDS round trip and a
// barrier a layer: 1024^2 grid 3145 -> 3090 us, 4096^2 6980 -> 6890, R-MAT 19
// 106.0 -> 104.8, 22 175.2 -> 173.5, 24 305.5 -> 302.9.
__device__ __forceinline__ uint32_t decide_compute(LevelCtl *ctl, const SchedLds &S, uint32_t idx,
                                               uint64_t n_cols, uint64_t nnz, uint64_t n_iso,
                                               uint32_t allow_mask, int first) {
  if (threadIdx.x >= 64) return 0;
  const float *W = S.w;
  const int l = threadIdx.x;
  float x;
  {
    // lanes i and 32 + i compute input i (x = log2((1+a)/(1+b))/d with a, b,
    // d picked per lane): one the logarithm of 1+a, one that of 1+b
    const int i = l & (IN - 1);
    const double F = ctl->q_count[idx];
    const double EF = (double)ctl->q_edges[idx];
    const double vv = (double)ctl->visited_vertices + (double)n_iso;
    const double UV = vv < (double)n_cols ? (double)n_cols - vv : 0.0;
    const double ve = (double)ctl->visited_edges;
    const double UE = ve < (double)nnz ? (double)nnz - ve : 0.0;
    const double n = (double)n_cols, m = (double)nnz;
    const double a = i == 0 ? F : i == 1 ? EF : i == 2 ? UV : i == 3 ? UE
                   : i == 4 ? (F > 0 ? EF / F : 0.0) : i == 5 ? (n > 0 ? m / n : 0.0) : n;
    const double b = (i == 0 || i == 2) ? n : (i == 1 || i == 3) ? m : 0.0;
    const double c = l < 32 ? a : b;
    const double lg = log2(1.0 + (c > 0 ? c : 0.0));
    const double other = __shfl_xor(lg, 32, 64);
    x = (float)(lg - other) / ((i == 4 || i == 5) ? 16.f : 32.f);
    if (i == 7) x = (!first && ctl->choice == BFSX_PULL) ? 1.f : 0.f;
  }
  float h, g, y;
  {
    const int r = l & (H1 - 1);
    float s = W[LDS_B1 + r];
#pragma unroll
    for (int k = 0; k < IN; k++) s = fmaf(W[LDS_W1 + r * (IN + 1) + k], lane_value(x, k), s);
    h = s > 0.f ? s : 0.f;
  }
  {
    const int r = l & (H2 - 1);
    float s = W[LDS_B2 + r];
#pragma unroll
    for (int k = 0; k < H1; k++) s = fmaf(W[LDS_W2 + r * (H1 + 1) + k], lane_value(h, k), s);
    g = s > 0.f ? s : 0.f;
  }
  {
    const int r = l & (OUT - 1);
    float s = W[LDS_B3 + r];
#pragma unroll
    for (int k = 0; k < H2; k++) s = fmaf(W[LDS_W3 + r * (H2 + 1) + k], lane_value(g, k), s);
    y = s;
  }
  uint32_t best = 0;
  float bv = INFINITY;
  bool ok = true;
#pragma unroll
  for (int j = 0; j < OUT; j++) {
    const float v = lane_value(y, j);
    if (!(v == v)) ok = false;  // NaN
    if (((allow_mask >> j) & 1u) && v < bv) {
      bv = v;
      best = (uint32_t)j;
    }
  }
  const uint32_t picked = ok && bv < INFINITY ? best : (uint32_t)BFSX_LLB;
  if (l < IN) ctl->sched_in[l] = x;
  if (l < OUT) ctl->sched_out[l] = y;
  if (l == 0) {
    ctl->choice = picked;
    ctl->decisions += 1;
  }
  return picked;
}

__device__ __forceinline__ void decide_wave(LevelCtl *ctl, const float *Wg, uint32_t idx,
                                            uint64_t n_cols, uint64_t nnz, uint64_t n_iso,
                                            uint32_t allow_mask, int first) {
  __shared__ SchedLds S;
  for (int j = threadIdx.x; j < NPARAM / 4; j += 64)
    stage_weights(S, j, reinterpret_cast<const float4 *>(Wg)[j]);
  __syncthreads();
  decide_compute(ctl, S, idx, n_cols, nnz, n_iso, allow_mask, first);
}

}  // namespace bfsx
