// The routing-weight gradient's direct form, shared by the launch that computes
// it alone (permute.hip) and the one that forms the whole logit gradient
// (router.hip).
#pragma once

#include "vmoe_common.h"

namespace vmoe {

// Routing weights below this magnitude (zero and every bf16 denormal among
// them) take the direct form of their gradient: the dH GEMM's row sums hold
// w * (G W2^T) * relu(z)^2 rounded through bf16(w * (G W2^T)), and dividing
// them by such a w is 0 / 0 at w = 0 and loses the gradient's bits below.
constexpr float kTinyWeight = 0x1p-64f;

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Operands of dL/dw = sum_c (G[t] . W2[ewo[e] + c]) * pre[row][c]^2, e the
// expert whose rows [eto[e], eto[e+1]) hold `row`.
struct DirectWgrad {
  const uint16_t* gy;
  int64_t ldgy, gy_rows;
  const uint16_t* grad_scale;  // nullable
  const uint16_t* w2;
  int64_t ldw2;
  const uint16_t* pre;
  int64_t ldp;
  const int32_t *eto, *ewo, *widths;
  int E;
  int64_t hidden;
};

// dL/dw of token tok's row r, by a whole wave (one fp32 dot of length hidden
// per column, summed across the wave); every lane returns it.
__device__ __forceinline__ float direct_wgrad(const DirectWgrad& p, int32_t r, int64_t tok) {
  const int lane = threadIdx.x & (kWave - 1);
  int lo = 0, hi = p.E;  // eto[lo] <= r < eto[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (p.eto[mid] <= r) lo = mid; else hi = mid;
  }
  const int width = p.widths[lo];
  const int64_t col0 = p.ewo[lo];
  float s = 0.0f;
  if (tok < p.gy_rows) {
    const uint16_t* g = p.gy + tok * p.ldgy;
    const uint16_t* pr = p.pre + (int64_t)r * p.ldp;
    for (int c = 0; c < width; ++c) {
      const uint16_t* wr = p.w2 + (col0 + c) * p.ldw2;
      float d = 0.0f;
      for (int64_t j = lane; j < p.hidden; j += kWave) d += bf16_to_f32(g[j]) * bf16_to_f32(wr[j]);
      d = wave_sum(d);
      const float pc = bf16_to_f32(pr[c]);
      s += d * (pc * pc);
    }
  }
  if (p.grad_scale) s *= bf16_to_f32(*p.grad_scale);
  return s;
}

// The whole logit gradient of vmoe_moe_backward with routing-weight gradients
// in one launch (router.hip): the routing weights' gradients from the dH GEMM's
// row sums (row_dot [row][block of 64 columns]) or their direct form, their
// chain into the logits, and the auxiliary losses' gradient, with the
// roundings of the separate launches (bf16 weight gradients, each logit term,
// their sum). Losses without a gradient are null; all null: the chain alone.
struct LogitGrad {
  const uint16_t* logits;  // [T, E] contiguous, as grad
  int64_t T;
  int E, k, norm;
  const int32_t* sel;
  const float *lse, *f_i32, *coef, *wn;
  const float *g_z, *g_lb, *g_cl;
  const float* row_dot;
  int64_t ld_rd;
  int max_blocks;  // blocks a row of row_dot has
  const float* row_weight;
  const int32_t* assignment_row;
  int64_t rows;
  DirectWgrad direct;
  uint16_t* grad;
};
int router_logit_grad(const LogitGrad& a, vmoe_stream_t stream);

}  // namespace vmoe
