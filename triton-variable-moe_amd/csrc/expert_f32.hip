// The float32 layer after its router Linear, one call per direction, as
// expert.hip has it for bf16: top-k (with the routing counts where
// vmoe_router_topk_hist_f32 applies), routing, fp32 grouped GEMMs, weighted
// combine and auxiliary losses (TritonMoEMLP.forward, triton_moe/moe.py:167-303
// of the reference, whose kernels are dtype-generic), and their backward.
// Host code only: the kernels, operands and order of the per-kernel path, whose
// Python wrappers took more time than the kernels of a small layer (4 x 64
// tokens, 128 wide, 4 experts of 256: 157 us of kernels in a step of 500-560).
//
// Buffers are the caller's (vmoe_moe_f32_layout): `saved` is kept for the
// backward, the scratch of each direction is not. Slots start on 256 bytes.
#include <algorithm>

#include "vmoe_common.h"

namespace vmoe {
namespace {

struct F32Layout {
  int64_t A = 0, cap = 0;
  bool counted = false;
  int64_t partial_rows = 0;
  size_t route_ws_bytes = 0;
  // saved
  int64_t row_src, gmap, arow, eto, ptpe, tpe, h, pre, wts, lse, f_i, saved;
  // forward scratch
  int64_t sel, bin_ids, indices, bins, pbins, info, y, partial, route_ws, p_i, f_scratch;
  // backward scratch: the gathered gradient rows, later the dX rows; GA
  int64_t rows, ga, b_scratch;
};

bool f32_layout(int64_t T, int E, int k, int b, int64_t d, int64_t w, F32Layout& L) {
  if (T < 0 || E <= 0 || k <= 0 || b <= 0 || d <= 0 || w <= 0 || E > 2048 || k > kWave)
    return false;
  L.A = T * k;
  L.cap = L.A + (int64_t)E * (b - 1);
  const int hist = T > 0 ? vmoe_router_topk_hist_blocks(T, E, k) : 0;
  L.counted = hist > 0;
  L.partial_rows = L.counted ? hist
                             : (int64_t)(vmoe_router_partial_floats(std::max<int64_t>(T, 1), E) /
                                         (size_t)(E + 1));
  L.route_ws_bytes = L.counted ? vmoe_route_counted_workspace_bytes(T, E, k)
                               : vmoe_route_workspace_bytes(L.A, E);
  int64_t off = 0;
  auto slot = [&](int64_t words) {
    const int64_t o = off;
    off += (std::max<int64_t>(4 * words, 4) + 255) / 256 * 256;
    return o;
  };
  L.row_src = slot(L.cap);
  L.gmap = slot(L.cap);
  L.arow = slot(L.A);
  L.eto = slot(E + 1);
  L.ptpe = slot(E);
  L.tpe = slot(E);
  L.h = slot(L.cap * w);
  L.pre = slot(L.cap * w);
  L.wts = slot(L.A);
  L.lse = slot(T);
  L.f_i = slot(E);
  L.saved = off;
  off = 0;
  L.sel = slot(L.A);
  L.bin_ids = slot(L.A);
  L.indices = slot(L.A);
  L.bins = slot(E);
  L.pbins = slot(E);
  L.info = slot(VMOE_INFO_LEN);
  L.y = slot(L.cap * d);
  L.partial = slot(L.partial_rows * ((int64_t)E + 1));
  L.route_ws = slot(((int64_t)L.route_ws_bytes + 3) / 4);
  L.p_i = slot(E);
  L.f_scratch = off;
  off = 0;
  L.rows = slot(L.cap * d);
  L.ga = slot(L.cap * w);
  L.b_scratch = off;
  return true;
}

template <typename T>
T* at(void* base, int64_t off) {
  return reinterpret_cast<T*>(static_cast<char*>(base) + off);
}
template <typename T>
const T* at(const void* base, int64_t off) {
  return reinterpret_cast<const T*>(static_cast<const char*>(base) + off);
}

}  // namespace
}  // namespace vmoe

using namespace vmoe;

#define VMOE_TRY(expr)              \
  do {                              \
    const int st_ = (expr);         \
    if (st_ != VMOE_OK) return st_; \
  } while (0)

extern "C" int vmoe_moe_f32_layout(int64_t num_tokens, int32_t num_experts, int32_t top_k,
                                   int32_t block_size, int64_t hidden, int64_t max_width,
                                   int64_t* out) {
  F32Layout L;
  if (!out || !f32_layout(num_tokens, num_experts, top_k, block_size, hidden, max_width, L))
    return VMOE_ERR_INVALID_ARG;
  out[0] = L.saved;
  out[1] = L.f_scratch;
  out[2] = L.b_scratch;
  return VMOE_OK;
}

extern "C" int vmoe_moe_f32_forward(const float* logits, int64_t num_tokens, int32_t num_experts,
                                    int32_t top_k, int32_t normalize, int32_t block_size,
                                    const float* x, int64_t ldx, const float* w1, int64_t ldw1,
                                    const float* w2, int64_t ldw2, const int32_t* ewo,
                                    const int32_t* widths, int64_t hidden, int64_t max_width,
                                    const float* coef, const float* widths_normalized,
                                    void* saved, void* scratch, float* out, int64_t ldo,
                                    float* z_loss, float* losses, float* f_i,
                                    vmoe_stream_t stream) {
  F32Layout L;
  if (!f32_layout(num_tokens, num_experts, top_k, block_size, hidden, max_width, L))
    return VMOE_ERR_INVALID_ARG;
  if (num_tokens == 0) return VMOE_OK;
  if (!logits || !x || !w1 || !w2 || !ewo || !widths || !coef || !widths_normalized || !saved ||
      !scratch || !out || !z_loss || !losses || !f_i)
    return VMOE_ERR_INVALID_ARG;
  const int E = num_experts, k = top_k;
  const int64_t T = num_tokens;
  int32_t* sel = at<int32_t>(scratch, L.sel);
  float* wts = at<float>(saved, L.wts);
  float* lse = at<float>(saved, L.lse);
  float* partial = at<float>(scratch, L.partial);
  void* rws = at<void>(scratch, L.route_ws);
  const size_t nfl = (size_t)L.partial_rows * (size_t)(E + 1);
  if (L.counted)
    VMOE_TRY(vmoe_router_topk_hist_f32(logits, E, T, E, k, normalize, wts, sel, nullptr, nullptr,
                                       lse, partial, nfl, nullptr, rws, L.route_ws_bytes, stream));
  else
    VMOE_TRY(vmoe_router_topk_f32(logits, E, T, E, k, normalize, wts, sel, nullptr, nullptr, lse,
                                  partial, nfl, nullptr, stream));
  int32_t* tpe = at<int32_t>(saved, L.tpe);
  int32_t* gmap = at<int32_t>(saved, L.gmap);
  int32_t* arow = at<int32_t>(saved, L.arow);
  int32_t* eto = at<int32_t>(saved, L.eto);
  int32_t* ptpe = at<int32_t>(saved, L.ptpe);
  // pad rows of the map are -1 (the GEMMs' gather reads zeros for them)
  VMOE_TRY((L.counted ? vmoe_route_counted : vmoe_route)(
      sel, 0, L.A, E, k, block_size, VMOE_ROUND_UP, at<int32_t>(scratch, L.bin_ids),
      at<int32_t>(scratch, L.indices), tpe, at<int32_t>(scratch, L.bins),
      at<int32_t>(scratch, L.pbins), at<int32_t>(saved, L.row_src), gmap, -1, L.cap, arow,
      at<int32_t>(scratch, L.info), eto, ptpe, nullptr, nullptr, rws, L.route_ws_bytes, stream));
  float* h = at<float>(saved, L.h);
  float* y = at<float>(scratch, L.y);
  VMOE_TRY(vmoe_gemm_f32_up_fwd(x, ldx, T, gmap, w1, ldw1, h, at<float>(saved, L.pre), nullptr,
                                max_width, VMOE_ACT_RELU_SQUARED, eto, ewo, widths, ptpe, E,
                                hidden, max_width, L.cap, stream));
  VMOE_TRY(vmoe_gemm_f32_down_fwd(h, max_width, w2, ldw2, y, hidden, eto, ewo, widths, ptpe, E,
                                  hidden, max_width, L.cap, stream));
  VMOE_TRY(vmoe_combine_f32(y, L.cap, hidden, arow, wts, k, out, ldo, T, hidden, stream));
  return vmoe_router_aux_f32(partial, (int32_t)L.partial_rows, T, E, tpe, coef,
                             widths_normalized, f_i, at<float>(saved, L.f_i),
                             at<float>(scratch, L.p_i), z_loss, losses, stream);
}

extern "C" int vmoe_moe_f32_backward(
    const void* saved, const float* logits, int64_t num_tokens, int32_t num_experts,
    int32_t top_k, int32_t block_size, const float* x, int64_t ldx, const float* w1, int64_t ldw1,
    const float* w2, int64_t ldw2, const int32_t* ewo, const int32_t* widths, int64_t hidden,
    int64_t max_width, const float* coef, const float* widths_normalized, const float* grad_out,
    int64_t ldg, const float* grad_z, const float* grad_lb, const float* grad_cl, float* grad_x,
    int64_t ldgx, float* grad_w1, int64_t ldgw1, float* grad_w2, int64_t ldgw2,
    float* grad_logits, void* scratch, vmoe_stream_t stream) {
  F32Layout L;
  if (!f32_layout(num_tokens, num_experts, top_k, block_size, hidden, max_width, L))
    return VMOE_ERR_INVALID_ARG;
  if (num_tokens == 0) return VMOE_OK;
  if (!saved || !scratch) return VMOE_ERR_INVALID_ARG;
  const int E = num_experts, k = top_k;
  const int64_t T = num_tokens;
  if (grad_out) {
    if (!x || !w1 || !w2 || !ewo || !widths || !grad_x || !grad_w1 || !grad_w2)
      return VMOE_ERR_INVALID_ARG;
    const int32_t* gmap = at<int32_t>(saved, L.gmap);
    const int32_t* eto = at<int32_t>(saved, L.eto);
    const int32_t* ptpe = at<int32_t>(saved, L.ptpe);
    const float* h = at<float>(saved, L.h);
    float* rows = at<float>(scratch, L.rows);
    float* ga = at<float>(scratch, L.ga);
    // GY[row] = w G[token]; dH with the relu^2 rule, dW2; dX into GY's place, dW1
    VMOE_TRY(vmoe_gather_f32(grad_out, T, ldg, at<int32_t>(saved, L.row_src), k,
                             at<float>(saved, L.wts), L.A, rows, hidden, L.cap, nullptr, hidden,
                             stream));
    VMOE_TRY(gemm_f32_down_bwd_ga(rows, hidden, w2, ldw2, at<float>(saved, L.pre), ga, max_width,
                                  eto, ewo, widths, ptpe, E, hidden, max_width, L.cap, stream));
    VMOE_TRY(vmoe_gemm_f32_down_bwd_dw(h, max_width, rows, hidden, grad_w2, ldgw2, eto, ewo,
                                       widths, ptpe, E, hidden, max_width, L.cap, stream));
    VMOE_TRY(vmoe_gemm_f32_up_bwd_dx(ga, nullptr, nullptr, max_width, VMOE_ACT_NONE, w1, ldw1,
                                     rows, hidden, eto, ewo, widths, ptpe, E, hidden, max_width,
                                     L.cap, stream));
    VMOE_TRY(vmoe_gemm_f32_up_bwd_dw(x, ldx, T, gmap, ga, nullptr, nullptr, max_width,
                                     VMOE_ACT_NONE, grad_w1, ldgw1, eto, ewo, widths, ptpe, E,
                                     hidden, max_width, L.cap, stream));
    VMOE_TRY(vmoe_combine_f32(rows, L.cap, hidden, at<int32_t>(saved, L.arow), nullptr, k, grad_x,
                              ldgx, T, hidden, stream));
  }
  if (!grad_logits) return VMOE_OK;
  if (!logits || !coef || !widths_normalized || (!grad_z && !grad_lb && !grad_cl))
    return VMOE_ERR_INVALID_ARG;
  return vmoe_router_aux_bwd_f32(logits, E, T, E, at<float>(saved, L.lse),
                                 at<float>(saved, L.f_i), coef, widths_normalized, grad_z,
                                 grad_lb, grad_cl, grad_logits, E, stream);
}
