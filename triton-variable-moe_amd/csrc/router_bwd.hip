// Backward of the router Linear (nn.Linear without bias, triton_moe/moe.py:78
// of the reference) from the logit gradient g [T, E]:
//   grad_w[e, n] = sum_t g[t, e] x[t, n]        (E x d over T tokens)
//   grad_x[t, n] (+)= sum_e g[t, e] w[e, n]     (T x d over E experts)
// bf16 operands, fp32 sums, one rounding of each result.
//
// Both products are thin (E <= 128), so what bounds them is reading x (2 T d
// bytes) and reading and writing grad_x (4 T d). grad_w as a plain GEMM has an
// output of E x d, a handful of tiles: hipBLASLt runs it on 16 to 57
// workgroups with the whole of T as their K (16384 x 1024, E = 64: 101 us,
// 0.33 TB/s; 32768 x 2048, E = 128: 182 us). Here T is cut into chunks so
// that about one workgroup per CU reads x once, the chunks' fp32 sums going
// through a workspace (chunks x E x d floats) to a second launch that adds
// them in chunk order. grad_x rides in the same launch as further workgroups
// and adds to the expert path's gradient in place, where two more launches
// (the GEMM and an elementwise add, 17 + 16 us at that size) wrote and re-read
// [T, d] twice; both gradients together take 29 and 107 us (77 at the first
// size where the launch also sums the expert path's rows, a combine of 52).
#include <algorithm>

#include "vmoe_common.h"

namespace vmoe {
namespace {

typedef __bf16 rb_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 rb_bf16x4 __attribute__((ext_vector_type(4)));
typedef float rb_f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t rb_u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char rb_lds;

constexpr int kRbThreads = 256;
constexpr int kRbCols = 128;    // columns of x / grad_x per workgroup
constexpr int kRbTokens = 128;  // tokens per stage of grad_w
constexpr int kRbRows = 128;    // tokens per workgroup and step of grad_x
constexpr int kRbOutStride = 64 + 4;  // floats per row of grad_x's result tiles
constexpr int kRbMaxExperts = 128;
// LDS row strides: 64 or 192 bytes past a multiple of 256, so the four rows of
// 64 bytes that one phase of the transposing read takes fall on different
// banks.
constexpr int kRbXStride = kRbCols * 2 + 64;
__host__ __device__ constexpr int rb_gstride(int mb) {  // rows of 32 mb experts
  return mb >= 3 ? 320 : mb == 2 ? 192 : 64;
}

// MFMA fragment of columns [col0, col0 + 32) and rows k0 .. k0 + 15 of a
// row-major LDS tile: lane l holds column col0 + l % 32, rows 8 (l / 32) .. +7.
__device__ __forceinline__ rb_bf16x8 rb_frag(const rb_lds* tile, int stride, int col0, int k0) {
  const int lane = threadIdx.x & 63, g = lane >> 4, L = lane & 15;
  const int off = (k0 + 8 * (g >> 1) + (L >> 2)) * stride + (col0 + 16 * (g & 1) + 4 * (L & 3)) * 2;
  typedef __attribute__((address_space(3))) rb_bf16x4 lds4;
  const rb_bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4*)(tile + off));
  const rb_bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds4*)(tile + off + 4 * stride));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

struct RbArgs {
  const uint16_t* g;  // [T, E] contiguous
  const uint16_t* x;
  int64_t ldx;
  const uint16_t* w;
  int64_t ldw;
  uint16_t* gx;  // nullable
  int64_t ldgx;
  uint16_t* gw;  // nullable
  int64_t ldgw;
  float* partial;  // [chunks][E][d], where chunks > 1
  int64_t T;
  int E, d, slabs, chunks, per, add;  // per: tokens per chunk
  int iters;  // grad_x: 128-token steps per workgroup
  // what grad_x is added to, instead of its old values: the combine of the
  // expert path's gradient rows, sum_j y[arow[t k + j]] (vmoe_combine)
  const uint16_t* y;
  int64_t ldy, y_rows;
  const int32_t* arow;
  int k;
};

// grad_w of columns [c0, c0 + 128) over the tokens of one chunk: stages of 128
// tokens go through registers (the next stage's loads are in flight while this
// one is multiplied) into LDS, row-major, and the transposing LDS reads give
// both operands with the tokens as K. Wave v owns columns 32 v .. +31.
template <int MB>
__device__ __forceinline__ void rb_grad_w(const RbArgs& p, int block, char* lds) {
  constexpr int GS = rb_gstride(MB);
  constexpr int XL = kRbTokens * (kRbCols / 8) / kRbThreads;     // 16-byte loads per thread
  constexpr int GL = kRbTokens * (32 * MB / 8) / kRbThreads;
  rb_lds* xs = (rb_lds*)lds;
  rb_lds* gs = (rb_lds*)(lds + kRbTokens * kRbXStride);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int slab = block % p.slabs, chunk = block / p.slabs;
  const int c0 = slab * kRbCols;
  const int64_t t_beg = (int64_t)chunk * p.per, t_end = min(p.T, t_beg + p.per);
  const int epr = p.E / 8;  // 16-byte pieces of a gradient row
  rb_u32x4 xr[XL], gr[GL];
  auto load = [&](int64_t t0) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int c = tid + i * kRbThreads, r = c / (kRbCols / 8), col = c0 + (c % (kRbCols / 8)) * 8;
      const rb_u32x4 z = {0, 0, 0, 0};
      xr[i] = t0 + r < t_end && col < p.d
                  ? *reinterpret_cast<const rb_u32x4*>(p.x + (t0 + r) * p.ldx + col) : z;
    }
#pragma unroll
    for (int i = 0; i < GL; ++i) {
      const int c = tid + i * kRbThreads;  // the stage's gradient rows are contiguous
      const rb_u32x4 z = {0, 0, 0, 0};
      gr[i] = c < kRbTokens * epr && t0 + c / epr < t_end
                  ? *reinterpret_cast<const rb_u32x4*>(p.g + t0 * p.E + c * 8) : z;
    }
  };
  rb_f32x16 acc[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[b][v] = 0.0f;
  load(t_beg);
  for (int64_t t0 = t_beg; t0 < t_end; t0 += kRbTokens) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int c = tid + i * kRbThreads;
      *reinterpret_cast<__attribute__((address_space(3))) rb_u32x4*>(
          xs + (c / (kRbCols / 8)) * kRbXStride + (c % (kRbCols / 8)) * 16) = xr[i];
    }
#pragma unroll
    for (int i = 0; i < GL; ++i) {
      const int c = tid + i * kRbThreads;
      if (c < kRbTokens * epr)
        *reinterpret_cast<__attribute__((address_space(3))) rb_u32x4*>(
            gs + (c / epr) * GS + (c % epr) * 16) = gr[i];
    }
    __syncthreads();
    if (t0 + kRbTokens < t_end) load(t0 + kRbTokens);
#pragma unroll
    for (int ks = 0; ks < kRbTokens / 16; ++ks) {
      const rb_bf16x8 b = rb_frag(xs, kRbXStride, 32 * wv, 16 * ks);
#pragma unroll
      for (int m = 0; m < MB; ++m)
        // (columns past E hold whatever LDS held: they only reach the
        // results of those experts, which are not stored)
        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rb_frag(gs, GS, 32 * m, 16 * ks), b,
                                                         acc[m], 0, 0, 0);
    }
    __syncthreads();
  }
  const int n = c0 + 32 * wv + (lane & 31);
  if (n >= p.d) return;
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int e = 32 * m + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
      if (e >= p.E) continue;
      if (p.chunks > 1)
        p.partial[((int64_t)chunk * p.E + e) * p.d + n] = acc[m][v];
      else
        p.gw[e * p.ldgw + n] = (uint16_t)f32_to_bf16(acc[m][v]);
    }
}

// The combine of 2 x 8 tokens' rows for 8 of the wave's columns per lane (8
// lanes to a token): every slot's 16 bytes are in flight before any is summed,
// the sum runs in slot order in fp32 and is rounded once, as in
// combine_k_kernel. idx: the lane's token's row for slot lane % 8 of each.
template <int KMAX>
__device__ __forceinline__ void rb_combine(const RbArgs& p, const int32_t (&idx)[2], int col,
                                           rb_u32x4 (&out)[2]) {
  const int lane = threadIdx.x & 63;
  rb_u32x4 v[2][KMAX];
  bool ok[2][KMAX];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
      const int32_t row = __shfl(idx[u], (lane & 56) + j, kWave);
      ok[u][j] = row >= 0 && col < p.d;
      const rb_u32x4 z = {0, 0, 0, 0};
      v[u][j] = ok[u][j] ? __builtin_nontemporal_load(reinterpret_cast<const rb_u32x4*>(
                               p.y + (int64_t)row * p.ldy + col))
                         : z;
    }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
#pragma unroll
    for (int j = 0; j < KMAX; ++j)
      if (ok[u][j]) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          acc[2 * q] += lo_f32(v[u][j][q]);
          acc[2 * q + 1] += hi_f32(v[u][j][q]);
        }
      }
#pragma unroll
    for (int q = 0; q < 4; ++q) out[u][q] = pack_bf16(acc[2 * q], acc[2 * q + 1]);
  }
}

// grad_x of 128 * p.iters tokens x 128 columns, 32 tokens per wave and step:
// w's columns stay in LDS (transposing reads), each wave reads its own gradient
// rows straight from memory as fragments, and its fp32 results go through a
// private piece of LDS, 64 columns at a time, so that grad_x is read and
// written 128 bytes of a row at a time; after w is staged no wave waits for
// another. (Waves that split the columns instead each read all of the
// gradient rows, and one step per workgroup reads w's columns, 32 KB at
// E = 128, for every 16 KB of grad_x: 108 and 130 us at 32768 x 2048,
// E = 128, against 60 here and 52 for its bytes.)
// KMAX > 0: the sum of the expert path's rows (at most KMAX per token) is formed
// here instead of by a combine launch that writes grad_x for this one to read
// back (combine and this launch, then this launch alone: 52 + 29 -> 74 us at
// 16384 x 1024, E = 64, k = 8; 15 + 19 -> 23 us at 16384 x 768, E = 16, k = 2).
// Up to 64 experts: at 128 the larger tile of w leaves fewer workgroups per CU
// for the row reads (32768 x 2048, k = 8: 213 + 107 against 323 us). Between
// them it depends on the slots and the tokens: training steps of 72 and 96
// experts, 512-2048 wide, took with the sum here 0.96-1.00 of their time at
// k = 2, 0.97-1.01 at k = 8 from 4096 tokens and up to 1.04 at 1024 tokens (the
// launch's few workgroups each wait for 8 rows a token), so the line stays.
template <int MB, int KMAX>
__device__ __forceinline__ void rb_grad_x(const RbArgs& p, int block, char* lds) {
  rb_lds* ws = (rb_lds*)lds;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  float* os = reinterpret_cast<float*>(lds + 32 * MB * kRbXStride) + wv * 32 * kRbOutStride;
  const int slab = block % p.slabs;
  const int64_t t_beg = (int64_t)(block / p.slabs) * kRbRows * p.iters + 32 * wv;
  const int c0 = slab * kRbCols;
  const int kpad = (p.E + 15) / 16 * 16;
  for (int c = tid; c < kpad * (kRbCols / 8); c += kRbThreads) {
    const int r = c / (kRbCols / 8), col = c0 + (c % (kRbCols / 8)) * 8;
    const rb_u32x4 z = {0, 0, 0, 0};
    *reinterpret_cast<__attribute__((address_space(3))) rb_u32x4*>(
        ws + r * kRbXStride + (c % (kRbCols / 8)) * 16) =
        r < p.E && col < p.d ? *reinterpret_cast<const rb_u32x4*>(p.w + r * p.ldw + col) : z;
  }
  __syncthreads();
  for (int it = 0; it < p.iters; ++it) {
    const int64_t t0 = t_beg + (int64_t)it * kRbRows;  // the wave's first token
    if (t0 >= p.T) break;
    rb_bf16x8 a[2 * MB];
#pragma unroll
    for (int ks = 0; ks < 2 * MB; ++ks) {
      const int64_t t = t0 + (lane & 31);
      const int k = 16 * ks + 8 * (lane >> 5);
      const rb_u32x4 z = {0, 0, 0, 0};
      a[ks] = __builtin_bit_cast(
          rb_bf16x8,
          t < p.T && k < p.E ? *reinterpret_cast<const rb_u32x4*>(p.g + t * p.E + k) : z);
    }
    rb_u32x4 old[2][4];  // (64-column half, 8 rows each)
    if constexpr (KMAX > 0) {
      int32_t idx[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t t = t0 + 8 * i + (lane >> 3);
        const int32_t row =
            t < p.T && (lane & 7) < p.k ? p.arow[t * p.k + (lane & 7)] : -1;
        idx[i] = row < p.y_rows ? row : -1;
      }
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          const int32_t two[2] = {idx[i], idx[i + 1]};
          rb_u32x4 sum[2];
          rb_combine<KMAX>(p, two, c0 + 64 * hf + (lane & 7) * 8, sum);
          old[hf][i] = sum[0];
          old[hf][i + 1] = sum[1];
        }
    } else {
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int64_t t = t0 + 8 * i + (lane >> 3);
          const int col = c0 + 64 * hf + (lane & 7) * 8;
          const rb_u32x4 z = {0, 0, 0, 0};
          old[hf][i] = p.add && t < p.T && col < p.d
                           ? *reinterpret_cast<const rb_u32x4*>(p.gx + t * p.ldgx + col) : z;
        }
    }
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      rb_f32x16 acc[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[j][v] = 0.0f;
#pragma unroll
      for (int ks = 0; ks < 2 * MB; ++ks) {
        if (16 * ks >= kpad) break;
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              a[ks], rb_frag(ws, kRbXStride, 64 * hf + 32 * j, 16 * ks), acc[j], 0, 0, 0);
      }
      asm volatile("" ::: "memory");  // the wave's LDS accesses complete in order
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          os[(8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)) * kRbOutStride + 32 * j + (lane & 31)] =
              acc[j][v];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 8 * i + (lane >> 3), cc = 64 * hf + (lane & 7) * 8;
        const float4 u = *reinterpret_cast<const float4*>(os + r * kRbOutStride + (lane & 7) * 8);
        const float4 v =
            *reinterpret_cast<const float4*>(os + r * kRbOutStride + (lane & 7) * 8 + 4);
        // the product rounded, then the sum: the bits of a linear layer's
        // gradient added to the other one's by autograd
        rb_u32x4 res = {pack_bf16(u.x, u.y), pack_bf16(u.z, u.w), pack_bf16(v.x, v.y),
                        pack_bf16(v.z, v.w)};
        if (KMAX > 0 || p.add) {
          const rb_u32x4 o = old[hf][i];
#pragma unroll
          for (int q = 0; q < 4; ++q)
            res[q] = pack_bf16(lo_f32(o[q]) + lo_f32(res[q]), hi_f32(o[q]) + hi_f32(res[q]));
        }
        if (t0 + r < p.T && c0 + cc < p.d)
          __builtin_nontemporal_store(
              res, reinterpret_cast<rb_u32x4*>(p.gx + (t0 + r) * p.ldgx + c0 + cc));
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

template <int MB, int KMAX>
__global__ __launch_bounds__(kRbThreads) void router_linear_bwd_kernel(RbArgs p) {
  constexpr int DW = kRbTokens * (kRbXStride + rb_gstride(MB));
  constexpr int DX = 32 * MB * kRbXStride + kRbRows * kRbOutStride * 4;
  __shared__ __align__(16) char lds[DW > DX ? DW : DX];
  const int ndw = p.gw ? p.slabs * p.chunks : 0;
  if ((int)blockIdx.x < ndw)
    rb_grad_w<MB>(p, blockIdx.x, lds);
  else
    rb_grad_x<MB, KMAX>(p, blockIdx.x - ndw, lds);
}

// grad_w = bf16(sum over the chunks, in order), four columns per thread.
__global__ __launch_bounds__(256) void router_linear_sum_kernel(const float* __restrict__ partial,
                                                                int chunks, int E, int d,
                                                                uint16_t* __restrict__ gw,
                                                                int64_t ldgw) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4, n = (int64_t)E * d;
  if (i >= n) return;
  float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 8
  for (int c = 0; c < chunks; ++c) {
    const float4 v = *reinterpret_cast<const float4*>(partial + c * n + i);
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  *reinterpret_cast<uint2*>(gw + (i / d) * ldgw + i % d) =
      make_uint2(pack_bf16(s.x, s.y), pack_bf16(s.z, s.w));
}

// About one grad_w workgroup per CU of a whole MI355X (256; a part of one runs
// them in turn), at least one stage of tokens each.
void rb_split(int64_t T, int64_t d, int& slabs, int& chunks, int& per) {
  slabs = (int)((d + kRbCols - 1) / kRbCols);
  const int64_t stages = (T + kRbTokens - 1) / kRbTokens;
  const int64_t want = std::max<int64_t>(1, std::min<int64_t>(stages, 256 / slabs));
  const int64_t sper = (stages + want - 1) / want;
  per = (int)(sper * kRbTokens);
  chunks = (int)((stages + sper - 1) / sper);
}

bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace vmoe

using namespace vmoe;

extern "C" size_t vmoe_router_linear_bwd_workspace_bytes(int64_t num_tokens, int64_t hidden,
                                                         int32_t num_experts) {
  if (num_tokens <= 0 || hidden <= 0 || num_experts <= 0 || num_tokens > INT32_MAX ||
      hidden > INT32_MAX)
    return 0;
  int slabs, chunks, per;
  rb_split(num_tokens, hidden, slabs, chunks, per);
  return chunks > 1 ? (size_t)chunks * (size_t)num_experts * (size_t)hidden * sizeof(float) : 0;
}

namespace vmoe {
namespace {
// The argument checks of router_linear_bwd and its kernel's operands; kmax: the
// slots of the kernel instance that sums rows (0: none).
int rb_args(const uint16_t* grad_logits, const uint16_t* x, int64_t ldx, const uint16_t* weight,
            int64_t ldw, int64_t num_tokens, int64_t hidden, int32_t num_experts,
            uint16_t* grad_x, int64_t ldgx, int32_t accumulate, uint16_t* grad_weight,
            int64_t ldgw, void* workspace, size_t workspace_bytes, const RowSum* sum, RbArgs& p,
            int& kmax) {
  if (num_tokens < 0 || hidden <= 0 || num_experts <= 0) return VMOE_ERR_INVALID_ARG;
  if (!grad_x && !grad_weight) return VMOE_OK;
  if (num_tokens == 0) return VMOE_ERR_INVALID_ARG;  // grad_weight would be left unwritten
  if (!grad_logits || (grad_weight && !x) || (grad_x && !weight)) return VMOE_ERR_INVALID_ARG;
  if (num_experts % 8 != 0 || num_experts > kRbMaxExperts || hidden % 8 != 0 ||
      hidden > INT32_MAX / 2 || num_tokens > INT32_MAX / 2 || !a16(grad_logits))
    return VMOE_ERR_UNSUPPORTED;
  // (ldx 0: one row for every token)
  if (grad_weight &&
      ((ldx != 0 && ldx < hidden) || ldx % 8 != 0 || !a16(x) || ldgw < hidden || ldgw % 4 != 0 ||
       (reinterpret_cast<uintptr_t>(grad_weight) & 7) != 0))
    return VMOE_ERR_UNSUPPORTED;
  if (grad_x && (ldw < hidden || ldw % 8 != 0 || !a16(weight) || ldgx < hidden ||
                 ldgx % 8 != 0 || !a16(grad_x)))
    return VMOE_ERR_UNSUPPORTED;
  p.g = grad_logits;
  p.x = x; p.ldx = ldx;
  p.w = weight; p.ldw = ldw;
  p.gx = grad_x; p.ldgx = ldgx; p.add = accumulate != 0;
  p.gw = grad_weight; p.ldgw = ldgw;
  p.T = num_tokens; p.E = num_experts; p.d = (int)hidden;
  kmax = 0;
  if (grad_x && sum) {
    if (!sum->y || !sum->arow || sum->k <= 0 || sum->ldy < hidden) return VMOE_ERR_INVALID_ARG;
    if (sum->k > kRowSumSlots || num_experts > kRowSumExperts || sum->ldy % 8 != 0 ||
        !a16(sum->y))
      return VMOE_ERR_UNSUPPORTED;
    p.y = sum->y; p.ldy = sum->ldy; p.y_rows = sum->rows; p.arow = sum->arow; p.k = sum->k;
    kmax = sum->k <= 2 ? 2 : 8;
  }
  rb_split(num_tokens, hidden, p.slabs, p.chunks, p.per);
  if (grad_weight && p.chunks > 1) {
    if (workspace_bytes < vmoe_router_linear_bwd_workspace_bytes(num_tokens, hidden, num_experts) ||
        !workspace || !a16(workspace))
      return VMOE_ERR_WORKSPACE;
    p.partial = reinterpret_cast<float*>(workspace);
  }
  return VMOE_OK;
}
}  // namespace

int router_linear_bwd_check(const uint16_t* grad_logits, const uint16_t* x, int64_t ldx,
                            const uint16_t* weight, int64_t ldw, int64_t num_tokens,
                            int64_t hidden, int32_t num_experts, uint16_t* grad_x, int64_t ldgx,
                            uint16_t* grad_weight, int64_t ldgw, void* workspace,
                            size_t workspace_bytes, const RowSum* sum) {
  RbArgs p{};
  int kmax = 0;
  return rb_args(grad_logits, x, ldx, weight, ldw, num_tokens, hidden, num_experts, grad_x, ldgx,
                 0, grad_weight, ldgw, workspace, workspace_bytes, sum, p, kmax);
}

int router_linear_bwd(const uint16_t* grad_logits, const uint16_t* x, int64_t ldx,
                      const uint16_t* weight, int64_t ldw, int64_t num_tokens, int64_t hidden,
                      int32_t num_experts, uint16_t* grad_x, int64_t ldgx, int32_t accumulate,
                      uint16_t* grad_weight, int64_t ldgw, void* workspace,
                      size_t workspace_bytes, const RowSum* sum, vmoe_stream_t stream) {
  RbArgs p{};
  int kmax = 0;
  const int st = rb_args(grad_logits, x, ldx, weight, ldw, num_tokens, hidden, num_experts, grad_x,
                         ldgx, accumulate, grad_weight, ldgw, workspace, workspace_bytes, sum, p,
                         kmax);
  if (st != VMOE_OK || (!grad_x && !grad_weight)) return st;
  // up to 4 steps per workgroup while at least 4 workgroups per CU are left
  const int64_t steps = (num_tokens + kRbRows - 1) / kRbRows;
  p.iters = (int)std::max<int64_t>(1, std::min<int64_t>(4, steps * p.slabs / 1024));
  const int64_t blocks = (grad_weight ? (int64_t)p.slabs * p.chunks : 0) +
                         (grad_x ? (steps + p.iters - 1) / p.iters * p.slabs : 0);
  if (blocks > INT32_MAX) return VMOE_ERR_UNSUPPORTED;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)blocks), wg(kRbThreads);
  switch ((num_experts + 31) / 32 * 16 + kmax) {
#define VMOE_RB_CASE(M, K)                                                        \
  case M * 16 + K:                                                                \
    VMOE_LAUNCH((router_linear_bwd_kernel<M, K>), grid, wg, 0, s, p);             \
    break;
    VMOE_RB_CASE(1, 0)
    VMOE_RB_CASE(1, 2)
    VMOE_RB_CASE(1, 8)
    VMOE_RB_CASE(2, 0)
    VMOE_RB_CASE(2, 2)
    VMOE_RB_CASE(2, 8)
    VMOE_RB_CASE(3, 0)
    VMOE_RB_CASE(4, 0)
#undef VMOE_RB_CASE
    default: return VMOE_ERR_UNSUPPORTED;
  }
  VMOE_CHECK_LAUNCH();
  if (grad_weight && p.chunks > 1) {
    const int64_t n = (int64_t)num_experts * hidden / 4;
    VMOE_LAUNCH(router_linear_sum_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                p.partial, p.chunks, (int)num_experts, (int)hidden, grad_weight, ldgw);
    VMOE_CHECK_LAUNCH();
  }
  return VMOE_OK;
}
}  // namespace vmoe

extern "C" int vmoe_router_linear_bwd(const uint16_t* grad_logits, const uint16_t* x, int64_t ldx,
                                      const uint16_t* weight, int64_t ldw, int64_t num_tokens,
                                      int64_t hidden, int32_t num_experts, uint16_t* grad_x,
                                      int64_t ldgx, int32_t accumulate, uint16_t* grad_weight,
                                      int64_t ldgw, void* workspace, size_t workspace_bytes,
                                      vmoe_stream_t stream) {
  return router_linear_bwd(grad_logits, x, ldx, weight, ldw, num_tokens, hidden, num_experts,
                           grad_x, ldgx, accumulate, grad_weight, ldgw, workspace,
                           workspace_bytes, nullptr, stream);
}
