// fp32 grouped GEMMs: the float32 inputs of the public grouped-GEMM API and
// the float32 module.
//
// The reference's grouped-GEMM kernels take fp32 as well as bf16 operands
// (triton_moe/kernels/grouped_gemm.py:217-1162, dtype-generic tl.dot with an
// fp32 accumulator); its autograd tests and forward/backward benchmark run
// them in fp32 (tests/test_grouped_gemm_backward.py:151-208). The bf16 kernels
// of gemm.hip stage bf16 tiles and cannot take fp32, so this file holds one
// LDS-tiled kernel for all six forms (up forward with its activation, down
// forward, and both backward GEMMs of each) on v_mfma_f32_32x32x2_f32: fp32
// products and sums, nothing narrower. The activation gradients (SwiGLU's
// [dG | dU]) are formed from grad/pre/up as the operand tile is loaded, as the
// reference's backward kernels do (grouped_gemm.py:751-764, 914-927).
//
// What bounds it: the fp32 matrix rate (256 flop per cycle and CU, 157 TFLOP/s
// at 2.4 GHz; the vector pipe without packed fp32, which this build does not
// use, has half of it: the fma kernel this replaced ran cfg-like shapes of
// 8192 rows x 768 x 512 at 42 TFLOP/s). That rate is low enough that a 64 x 64 tile
// per 256-thread workgroup, one 32 x 32 block per wave, needs only 16 bytes
// per cycle and CU from L2 and 32 from LDS, so the tile is chosen small for
// balance and occupancy: four workgroups share a CU and hide each other's
// loads, and the widths and row counts of real experts leave little of a tile
// empty. The six forms at 8192 rows x 768 x 512: 793 us with fma, 473 - 486 now
// (80 TFLOP/s; 101 at 131072 rows x 1024 x 256).
#include <algorithm>
#include <type_traits>

#include "vmoe_common.h"

namespace vmoe {
namespace {

enum F32Form { F_UP_FWD, F_DOWN_FWD, F_UP_DX, F_UP_DW, F_DOWN_DH, F_DOWN_DW };

constexpr int kT = 64;        // tile edge
constexpr int kBK = 32;       // k per LDS stage
constexpr int kThreads = 256;
constexpr int kRuns = kT * kBK / 4 / kThreads;  // runs of 4 floats per thread and operand stage
// LDS rows (floats). An operand that is contiguous along k is held as [x][k],
// one 16-byte read giving a lane 4 consecutive k: rows of 36 floats put the 16
// rows one phase reads on different banks. Any other is held as [k][x], one
// 4-byte read per k: rows of 72 floats put the two rows 4 apart that the
// halves of a wave read on different banks.
constexpr int kRowK = kBK + 4, kRowX = kT + 8;
constexpr int kStage = kT * kRowK > kBK * kRowX ? kT * kRowK : kBK * kRowX;
typedef float f32x16_t __attribute__((ext_vector_type(16)));

struct F32Args {
  // token-row operand: x (up forms), h (down forms) or grad_y (dH)
  const float* a;
  int64_t lda, a_rows;
  const int32_t* a_map;  // x rows through a gather map (up forms), may be null
  // weights: w1 or w2 (forward, dX and dH), or grad_y (down dW)
  const float* b;
  int64_t ldb;
  // gradient of the up projection's output with pre (relu(z) or the gate)
  // and up (SwiGLU), all [rows, max_width] with leading dimension ldg
  const float *g, *pre, *up;
  int64_t ldg;
  float *c, *c2, *c3;
  int64_t ldc;
  const int32_t *eto, *ewo, *widths, *tpe;
  int E, act;
  int64_t hidden, max_width, rows_bound;
};

struct F32Prob {
  int64_t M, N, K, t0, w0, w;
};

__device__ __forceinline__ int64_t cdiv64(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Rows of expert e: [t0, t0 + rows), rows = min(tpe, eto[e+1] - eto[e]) and
// inside [0, rows_bound).
template <int F>
__device__ F32Prob f32_prob(const F32Args& p, int e) {
  F32Prob q;
  const int64_t t0 = p.eto[e];
  const int64_t t1 = min((int64_t)p.eto[e + 1], p.rows_bound);
  int64_t rows = min((int64_t)p.tpe[e], t1 - t0);
  if (t0 < 0 || rows < 0) rows = 0;
  const int64_t w = max((int64_t)0, min((int64_t)p.widths[e], p.max_width));
  // the SwiGLU backward GEMMs run over the expert's gate and up columns
  const int64_t wg = p.act == VMOE_ACT_SWIGLU ? 2 * w : w;
  q.t0 = t0;
  q.w0 = p.ewo[e];
  q.w = w;
  switch (F) {
    case F_UP_FWD: q.M = rows; q.N = w; q.K = p.hidden; break;
    case F_DOWN_FWD: q.M = rows; q.N = p.hidden; q.K = w; break;
    case F_UP_DX: q.M = rows; q.N = p.hidden; q.K = wg; break;
    case F_UP_DW: q.M = p.hidden; q.N = wg; q.K = rows; break;
    case F_DOWN_DH: q.M = rows; q.N = w; q.K = p.hidden; break;
    default: q.M = w; q.N = p.hidden; q.K = rows; break;  // F_DOWN_DW
  }
  return q;
}

__device__ __forceinline__ float sigmoid32(float v) { return 1.0f / (1.0f + expf(-v)); }

// The gradient w.r.t. the up projection's pre-activation at row r, column c
// (c < 2w for SwiGLU: c < w is the gate's, c >= w the up half's).
__device__ __forceinline__ float act_grad(const F32Args& p, int64_t r, int64_t c, int64_t w) {
  if (p.act == VMOE_ACT_SWIGLU) {
    const int64_t cc = c < w ? c : c - w;
    const int64_t o = r * p.ldg + cc;
    const float gr = p.g[o], gate = p.pre[o], s = sigmoid32(gate);
    return c < w ? gr * p.up[o] * s * (1.0f + gate * (1.0f - s)) : gr * gate * s;
  }
  const int64_t o = r * p.ldg + c;
  const float gr = p.g[o];
  if (p.act == VMOE_ACT_RELU_SQUARED) {
    const float pr = p.pre[o];
    return pr > 0.0f ? gr * 2.0f * pr : 0.0f;
  }
  return gr;
}

// x row of padded row r (through the gather map when there is one; a map
// entry outside [0, a_rows) reads zeros).
__device__ __forceinline__ const float* token_row(const F32Args& p, int64_t r) {
  if (!p.a_map) return p.a + r * p.lda;
  const int64_t s = p.a_map[r];
  return s >= 0 && s < p.a_rows ? p.a + s * p.lda : nullptr;
}

// A(m, k) of the tile's problem (0 outside M x K).
template <int F>
__device__ __forceinline__ float f32_a(const F32Args& p, const F32Prob& q, int64_t m, int64_t k) {
  if (m >= q.M || k >= q.K) return 0.0f;
  switch (F) {
    case F_UP_FWD: {
      const float* row = token_row(p, q.t0 + m);
      return row ? row[k] : 0.0f;
    }
    case F_DOWN_FWD:
    case F_DOWN_DH: return p.a[(q.t0 + m) * p.lda + k];
    case F_UP_DX: return act_grad(p, q.t0 + m, k, q.w);
    case F_UP_DW: {
      const float* row = token_row(p, q.t0 + k);
      return row ? row[m] : 0.0f;
    }
    default: return p.a[(q.t0 + k) * p.lda + m];  // F_DOWN_DW: h^T
  }
}

// B(k, n); `second` selects the SwiGLU up half of W1 in the up forward.
template <int F>
__device__ __forceinline__ float f32_b(const F32Args& p, const F32Prob& q, int64_t k, int64_t n,
                                       bool second) {
  if (k >= q.K || n >= q.N) return 0.0f;
  switch (F) {
    case F_UP_FWD: return p.b[k * p.ldb + q.w0 + (second ? q.w : 0) + n];
    case F_DOWN_FWD: return p.b[(q.w0 + k) * p.ldb + n];
    case F_UP_DX: return p.b[n * p.ldb + q.w0 + k];  // W1^T
    case F_UP_DW: return act_grad(p, q.t0 + k, n, q.w);
    case F_DOWN_DH: return p.b[(q.w0 + n) * p.ldb + k];  // W2^T
    default: return p.b[(q.t0 + k) * p.ldb + n];  // F_DOWN_DW: grad_y
  }
}

// Whether A / B are contiguous along k (decides which thread loads what).
template <int F>
constexpr bool a_k_contig() { return F == F_UP_FWD || F == F_DOWN_FWD || F == F_UP_DX || F == F_DOWN_DH; }
template <int F>
constexpr bool b_k_contig() { return F == F_UP_DX || F == F_DOWN_DH; }

// Four consecutive floats from ptr of which `valid` are in range (the rest
// read as 0): one 16-byte load when all four are and the address allows it.
__device__ __forceinline__ float4 load_run(const float* ptr, int64_t valid) {
  float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (!ptr || valid <= 0) return v;
  if (valid >= 4 && (reinterpret_cast<uintptr_t>(ptr) & 15) == 0)
    return *reinterpret_cast<const float4*>(ptr);
  v.x = ptr[0];
  if (valid > 1) v.y = ptr[1];
  if (valid > 2) v.z = ptr[2];
  if (valid > 3) v.w = ptr[3];
  return v;
}

// Four elements of A from (m, k) along its contiguous dimension (k for the
// K-contiguous forms, m otherwise); up dX only without an activation (with
// one, its A is formed element by element).
template <int F>
__device__ __forceinline__ float4 f32_a_run(const F32Args& p, const F32Prob& q, int64_t m,
                                            int64_t k) {
  const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  switch (F) {
    case F_UP_FWD: {
      if (m >= q.M) return z;
      const float* row = token_row(p, q.t0 + m);
      return load_run(row ? row + k : nullptr, q.K - k);
    }
    case F_UP_DX:  // the gradient itself (no activation)
      return m < q.M ? load_run(p.g + (q.t0 + m) * p.ldg + k, q.K - k) : z;
    case F_DOWN_FWD:
    case F_DOWN_DH:
      return m < q.M ? load_run(p.a + (q.t0 + m) * p.lda + k, q.K - k) : z;
    case F_UP_DW: {
      if (k >= q.K) return z;
      const float* row = token_row(p, q.t0 + k);
      return load_run(row ? row + m : nullptr, q.M - m);
    }
    default:  // F_DOWN_DW: h^T
      return k < q.K ? load_run(p.a + (q.t0 + k) * p.lda + m, q.M - m) : z;
  }
}

// Four elements of B from (k, n) along its contiguous dimension (k for up dX
// and down dH, n otherwise); up dW only without an activation.
template <int F>
__device__ __forceinline__ float4 f32_b_run(const F32Args& p, const F32Prob& q, int64_t k,
                                            int64_t n, bool second) {
  const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  switch (F) {
    case F_UP_FWD:
      return k < q.K ? load_run(p.b + k * p.ldb + q.w0 + (second ? q.w : 0) + n, q.N - n) : z;
    case F_DOWN_FWD:
      return k < q.K ? load_run(p.b + (q.w0 + k) * p.ldb + n, q.N - n) : z;
    case F_UP_DX:  // W1^T
      return n < q.N ? load_run(p.b + n * p.ldb + q.w0 + k, q.K - k) : z;
    case F_UP_DW:  // the gradient itself (no activation)
      return k < q.K ? load_run(p.g + (q.t0 + k) * p.ldg + n, q.N - n) : z;
    case F_DOWN_DH:  // W2^T
      return n < q.N ? load_run(p.b + (q.w0 + n) * p.ldb + k, q.K - k) : z;
    default:  // F_DOWN_DW: grad_y
      return k < q.K ? load_run(p.b + (q.t0 + k) * p.ldb + n, q.N - n) : z;
  }
}

// Runs of 4 elements of a kBK x kT operand stage: thread -> (k, x) of run i,
// along the operand's contiguous dimension (k when KCONTIG).
template <bool KCONTIG>
__device__ __forceinline__ void run_at(int i, int& k, int& x) {
  const int tid = threadIdx.x;
  if (KCONTIG) {
    x = (tid >> 3) + 32 * i;
    k = (tid & 7) * 4;
  } else {
    x = (tid & 15) * 4;
    k = (tid >> 4) + 16 * i;
  }
}

template <bool KCONTIG, typename Fn>
__device__ __forceinline__ void load_stage(float4 (&r)[kRuns], Fn&& run) {
#pragma unroll
  for (int i = 0; i < kRuns; ++i) {
    int k, x;
    run_at<KCONTIG>(i, k, x);
    r[i] = run(k, x);
  }
}

template <bool KCONTIG>
__device__ __forceinline__ void store_stage(float* lds, const float4 (&r)[kRuns]) {
#pragma unroll
  for (int i = 0; i < kRuns; ++i) {
    int k, x;
    run_at<KCONTIG>(i, k, x);
    *reinterpret_cast<float4*>(lds + (KCONTIG ? x * kRowK + k : k * kRowX + x)) = r[i];
  }
}

// The lane's operand values of 8 consecutive k from kk: element j is (x = x0 +
// lane % 32, k = kk + 4 (lane / 32) + j), so MFMA j takes k = kk + j from the
// lower and kk + 4 + j from the upper half of the wave.
template <bool KCONTIG>
__device__ __forceinline__ float4 frag(const float* lds, int x0, int kk) {
  const int lane = threadIdx.x & 63;
  const int x = x0 + (lane & 31), k = kk + 4 * (lane >> 5);
  if (KCONTIG) return *reinterpret_cast<const float4*>(lds + x * kRowK + k);
  const float* c = lds + k * kRowX + x;
  return make_float4(c[0], c[kRowX], c[2 * kRowX], c[3 * kRowX]);
}

__device__ __forceinline__ void mfma4(f32x16_t& acc, const float4& a, const float4& b) {
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, acc, 0, 0, 0);
}

// The expert and tile of item j of this workgroup's XCD: each wave counts the
// tiles of 64 experts at a time, one per lane, and scans them (a walk over the
// experts one by one costs a dependent load per expert). XCD x takes a contiguous eighth
// of the tiles, so the tiles that share rows or columns share an L2. Returns
// false past the last tile.
template <int F>
__device__ __forceinline__ bool find_tile(const F32Args& p, int64_t j, int& expert,
                                          int64_t& local) {
  const int lane = threadIdx.x & 63;
  auto tiles_of = [&](int e) -> int {
    if (e >= p.E) return 0;
    const F32Prob q = f32_prob<F>(p, e);
    return (int)(cdiv64(q.M, kT) * cdiv64(q.N, kT));
  };
  int64_t total = 0;
  int first = 0;  // the lane's count and its wave's inclusive scan for experts 0 .. 63
  for (int e0 = 0; e0 < p.E; e0 += kWave) {
    const int inc = wave_inclusive_scan(tiles_of(e0 + lane));
    if (e0 == 0) first = inc;
    total += __shfl(inc, kWave - 1);
  }
  const int64_t per = (total + 7) / 8;
  const int64_t t = (blockIdx.x & 7) * per + j;
  if (j >= per || t >= total) return false;
  int64_t before = 0;
  for (int e0 = 0; e0 < p.E; e0 += kWave) {
    const int inc = e0 == 0 ? first : wave_inclusive_scan(tiles_of(e0 + lane));
    const uint64_t past = ballot64(before + inc > t);
    if (past) {
      const int l = __builtin_ctzll(past);
      expert = __builtin_amdgcn_readfirstlane(e0 + l);
      local = t - before - (l > 0 ? __shfl(inc, l - 1) : 0);
      return true;
    }
    before += __shfl(inc, kWave - 1);
  }
  return false;
}

// Operand sources of a form: the matrix its A and B come from and the leading
// dimensions (the gradient g for up dX's A and up dW's B).
template <int F>
__device__ __forceinline__ const float* a_src(const F32Args& p) { return F == F_UP_DX ? p.g : p.a; }
template <int F>
__device__ __forceinline__ int64_t a_ld(const F32Args& p) { return F == F_UP_DX ? p.ldg : p.lda; }
template <int F>
__device__ __forceinline__ const float* b_src(const F32Args& p) { return F == F_UP_DW ? p.g : p.b; }
template <int F>
__device__ __forceinline__ int64_t b_ld(const F32Args& p) { return F == F_UP_DW ? p.ldg : p.ldb; }

// Stage loads without branches: buffer loads at 32-bit offsets from the tile's
// corner, where an offset past the resource reads zeros. `wide` (tile_wide)
// tiles have every run of 4 floats wholly inside or outside the operand and
// 16-byte aligned and load it at once, the others element by element. (The
// general loads, f32_a_run and f32_b_run, test every run's alignment and every
// element of a cut one behind branches, at 64-bit addresses; that code took
// longer than the stage's MFMAs: 8192 rows x 768 x 512, 106 us a GEMM with it,
// 79-90 without.)
constexpr uint32_t kOob = 0x80000000u;

// A workgroup-uniform value in scalar registers.
__device__ __forceinline__ int64_t uniform(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// b in scalar registers (uniform)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t f32_rsrc(const float* b) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(b), 0, 0x7FFFFFFF, 0x00020000);
}

// The 4 floats at byte offset off, of which the first n are in the operand.
template <bool WIDE>
__device__ __forceinline__ float4 f32_run(__amdgpu_buffer_rsrc_t rs, uint32_t off, int n) {
  if (WIDE) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, n > 0 ? off : kOob, 0, 0);
    return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z),
                       __uint_as_float(v.w));
  }
  float v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    v[j] = __uint_as_float(
        __builtin_amdgcn_raw_buffer_load_b32(rs, j < n ? off + 4 * j : kOob, 0, 0));
  return make_float4(v[0], v[1], v[2], v[3]);
}

template <bool KCONTIG>
struct VecOp {
  const float* base;    // the tile's corner at k = 0
  int64_t step;         // floats from one k to the next
  uint32_t off[kRuns];  // bytes from base (+ k0 * step) of the thread's runs
  int n[kRuns];         // KCONTIG: row inside; else elements of the run inside
  __device__ __forceinline__ void init(const float* corner, int64_t ld, int64_t extent) {
    base = reinterpret_cast<const float*>(uniform(reinterpret_cast<int64_t>(corner)));
    step = KCONTIG ? 1 : uniform(ld);
#pragma unroll
    for (int i = 0; i < kRuns; ++i) {
      int k, x;
      run_at<KCONTIG>(i, k, x);
      n[i] = extent - x < 4 ? (int)(extent - x) : 4;
      off[i] = (uint32_t)((KCONTIG ? x * ld + k : k * ld + x) * 4);
    }
  }
  // 32-bit tests on `left`, the stage's k still inside (int64_t min compiles to
  // conversions and a minimum in double).
  template <bool WIDE>
  __device__ __forceinline__ void load(float4 (&r)[kRuns], int64_t k0, int64_t K) const {
    const auto rs = f32_rsrc(base + k0 * step);
    const int left = K - k0 < kBK ? (int)(K - k0) : kBK;
#pragma unroll
    for (int i = 0; i < kRuns; ++i) {
      int k, x;
      run_at<KCONTIG>(i, k, x);
      const int in = min(left - k, 4);
      r[i] = f32_run<WIDE>(rs, off[i], KCONTIG ? (n[i] > 0 ? in : 0) : (in > 0 ? n[i] : 0));
    }
  }
};

// Whether a launch's offsets from a tile's corner, or from the gathered matrix,
// stay below 2^31 bytes and its gradient operand is stored as it is used (host).
template <int F>
bool f32_vec(const F32Args& p) {
  if ((F == F_UP_DX || F == F_UP_DW) && p.act != VMOE_ACT_NONE) return false;
  const int64_t la = F == F_UP_DX ? p.ldg : p.lda, lb = F == F_UP_DW ? p.ldg : p.ldb;
  return la < (1 << 22) && lb < (1 << 22) && (!p.a_map || p.a_rows * la < (int64_t)1 << 29);
}

template <int F>
__device__ __forceinline__ bool tile_wide(const F32Args& p, const F32Prob& q) {
  const uint64_t bits =
      reinterpret_cast<uint64_t>(a_src<F>(p)) | reinterpret_cast<uint64_t>(b_src<F>(p)) |
      (uint64_t)((a_ld<F>(p) | b_ld<F>(p) | p.hidden | q.w | q.w0) * 4);
  return (bits & 15) == 0;
}

// GLU: the SwiGLU up forward (a second accumulator over the up columns); its
// own instance, so the other forms do not carry its registers. VEC: f32_vec.
template <int F, bool GLU, bool VEC>
__global__ __launch_bounds__(kThreads) void grouped_gemm_f32_kernel(F32Args p) {
  __shared__ __align__(16) float As[2][kStage];
  __shared__ __align__(16) float Bs[2][kStage];
  __shared__ __align__(16) float Us[2][GLU ? kStage : 4];  // SwiGLU up half
  constexpr bool glu = GLU && F == F_UP_FWD;
  constexpr bool AK = a_k_contig<F>(), BKC = b_k_contig<F>();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  int e;
  int64_t local;
  for (int64_t j = blockIdx.x >> 3; find_tile<F>(p, j, e, local); j += gridDim.x >> 3) {
    F32Prob q = f32_prob<F>(p, e);
    q.M = uniform(q.M); q.N = uniform(q.N); q.K = uniform(q.K);
    q.t0 = uniform(q.t0); q.w0 = uniform(q.w0); q.w = uniform(q.w);
    const int64_t tn_count = cdiv64(q.N, kT);
    const int64_t m0 = uniform((local / tn_count) * kT), n0 = uniform((local % tn_count) * kT);
    f32x16_t acc, acc_up;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = acc_up[v] = 0.0f;
    float4 ra[kRuns], rb[kRuns], ru[glu ? kRuns : 1];
    // Multiplies stage by stage, the next stage's loads in flight meanwhile;
    // two LDS buffers, so one barrier per stage: a wave that has passed stage
    // s's barrier has every wave behind it past stage s - 1's reads.
    auto multiply = [&](auto&& load) {
      int buf = 0;
      if (q.K > 0) load(0);
      for (int64_t k0 = 0; k0 < q.K; k0 += kBK, buf ^= 1) {
        store_stage<AK>(As[buf], ra);
        store_stage<BKC>(Bs[buf], rb);
        if constexpr (glu) store_stage<BKC>(Us[buf], ru);
        __syncthreads();
        if (k0 + kBK < q.K) load(k0 + kBK);
        float4 fa[kBK / 8], fb[kBK / 8];
#pragma unroll
        for (int u = 0; u < kBK / 8; ++u) {
          fa[u] = frag<AK>(As[buf], wm, 8 * u);
          fb[u] = frag<BKC>(Bs[buf], wn, 8 * u);
        }
#pragma unroll
        for (int u = 0; u < kBK / 8; ++u) {
          mfma4(acc, fa[u], fb[u]);
          if constexpr (glu) mfma4(acc_up, fa[u], frag<BKC>(Us[buf], wn, 8 * u));
        }
      }
      __syncthreads();  // before the next tile's first stage
    };
    if constexpr (VEC) {
      const bool wide = tile_wide<F>(p, q);
      VecOp<AK> va;
      VecOp<BKC> vb, vu;
      const float* a = a_src<F>(p);
      const float* b = b_src<F>(p);
      const int64_t la = a_ld<F>(p), lb = b_ld<F>(p);
      const int32_t* map = F == F_UP_FWD || F == F_UP_DW ? p.a_map : nullptr;
      va.init(map ? a + (AK ? 0 : m0) : a + (AK ? (q.t0 + m0) * la : q.t0 * la + m0), la,
              q.M - m0);
      if constexpr (F == F_UP_FWD) {
        if (map) {  // the rows of the tile, the same for every stage
#pragma unroll
          for (int i = 0; i < kRuns; ++i) {
            int k, x;
            run_at<true>(i, k, x);
            const int64_t s = m0 + x < q.M ? map[q.t0 + m0 + x] : -1;
            va.n[i] = s >= 0 && s < p.a_rows ? 4 : 0;
            va.off[i] = (uint32_t)((s * la + k) * 4);
          }
        }
      }
      switch (F) {
        case F_UP_FWD: vb.init(b + q.w0 + n0, lb, q.N - n0); break;
        case F_DOWN_FWD: vb.init(b + q.w0 * lb + n0, lb, q.N - n0); break;
        case F_UP_DX: vb.init(b + n0 * lb + q.w0, lb, q.N - n0); break;
        case F_DOWN_DH: vb.init(b + (q.w0 + n0) * lb, lb, q.N - n0); break;
        default: vb.init(b + q.t0 * lb + n0, lb, q.N - n0); break;  // both dW
      }
      if constexpr (glu) vu.init(b + q.w0 + q.w + n0, lb, q.N - n0);
      if (F == F_UP_DW && map) {
        // gathered token rows as K: each stage's map entries are read a stage
        // ahead of its rows
        int32_t tok[kRuns];
        auto entries = [&](int64_t k0) {
#pragma unroll
          for (int i = 0; i < kRuns; ++i) {
            int k, x;
            run_at<false>(i, k, x);
            tok[i] = k0 + k < q.K ? map[q.t0 + k0 + k] : -1;
          }
        };
        entries(0);
        const auto rs = f32_rsrc(va.base);
        auto run = [&](auto w) {
          constexpr bool WIDE = decltype(w)::value;
          multiply([&](int64_t k0) {
#pragma unroll
            for (int i = 0; i < kRuns; ++i) {
              int k, x;
              run_at<false>(i, k, x);
              const bool ok = tok[i] >= 0 && tok[i] < p.a_rows;
              ra[i] = f32_run<WIDE>(rs, (uint32_t)((tok[i] * la + x) * 4), ok ? va.n[i] : 0);
            }
            entries(k0 + kBK);
            vb.template load<WIDE>(rb, k0, q.K);
          });
        };
        if (wide) run(std::true_type{}); else run(std::false_type{});
      } else {
        auto run = [&](auto w) {
          constexpr bool WIDE = decltype(w)::value;
          multiply([&](int64_t k0) {
            va.template load<WIDE>(ra, k0, q.K);
            vb.template load<WIDE>(rb, k0, q.K);
            if constexpr (glu) vu.template load<WIDE>(ru, k0, q.K);
          });
        };
        if (wide) run(std::true_type{}); else run(std::false_type{});
      }
    } else {
      multiply([&](int64_t k0) {
        if (F == F_UP_DX && p.act != VMOE_ACT_NONE)
          load_stage<AK>(ra, [&](int k, int x) {
            return make_float4(f32_a<F>(p, q, m0 + x, k0 + k), f32_a<F>(p, q, m0 + x, k0 + k + 1),
                               f32_a<F>(p, q, m0 + x, k0 + k + 2),
                               f32_a<F>(p, q, m0 + x, k0 + k + 3));
          });
        else
          load_stage<AK>(ra, [&](int k, int x) { return f32_a_run<F>(p, q, m0 + x, k0 + k); });
        if (F == F_UP_DW && p.act != VMOE_ACT_NONE)
          load_stage<BKC>(rb, [&](int k, int x) {
            return make_float4(f32_b<F>(p, q, k0 + k, n0 + x, false),
                               f32_b<F>(p, q, k0 + k, n0 + x + 1, false),
                               f32_b<F>(p, q, k0 + k, n0 + x + 2, false),
                               f32_b<F>(p, q, k0 + k, n0 + x + 3, false));
          });
        else
          load_stage<BKC>(rb,
                          [&](int k, int x) { return f32_b_run<F>(p, q, k0 + k, n0 + x, false); });
        if constexpr (glu)
          load_stage<BKC>(ru,
                          [&](int k, int x) { return f32_b_run<F>(p, q, k0 + k, n0 + x, true); });
      });
    }
    // acc[v]: row 8 (v / 4) + 4 (lane / 32) + v % 4, column lane % 32 of the block
    const int64_t n = n0 + wn + (lane & 31);
    if (n >= q.N) continue;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int64_t m = m0 + wm + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
      if (m >= q.M) continue;
      const float z = acc[v];
      if (F == F_UP_DW) {
        p.c[m * p.ldc + q.w0 + n] = z;
      } else if (F == F_DOWN_DW) {
        p.c[(q.w0 + m) * p.ldc + n] = z;
      } else {
        const int64_t o = (q.t0 + m) * p.ldc + n;
        if (F == F_UP_FWD && p.act == VMOE_ACT_RELU_SQUARED) {
          const float r = fmaxf(z, 0.0f);
          if (p.c2) p.c2[o] = r;
          p.c[o] = r * r;
        } else if constexpr (glu) {
          const float u = acc_up[v];
          if (p.c2) p.c2[o] = z;
          if (p.c3) p.c3[o] = u;
          if (p.c) p.c[o] = z * sigmoid32(z) * u;
        } else if (F == F_DOWN_DH && p.pre) {
          const float pr = p.pre[o];  // the relu^2 rule (pre shares c's layout)
          p.c[o] = pr > 0.0f ? z * 2.0f * pr : 0.0f;
        } else {
          p.c[o] = z;
        }
      }
    }
  }
}

// Upper bound of the tiles of one launch (sizes the grid; workgroups past
// the real count leave at once).
int64_t tile_bound(int64_t E, int64_t m_bound, int64_t n_bound, bool rows_m) {
  const int64_t tn = (n_bound + kT - 1) / kT;
  const int64_t tm = rows_m ? (m_bound + kT - 1) / kT + E : E * ((m_bound + kT - 1) / kT);
  return tm * tn;
}

template <int F, bool GLU = false>
int f32_launch(const F32Args& p, int64_t bound, hipStream_t s) {
  if (bound <= 0 || p.rows_bound == 0 || p.max_width == 0) return VMOE_OK;  // no work
  // one workgroup per tile in eight XCD ranges (find_tile), so that the
  // hardware deals tiles of unequal K to free slots; past the real count they
  // leave at once
  const int64_t grid = std::min<int64_t>((bound + 7) / 8 * 8, 1 << 22);
  if (f32_vec<F>(p))
    VMOE_LAUNCH((grouped_gemm_f32_kernel<F, GLU, true>), dim3((unsigned)grid), dim3(kThreads), 0,
                s, p);
  else
    VMOE_LAUNCH((grouped_gemm_f32_kernel<F, GLU, false>), dim3((unsigned)grid), dim3(kThreads), 0,
                s, p);
  VMOE_CHECK_LAUNCH();
  return VMOE_OK;
}

int f32_common(const int32_t* eto, const int32_t* ewo, const int32_t* widths,
               const int32_t* tpe, int32_t E, int64_t hidden, int64_t max_width,
               int64_t rows_bound) {
  if (!eto || !ewo || !widths || !tpe || E <= 0 || hidden <= 0 || max_width < 0 ||
      rows_bound < 0)
    return VMOE_ERR_INVALID_ARG;
  return VMOE_OK;
}

F32Args f32_args(const int32_t* eto, const int32_t* ewo, const int32_t* widths,
                 const int32_t* tpe, int32_t E, int64_t hidden, int64_t max_width,
                 int64_t rows_bound, int act) {
  F32Args p{};
  p.eto = eto; p.ewo = ewo; p.widths = widths; p.tpe = tpe;
  p.E = E; p.act = act; p.hidden = hidden; p.max_width = max_width; p.rows_bound = rows_bound;
  return p;
}

bool act_ok(int act) {
  return act == VMOE_ACT_NONE || act == VMOE_ACT_RELU_SQUARED || act == VMOE_ACT_SWIGLU;
}

// grad/pre/up of the backward GEMMs: pre is needed for relu^2, pre and up
// for SwiGLU.
bool grad_ok(const float* g, const float* pre, const float* up, int64_t ldg, int64_t max_width,
             int act) {
  if (!g || ldg < max_width || ldg <= 0) return false;
  if (act == VMOE_ACT_RELU_SQUARED && !pre) return false;
  if (act == VMOE_ACT_SWIGLU && (!pre || !up)) return false;
  return true;
}

__global__ __launch_bounds__(256) void f32_relu2_grad_kernel(const float* g, const float* pre,
                                                             int64_t ld, float* ga, int64_t ldo,
                                                             int64_t rows, int64_t cols) {
  const int64_t n = rows * cols;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / cols, c = i - r * cols;
    const float pr = pre[r * ld + c];
    ga[r * ldo + c] = pr > 0.0f ? g[r * ld + c] * 2.0f * pr : 0.0f;
  }
}

}  // namespace
}  // namespace vmoe

using namespace vmoe;

extern "C" int vmoe_f32_relu2_grad(const float* grad_h, const float* pre_act, int64_t ld,
                                   float* grad_act, int64_t ldo, int64_t rows, int64_t cols,
                                   vmoe_stream_t stream) {
  if (rows < 0 || cols < 0 || ld < cols || ldo < cols) return VMOE_ERR_INVALID_ARG;
  if (rows == 0 || cols == 0) return VMOE_OK;
  if (!grad_h || !pre_act || !grad_act) return VMOE_ERR_INVALID_ARG;
  const int64_t n = rows * cols;
  const int64_t blocks = std::min<int64_t>((n + 255) / 256, 8192);
  VMOE_LAUNCH(f32_relu2_grad_kernel, dim3((unsigned)blocks), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), grad_h, pre_act, ld, grad_act, ldo,
                     rows, cols);
  VMOE_CHECK_LAUNCH();
  return VMOE_OK;
}

extern "C" int vmoe_gemm_f32_up_fwd(const float* x, int64_t ldx, int64_t x_rows,
                                    const int32_t* gather_map, const float* w1, int64_t ldw1,
                                    float* out, float* pre_act, float* up, int64_t ldo,
                                    int32_t activation, const int32_t* eto, const int32_t* ewo,
                                    const int32_t* widths, const int32_t* tpe, int32_t E,
                                    int64_t hidden, int64_t max_width, int64_t rows_bound,
                                    vmoe_stream_t stream) {
  int st = f32_common(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound);
  if (st) return st;
  if (!act_ok(activation) || !x || !w1 || x_rows < 0 || ldx < hidden || ldw1 <= 0 ||
      ldo < max_width || ldo <= 0)
    return VMOE_ERR_INVALID_ARG;
  if (!out && !(activation == VMOE_ACT_SWIGLU && (pre_act || up))) return VMOE_ERR_INVALID_ARG;
  F32Args p = f32_args(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound, activation);
  p.a = x; p.lda = ldx; p.a_rows = x_rows; p.a_map = gather_map;
  p.b = w1; p.ldb = ldw1;
  p.c = out; p.ldc = ldo;
  p.c2 = activation == VMOE_ACT_NONE ? nullptr : pre_act;
  p.c3 = activation == VMOE_ACT_SWIGLU ? up : nullptr;
  const int64_t bound = tile_bound(E, rows_bound, max_width, true);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  return activation == VMOE_ACT_SWIGLU ? f32_launch<F_UP_FWD, true>(p, bound, s)
                                       : f32_launch<F_UP_FWD>(p, bound, s);
}

extern "C" int vmoe_gemm_f32_down_fwd(const float* h, int64_t ldh, const float* w2, int64_t ldw2,
                                      float* y, int64_t ldy, const int32_t* eto,
                                      const int32_t* ewo, const int32_t* widths,
                                      const int32_t* tpe, int32_t E, int64_t hidden,
                                      int64_t max_width, int64_t rows_bound,
                                      vmoe_stream_t stream) {
  int st = f32_common(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound);
  if (st) return st;
  if (!h || !w2 || !y || ldh < max_width || ldh <= 0 || ldw2 < hidden || ldy < hidden)
    return VMOE_ERR_INVALID_ARG;
  F32Args p = f32_args(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound, VMOE_ACT_NONE);
  p.a = h; p.lda = ldh;
  p.b = w2; p.ldb = ldw2;
  p.c = y; p.ldc = ldy;
  return f32_launch<F_DOWN_FWD>(p, tile_bound(E, rows_bound, hidden, true),
                                reinterpret_cast<hipStream_t>(stream));
}

extern "C" int vmoe_gemm_f32_up_bwd_dx(const float* grad_h, const float* pre_act,
                                       const float* up, int64_t ldg, int32_t activation,
                                       const float* w1, int64_t ldw1, float* grad_x,
                                       int64_t ldgx, const int32_t* eto, const int32_t* ewo,
                                       const int32_t* widths, const int32_t* tpe, int32_t E,
                                       int64_t hidden, int64_t max_width, int64_t rows_bound,
                                       vmoe_stream_t stream) {
  int st = f32_common(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound);
  if (st) return st;
  if (!act_ok(activation) || !grad_ok(grad_h, pre_act, up, ldg, max_width, activation) || !w1 ||
      ldw1 <= 0 || !grad_x || ldgx < hidden)
    return VMOE_ERR_INVALID_ARG;
  F32Args p = f32_args(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound, activation);
  p.g = grad_h; p.pre = pre_act; p.up = up; p.ldg = ldg;
  p.b = w1; p.ldb = ldw1;
  p.c = grad_x; p.ldc = ldgx;
  return f32_launch<F_UP_DX>(p, tile_bound(E, rows_bound, hidden, true),
                             reinterpret_cast<hipStream_t>(stream));
}

extern "C" int vmoe_gemm_f32_up_bwd_dw(const float* x, int64_t ldx, int64_t x_rows,
                                       const int32_t* gather_map, const float* grad_h,
                                       const float* pre_act, const float* up, int64_t ldg,
                                       int32_t activation, float* grad_w1, int64_t ldgw,
                                       const int32_t* eto, const int32_t* ewo,
                                       const int32_t* widths, const int32_t* tpe, int32_t E,
                                       int64_t hidden, int64_t max_width, int64_t rows_bound,
                                       vmoe_stream_t stream) {
  int st = f32_common(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound);
  if (st) return st;
  if (!act_ok(activation) || !grad_ok(grad_h, pre_act, up, ldg, max_width, activation) || !x ||
      x_rows < 0 || ldx < hidden || !grad_w1 || ldgw <= 0)
    return VMOE_ERR_INVALID_ARG;
  F32Args p = f32_args(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound, activation);
  p.a = x; p.lda = ldx; p.a_rows = x_rows; p.a_map = gather_map;
  p.g = grad_h; p.pre = pre_act; p.up = up; p.ldg = ldg;
  p.c = grad_w1; p.ldc = ldgw;
  const int64_t n_bound = activation == VMOE_ACT_SWIGLU ? 2 * max_width : max_width;
  return f32_launch<F_UP_DW>(p, tile_bound(E, hidden, n_bound, false),
                             reinterpret_cast<hipStream_t>(stream));
}

namespace vmoe {
int gemm_f32_down_bwd_ga(const float* grad_y, int64_t ldgy, const float* w2, int64_t ldw2,
                         const float* pre_act, float* ga, int64_t ldga, const int32_t* eto,
                         const int32_t* ewo, const int32_t* widths, const int32_t* tpe, int32_t E,
                         int64_t hidden, int64_t max_width, int64_t rows_bound,
                         vmoe_stream_t stream) {
  int st = f32_common(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound);
  if (st) return st;
  if (!grad_y || ldgy < hidden || !w2 || ldw2 < hidden || !ga || ldga < max_width || ldga <= 0)
    return VMOE_ERR_INVALID_ARG;
  F32Args p = f32_args(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound, VMOE_ACT_NONE);
  p.a = grad_y; p.lda = ldgy;
  p.b = w2; p.ldb = ldw2;
  p.pre = pre_act;
  p.c = ga; p.ldc = ldga;
  return f32_launch<F_DOWN_DH>(p, tile_bound(E, rows_bound, max_width, true),
                               reinterpret_cast<hipStream_t>(stream));
}
}  // namespace vmoe

extern "C" int vmoe_gemm_f32_down_bwd_dh(const float* grad_y, int64_t ldgy, const float* w2,
                                         int64_t ldw2, float* grad_h, int64_t ldgh,
                                         const int32_t* eto, const int32_t* ewo,
                                         const int32_t* widths, const int32_t* tpe, int32_t E,
                                         int64_t hidden, int64_t max_width, int64_t rows_bound,
                                         vmoe_stream_t stream) {
  return gemm_f32_down_bwd_ga(grad_y, ldgy, w2, ldw2, nullptr, grad_h, ldgh, eto, ewo, widths, tpe,
                              E, hidden, max_width, rows_bound, stream);
}

extern "C" int vmoe_gemm_f32_down_bwd_dw(const float* h, int64_t ldh, const float* grad_y,
                                         int64_t ldgy, float* grad_w2, int64_t ldgw,
                                         const int32_t* eto, const int32_t* ewo,
                                         const int32_t* widths, const int32_t* tpe, int32_t E,
                                         int64_t hidden, int64_t max_width, int64_t rows_bound,
                                         vmoe_stream_t stream) {
  int st = f32_common(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound);
  if (st) return st;
  if (!h || ldh < max_width || ldh <= 0 || !grad_y || ldgy < hidden || !grad_w2 ||
      ldgw < hidden)
    return VMOE_ERR_INVALID_ARG;
  F32Args p = f32_args(eto, ewo, widths, tpe, E, hidden, max_width, rows_bound, VMOE_ACT_NONE);
  p.a = h; p.lda = ldh;
  p.b = grad_y; p.ldb = ldgy;
  p.c = grad_w2; p.ldc = ldgw;
  return f32_launch<F_DOWN_DW>(p, tile_bound(E, max_width, hidden, false),
                               reinterpret_cast<hipStream_t>(stream));
}
