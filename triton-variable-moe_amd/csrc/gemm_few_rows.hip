// The layer's up and down projections where its experts get few tokens each (a
// generation step), with the bits of the 128 x 256 kernels in gemm.hip.
//
// What bounds them is reading the weights of the experts that got tokens, and
// how much of it is in flight. The 128 x 256 kernel has one tile per expert and
// 256 columns, so 64 experts of 256 columns use 64 CUs, and each walks K in
// stages of 32, three in flight. Here a workgroup takes 64 rows x 64 columns,
// so four times the CUs read, and a stage is 128 deep: 16 KB of weights and 16
// KB of activations, three stages in flight behind the one in work. The tile
// of 32 x 32 per wave takes the k-steps in the same order with the same
// operands as gemm.hip's, so each sum has the same bits and the layer's other
// paths (and its backward) see no difference. Measured us a launch, before and
// now: up 16.7 and 9.7, down 12.4 and 6.6 with 16 assignments through 8 experts
// 768 -> 512; up 21.2 and 12.0 with 512 through 64 experts 1024 -> 256 (33 MB of
// weights: 2.8 TB/s; what is left is the chain of table, row map, first stage).
#include <algorithm>

#include "vmoe_common.h"

namespace vmoe {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) bf16x8_t lds_bf16x8;
typedef __attribute__((address_space(3))) bf16x4_t lds_bf16x4;

constexpr int kThreads = 256;
constexpr int kTile = 64;  // rows and columns of a workgroup, 2 x 2 waves
constexpr int kDepth = 128;
constexpr int kABytes = kTile * kDepth * 2, kBBytes = kDepth * kTile * 2;
constexpr int kStageBytes = kABytes + kBBytes;
constexpr int kDmas = 8;  // of one wave and stage: four of A, four of B
constexpr uint32_t kOob = 0x80000000u;

struct Args {
  const uint16_t* a;  // x (through map) or H
  int64_t lda;
  const int32_t* map;
  int64_t a_rows;
  const uint16_t* b;  // W1 or W2
  int64_t ldb;
  uint16_t *c, *pre;
  int64_t ldc;
  const float* row_scale;
  const int32_t *eto, *ewo, *widths, *tpe;
  int E, hidden;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), 0,
                                           0x7FFFFFFF, 0x00020000);
}

// 16 bytes per lane into LDS at lds + 16 * lane; the data never passes through
// registers, so completion is ordered by the waits in the loop.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
               :: "v"(voff), "s"(r), "s"(lds) : "memory", "m0");
}

// Workgroup -> expert, 64-row block, 64-column slab. An XCD (blockIdx % 8) takes
// a contiguous eighth of the items, the slabs of a row block one after the
// other: they share its activations in the XCD's L2. False past the last item.
template <bool UP>
__device__ __forceinline__ bool find_item(const Args& p, int& expert, int& mblk, int& slab) {
  const int lane = threadIdx.x & (kWave - 1);
  auto slabs_of = [&](int e) { return ((UP ? p.widths[e] : p.hidden) + kTile - 1) / kTile; };
  auto items_of = [&](int e) {
    return e < p.E ? (p.tpe[e] + kTile - 1) / kTile * slabs_of(e) : 0;
  };
  int total = 0, first = 0;
  for (int e0 = 0; e0 < p.E; e0 += kWave) {
    const int inc = wave_inclusive_scan(items_of(e0 + lane));
    if (e0 == 0) first = inc;
    total += __shfl(inc, kWave - 1);
  }
  const int per = (total + 7) / 8;
  const int j = blockIdx.x >> 3, t = (blockIdx.x & 7) * per + j;
  if (j >= per || t >= total) return false;
  int before = 0;
  for (int e0 = 0; e0 < p.E; e0 += kWave) {
    const int inc = e0 == 0 ? first : wave_inclusive_scan(items_of(e0 + lane));
    const uint64_t past = ballot64(before + inc > t);
    if (past) {
      const int l = __builtin_ctzll(past);
      const int prev = __shfl(inc, max(l - 1, 0));
      expert = __builtin_amdgcn_readfirstlane(e0 + l);
      const int local = __builtin_amdgcn_readfirstlane(t - before - (l > 0 ? prev : 0));
      const int slabs = slabs_of(expert);
      mblk = __builtin_amdgcn_readfirstlane(local / slabs);
      slab = __builtin_amdgcn_readfirstlane(local % slabs);
      return true;
    }
    before += __shfl(inc, kWave - 1);
  }
  return false;
}

// Waits until all but the last `stages` issued stages of this wave are in LDS
// and this wave's own LDS reads are done.
__device__ __forceinline__ void wait_stages(int stages) {
  if (stages >= 3)
    asm volatile("s_waitcnt vmcnt(24) lgkmcnt(0)" ::: "memory");
  else if (stages == 2)
    asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)" ::: "memory");
  else if (stages == 1)
    asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
  else
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}
static_assert(kDmas == 8, "wait_stages counts eight DMAs a stage");

__device__ __forceinline__ void block_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// S: stages in LDS. 4 (128 KB, one workgroup to a CU), or 2 (two to a CU) where
// K is at most two stages.
template <bool UP, int S>
__global__ __launch_bounds__(kThreads) void few_rows_kernel(Args p) {
  static_assert(S >= 2 && S <= 4, "wait_stages covers up to three stages in flight");
  __shared__ __align__(1024) char lds[S * kStageBytes];
  int e, mblk, slab;
  if (!find_item<UP>(p, e, mblk, slab)) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m0 = mblk * kTile, n0 = slab * kTile;
  const int t0 = __builtin_amdgcn_readfirstlane(p.eto[e]) + m0;  // the block's first row
  const int ew = __builtin_amdgcn_readfirstlane(p.ewo[e]);
  const int width = __builtin_amdgcn_readfirstlane(p.widths[e]);
  const int rows = __builtin_amdgcn_readfirstlane(min(kTile, p.tpe[e] - m0));
  // Real rows come first. A block of pad rows is zeros in PRE and H'
  // (relu(0) whatever the weights hold), so K = 0; its Y rows are read by no one.
  const bool pad = __builtin_amdgcn_readfirstlane(p.map[t0]) < 0;
  if (!UP && pad) return;
  const int N = (UP ? width : p.hidden) - n0, K = UP ? (pad ? 0 : p.hidden) : width;
  const int stages = (K + kDepth - 1) / kDepth;

  // A stage: 64 rows of 256 bytes, 16-byte piece q of row r at q ^ (r % 16), so
  // the 16 rows that one cycle of a fragment read takes lie on all 64 banks.
  // DMA i of a wave: rows 16 wave + 4 i .. + 3, 16 lanes each.
  const auto ars = make_rsrc(UP ? p.a : p.a + (int64_t)t0 * p.lda);
  uint32_t aoff[4];
  int ak[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 16 * wave + 4 * i + (lane >> 4);
    int64_t src = r;
    bool ok = r < rows;
    if (UP && ok) {
      src = p.map[t0 + r];
      ok = src >= 0 && src < p.a_rows;
    }
    ak[i] = ((lane & 15) ^ (r & 15)) * 8;
    aoff[i] = ok ? (uint32_t)((src * p.lda + ak[i]) * 2) : kOob;
  }
  // B stage: 128 k-rows of 128 bytes, piece q of k-row k at q ^ 4 ((k / 2) % 2)
  // for the transposing reads. DMA i: k-rows 32 wave + 8 i .. + 7, 8 lanes each.
  const auto brs = make_rsrc(UP ? p.b + ew + n0 : p.b + (int64_t)ew * p.ldb + n0);
  const int bk = 32 * wave + (lane >> 3);
  const int bn = ((lane & 7) ^ ((bk >> 1 & 1) << 2)) * 8;
  const uint32_t boff = (uint32_t)((bk * p.ldb + bn) * 2), bstep = (uint32_t)(8 * p.ldb * 2);
  const uint32_t base = __builtin_amdgcn_readfirstlane(
      (uint32_t)reinterpret_cast<uintptr_t>((lds_char*)lds));
  auto issue = [&](int c) {
    const uint32_t dst = base + (c % S) * kStageBytes + wave * 4096;
    const int k0 = c * kDepth;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      dma16(brs, k0 + bk + 8 * i < K && bn < N
                     ? boff + (uint32_t)k0 * (uint32_t)(p.ldb * 2) + i * bstep : kOob,
            dst + kABytes + i * 1024);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      dma16(ars, aoff[i] != kOob && k0 + ak[i] < K ? aoff[i] + (uint32_t)(k0 * 2) : kOob,
            dst + i * 1024);
  };

  const int wm = wave >> 1, wn = wave & 1;
  const int arow = 32 * wm + (lane & 31);
  const int bcol = 32 * wn + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const int brow = 8 * (lane >> 5) + ((lane & 15) >> 2);
  f32x16_t acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  for (int c = 0; c < S && c < stages; ++c) issue(c);
  for (int c = 0; c < stages; ++c) {
    // issued so far: stages 0 .. max(S, c - 1 + S) - 1
    wait_stages(min(stages, c == 0 ? S : c - 1 + S) - 1 - c);
    block_barrier();  // stage c is whole, and all waves have read stage c - 1
    if (c > 0 && c - 1 + S < stages) issue(c - 1 + S);
    const lds_char* sa = (lds_char*)lds + (c % S) * kStageBytes;
    const lds_char* sb = sa + kABytes;
    const int steps = min(kDepth, K - c * kDepth + 15) / 16;
#pragma unroll
    for (int ks = 0; ks < kDepth / 16; ++ks) {
      if (ks >= steps) break;
      const bf16x8_t af = *reinterpret_cast<const lds_bf16x8*>(
          sa + arow * 256 + (((2 * ks + (lane >> 5)) ^ (arow & 15)) << 4));
      const int kr = 16 * ks + brow;
      const lds_char* b =
          sb + kr * 128 + (((bcol >> 3) ^ ((kr >> 1 & 1) << 2)) << 4) + (bcol & 7) * 2;
      const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)b);
      const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(b + 4 * 128));
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), af, acc, 0, 0, 0);
    }
  }
  // acc[4 g + r]: row 32 wm + lane % 32, column 32 wn + 8 g + 4 (lane / 32) + r
  if (arow >= rows) return;
  const int64_t out = (int64_t)t0 + arow;
  const float sc = UP ? p.row_scale[out] : 1.0f;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int n = 32 * wn + 8 * g + 4 * (lane >> 5);
    if (n >= N) break;
    float v[4] = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    if (UP) {
      // PRE = bf16(relu(z)), H' = bf16(w relu(z)^2), as gemm.hip's epilogue
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = fmaxf(v[r], 0.0f);
      *reinterpret_cast<uint2*>(p.pre + out * p.ldc + n0 + n) =
          make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = sc * (v[r] * v[r]);
    }
    *reinterpret_cast<uint2*>(p.c + out * p.ldc + n0 + n) =
        make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
  }
}

template <bool UP>
int launch(const Args& p, int64_t blocks, int64_t N, int64_t K, hipStream_t s) {
  const int64_t items = blocks * ((N + kTile - 1) / kTile);
  if (items <= 0) return VMOE_OK;
  const int64_t grid = (items + 7) / 8 * 8;
  if (grid > INT32_MAX / kThreads) return VMOE_ERR_UNSUPPORTED;
  if (K <= 2 * kDepth)
    VMOE_LAUNCH((few_rows_kernel<UP, 2>), dim3((unsigned)grid), dim3(kThreads), 0, s, p);
  else
    VMOE_LAUNCH((few_rows_kernel<UP, 4>), dim3((unsigned)grid), dim3(kThreads), 0, s, p);
  VMOE_CHECK_LAUNCH();
  return VMOE_OK;
}

// At most so many row blocks with tokens in them: every expert's count of
// tokens rounded up to 64.
inline int64_t live_blocks(int64_t assignments, int64_t E) {
  return assignments / kTile + std::min(E, assignments);
}

// A grid bound: blocks of padded rows too. At most min(E, assignments) experts
// have rows, each padded by less than block_size; a padded count that is no
// multiple of 64 ends in a part of a block.
inline int64_t grid_blocks(int64_t assignments, int64_t E, int64_t block_size) {
  const int64_t live = std::min(E, assignments);
  return (assignments + live * (block_size - 1)) / kTile + (block_size % kTile ? live : 0);
}

inline bool a16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }
inline bool ld_ok(int64_t ld, int64_t cols, bool zero) {
  return (zero && ld == 0) || (ld >= cols && ld % 8 == 0);
}
// byte offsets of a source stay below the 31 bits that a DMA takes
inline bool span_ok(int64_t rows, int64_t ld) { return rows * ld * 2 < ((int64_t)1 << 31); }

}  // namespace

// A workgroup here does one tile, started cold, and ends, where the persistent
// 128 x 256 kernel loads its next tile during the last one's k-steps. So these
// win while one round of the 256 CUs, or a little more, takes all tiles. Whole
// forward in a graph, us with 128 x 256 tiles and with these: 8 experts 768 ->
// 512 at 24 row blocks (192 + 288 tiles) 47.8 and 34.1, at 40 (up 320 of these,
// down 480 of the old) 49.7 and 47.4; 64 experts 1024 -> 256 at 72 - 96 blocks
// (up 288 - 384) 56.7 and 48.9, 58.9 and 50.2. Without the line: 64 experts at
// 128 blocks (512 and 2048 tiles) 61.8 and 61.6, at 192 69.5 and 79.6; 128
// experts 2048 -> 1024 / 512 / 256 185 and 258. With it, 140 forwards drawn over
// 1-128 experts, widths 64-1024, 64-2048 hidden columns and 1-512 tokens are
// 0.98-1.4 times as fast as without, 1.20 in the mean (below 1 where neither
// projection takes these tiles).
bool few_rows_fits(int64_t assignments, int64_t E, int64_t cols) {
  return cols > 0 && live_blocks(assignments, E) * ((cols + kTile - 1) / kTile) <= kFewRowsItems;
}

int few_rows_up(const uint16_t* x, int64_t ldx, int64_t x_rows, const int32_t* map,
                const uint16_t* w1, int64_t ldw1, uint16_t* h, uint16_t* pre, int64_t ldh,
                const float* row_scale, const int32_t* eto, const int32_t* ewo,
                const int32_t* widths, const int32_t* tpe, int E, int64_t hidden,
                int64_t max_width, int64_t assignments, int block_size, vmoe_stream_t stream) {
  if (hidden % 8 || max_width % 8 || !ld_ok(ldx, hidden, true) || !ld_ok(ldw1, 1, false) ||
      !ld_ok(ldh, max_width, false) || !a16(x) || !a16(w1) || !a16(h) || !a16(pre) ||
      !span_ok(x_rows, ldx) || !span_ok(hidden, ldw1))
    return VMOE_ERR_UNSUPPORTED;
  Args p{};
  p.a = x; p.lda = ldx; p.map = map; p.a_rows = x_rows;
  p.b = w1; p.ldb = ldw1;
  p.c = h; p.pre = pre; p.ldc = ldh;
  p.row_scale = row_scale;
  p.eto = eto; p.ewo = ewo; p.widths = widths; p.tpe = tpe;
  p.E = E; p.hidden = (int)hidden;
  return launch<true>(p, grid_blocks(assignments, E, block_size), max_width, hidden,
                      reinterpret_cast<hipStream_t>(stream));
}

int few_rows_down(const uint16_t* h, int64_t ldh, const int32_t* map, const uint16_t* w2,
                  int64_t ldw2, uint16_t* y, int64_t ldy, const int32_t* eto,
                  const int32_t* ewo, const int32_t* widths, const int32_t* tpe, int E,
                  int64_t hidden, int64_t max_width, int64_t assignments, int block_size,
                  vmoe_stream_t stream) {
  if (hidden % 8 || max_width % 8 || !ld_ok(ldh, max_width, false) ||
      !ld_ok(ldw2, hidden, false) || !ld_ok(ldy, hidden, false) || !a16(h) || !a16(w2) ||
      !a16(y) || !span_ok(max_width, ldw2))
    return VMOE_ERR_UNSUPPORTED;
  Args p{};
  p.a = h; p.lda = ldh; p.map = map;
  p.b = w2; p.ldb = ldw2;
  p.c = y; p.ldc = ldy;
  p.eto = eto; p.ewo = ewo; p.widths = widths; p.tpe = tpe;
  p.E = E; p.hidden = (int)hidden;
  return launch<false>(p, grid_blocks(assignments, E, block_size), hidden, max_width,
                       reinterpret_cast<hipStream_t>(stream));
}

}  // namespace vmoe

extern "C" int vmoe_moe_few_rows(int64_t num_assignments, int32_t num_experts, int64_t cols) {
  return num_assignments > 0 && num_experts > 0 &&
                 vmoe::few_rows_fits(num_assignments, num_experts, cols)
             ? 1 : 0;
}
