// Matrix products of a few tokens (up to 16: decoding at small batch) whose activations
// are made by the kernel itself instead of being read from memory.
//
// A decode step of a small model is a chain of short dependent kernels, and each link
// costs a few microseconds whatever it computes.  Two links per layer go away when the
// product that follows a norm computes the norm itself, and one more when the output
// product of the attention merges the split-KV partitions itself:
//  * norm prologue: every workgroup adds the not-yet-added delta (a bfloat16 tensor, or
//    float32 partial sums of a K-sliced product, in slice order) to the float32 residual
//    stream, takes the RMSNorm of the sum (src/mini_llm_runtime/qwen_model_runner.py:22-26,
//    statistics in 32-bit) and keeps the normed rows as bfloat16 in LDS; the workgroups whose
//    index matches a row also write that row of the updated stream to `x_out` (a buffer of
//    its own: other workgroups still read `x_in`).  The few rows are re-read by every
//    workgroup, from L2.
//  * merge prologue: every workgroup merges the partitions of the attention of its slice
//    of K (m = max m_j, O = sum w_j a_j / sum w_j l_j, w_j = exp2(m_j - m),
//    csrc/paged_attention_split_cuda.cu:66-88 of the reference) into LDS.
// Behind the norm the weights stream as in gemm_lines (gemm_norm_lines): whole lines straight into LDS, asked for by four wavefronts before
// the norm is there, which others make.  A workgroup has as many rows as make one round of the compute units, and one prologue.  Against 16 rows a
// workgroup through registers, 64 bytes of a row a load, the norm by the same wavefronts (one token, 4 slices to add up, microseconds in a replayed graph, weights from
// memory): 9,728 x 896 8.7 to 6.0 (4 tokens 10.7 to 6.5), 4,864 x 896 6.7 to 4.5, 5,120 x 2,048 11.0 to 6.7, 6,144 x 1,536 10.2 to 6.1, 2,048 x 2,048 7.5 to 5.3;
// query/key/value 1,152 x 896 5.4 to 4.4, 2,560 x 2,048 7.9 to 6.1.  Over 972 products of all forms (1 to 4 tokens, up to 16 slices) 0.75 of the time,
// two slower by more than 2 % (18,000 x 520, 4 tokens, 2 slices 11.0 to 11.5).
// In one round the norm's loads go first: its rows come from L2, and behind some 30 KB of weights from memory they would wait for those
// (9,728 x 896 7.3 instead of 6.0; query/key/value 3,072 x 1,024, 4 tokens, 8 slices 7.0 instead of 5.7, 6.2 through registers).
// Beyond one round (MANY) other workgroups' loads fill that time, and what counts is how many fit a unit: no more LDS than the steps of k fill
// (16 KB up to 256 columns) and one partial sum at a time (65 registers).  17,920 x 560 10.1 to 9.4 (10.5 with two workgroups a unit), 40,000 x
// 256 13.5 to 7.6 (11.8).
// Behind the merge they stream as in gemm_skinny_split: a workgroup owns 16 * NT output
// features and one slice of K, its four wavefronts split K, range-checked buffer loads
// keep two batches of eight 16-byte loads per lane in flight, the first of them issued
// before the prologue, and the wavefronts' sums meet in LDS.  Epilogues are those of
// gemm_mfma.hip: bias, SwiGLU, partial sums, or the query/key/value product's rotation and
// cache write.
#include "api.h"
#include "common.h"
#include "gemm_epilogue.h"
#include "mfma.h"

namespace mlr {

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct NormPrologue {
  const float* x_in;     // [M, K] residual stream
  float* x_out;          // [M, K] the stream with the delta added; null when there is no delta
  const bf16* delta;     // [M, K] or null
  const float* partial;  // [slices, M, K] or null
  int slices;
  const void* weight;  // [K]
  int weight_is_f32;
  float eps;
};

struct MergePrologue {
  const float* partial;     // [M, heads, all_splits, head_dim + 2]: numerator, max, denominator
  const int* context_lens;  // [M]
  int heads, head_dim, window, part, all_splits;
  unsigned bytes;  // of `partial`
};

constexpr int kFusedWaves = 4;
// k-steps per batch of loads and wavefront: eight 16-byte loads of a lane per batch and row block
constexpr int fused_depth(int row_blocks) { return row_blocks == 1 ? 8 : 4; }

// ---- norm prologue ------------------------------------------------------------------------
// A wavefront takes one row (so the kernels take up to four tokens).  Its work comes in two
// halves so that others can send loads between them: `issue` sends every load of the
// row (the stream, the delta, up to a batch of partial sums, the norm's weights), `finish` adds
// up, takes the statistics and writes the normed row to LDS: one trip to L2.  Columns past the end are range-checked
// away; what is absent (no delta, fewer partial sums than the batch holds) is not asked for: a load of an empty range
// costs as much of the unit's way to memory as any (query/key/value 1,152 x 896, 4 tokens, nothing to add, microseconds: 5.7 so, 5.3 without).
//
// Every workgroup reads the same few rows; were they all to read them in the same order, the
// whole chip would ask the same few L2 channels for the same lines at the same moment.  So a
// workgroup starts at a column of its own and wraps around.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x4 buffer_load_f32x4(__amdgpu_buffer_rsrc_t rsrc, unsigned byte_offset) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, byte_offset, 0, 0));
}
__device__ __forceinline__ u32x2 buffer_load_u32x2(__amdgpu_buffer_rsrc_t rsrc, unsigned byte_offset) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, byte_offset, 0, 0));
}
__device__ __forceinline__ float bf16_low(uint32_t pair) { return __builtin_bit_cast(float, pair << 16); }
__device__ __forceinline__ float bf16_high(uint32_t pair) { return __builtin_bit_cast(float, pair & 0xffff0000u); }

// SB: partial sums per trip: 8 of rows of up to 1,024 columns, 4 of longer ones (two wavefronts a SIMD have the registers for them), or 1.
template <int VPT, int SB>
struct NormRow {
  unsigned at[VPT];  // byte offset of this lane's columns within a float32 row, out of range past the end
  f32x4 v[VPT];
  f32x4 p[VPT][SB];
  u32x2 d[VPT];
  u32x4 w[VPT];  // four float32 weights, or four bfloat16 ones in the first half
};

template <int VPT, int SB>
__device__ __forceinline__ void norm_issue(const NormPrologue& np, NormRow<VPT, SB>& t, int row, int M, int K) {
  const int lane = threadIdx.x % kWave;
  const int quads = K / 4;
  const int rot = static_cast<int>((static_cast<unsigned>(blockIdx.x) * 40503u) % static_cast<unsigned>(quads));
  const unsigned row_bytes = static_cast<unsigned>(K) * 4u;
  const unsigned slab = static_cast<unsigned>(M) * row_bytes;
  const __amdgpu_buffer_rsrc_t x_buf = make_buffer(np.x_in + static_cast<int64_t>(row) * K, row_bytes);
  const __amdgpu_buffer_rsrc_t d_buf = make_buffer(np.delta + static_cast<int64_t>(row) * K, row_bytes / 2);
  const __amdgpu_buffer_rsrc_t p_buf =
      make_buffer(np.partial + static_cast<int64_t>(row) * K, static_cast<unsigned>(np.slices - 1) * slab + row_bytes);
  const __amdgpu_buffer_rsrc_t w_buf = make_buffer(np.weight, np.weight_is_f32 ? row_bytes : row_bytes / 2);
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int idx = lane + kWave * j;
    const int i = idx + rot;
    t.at[j] = idx < quads ? static_cast<unsigned>(i >= quads ? i - quads : i) * 16u : kOutOfBuffer;
  }
#pragma unroll
  for (int j = 0; j < VPT; ++j) t.v[j] = buffer_load_f32x4(x_buf, t.at[j]);
  if (np.delta != nullptr) {
#pragma unroll
    for (int j = 0; j < VPT; ++j) t.d[j] = buffer_load_u32x2(d_buf, t.at[j] / 2);
  }
#pragma unroll
  for (int u = 0; u < SB; ++u) {
    if (u >= np.slices) break;
#pragma unroll
    for (int j = 0; j < VPT; ++j) t.p[j][u] = buffer_load_f32x4(p_buf, t.at[j] + static_cast<unsigned>(u) * slab);
  }
  if (np.weight_is_f32) {
#pragma unroll
    for (int j = 0; j < VPT; ++j) t.w[j] = __builtin_bit_cast(u32x4, buffer_load_f32x4(w_buf, t.at[j]));
  } else {
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      const u32x2 pair = buffer_load_u32x2(w_buf, t.at[j] / 2);
      t.w[j] = u32x4{pair[0], pair[1], 0u, 0u};
    }
  }
  __builtin_amdgcn_sched_barrier(0);
}

template <int VPT, int SB>
__device__ __forceinline__ void norm_finish(const NormPrologue& np, NormRow<VPT, SB>& t, bf16* hb, int ldk, int row, int M,
                                            int K, int kcols) {
  const int lane = threadIdx.x % kWave;
  auto add_slices = [&](int first) {  // in order
#pragma unroll
    for (int u = 0; u < SB; ++u) {
      if (first + u >= np.slices) break;
#pragma unroll
      for (int j = 0; j < VPT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) t.v[j][e] += t.p[j][u][e];
    }
  };
  if (np.delta != nullptr) {
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      t.v[j][0] += bf16_low(t.d[j][0]);
      t.v[j][1] += bf16_high(t.d[j][0]);
      t.v[j][2] += bf16_low(t.d[j][1]);
      t.v[j][3] += bf16_high(t.d[j][1]);
    }
  }
  add_slices(0);
  if (np.slices > SB) {  // more partial sums than the first batch held
    const unsigned row_bytes = static_cast<unsigned>(K) * 4u;
    const unsigned slab = static_cast<unsigned>(M) * row_bytes;
    const __amdgpu_buffer_rsrc_t p_buf =
        make_buffer(np.partial + static_cast<int64_t>(row) * K, static_cast<unsigned>(np.slices - 1) * slab + row_bytes);
    for (int s0 = SB; s0 < np.slices; s0 += SB) {
#pragma unroll
      for (int u = 0; u < SB; ++u) {
        if (s0 + u >= np.slices) break;
#pragma unroll
        for (int j = 0; j < VPT; ++j) t.p[j][u] = buffer_load_f32x4(p_buf, t.at[j] + static_cast<unsigned>(s0 + u) * slab);
      }
      add_slices(s0);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < VPT; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) ss += t.v[j][e] * t.v[j][e];  // columns past the end read zeros
  const float total = wave_sum(ss);
  const float inv = 1.0f / sqrtf(total / static_cast<float>(K) + np.eps);
  const bool writes_stream = np.x_out != nullptr && row % static_cast<int>(gridDim.x) == static_cast<int>(blockIdx.x);
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (t.at[j] == kOutOfBuffer) continue;
    const unsigned col = t.at[j] / 4;
    if (writes_stream) *reinterpret_cast<f32x4*>(np.x_out + static_cast<int64_t>(row) * K + col) = t.v[j];
    const f32x4 wide = __builtin_bit_cast(f32x4, t.w[j]);
    float w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = np.weight_is_f32 ? wide[e] : e % 2 ? bf16_high(t.w[j][e / 2]) : bf16_low(t.w[j][e / 2]);
    const u32x2 packed = {pack_bf16x2(w[0] * (t.v[j][0] * inv), w[1] * (t.v[j][1] * inv)),
                          pack_bf16x2(w[2] * (t.v[j][2] * inv), w[3] * (t.v[j][3] * inv))};
    *reinterpret_cast<u32x2*>(hb + row * ldk + col) = packed;
  }
  // the tail of the last k-step: zeros (0 * whatever LDS held could be NaN)
  for (int c = K + lane; c < kcols; c += kWave) hb[row * ldk + c].bits = 0;
}

// ---- merge prologue -----------------------------------------------------------------------
// Merged attention of the tokens' heads that fall into columns [k_begin, k_end) into LDS.
// A thread makes 8 consecutive columns of one token (inside one head: the head size is a
// multiple of 8) from all partitions of that head, eight partitions per trip to L2, keeping a
// running maximum as the attention kernels do.  There is at most one such item per thread (the
// host sees to it).  `issue` sends the loads of the first eight partitions.
typedef float f32x2 __attribute__((ext_vector_type(2)));
constexpr int kMergeBatch = 8;

struct MergeItem {
  int m, c, splits;  // token, chunk of 8 columns within the slice, partitions of the token's entry
  unsigned at;       // byte offset of the chunk's first column within partition 0 of (token, head)
  unsigned tail;     // byte offset of (maximum, denominator) within partition 0
  f32x2 ml[kMergeBatch];
  f32x4 piece[kMergeBatch][2];
};

__device__ __forceinline__ void merge_load(const MergePrologue& mp, MergeItem& t, int s0) {
  const unsigned stride = static_cast<unsigned>(mp.head_dim + 2) * 4u;
  // one resource over all tokens' partitions (the same for every lane); partitions past an
  // entry's own read as zeros (out of range)
  const __amdgpu_buffer_rsrc_t buf = make_buffer(mp.partial, mp.bytes);
#pragma unroll
  for (int u = 0; u < kMergeBatch; ++u) {
    const unsigned off = s0 + u < t.splits ? static_cast<unsigned>(s0 + u) * stride : kOutOfBuffer;
    t.ml[u] = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(buf, t.tail + off, 0, 0));
    // rows of head_dim + 2 floats are 8-byte aligned only
    const u32x2 a = buffer_load_u32x2(buf, t.at + off), b = buffer_load_u32x2(buf, t.at + off + 8u);
    const u32x2 c = buffer_load_u32x2(buf, t.at + off + 16u), d = buffer_load_u32x2(buf, t.at + off + 24u);
    t.piece[u][0] = __builtin_bit_cast(f32x4, u32x4{a[0], a[1], b[0], b[1]});
    t.piece[u][1] = __builtin_bit_cast(f32x4, u32x4{c[0], c[1], d[0], d[1]});
  }
}

__device__ __forceinline__ void merge_issue(const MergePrologue& mp, MergeItem& t, int item, int M, int k_begin,
                                            int k_end, int kcols) {
  const int per_row = kcols / 8;
  t.m = item / per_row;
  t.c = item - t.m * per_row;
  const int k = min(k_begin + t.c * 8, k_end - 8);  // chunks past the end of K become zeros; their loads stay inside
  const int D = mp.head_dim;
  const int h = k / D;
  // the partitions that hold keys of this entry, as attn_decode cuts them
  const int ctx = mp.context_lens[t.m];
  const int first = mp.window > 0 ? max(0, ctx - mp.window) : 0;
  t.splits = min(mp.all_splits, (ctx - (first / 16) * 16 + mp.part - 1) / mp.part);
  const unsigned head_at = (static_cast<unsigned>(t.m) * mp.heads + h) * mp.all_splits * (D + 2) * 4u;
  t.at = head_at + static_cast<unsigned>(k - h * D) * 4u;
  t.tail = head_at + static_cast<unsigned>(D) * 4u;
  merge_load(mp, t, 0);
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void merge_finish(const MergePrologue& mp, MergeItem& t, bf16* hb, int ldk, int k_begin,
                                             int k_end) {
  float mstar = -INFINITY, den = 0.f;
  float num[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < t.splits; s0 += kMergeBatch) {
    if (s0 > 0) merge_load(mp, t, s0);
    float batch_max = -INFINITY;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) batch_max = fmaxf(batch_max, s0 + u < t.splits ? t.ml[u][0] : -INFINITY);
    const float m_new = fmaxf(mstar, batch_max);
    const float rescale = (mstar == -INFINITY) ? 0.f : fast_exp2(mstar - m_new);
    den *= rescale;
#pragma unroll
    for (int e = 0; e < 8; ++e) num[e] *= rescale;
    mstar = m_new;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      const float wgt = (s0 + u >= t.splits || t.ml[u][0] == -INFINITY) ? 0.f : fast_exp2(t.ml[u][0] - mstar);
      den += wgt * t.ml[u][1];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        num[e] += wgt * t.piece[u][0][e];
        num[4 + e] += wgt * t.piece[u][1][e];
      }
    }
  }
  u32x4 packed = {0u, 0u, 0u, 0u};
  if (k_begin + t.c * 8 < k_end && t.splits > 0) {
    const float inv = 1.0f / den;
#pragma unroll
    for (int e = 0; e < 4; ++e) packed[e] = pack_bf16x2(num[2 * e] * inv, num[2 * e + 1] * inv);
  }
  *reinterpret_cast<u32x4*>(hb + t.m * ldk + t.c * 8) = packed;
}

// The merge prologue.  A workgroup owns 16 * NT output features and a slice of K, its four wavefronts split K.
template <int NT>
__global__ __launch_bounds__(kFusedWaves* kWave) void gemm_few_fused_kernel(const bf16* __restrict__ w, GemmEpilogue ep, MergePrologue mp, int ldk,
                                                                            int M, int N, int K) {
  constexpr int U = fused_depth(NT);
  extern __shared__ __attribute__((aligned(16))) unsigned char fused_lds[];
  bf16* const hb = reinterpret_cast<bf16*>(fused_lds);
  __shared__ float red[kFusedWaves][NT][kWave][4];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // uniform, and said so: it picks buffers
  const int r = lane % 16;
  const int q = lane / 16;
  const int n0 = blockIdx.x * 16 * NT;
  const int slices = gridDim.y;
  const int chunks = K / 8;
  const int ksteps = (chunks + 3) / 4;
  const int per = (ksteps + slices - 1) / slices;
  const int sb = blockIdx.y * per;
  const int se = max(sb, min(ksteps, sb + per));  // a slice past the end of K is empty: its partial sums are zeros
  const int kcols = (se - sb) * 32;

  // Weights through a buffer resource: rows past the end of the matrix, chunks past the end of
  // K and k-steps past this slice read as zeros, without a branch around any load.
  const unsigned row_bytes = static_cast<unsigned>(K) * 2u;
  const __amdgpu_buffer_rsrc_t w_buf =
      make_buffer(w + static_cast<int64_t>(n0) * K, static_cast<unsigned>(min(16 * NT, N - n0)) * row_bytes);
  unsigned row_off[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) row_off[nt] = static_cast<unsigned>(nt * 16 + r) * row_bytes;
  auto load_weights = [&](int s0, bf16x8_t (&a)[U][NT]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u * kFusedWaves;
      const int c = s * 4 + q;
      const bool in = s < se && c < chunks;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        a[u][nt] = __builtin_bit_cast(
            bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(w_buf, in ? row_off[nt] + c * 16u : kOutOfBuffer, 0, 2));
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // Order of the loads: the prologue's own first (they come from L2 and are waited for first;
  // loads return in the order they were sent), then the first batch of weights, which streams
  // from memory while the activations are made.
  bf16x8_t a0[U][NT], a1[U][NT];
  MergeItem item;
  const int k_begin = sb * 32, k_end = min(K, se * 32);
  const int items = M * (kcols / 8);
  // a workgroup starts at an item of its own (see the norm prologue: everybody reads the same rows)
  const int turn = static_cast<int>((static_cast<unsigned>(blockIdx.x) * 40503u) % static_cast<unsigned>(max(items, 1)));
  const int mine = static_cast<int>(threadIdx.x) + turn >= items ? static_cast<int>(threadIdx.x) + turn - items
                                                                    : static_cast<int>(threadIdx.x) + turn;
  const bool has = static_cast<int>(threadIdx.x) < items;
  if (has) merge_issue(mp, item, mine, M, k_begin, k_end, kcols);
  load_weights(sb + wave, a0);
  if (has) merge_finish(mp, item, hb, ldk, k_begin, k_end);
  __syncthreads();

  f32x4_t acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const bf16* brow = hb + min(r, M - 1) * ldk + q * 8;  // columns past M repeat the last row; their sums are dropped
  auto multiply = [&](int s0, const bf16x8_t (&a)[U][NT]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = min(s0 + u * kFusedWaves, se - 1);  // past the slice: the weights are zeros
      const bf16x8_t b = load_bf16x8(brow + (s - sb) * 32);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[nt] = mfma_16x16x32(a[u][nt], b, acc[nt]);
    }
  };
  constexpr int kBatch = kFusedWaves * U;
  for (int s0 = sb + wave; s0 < se; s0 += 2 * kBatch) {
    load_weights(s0 + kBatch, a1);
    multiply(s0, a0);
    if (s0 + kBatch >= se) break;
    load_weights(s0 + 2 * kBatch, a0);
    multiply(s0 + kBatch, a1);
  }

#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][nt][lane][i] = acc[nt][i];
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ww = 0; ww < kFusedWaves; ++ww)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += red[ww][nt][lane][i];
    finish4(ep, blockIdx.y, slices, r, n0 + nt * 16 + q * 4, M, N, v);
  }
}

// ---- the norm ahead of a product, whole lines of weights -----------------------------------------------
// The norm prologue with the weights streamed as by gemm_lines (gemm_mfma.hip): four wavefronts bring whole lines of 128 bytes of RUNS * 8
// rows straight into LDS, each the lines of its own steps of 64 k through buffers of its own, and up to four others
// norm a token's row each meanwhile.  (Wavefronts of their own: loads into registers and into LDS do not return in one order.)
// BUF: slices of LDS a wavefront.  MANY: more workgroups than one round of the compute units.
constexpr int norm_line_buffers(int runs) { return runs > 6 ? 3 : 4; }
constexpr int norm_line_bytes(int runs, int buffers) { return kFusedWaves * buffers * runs * 1024; }
constexpr int norm_slice_batch(int vpt, bool many) { return many ? 1 : 32 / vpt; }

template <int RUNS, int VPT, bool QKV, int BUF, bool MANY>
__device__ __forceinline__ void norm_lines(const bf16* __restrict__ w, const GemmEpilogue& ep, const QkvTarget& qkv, const NormPrologue& np, int ldk, int M, int N, int K) {
  constexpr int NB = (RUNS + 1) / 2;
  static_assert(!QKV || RUNS % 2 == 0, "a block of 16 holds 8 dims and their partners");
  extern __shared__ __attribute__((aligned(16))) unsigned char fused_lds[];
  bf16* const hb = reinterpret_cast<bf16*>(fused_lds + norm_line_bytes(RUNS, BUF));
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int steps = (K + 63) / 64;
  if (wave >= kFusedWaves) {
    const int row = wave - kFusedWaves;
    NormRow<VPT, norm_slice_batch(VPT, MANY)> t;
    norm_issue(np, t, row, M, K);
    if (!MANY) __builtin_amdgcn_s_barrier();  // from here on the others send theirs
    norm_finish(np, t, hb, ldk, row, M, K, steps * 64);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    return;
  }
  const int r = lane % 16, q = lane / 16;
  const int n0 = blockIdx.x * (RUNS * 8);
  const int chunks = K / 8;
  // the weight row behind row 0 of run `run` of 8
  auto run_row = [&](int run) {
    int first = n0 + run * 8;
    if (QKV) {
      const int at = blockIdx.x * NB + run / 2, per_head = qkv.head_dim / 16, head = at / per_head;
      if (qkv.cos != nullptr && head < qkv.heads + qkv.kv_heads)
        first = head * qkv.head_dim + (at - head * per_head) * 8 + run % 2 * (qkv.head_dim / 2);
    }
    return first;
  };
  const unsigned row_bytes = static_cast<unsigned>(K) * 2u;
  // query/key/value rows lie anywhere in the matrix, other rows follow one another
  const __amdgpu_buffer_rsrc_t w_buf = QKV ? make_buffer(w, static_cast<unsigned>(N) * row_bytes)
                                           : make_buffer(w + static_cast<int64_t>(n0) * K, static_cast<unsigned>(min(RUNS * 8, N - n0)) * row_bytes);
  const int row = lane / 8;  // pieces of a row in the order piece ^ (row / 2) % 8, rows counted over the runs
  unsigned from_row[RUNS];
#pragma unroll
  for (int p = 0; p < RUNS; ++p) {
    const int at = run_row(p) + row;
    from_row[p] = at < N ? static_cast<unsigned>(QKV ? at : at - n0) * row_bytes : kOutOfBuffer;
  }
  auto fetch = [&](int it) {
    const int s = it * kFusedWaves + wave;
#pragma unroll
    for (int p = 0; p < RUNS; ++p) {
      const int piece = (lane % 8) ^ ((4 * (p % 2) + row / 2) % 8);
      const unsigned at = s * 8 + piece < chunks ? from_row[p] + static_cast<unsigned>(s) * 128u + piece * 16u : kOutOfBuffer;  // a row past the end stays past it
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          w_buf, (__attribute__((address_space(3))) void*)(fused_lds + ((wave * BUF + it % BUF) * RUNS + p) * 1024), 16, at, 0, 0, 2);
    }
  };
  if (!MANY) __builtin_amdgcn_s_barrier();  // the norm's loads are on their way: behind these they would wait for memory
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < BUF; ++i) fetch(i);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();  // the normed rows are in LDS
  asm volatile("" ::: "memory");
  f32x4_t acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const bf16* const brow = hb + min(r, M - 1) * ldk + q * 8;  // columns past M repeat the last row; their sums are dropped
  const int swz = (r / 2) % 8;
  const int iterations = (steps + kFusedWaves - 1) / kFusedWaves;
  for (int it = 0; it < iterations; ++it) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((BUF - 1) * RUNS) : "memory");  // the oldest slice has landed; only this wavefront reads it
    const unsigned char* const base = fused_lds + (wave * BUF + it % BUF) * RUNS * 1024;
    const int s = min(it * kFusedWaves + wave, steps - 1);  // past the last step: the weights are zeros
    bf16x8_t a[2][NB], b[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int i = 0; i < NB; ++i) a[kk][i] = load_bf16x8(base + min(i * 16 + r, RUNS * 8 - 1) * 128 + (((kk * 4 + q) ^ swz) * 16));
      b[kk] = load_bf16x8(brow + s * 64 + kk * 32);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    fetch(it + BUF);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < NB; ++i) acc[i] = mfma_16x16x32(a[kk][i], b[kk], acc[i]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be on its way into LDS
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NB; ++i) *reinterpret_cast<f32x4_t*>(fused_lds + ((wave * NB + i) * kWave + lane) * 16) = acc[i];
  __syncthreads();
  if (wave >= NB) return;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ww = 0; ww < kFusedWaves; ++ww) {
    const f32x4_t part = *reinterpret_cast<const f32x4_t*>(fused_lds + ((ww * NB + wave) * kWave + lane) * 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += part[i];
  }
  if constexpr (QKV) {
    if (n0 + wave * 16 >= N) return;
    const int per_head = qkv.head_dim / 16, block = blockIdx.x * NB + wave, head = block / per_head;
    const bool rotated = qkv.cos != nullptr && head < qkv.heads + qkv.kv_heads;
    qkv_finish(ep, qkv, head, block - head * per_head, rotated, run_row(2 * wave + q / 2) + q % 2 * 4 - head * qkv.head_dim, q, min(r, M - 1), r < M, v);
  } else {
    if (wave * 16 + q * 4 < RUNS * 8) finish4(ep, 0, 1, r, n0 + wave * 16 + q * 4, M, N, v);
  }
}

template <int RUNS, int VPT, bool QKV, int BUF, bool MANY>
__global__ __launch_bounds__(2 * kFusedWaves* kWave) void gemm_norm_lines_kernel(const bf16* __restrict__ w, GemmEpilogue ep, QkvTarget qkv, NormPrologue np,
                                                                                 int ldk, int M, int N, int K) {
  norm_lines<RUNS, VPT, QKV, BUF, MANY>(w, ep, qkv, np, ldk, M, N, K);
}

template <int RUNS, int VPT, bool QKV, int BUF = norm_line_buffers(RUNS), bool MANY = false>
static int launch_norm_lines(const bf16* w, const GemmEpilogue& ep, const QkvTarget& qkv, const NormPrologue& np, int m, int n, int k,
                             hipStream_t stream, const char* who) {
  const int ldk = (k + 63) / 64 * 64 + 8;  // padded so that the rows of an operand load fall into different banks
  const int lds = norm_line_bytes(RUNS, BUF) + m * ldk * 2;
  constexpr int kMost = norm_line_bytes(RUNS, BUF) + kFusedWaves * (2048 + 8) * 2;
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_norm_lines_kernel<RUNS, VPT, QKV, BUF, MANY>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kMost);
    if (e != hipSuccess) {
      set_error(std::string(who) + ": cannot raise the LDS limit: " + hipGetErrorString(e));
      return -1;
    }
    configured = true;
  }
  gemm_norm_lines_kernel<RUNS, VPT, QKV, BUF, MANY>
      <<<(n + RUNS * 8 - 1) / (RUNS * 8), (kFusedWaves + m) * kWave, lds, stream>>>(w, ep, qkv, np, ldk, m, n, k);
  return 0;
}

// Runs of 8 rows a workgroup: the fewest that make one round of the compute units, 4 where none does.  Microseconds in a replayed
// graph, weights from memory, one token (before the norm's loads went first, and with 64 KB of LDS beyond one round), with 1, 2, 3, 4, 5, 6 and 8 runs: 9,728 x 896 (1,216 runs) -, 9.7, 7.3, 7.8, 7.0, 7.1, 7.6; 4,864 x 896 -, 5.9, 5.5, 5.6, 6.1,
// 6.4, 7.2; 2,048 x 2,048 5.9, 6.2, 6.7, 7.5, 8.2, 8.8, 10; 10,000 x 1,000 12.1, 10.4, 8.6, 9.3, 8.0, 8.5, 9.5; 14,336 x 512 11.7, 9.2, 8.2, 6.5, 9.3, 9.6, 6.5;
// 20,000 x 512 15.9, 11.3, 10.4, 9.1, 10.1, 10.1, 10.8.
static int norm_runs(int n, int multiple) {
  for (int runs : {1, 2, 3, 4, 5, 6, 8})
    if (runs % multiple == 0 && (n + runs * 8 - 1) / (runs * 8) <= 256) return runs;
  return 4;
}

template <bool QKV>
static int norm_lines_any(int runs, const bf16* w, const GemmEpilogue& ep, const QkvTarget& qkv, const NormPrologue& np, int m, int n, int k,
                          hipStream_t stream, const char* who) {
  if (n > 256 * 64) {  // more than one round: four runs
    const int iterations = ((k + 63) / 64 + kFusedWaves - 1) / kFusedWaves;
    if (k > 1024) return launch_norm_lines<4, 8, QKV, 4, true>(w, ep, qkv, np, m, n, k, stream, who);
    if (iterations == 1) return launch_norm_lines<4, 4, QKV, 1, true>(w, ep, qkv, np, m, n, k, stream, who);
    if (iterations == 2) return launch_norm_lines<4, 4, QKV, 2, true>(w, ep, qkv, np, m, n, k, stream, who);
    if (iterations == 3) return launch_norm_lines<4, 4, QKV, 3, true>(w, ep, qkv, np, m, n, k, stream, who);
    return launch_norm_lines<4, 4, QKV, 4, true>(w, ep, qkv, np, m, n, k, stream, who);
  }
#define MLR_NORM_LINES(RUNS)                                                                              \
  case RUNS:                                                                                              \
    return k <= 1024 ? launch_norm_lines<RUNS, 4, QKV>(w, ep, qkv, np, m, n, k, stream, who)              \
                     : launch_norm_lines<RUNS, 8, QKV>(w, ep, qkv, np, m, n, k, stream, who)
  switch (runs) {
    MLR_NORM_LINES(2);
    MLR_NORM_LINES(4);
    MLR_NORM_LINES(6);
    MLR_NORM_LINES(8);
    default: break;
  }
  if constexpr (!QKV) {
    switch (runs) {
      MLR_NORM_LINES(1);
      MLR_NORM_LINES(3);
      MLR_NORM_LINES(5);
      default: break;
    }
  }
#undef MLR_NORM_LINES
  set_error(std::string(who) + ": no such number of rows a workgroup");
  return -1;
}

constexpr int kFusedMaxLds = 140 * 1024;  // the device's 160 KB less the wavefronts' meeting place (up to 16 KB) and slack

template <int NT>
static int launch_fused(const bf16* w, const GemmEpilogue& ep, const MergePrologue& mp, int m, int n, int k, int slices, hipStream_t stream,
                        const char* who) {
  const int ksteps = (k / 8 + 3) / 4;
  const int per = (ksteps + slices - 1) / slices;
  const int ldk = per * 32 + 8;  // padded so that the 16 rows of an operand load fall into different banks
  const int lds = m * ldk * 2;
  if (lds > kFusedMaxLds) {
    set_error(std::string(who) + ": the activations do not fit LDS (" + std::to_string(lds) + " bytes)");
    return -1;
  }
  static int configured = 0;
  if (lds > configured) {
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_few_fused_kernel<NT>), hipFuncAttributeMaxDynamicSharedMemorySize, kFusedMaxLds);
    if (e != hipSuccess) {
      set_error(std::string(who) + ": cannot raise the LDS limit: " + hipGetErrorString(e));
      return -1;
    }
    configured = kFusedMaxLds;
  }
  const dim3 grid(static_cast<unsigned>((n + 16 * NT - 1) / (16 * NT)), static_cast<unsigned>(slices));
  gemm_few_fused_kernel<NT><<<grid, kFusedWaves * kWave, lds, stream>>>(w, ep, mp, ldk, m, n, k);
  return 0;
}

// Row blocks per workgroup: as many as still leave a workgroup for every compute unit.
static int choose_row_blocks(int n, int slices) {
  return static_cast<int64_t>((n + 31) / 32) * slices >= 256 ? 2 : 1;
}

static bool norm_arguments_ok(const void* x_in, const void* x_out, const void* delta, const void* partial,
                              int slices_in, const void* norm_weight, int m, int k, std::string& why) {
  if (!x_in || !norm_weight) why = "null pointer";
  else if (m <= 0 || m > kFusedWaves) why = "takes 1..4 tokens (a wavefront per row)";
  else if (k <= 0 || k % 8 != 0 || k > 2048) why = "k must be a multiple of 8, at most 2048";
  else if (delta != nullptr && partial != nullptr) why = "one kind of delta at a time";
  else if ((partial != nullptr) != (slices_in > 0) || slices_in < 0 || slices_in > 64) why = "partial sums and their count come together (at most 64)";
  else if ((delta != nullptr || partial != nullptr) != (x_out != nullptr)) why = "x_out is needed exactly when something is added";
  else if (x_out == x_in) why = "x_out must not be x_in (other workgroups still read it)";
  else if (reinterpret_cast<uintptr_t>(x_in) % 16 || reinterpret_cast<uintptr_t>(x_out) % 16 ||
           reinterpret_cast<uintptr_t>(delta) % 8 || reinterpret_cast<uintptr_t>(partial) % 16)
    why = "operands must be 16-byte aligned";
  return why.empty();
}

}  // namespace mlr

using namespace mlr;

extern "C" {

int mlr_gemm_norm_fused_bf16(const float* x_in, float* x_out, const void* delta, const float* partial, int slices_in,
                             const void* norm_weight, int norm_weight_is_f32, float eps, const void* w,
                             const void* bias, int bias_is_f32, void* y, int out_is_f32, int swiglu, int m, int n, int k,
                             hipStream_t stream) {
  std::string why;
  if (!norm_arguments_ok(x_in, x_out, delta, partial, slices_in, norm_weight, m, k, why)) {
    set_error("mlr_gemm_norm_fused_bf16: " + why);
    return -1;
  }
  MLR_REQUIRE(w && y && n > 0, "null pointer or empty product");
  MLR_REQUIRE(reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0, "w and y must be 16-byte aligned");
  MLR_REQUIRE(swiglu >= kEpNone && swiglu <= kEpGeluTanh, "unknown epilogue");
  MLR_REQUIRE(swiglu != kEpSwiglu || (n % 4 == 0 && bias == nullptr), "swiglu needs n % 4 == 0 and no bias");
  const GemmEpilogue ep{bias, bias_is_f32, y, out_is_f32, swiglu};
  const NormPrologue np{x_in, x_out, static_cast<const bf16*>(delta), partial, slices_in, norm_weight, norm_weight_is_f32, eps};
  const bf16* wb = static_cast<const bf16*>(w);
  const int status = norm_lines_any<false>(norm_runs(n, 1), wb, ep, QkvTarget{}, np, m, n, k, stream, __func__);
  if (status != 0) return -1;
  MLR_LAUNCH_CHECK();
  return 0;
}

int mlr_qkv_norm_fused_bf16(const float* x_in, float* x_out, const void* delta, const float* partial, int slices_in,
                            const void* norm_weight, int norm_weight_is_f32, float eps, const void* w,
                            const void* bias, int bias_is_f32, const float* cos, const float* sin, const int* slots,
                            void* key_pages, void* value_pages, void* q_out, int m, int k, int heads, int kv_heads,
                            int head_dim, int block_size, int num_pages, int write, hipStream_t stream) {
  std::string why;
  if (!norm_arguments_ok(x_in, x_out, delta, partial, slices_in, norm_weight, m, k, why)) {
    set_error("mlr_qkv_norm_fused_bf16: " + why);
    return -1;
  }
  MLR_REQUIRE(w && q_out, "null pointer");
  MLR_REQUIRE(heads > 0 && kv_heads > 0 && head_dim >= 16 && head_dim % 16 == 0, "head_dim must be a multiple of 16");
  MLR_REQUIRE((cos == nullptr) == (sin == nullptr), "cos and sin come together");
  MLR_REQUIRE(!write || (slots && key_pages && value_pages && block_size > 0 && num_pages > 0),
              "a cache write needs slots, pages and their sizes");
  MLR_REQUIRE(reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(q_out) % 8 == 0 &&
                  reinterpret_cast<uintptr_t>(key_pages) % 8 == 0 && reinterpret_cast<uintptr_t>(cos) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(sin) % 16 == 0,
              "operands must be 16-byte aligned");
  const int64_t n = static_cast<int64_t>(heads + 2 * kv_heads) * head_dim;
  MLR_REQUIRE(n * k * 2 < (1ll << 32) && n / 16 < (1ll << 31), "the weight matrix is too large");
  const GemmEpilogue ep{bias, bias_is_f32, nullptr, 0, 0};
  const QkvTarget target{cos, sin, write ? slots : nullptr, static_cast<bf16*>(key_pages), static_cast<bf16*>(value_pages),
                         static_cast<bf16*>(q_out), heads, kv_heads, head_dim, block_size, num_pages};
  const NormPrologue np{x_in, x_out, static_cast<const bf16*>(delta), partial, slices_in, norm_weight, norm_weight_is_f32, eps};
  const bf16* wb = static_cast<const bf16*>(w);
  const int status = norm_lines_any<true>(norm_runs(static_cast<int>(n), 2), wb, ep, target, np, m, static_cast<int>(n), k, stream, __func__);
  if (status != 0) return -1;
  MLR_LAUNCH_CHECK();
  return 0;
}

int mlr_gemm_merge_fused_bf16(const float* attn_partial, const int* context_lens, int heads, int head_dim, int window,
                              int part, int splits, const void* w, const void* bias, int bias_is_f32, void* y,
                              int out_is_f32, int slices, int m, int n, hipStream_t stream) {
  MLR_REQUIRE(attn_partial && context_lens && w && y, "null pointer");
  MLR_REQUIRE(m > 0 && m <= 16, "takes 1..16 tokens (one per entry)");
  MLR_REQUIRE(slices >= 1 && static_cast<int64_t>(m) * ((((heads * head_dim / 8 + 3) / 4 + slices - 1) / slices) * 4) <= kFusedWaves * kWave,
              "a workgroup merges at most 256 chunks of 8 columns: more K slices or fewer tokens");
  MLR_REQUIRE(heads > 0 && head_dim > 0 && head_dim % 8 == 0 && head_dim <= 256, "head_dim must be a multiple of 8, at most 256");
  MLR_REQUIRE(splits >= 1 && splits <= 64, "takes 1..64 partitions");
  MLR_REQUIRE(part > 0 && window >= 0, "bad partition size or window");
  MLR_REQUIRE(n > 0 && slices >= 1 && slices <= 64, "bad sizes");
  MLR_REQUIRE(slices == 1 || out_is_f32, "partial sums are float32");
  MLR_REQUIRE(reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0, "w and y must be 16-byte aligned");
  const int k = heads * head_dim;
  const GemmEpilogue ep{bias, bias_is_f32, y, out_is_f32, 0};
  const int64_t partial_bytes = static_cast<int64_t>(m) * heads * splits * (head_dim + 2) * 4;
  MLR_REQUIRE(partial_bytes < (1ll << 31), "the partitions are too large for 32-bit offsets");
  const MergePrologue mp{attn_partial, context_lens, heads, head_dim, window, part, splits, static_cast<unsigned>(partial_bytes)};
  const bf16* wb = static_cast<const bf16*>(w);
  const int nt = choose_row_blocks(n, slices);
  int status;
  if (nt == 2) status = launch_fused<2>(wb, ep, mp, m, n, k, slices, stream, __func__);
  else status = launch_fused<1>(wb, ep, mp, m, n, k, slices, stream, __func__);
  if (status != 0) return -1;
  MLR_LAUNCH_CHECK();
  return 0;
}

}  // extern "C"
