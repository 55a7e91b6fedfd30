// bfloat16 matrix products on the matrix cores: y[M, N] = x[M, K] * w[N, K]^T (+ bias).
//
// Both operands have k as their fastest index, which is what MFMA wants of both
// inputs, so tiles go from memory to the operand registers without a transpose.
// The weight tile is the A operand and the activation tile the B operand: the
// accumulator then holds four consecutive output features of one token per lane,
// which gives 8-byte stores and lets an epilogue see neighbouring features.
//
// Kernels:
//  * gemm_lines: up to 16 tokens (decode at small batch).  Bound by streaming w once, and a single compute
//    unit can only keep a few dozen cache lines in flight, so the stream has to be spread over all of
//    them: a workgroup owns 16 to 64 output features and one slice of K (grid.y slices), and its
//    wavefronts bring whole lines of the weight rows straight into LDS, each for itself.
//  * gemm_skinny_split: the fused query/key/value product of 17 to 64 tokens, and small matrices at as
//    many: 16 output features and a slice of K a workgroup, its wavefronts split the slice between them
//    (interleaved), keep eight 16-byte loads in flight per lane, and add their partial sums through LDS.
//  * gemm_tiled: everything else.  An output tile per workgroup (256 x 256 with
//    sixteen wavefronts for large products, 128 x 128 or 64 x 64 with four, whichever
//    is the largest that still keeps the compute units busy), K in
//    slices of 64 staged through double-buffered LDS by range-checked
//    buffer loads (edge tiles and the tail of K read zeros, no branches),
//    32x32x16 MFMA.  Beyond 64 tokens the larger tilings run gemm_direct (16x16x32 MFMA, as the kernels below): tiles
//    loaded straight into LDS (no registers, no LDS stores; rows swizzled instead of padded),
//    with a step's barrier ahead of its last quarter of products; and the 256 x 256 tile gemm_phased, whose
//    two groups of wavefronts read and multiply in turn.  Workgroups are placed so that those resident on
//    one XCD share operands in its L2.  Up to 16 tokens take this kernel too once
//    its tiles fill the compute units (it streams a wide weight fastest).
//    With more than one K slice both kernels write float32 partial sums
//    [slice, M, N]; the consumer (the residual-adding norm kernel) sums them in a
//    fixed order, so results do not depend on which slice finishes first.
//  * They also run the query/key/value product with bias, rotation and the cache write as
//    their epilogue (QkvTarget): the streaming kernels for up to 64 tokens (in slabs of 16 beyond 16),
//    the tiled one beyond, and the 128 x 128 tiles (staged_qkv_kernel).
// K must be a multiple of 8 (16-byte rows); other shapes take the FMA kernel.
//
// SwiGLU epilogue: with gate and up rows interleaved in pairs
// (g0 g1 u0 u1 g2 g3 u2 u3 ...) a lane holds two gate sums and their two up sums
// and stores silu(gate) * up (src/mini_llm_runtime/qwen_model_runner.py:215-216)
// directly, which saves a kernel and a round trip of the widest activation.
#include "api.h"
#include "common.h"
#include "mfma.h"
#include "gemm_epilogue.h"

namespace mlr {

// ---- skinny, wavefronts split K ------------------------------------------
// MT: slabs of 16 tokens a workgroup multiplies its weight rows with.
template <int WAVES, bool QKV, int MT>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_split_kernel(const bf16* __restrict__ x,
                                                                       const bf16* __restrict__ w,
                                                                       GemmEpilogue ep, QkvTarget qkv, int M, int N,
                                                                       int K) {
  constexpr int U = MT > 2 ? 4 : 8;  // k-steps in flight per wavefront
  __shared__ float red[WAVES][MT][kWave][4];
  __shared__ float scales[MT * 16];
  RowScaleLoads<MT * 16 / WAVES, 4 / MT> owed;  // up to 256 partial sums a row for 16 tokens, 64 for 64 tokens
  const int token0 = blockIdx.z * (MT * 16);  // grid.z: further groups of MT slabs, a workgroup each
  if (ep.row_sumsq != nullptr) row_scales_issue(ep, owed, token0, min(M - token0, MT * 16), M);
  const int lane = threadIdx.x % kWave;
  const int wave = threadIdx.x / kWave;
  const int r = lane % 16;
  const int q = lane / 16;
  const int n0 = blockIdx.x * 16;
  const int slices = gridDim.y;
  const int chunks = K / 8;             // 16-byte chunks per row
  const int ksteps = (chunks + 3) / 4;  // one MFMA consumes 4 chunks (32 elements of k)
  const int per = (ksteps + slices - 1) / slices;
  const int sb = blockIdx.y * per;
  const int se = min(ksteps, sb + per);
  // the weight row behind accumulator row `slot` of this workgroup
  int head = 0, block_in_head = 0;
  bool rotated = false;
  if constexpr (QKV) {
    const int per_head = qkv.head_dim / 16;
    head = blockIdx.x / per_head;
    block_in_head = blockIdx.x - head * per_head;
    rotated = qkv.cos != nullptr && head < qkv.heads + qkv.kv_heads;
  }
  auto row_of = [&](int slot) {
    if (!rotated) return n0 + slot;
    return head * qkv.head_dim + block_in_head * 8 + (slot < 8 ? slot : qkv.head_dim / 2 + slot - 8);
  };
  const bf16x8_t* wp = reinterpret_cast<const bf16x8_t*>(w + static_cast<int64_t>(min(row_of(r), N - 1)) * K);
  const bf16x8_t* xp[MT];
  bool xok[MT];
  f32x4_t acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    xp[mt] = reinterpret_cast<const bf16x8_t*>(x + static_cast<int64_t>(min(token0 + mt * 16 + r, M - 1)) * K);
    xok[mt] = token0 + mt * 16 + r < M;
    acc[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  for (int s0 = sb + wave; s0 < se; s0 += WAVES * U) {
    bf16x8_t a[U], b[U][MT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u * WAVES;
      const int c = s * 4 + q;
      a[u] = (s < se && c < chunks) ? __builtin_nontemporal_load(wp + c) : zero_bf16x8();
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u * WAVES;
      const int c = s * 4 + q;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) b[u][mt] = (xok[mt] && s < se && c < chunks) ? xp[mt][c] : zero_bf16x8();
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma_16x16x32(a[u], b[u][mt], acc[mt]);
  }

#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][mt][lane][i] = acc[mt][i];
  if (ep.row_sumsq != nullptr) row_scales_finish(ep, owed, token0, min(M - token0, MT * 16), M, K, scales);
  __syncthreads();
  // Slab mt is finished by wavefront mt % WAVES: the epilogue of a slab waits for memory more than once
  // (rotation tables, cache slots, the stores), and one wavefront doing four slabs in turn was a third
  // of the kernel's time at 64 tokens.
  if (wave >= MT) return;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    if (mt % WAVES != wave) continue;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    for (int ww = 0; ww < WAVES; ++ww)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += red[ww][mt][lane][i];
    const int token = token0 + mt * 16 + r;
    if (ep.row_sumsq != nullptr && token < M) {
      const float scale = scales[mt * 16 + r];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] *= scale;
    }
    if constexpr (!QKV) {
      finish4(ep, blockIdx.y, slices, token, n0 + q * 4, M, N, v);
    } else {
      // the lane holds accumulator rows 4q..4q+3 of its token: four consecutive dims of one head
      qkv_finish(ep, qkv, head, block_in_head, rotated, row_of(q * 4) - head * qkv.head_dim, q, min(token, M - 1),
                 token < M, v);
    }
  }
}

// ---- up to 16 tokens, whole lines through LDS ------------------------------------------------------------
// A workgroup owns 16 NB features and a slice of k; its four wavefronts take steps of 64 k in turn, each through LDS buffers of its own, so
// nothing is waited for but a wavefront's own loads: eight rows' whole lines of 128 bytes an instruction, three or four steps on
// their way.  At the end the wavefronts' sums meet in LDS.  Bound by what a compute unit takes in: reading 64 bytes of 16 rows an
// instruction into registers, as gemm_skinny_split does, it was half of this, and every 16 features read the tokens again.
// Against gemm_skinny_split, 8 tokens in a replayed graph, weights from memory: 0.5B gate-up (9,728 x 896) 8.1 to 6.7 us, down (896 x 4,864)
// 5.3 in 8 slices to 4.3 in 4, 1.5B down 10.8 to 8.3, 2,048 x 2,048 5.1 to 4.3, 896 x 896 3.2 to 3.3.
constexpr int line_buffers(int nb) { return nb % 2 == 0 ? 3 : 4; }
constexpr int line_lds_bytes(int nb) { return 4 * line_buffers(nb) * (nb * 16 + 16) * 128; }  // 64, 72, 128 and 120 KB

template <int NB, bool QKV>
__global__ __launch_bounds__(256) void gemm_lines_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, GemmEpilogue ep,
                                                        QkvTarget qkv, int M, int N, int K) {
  constexpr int BUF = line_buffers(NB);
  constexpr int kRowsInSlice = NB * 16 + 16;  // weights, then tokens
  constexpr int kSlice = kRowsInSlice * 128;
  constexpr int kLoads = kRowsInSlice / 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float scales[16];
  RowScaleLoads<4, 4> owed;
  if (ep.row_sumsq != nullptr) row_scales_issue(ep, owed, 0, M, M);
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r = lane % 16, q = lane / 16;
  const int n0 = blockIdx.x * (NB * 16);
  const int slices = gridDim.y;
  const int chunks = K / 8;
  const int k_slices = (K + 63) / 64;
  const int per = (k_slices + slices - 1) / slices;
  const int sb = blockIdx.y * per, se = min(k_slices, sb + per);
  // The weight row behind row 8 * half of block `block` of 16.  Query/key/value: a block of a rotated head is 8 of its dims and the 8
  // they are rotated with.
  auto run_row = [&](int block, int half) {
    const int at = blockIdx.x * NB + block;
    int first = at * 16 + half * 8;
    if (QKV) {
      const int per_head = qkv.head_dim / 16, head = at / per_head;
      if (qkv.cos != nullptr && head < qkv.heads + qkv.kv_heads)
        first = head * qkv.head_dim + (at - head * per_head) * 8 + half * (qkv.head_dim / 2);
    }
    return first;
  };
  __amdgpu_buffer_rsrc_t w_buf[8];  // rows in one piece, or 8 at a time
  if constexpr (QKV) {
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      if (p >= 2 * NB) break;
      const bool there = n0 + p / 2 * 16 < N;  // N is a multiple of 16
      w_buf[p] = make_buffer(w + (there ? static_cast<int64_t>(run_row(p / 2, p % 2)) * K : 0), there ? 16u * K : 0u);
    }
  } else {
    w_buf[0] = make_buffer(w + static_cast<int64_t>(n0) * K, static_cast<unsigned>(min(NB * 16, N - n0)) * K * 2u);
  }
  const __amdgpu_buffer_rsrc_t x_buf = make_buffer(x, static_cast<unsigned>(M) * K * 2u);
  const int piece0 = lane % 8, row = lane / 8;  // load p brings rows 8 p .. + 8; pieces in the order piece ^ (row / 2) % 8
  auto fetch = [&](int it) {
    const int s = sb + it * 4 + wave;
#pragma unroll
    for (int p = 0; p < 10; ++p) {
      if (p >= kLoads) break;
      const bool weights = p < NB * 2;
      const int piece = piece0 ^ ((4 * (p % 2) + row / 2) % 8);
      const unsigned at = static_cast<unsigned>((weights ? (QKV ? 0 : 8 * p) : 8 * (p - NB * 2)) + row) * K * 2u + s * 128u + piece * 16u;
      const unsigned from = s < se && s * 8 + piece < chunks ? at : kOutOfBuffer;
      auto* const to = (__attribute__((address_space(3))) void*)(smem + (wave * BUF + it % BUF) * kSlice + p * 1024);
      if (weights)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(w_buf[QKV ? p % 8 : 0], to, 16, from, 0, 0, 2);  // non-temporal: read once a step
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(x_buf, to, 16, from, 0, 0, 0);
    }
  };
  f32x4_t acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < BUF; ++i) fetch(i);
  const int iterations = (per + 3) / 4;
  const int swz = (r / 2) % 8;
  for (int it = 0; it < iterations; ++it) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((BUF - 1) * kLoads) : "memory");  // the oldest slice has landed; only this wavefront reads it
    const unsigned char* const base = smem + (wave * BUF + it % BUF) * kSlice;
    bf16x8_t a[2][NB], b[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int at = ((kk * 4 + q) ^ swz) * 16;
#pragma unroll
      for (int i = 0; i < NB; ++i) a[kk][i] = load_bf16x8(base + (i * 16 + r) * 128 + at);
      b[kk] = load_bf16x8(base + (NB * 16 + r) * 128 + at);
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
  if (ep.row_sumsq != nullptr) row_scales_finish(ep, owed, 0, M, M, K, scales);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NB; ++i) *reinterpret_cast<f32x4_t*>(smem + ((wave * NB + i) * kWave + lane) * 16) = acc[i];
  __syncthreads();
  if (wave >= NB) return;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ww = 0; ww < 4; ++ww) {
    const f32x4_t part = *reinterpret_cast<const f32x4_t*>(smem + ((ww * NB + wave) * kWave + lane) * 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += part[i];
  }
  if (ep.row_sumsq != nullptr && r < M) {
    const float scale = scales[r];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= scale;
  }
  if constexpr (QKV) {
    if (n0 + wave * 16 >= N) return;
    const int per_head = qkv.head_dim / 16, block = blockIdx.x * NB + wave, head = block / per_head;
    const bool rotated = qkv.cos != nullptr && head < qkv.heads + qkv.kv_heads;
    // the lane holds rows 4q .. 4q + 3 of the block: four consecutive dims of one head
    qkv_finish(ep, qkv, head, block - head * per_head, rotated, run_row(wave, q / 2) + q % 2 * 4 - head * qkv.head_dim, q, min(r, M - 1), r < M, v);
  } else {
    finish4(ep, blockIdx.y, slices, r, n0 + wave * 16 + q * 4, M, N, v);
  }
}
template <int NB, bool QKV = false>
static int launch_lines(const bf16* xb, const bf16* wb, const GemmEpilogue& ep, int m, int n, int k, int slices, hipStream_t stream,
                        const QkvTarget& qkv = QkvTarget{}) {
  constexpr int kLds = line_lds_bytes(NB);
  static bool configured = false;
  if (m > 16) {
    set_error("mlr_gemm_bf16: kernels 71 to 74 take up to 16 tokens");
    return -1;
  }
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_lines_kernel<NB, QKV>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e != hipSuccess) {
      set_error(std::string("mlr_gemm_bf16: cannot raise the LDS limit: ") + hipGetErrorString(e));
      return -1;
    }
    configured = true;
  }
  gemm_lines_kernel<NB, QKV><<<dim3((n + NB * 16 - 1) / (NB * 16), slices), 256, kLds, stream>>>(xb, wb, ep, qkv, m, n, k);
  return 0;
}

// ---- skinny fused query/key/value product, up to 8 tokens: 8 weight rows a workgroup ----------
// The 16 x 16 matrix-core block is filled with two halves of K instead of 16 weight rows: lane
// rows 0..7 multiply the 8 weight rows with the tokens over the first half of K, rows 8..15 the
// same weight rows over the second half; tokens 0..7 stand in columns 0..7 and again in 8..15.
// The two diagonal quadrants of the result are the two partial sums, the others are not used.
// Every lane still streams weights, and there are twice as many workgroups as with 16 rows each,
// which counts where those leave compute units without work or give a few of them two.
template <int WAVES>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_qkv8_kernel(const bf16* __restrict__ x,
                                                                      const bf16* __restrict__ w, GemmEpilogue ep,
                                                                      QkvTarget qkv, int M, int N, int K) {
  constexpr int U = 8;  // k-steps in flight per wavefront
  __shared__ float red[WAVES][kWave][4];
  __shared__ float scales[8];
  RowScaleLoads<8 / WAVES, 4> owed;
  if (ep.row_sumsq != nullptr) row_scales_issue(ep, owed, 0, min(M, 8), M);
  const int lane = threadIdx.x % kWave;
  const int wave = threadIdx.x / kWave;
  const int r = lane % 16;
  const int q = lane / 16;
  const int r8 = r % 8;
  const int n0 = blockIdx.x * 8;
  const int chunks = K / 8;
  const int ksteps = (chunks + 3) / 4;
  const int half_steps = (ksteps + 1) / 2;
  const int shift = (r / 8) * half_steps;  // the k-step this lane's half of K starts at
  const int per_head = qkv.head_dim / 8;
  const int head = blockIdx.x / per_head;
  const int block_in_head = blockIdx.x - head * per_head;
  const bool rotated = qkv.cos != nullptr && head < qkv.heads + qkv.kv_heads;
  // the weight row behind slot 0..7: four low halves of rotation pairs, then their high halves
  auto row_of = [&](int slot) {
    if (!rotated) return n0 + slot;
    return head * qkv.head_dim + block_in_head * 4 + (slot < 4 ? slot : qkv.head_dim / 2 + slot - 4);
  };
  const bf16x8_t* wp = reinterpret_cast<const bf16x8_t*>(w + static_cast<int64_t>(min(row_of(r8), N - 1)) * K);
  const bf16x8_t* xp = reinterpret_cast<const bf16x8_t*>(x + static_cast<int64_t>(min(r8, M - 1)) * K);
  const bool xok = r8 < M;
  f32x4_t acc{0.f, 0.f, 0.f, 0.f};

  for (int s0 = wave; s0 < half_steps; s0 += WAVES * U) {
    bf16x8_t a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u * WAVES;
      const int c = (s + shift) * 4 + q;
      a[u] = (s < half_steps && s + shift < ksteps && c < chunks) ? __builtin_nontemporal_load(wp + c) : zero_bf16x8();
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u * WAVES;
      const int c = (s + shift) * 4 + q;
      b[u] = (xok && s < half_steps && s + shift < ksteps && c < chunks) ? xp[c] : zero_bf16x8();
    }
#pragma unroll
    for (int u = 0; u < U; ++u) acc = mfma_16x16x32(a[u], b[u], acc);
  }

#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][lane][i] = acc[i];
  if (ep.row_sumsq != nullptr) row_scales_finish(ep, owed, 0, min(M, 8), M, K, scales);
  __syncthreads();
  if (wave != 0) return;
  // lane (r < 8, q < 2) owns weight slots 4q..4q+3 of token r: its own quadrant over the first
  // half of K plus the quadrant of lane (r + 8, q + 2) over the second half
  const bool owner = r < 8 && q < 2;
  const int other = owner ? lane + 8 + 32 : lane;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  for (int ww = 0; ww < WAVES; ++ww)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += red[ww][lane][i] + red[ww][other][i];
  if (ep.row_sumsq != nullptr && r8 < M) {
    const float scale = scales[r8];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= scale;
  }
  const int qq = q & 1;
  qkv_finish_pairs(ep, qkv, head, rotated, row_of(qq * 4) - head * qkv.head_dim, block_in_head * 4, qq == 0, 16,
                   min(r8, M - 1), owner && r8 < M, v);
}

// ---- tiled: more than 16 tokens, and wide products of fewer ---------------------------------
// Four wavefronts in a 2 x 2 arrangement; each owns WM x WN blocks of 32 x 32 (tokens x
// features), so the workgroup tile is (64 WM) tokens x (64 WN) features.  K in slices of 64
// through double-buffered LDS (one barrier per slice).  grid.z cuts K into slices whose
// float32 partial sums go to [slice, M, N].
constexpr int kBK = 64;       // k per LDS slice
constexpr int kLd = kBK + 8;  // padded LDS row, in elements (144 bytes)

template <int WM, int WN, int GM = 2, int GN = 2>
struct TiledShape {
  static constexpr int kThreads = 64 * GM * GN;
  static constexpr int BM = 32 * WM * GM;
  static constexpr int BN = 32 * WN * GN;
  static constexpr int kPieces = (BM + BN) * (kBK / 8) / kThreads;  // 16-byte pieces per thread and slice
  static constexpr int kLds = 2 * (BM + BN) * kLd * 2;              // bytes, two buffers
  // slices of K in flight ahead of the one in LDS: one for the large tiles, two for the small ones
  // (a slice of their work is shorter than a trip to memory; four were no faster, also for the
  // tile of few tokens, which only streams weights)
  static constexpr int kDepth = WM * WN >= 4 || GM * GN > 4 ? 1 : 2;
};

// Workgroup -> (slice, token tile, feature tile).  Consecutive workgroups go to the eight
// XCDs in turn, each with an L2 of its own: the ones that land on one XCD take a contiguous
// run of the tile order, and that order walks groups of eight token tiles feature tile by
// feature tile, so that the workgroups resident on an XCD at one time form a compact block
// of the output and share their operands in its L2.
// `light`: the last token tile holds so few tokens that only the first row of wavefronts has any
// (a prompt portion of 2,048 tokens beside 32 decoding requests: the ninth tile of 256).  Such
// tiles cost a fraction of a full one, and at the end of the order they would all land on the last
// XCD, which would then idle while the others work: they are dealt out evenly instead, behind each
// XCD's share of the full tiles.
struct TileOrder {
  int m_tiles, n_tiles, slices, light;
};
__host__ __device__ inline TileOrder make_tile_order(int m, int n_tiles, int slices, int tile_tokens, int wave_rows) {
  const int m_tiles = (m + tile_tokens - 1) / tile_tokens;
  const int last = m - (m_tiles - 1) * tile_tokens;
  return TileOrder{m_tiles, n_tiles, slices, m_tiles > 1 && last * wave_rows <= tile_tokens ? 1 : 0};
}
__device__ __forceinline__ void place_workgroup(const TileOrder& order, int id, int& slice, int& mt, int& nt) {
  constexpr int kXcds = 8, kGroup = 8;
  const int full_rows = order.m_tiles - order.light;
  const int tiles = full_rows * order.n_tiles;  // full tiles of a slice
  const int full = tiles * order.slices;
  const int total = full + order.light * order.n_tiles * order.slices;
  const int q = total / kXcds, r = total % kXcds;
  const int qf = full / kXcds, rf = full % kXcds;
  const int xcd = id % kXcds, local = id / kXcds;
  const int full_here = qf + (xcd < rf ? 1 : 0);
  if (local >= full_here) {  // one of this XCD's light tiles
    const int before = (xcd * q + min(xcd, r)) - (xcd * qf + min(xcd, rf));
    const int pos = before + local - full_here;
    slice = pos / order.n_tiles;
    nt = pos - slice * order.n_tiles;
    mt = order.m_tiles - 1;
    return;
  }
  int pos = xcd * qf + min(xcd, rf) + local;
  slice = pos / tiles;
  pos -= slice * tiles;
  const int per_group = kGroup * order.n_tiles;
  const int group = pos / per_group;
  const int first = group * kGroup;
  const int size = min(full_rows - first, kGroup);
  const int in_group = pos - group * per_group;
  mt = first + in_group % size;
  nt = in_group / size;
}

// QKV: the fused query/key/value product (see QkvTarget).  The 32-feature blocks of a tile of
// the rotated part (query and key heads) come in pairs: an even block holds 32 dims j of the
// first half of their heads, the odd block after it their partners j + head_dim/2; tiles of the
// value heads (and all tiles, without rotation) hold consecutive rows.
template <int WM, int WN, int DEPTH, int GM = 2, int GN = 2, bool QKV = false, bool ONCE = false>
__global__ __launch_bounds__(64 * GM * GN) void gemm_tiled_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                                  GemmEpilogue ep, QkvTarget qkv, TileOrder order, int M,
                                                                  int N, int K) {
  using Shape = TiledShape<WM, WN, GM, GN>;
  constexpr int BM = Shape::BM, BN = Shape::BN, PIECES = Shape::kPieces, THREADS = Shape::kThreads;
  // Two LDS buffers, each BN rows of w and then BM rows of x.  Addressed as offsets from
  // the one shared array so that every access stays an LDS instruction.
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16* const lds = reinterpret_cast<bf16*>(smem);
  constexpr int kBuffer = (BM + BN) * kLd;
  __shared__ float scales[BM];  // of the tile's token rows, when their normalisation is still owed

  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = tid / kWave;
  const int wn = wave % GN;
  const int wm = wave / GN;
  const int r32 = lane % 32;
  const int h = lane / 32;
  int slice, mt, nt;
  place_workgroup(order, blockIdx.x, slice, mt, nt);
  const int n0 = nt * BN;
  const int m0 = mt * BM;
  // (tiles of up to 64 tokens hold their rows' partial sums in registers over the loop; larger
  // tiles never see such rows in practice and fetch them the slow way)
  RowScaleLoads<(BM <= 64 ? BM / (GM * GN) : 1), (BM <= 64 ? 2 : 1)> owed;
  if (ep.row_sumsq != nullptr) row_scales_issue(ep, owed, m0, BM, M);
  const int chunks = K / 8;
  const int slices = order.slices;
  const int k_slices = (K + kBK - 1) / kBK;
  const int per = (k_slices + slices - 1) / slices;
  const int s_begin = slice * per;
  const int s_end = min(k_slices, s_begin + per);

  // which weight row stands behind feature slot `slot` of this tile (-1: none)
  bool rotated = false;
  int pair_base = 0, row_base = n0, rot_pairs = 0;
  if constexpr (QKV) {
    rot_pairs = qkv.cos != nullptr ? (qkv.heads + qkv.kv_heads) * (qkv.head_dim / 2) : 0;
    const int rot_tiles = (rot_pairs + BN / 2 - 1) / (BN / 2);
    rotated = nt < rot_tiles;
    pair_base = nt * (BN / 2);
    row_base = 2 * rot_pairs + (nt - rot_tiles) * BN;
  }
  auto row_of = [&](int slot) {
    if constexpr (QKV) {
      if (rotated) {
        const int block = slot / 32;
        const int pair = pair_base + (block / 2) * 32 + slot % 32;
        if (pair >= rot_pairs) return -1;
        const int half = qkv.head_dim / 2;
        const int head = pair / half;
        return head * qkv.head_dim + (pair - head * half) + ((block & 1) ? half : 0);
      }
    }
    return row_base + slot < N ? row_base + slot : -1;
  };

  // global -> register staging through two buffer resources: rows past the end of the
  // matrix, and the tail of K, read as zeros.  The weight resource covers this tile's rows
  // (QKV: the whole matrix, since a tile's rows lie apart).
  const int w_rows = min(BN, N - n0), x_rows = min(BM, M - m0);
  const __amdgpu_buffer_rsrc_t w_buf =
      QKV ? make_buffer(w, static_cast<unsigned>(N) * K * 2u)
          : make_buffer(w + static_cast<int64_t>(n0) * K, static_cast<unsigned>(w_rows) * K * 2u);
  const __amdgpu_buffer_rsrc_t x_buf = make_buffer(x + static_cast<int64_t>(m0) * K, static_cast<unsigned>(x_rows) * K * 2u);
  unsigned piece_off[PIECES];  // byte offset of the piece in slice 0
  int lds_off[PIECES];
  int piece_chunk[PIECES];
#pragma unroll
  for (int it = 0; it < PIECES; ++it) {
    const int idx = tid + it * THREADS;
    const int row = idx / (kBK / 8);
    const int ch = idx % (kBK / 8);
    piece_off[it] = static_cast<unsigned>(row < BN ? row : row - BN) * K * 2u + ch * 16u;
    if constexpr (QKV) {
      if (row < BN) {
        const int weight_row = row_of(row);
        piece_off[it] = weight_row >= 0 ? static_cast<unsigned>(weight_row) * K * 2u + ch * 16u : kOutOfBuffer;
      }
    }
    lds_off[it] = row * kLd + ch * 8;
    piece_chunk[it] = ch;
  }

  f32x16_t acc[WN][WM];
#pragma unroll
  for (int i = 0; i < WN; ++i)
#pragma unroll
    for (int j = 0; j < WM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // The LDS buffers run one slice ahead of the matrix cores, and DEPTH register sets hold the
  // slices behind it on their way from memory (with a small tile one slice of work is shorter
  // than a trip to memory).  A slice past the end reads zeros through the range check, so the
  // loop bodies need no conditions on it.
  bf16x8_t regs[DEPTH][PIECES];
  auto fetch = [&](int slice, auto& reg) {
    const int left = slice < s_end ? chunks - slice * (kBK / 8) : 0;  // chunks of K from this slice on
#pragma unroll
    for (int it = 0; it < PIECES; ++it) {
      const unsigned off = piece_chunk[it] < left ? piece_off[it] + slice * (kBK * 2u) : kOutOfBuffer;
      // ONCE: one tile of tokens, so every weight byte is read once and need not stay in a cache
      // (the tokens are read by every workgroup and do stay)
      if (ONCE && it * THREADS / (kBK / 8) < BN)
        reg[it] = buffer_load_bf16x8_once(w_buf, off);
      else
        reg[it] = buffer_load_bf16x8(it * THREADS / (kBK / 8) < BN ? w_buf : x_buf, off);
    }
    // the loads are issued here, ahead of the products: the instruction scheduler would
    // otherwise move them down next to the LDS stores that consume them
    __builtin_amdgcn_sched_barrier(0);
  };
  auto stash = [&](int buf, const auto& reg) {
#pragma unroll
    for (int it = 0; it < PIECES; ++it) *reinterpret_cast<bf16x8_t*>(lds + buf * kBuffer + lds_off[it]) = reg[it];
  };
  // A tile at the lower edge of the matrix may have tokens for its first rows of wavefronts only:
  // the others skip the products and only help to stage the operands.
  const bool idle = __builtin_amdgcn_readfirstlane(static_cast<int>(wm * 32 * WM >= x_rows)) != 0;
  auto multiply = [&](int buf) {
    if (idle) return;
    const bf16* wt = lds + buf * kBuffer + (wn * 32 * WN + r32) * kLd + h * 8;
    const bf16* xt = lds + buf * kBuffer + (BN + wm * 32 * WM + r32) * kLd + h * 8;
#pragma unroll
    for (int kk = 0; kk < kBK / 16; ++kk) {
      bf16x8_t a[WN], b[WM];
#pragma unroll
      for (int i = 0; i < WN; ++i) a[i] = load_bf16x8(wt + i * 32 * kLd + kk * 16);
#pragma unroll
      for (int j = 0; j < WM; ++j) b[j] = load_bf16x8(xt + j * 32 * kLd + kk * 16);
#pragma unroll
      for (int i = 0; i < WN; ++i)
#pragma unroll
        for (int j = 0; j < WM; ++j) acc[i][j] = mfma_32x32x16(a[i], b[j], acc[i][j]);
    }
  };

  // set j holds slice s + 1 + j while slice s is multiplied; the set that was stashed is loaded
  // again at once, DEPTH slices further on
#pragma unroll
  for (int j = 0; j < DEPTH; ++j) fetch(s_begin + j, regs[j]);
  stash(0, regs[0]);
  __syncthreads();
  for (int s = s_begin; s < s_end; s += DEPTH) {
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      if (s + j >= s_end) break;
      const int buf = (s + j - s_begin) & 1;
      fetch(s + j + DEPTH, regs[j]);
      multiply(buf);
      stash(buf ^ 1, regs[(j + 1) % DEPTH]);  // slice s + j + 1
      __syncthreads();
    }
  }

  if (ep.row_sumsq != nullptr) {
    row_scales_finish(ep, owed, m0, BM, M, K, scales);
    __syncthreads();
  }
  if constexpr (!QKV) {
#pragma unroll
    for (int i = 0; i < WN; ++i)
#pragma unroll
      for (int j = 0; j < WM; ++j) {
        const int m = m0 + (wm * WM + j) * 32 + r32;
        const float scale = ep.row_sumsq != nullptr ? scales[(wm * WM + j) * 32 + r32] : 1.f;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int n = n0 + (wn * WN + i) * 32 + g * 8 + h * 4;
          const float v[4] = {acc[i][j][g * 4 + 0] * scale, acc[i][j][g * 4 + 1] * scale, acc[i][j][g * 4 + 2] * scale,
                              acc[i][j][g * 4 + 3] * scale};
          finish4(ep, slice, slices, m, n, M, N, v);
        }
      }
  } else {
    // sums -> bias -> bfloat16 (as the unfused kernels hand the product on)
    int row0[WN][4];  // weight row of the lane's first feature in group g of block i
#pragma unroll
    for (int i = 0; i < WN; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        row0[i][g] = row_of((wn * WN + i) * 32 + g * 8 + h * 4);
#pragma unroll
        for (int j = 0; j < WM; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v = acc[i][j][g * 4 + e];
            if (ep.row_sumsq != nullptr) v *= scales[(wm * WM + j) * 32 + r32];
            if (ep.bias != nullptr && row0[i][g] >= 0) v += load_as_f32(ep.bias, row0[i][g] + e, ep.bias_is_f32);
            acc[i][j][g * 4 + e] = to_f32(f32_to_bf16(v));
          }
      }
    // a rotated block needs its partner block: in the same wavefront when it holds two blocks
    // side by side, else in the neighbouring wavefront, through LDS (the tiles are done with)
    float* const exchange = reinterpret_cast<float*>(smem);
    if constexpr (WN == 1) {
      if (rotated) {
        __syncthreads();  // every wavefront has read its last tile
#pragma unroll
        for (int j = 0; j < WM; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) exchange[((wave * WM + j) * 16 + e) * kWave + lane] = acc[0][j][e];
        __syncthreads();
      }
    }
#pragma unroll
    for (int i = 0; i < WN; ++i)
#pragma unroll
      for (int j = 0; j < WM; ++j) {
        const int m = m0 + (wm * WM + j) * 32 + r32;
        const int token = min(m, M - 1);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if (row0[i][g] < 0) continue;
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[i][j][g * 4 + e];
          if (rotated) {
            const int D = qkv.head_dim, half = D / 2;
            const int d = row0[i][g] % D;
            const bool low = d < half;
            const float* cs = qkv.cos + static_cast<int64_t>(token) * half + (low ? d : d - half);
            const float* sn = qkv.sin + static_cast<int64_t>(token) * half + (low ? d : d - half);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float partner;
              if constexpr (WN == 1)
                partner = exchange[(((wave ^ 1) * WM + j) * 16 + g * 4 + e) * kWave + lane];
              else
                partner = acc[i ^ 1][j][g * 4 + e];
              v[e] = low ? v[e] * cs[e] - partner * sn[e] : v[e] * cs[e] + partner * sn[e];
            }
          }
          if (m >= M) continue;
          u16x4_t packed;
#pragma unroll
          for (int e = 0; e < 4; ++e) packed[e] = f32_to_bf16(v[e]).bits;
          qkv_store4(qkv, row0[i][g], m, packed);
        }
      }
  }
}

// ---- tiled, tiles loaded straight into LDS ---------------------------------------------------------
// The tiles of gemm_tiled_kernel (wavefronts of WM x WN blocks of 32 x 32 in a GM x GN arrangement; square
// ones and, for products whose square tiles would not go round the compute units, 256 tokens x 192 or
// x 160 features) with two changes to what a step of k costs beside its products.
//  * The tiles go from memory into LDS without passing registers.  A lane's 16 bytes land at wavefront
//    base + 16 * lane, so a row of a slice (BKT * 2 bytes) has no padding; instead its 16-byte pieces
//    are stored in the order piece ^ key.  LDS serves sixteen lanes' 16 bytes a cycle from 64 banks
//    (256 bytes: two rows of a 64-wide slice), so the key is (row / 2) % 8 there: the operand reads of
//    sixteen consecutive rows fall on sixteen different places.  (With row % 8 as the key the bank
//    conflict counter showed a third of the kernel's cycles.)
//  * The one barrier of a step stands before its last quarter of products: behind it every wavefront
//    first asks for the next slice's first operands and for the slice NBUF slices on, then multiplies
//    the quarter it kept, so the matrix cores have work while those arrive.
// Measured against the register-staged kernel on one matrix streamed again and again: 7B gate-up at
// 2,048 tokens 592 to 527 us (the vendor library: 584), 7B down in two slices 262 to 247, 32B down in
// three slices 541 to 493, 0.5B gate-up 57 to 51 (the library: 53); on a model's weights, which come
// from memory, 1 to 10 %.  (The 256 x 256 tile has since moved on to gemm_phased_kernel.)  Results of whole products
// leave through LDS (stage_tile), which took 128 x 128 tiles of the 0.5B gate-up from 57 to 47 us, 256 x 320 from 48 to 41,
// 256 x 192 tiles of 2,048 x 4,608 x 3,584 from 73 to 70.  With products of 32 x 32 x 16 (see mfma.h), each quarter 16 of k of all blocks,
// 8,191 x 4,608 x 3,584 took 251 us in tiles of 192 features (238 here), 7B gate-up at 512 tokens 135 in tiles of 320 (129), products of
// up to 64 tokens the same within 2 %.  Variants that lost: two quarters kept (spills a register, no gain);
// slices of 32 in four buffers or of 64 in three (NBUF - 1 slices on their way: 5 to 25 %
// slower from 512 tokens on, up to 16 % faster at 128 to 256, where other tilings are chosen); a 64 x 64
// tile (7 to 15 % slower than the staged kernel, which has two slices on their way, at up to 512 tokens
// of weights that come from memory; equal beyond); eight wavefronts of 128 x 64 or 64 x 128 on the
// 256 x 256 tile (like sixteen of 64 x 64), four of 128 x 128 (7B gate-up 791 us against 571: one wavefront
// per SIMD has nobody to fill its waits); sixteen of 32 x 32 on the 128 x 128 tile (slower than four).

// LDS of a tile of `tokens` x `features` under `waves` wavefronts: a buffer holds the tile's 1 KB runs
// and, where they do not go round the wavefronts, one more for the surplus loads (see kPieces).
constexpr int direct_lds_bytes(int tokens, int features, int waves, int buffers) {
  const int runs = (tokens + features) * kBK * 2 / 1024;
  return buffers * (runs + (runs % waves != 0 ? 1 : 0)) * 1024;
}

// FIXED: an epilogue fixed at compile time (kEpGeglu, for the tile that has no room for a choice), or -1.
// QKV: the query/key/value product, with its epilogue (stage_qkv).
template <int WM, int WN, int GM, int GN, int NBUF = 2, bool ONCE = false, int FIXED = -1, bool QKV = false>
__global__ __launch_bounds__(64 * GM * GN) void gemm_direct_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                                  GemmEpilogue ep, QkvTarget qkv, TileOrder order, int M, int N,
                                                                  int K) {
  constexpr int BM = 32 * WM * GM, BN = 32 * WN * GN, WAVES = GM * GN;
  constexpr int kRowBytes = kBK * 2;
  constexpr int kRowPieces = kBK / 8;           // 16-byte pieces of a row
  constexpr int kRunRows = 1024 / kRowBytes;    // rows of a 1 KB run, the unit a wavefront loads
  constexpr int kBankRows = 256 / kRowBytes;    // rows that LDS serves side by side in one cycle
  constexpr int kRuns = (BM + BN) / kRunRows;   // dealt out to the wavefronts in turn
  constexpr int kWeightRuns = BN / kRunRows;    // the first of them are weight rows, the others token rows
  // Every wavefront issues kPieces loads per slice (the wait counters count instructions); where the
  // runs do not go round, the last wavefronts' surplus loads are out of range and bring zeros to one
  // spare run behind the tile, which nobody reads.
  constexpr int kPieces = (kRuns + WAVES - 1) / WAVES;
  // (loops over a wavefront's runs go to this fixed bound and break: with a bound that depends on the
  // template's parameters the host pass left the kernel uninstantiated, without a message)
  constexpr int kMostPieces = 16;               // at most this many per wavefront
  constexpr bool kSplitFeatures = WN > WM;      // the side whose operands come in two halves (see below)
  static_assert(kPieces <= kMostPieces && BN % 32 == 0 && BM % 32 == 0, "whole runs of weight rows and of token rows");
  static_assert(WAVES % 2 == 0 && NBUF >= 2, "see the swizzle key and the loop");
  constexpr int kInFlight = (NBUF - 2) * kPieces;  // loads of this wavefront that may still be out when a slice is needed
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int kBufferBytes = (kRuns + (kRuns % WAVES != 0 ? 1 : 0)) * 1024;
  __shared__ float scales[BM];

  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wn = wave % GN;
  const int wm = wave / GN;
  const int c16 = lane % 16;
  const int quad = lane / 16;
  int slice, mt, nt;
  place_workgroup(order, blockIdx.x, slice, mt, nt);
  const int n0 = nt * BN;
  const int m0 = mt * BM;
  RowScaleLoads<1, 1> owed;
  if (ep.row_sumsq != nullptr) row_scales_issue(ep, owed, m0, BM, M);
  const int chunks = K / 8;
  const int slices = order.slices;
  const int k_slices = (K + kBK - 1) / kBK;
  const int per = (k_slices + slices - 1) / slices;
  const int s_begin = slice * per;
  const int s_end = min(k_slices, s_begin + per);

  const int w_rows = min(BN, N - n0), x_rows = min(BM, M - m0);
  const __amdgpu_buffer_rsrc_t w_buf = make_buffer(w + static_cast<int64_t>(n0) * K, static_cast<unsigned>(w_rows) * K * 2u);
  const __amdgpu_buffer_rsrc_t x_buf = make_buffer(x + static_cast<int64_t>(m0) * K, static_cast<unsigned>(x_rows) * K * 2u);
  // piece p of this wavefront fills the run of rows kRunRows * (WAVES p + wave) .. of a buffer (its first
  // half: weights, its second: tokens): lane l brings row + l / kRowPieces, piece (l % kRowPieces) ^ key to
  // slot l % kRowPieces, key = (row / kBankRows) % kRowPieces (the same for every p)
  const int lane_row = lane / kRowPieces;
  const int lane_chunk = (lane % kRowPieces) ^ (((kRunRows / kBankRows) * wave + lane_row / kBankRows) % kRowPieces);
  unsigned piece_off[kMostPieces];
#pragma unroll
  for (int p = 0; p < kMostPieces; ++p) {
    const int run = WAVES * p + wave;
    const int row = kRunRows * run + lane_row;  // rows of the buffer: BN weight rows, then BM token rows
    piece_off[p] = run >= kRuns ? kOutOfBuffer : static_cast<unsigned>(row < BN ? row : row - BN) * K * 2u + lane_chunk * 16u;
  }
  auto fetch = [&](int s, int buf) {
    const int left = s < s_end ? chunks - s * kRowPieces : 0;
    const unsigned off_ok = lane_chunk < left ? 0u : kOutOfBuffer;
#pragma unroll
    for (int p = 0; p < kMostPieces; ++p) {
      if (p >= kPieces) break;
      __attribute__((address_space(3))) void* dst =
          (__attribute__((address_space(3))) void*)(smem + buf * kBufferBytes + min(WAVES * p + wave, kRuns) * 1024);
      const bool weights = (p + 1) * WAVES <= kWeightRuns || (p * WAVES < kWeightRuns && WAVES * p + wave < kWeightRuns);
      const unsigned off = (piece_off[p] + s * (kBK * 2u)) | off_ok;
      if (ONCE && weights) __builtin_amdgcn_raw_ptr_buffer_load_lds(w_buf, dst, 16, off, 0, 0, 2);  // read once: non-temporal
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(weights ? w_buf : x_buf, dst, 16, off, 0, 0, 0);
    }
  };

  f32x4_t acc[2 * WN][2 * WM];  // blocks of 16 features, of 16 tokens
#pragma unroll
  for (int i = 0; i < 2 * WN; ++i)
#pragma unroll
    for (int j = 0; j < 2 * WM; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const bool idle = __builtin_amdgcn_readfirstlane(static_cast<int>(wm * 32 * WM >= x_rows)) != 0;
  // operand rows of this lane: weight rows wn * 32 WN + i * 16 + c16, token rows BN + wm * 32 WM + j * 16 + c16; piece
  // kk * 4 + quad of a row sits in slot (kk * 4 + quad) ^ key, and the key is (c16 / kBankRows) % kRowPieces for all of them.
  // A slice's products come in quarters: 32 of k, all blocks of one side (`whole`) with half the blocks of the other (`part`), the
  // one with more of them, so that the operands of two quarters fit the registers.
  constexpr int kWhole = 2 * (kSplitFeatures ? WM : WN), kPart = kSplitFeatures ? WN : WM;
  const int swz = (c16 / kBankRows) % kRowPieces;
  const int a_base = (wn * 32 * WN + c16) * kRowBytes;
  const int b_base = (BN + wm * 32 * WM + c16) * kRowBytes;
  struct Whole {
    bf16x8_t v[kWhole];
  };
  struct Part {
    bf16x8_t v[kPart];
  };
  auto read_whole = [&](int buf, int kk) {
    Whole f;
    const unsigned char* base = smem + buf * kBufferBytes + (((kk * 4 + quad) ^ swz) * 16) + (kSplitFeatures ? b_base : a_base);
#pragma unroll
    for (int i = 0; i < kWhole; ++i) f.v[i] = load_bf16x8(base + i * 16 * kRowBytes);
    return f;
  };
  auto read_part = [&](int buf, int kk, int half) {
    Part f;
    const unsigned char* base = smem + buf * kBufferBytes + (((kk * 4 + quad) ^ swz) * 16) + (kSplitFeatures ? a_base : b_base);
#pragma unroll
    for (int i = 0; i < kPart; ++i) f.v[i] = load_bf16x8(base + (half * kPart + i) * 16 * kRowBytes);
    return f;
  };
  auto multiply = [&](const Whole& u, const Part& v, int half) {
    constexpr int kTokens = kSplitFeatures ? kWhole : kPart, kFeatures = kSplitFeatures ? kPart : kWhole;
#pragma unroll
    for (int j = 0; j < kTokens; ++j)
#pragma unroll
      for (int f = 0; f < kFeatures; ++f) {
        const int i = turn_at(f, j, kFeatures);
        f32x4_t& sum = kSplitFeatures ? acc[half * kPart + i][j] : acc[i][half * kPart + j];
        sum = kSplitFeatures ? mfma_16x16x32(v.v[i], u.v[j], sum) : mfma_16x16x32(u.v[i], v.v[j], sum);
      }
  };

  // NBUF - 1 slices are on their way or in LDS ahead of the one that is multiplied
#pragma unroll
  for (int b = 0; b < NBUF; ++b) fetch(s_begin + b, b);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NBUF - 1) * kPieces) : "memory");
  __syncthreads();
  Whole whole = read_whole(0, 0);
  Part part = read_part(0, 0, 0);
  int buf = 0;
  for (int s = s_begin; s < s_end; ++s) {
    if (!idle) {
      const Part second = read_part(buf, 0, 1);
      multiply(whole, part, 0);
      const Whole whole1 = read_whole(buf, 1);
      const Part third = read_part(buf, 1, 0);
      multiply(whole, second, 1);
      part = read_part(buf, 1, 1);
      multiply(whole1, third, 0);
      whole = whole1;
    }
    // the slice after this one has landed (this wavefront's share; the barrier answers for the others),
    // and nobody reads this slice's buffer any more
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kInFlight) : "memory");
    __syncthreads();
    fetch(s + NBUF, buf);
    const int next_buf = buf + 1 == NBUF ? 0 : buf + 1;
    if (!idle) {
      const Whole kept_whole = whole;
      const Part kept = part;
      whole = read_whole(next_buf, 0);
      part = read_part(next_buf, 0, 0);
      multiply(kept_whole, kept, 1);  // the quarter kept for behind the barrier
    }
    buf = next_buf;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be on its way into LDS when the workgroup ends

  if (ep.row_sumsq != nullptr) {
    row_scales_finish(ep, owed, m0, BM, M, K, scales);
    __syncthreads();
  }
  // finished tiles of many tokens leave through LDS where they fit it (see stage_tile)
  constexpr int kLds = NBUF * kBufferBytes;
  if constexpr (QKV) {
    static_assert(staged_tile_bytes(BM, BN) <= kLds, "the staged tile fits");
    __syncthreads();  // everybody's loads have landed and nobody reads the slices any more
    stage_qkv<64 * GM * GN, BM, BN>(ep, qkv, acc, smem, scales, wn * 32 * WN, wm * 32 * WM, m0, n0, M, N);
    return;
  }
  constexpr bool kStagesPairs = BM >= 128 && staged_tile_bytes(BM, BN / 2) <= kLds;
  constexpr bool kStagesPlain = BM >= 128 && FIXED < 0 && staged_tile_bytes(BM, BN) <= kLds;
  constexpr int kSumRows = BM >= 128 && FIXED < 0 && WM * WN < 10 ? staged_sums_rows(BM, BN, 32 * WM, kLds) : 0;
  if constexpr (kSumRows > 0) {
    if (stages_sums(ep, N)) {
      __syncthreads();  // as below
      stage_sums<64 * GM * GN, BM, BN, kSumRows>(ep, acc, smem, scales, wn * 32 * WN, wm * 32 * WM, slice, m0, n0, M, N);
      return;
    }
  }
  if constexpr (kStagesPairs) {
    if (stages_tile(ep, slices, N) && (kStagesPlain || ep.swiglu != kEpNone)) {
      __syncthreads();  // everybody's loads have landed and nobody reads the slices any more
      constexpr int kThreads = 64 * GM * GN;
      if constexpr (FIXED < 0) {
        if (ep.swiglu == kEpSwiglu) {
          stage_tile<kEpSwiglu, kThreads, BM, BN>(ep, acc, smem, scales, wn * 32 * WN, wm * 32 * WM, m0, n0, M, N);
          return;
        }
      }
      if constexpr (kStagesPlain) {
        if (ep.swiglu == kEpNone) {
          stage_tile<kEpNone, kThreads, BM, BN>(ep, acc, smem, scales, wn * 32 * WN, wm * 32 * WM, m0, n0, M, N);
          return;
        }
      }
      stage_tile<kEpGeglu, kThreads, BM, BN>(ep, acc, smem, scales, wn * 32 * WN, wm * 32 * WM, m0, n0, M, N);
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < 2 * WN; ++i)
#pragma unroll
    for (int j = 0; j < 2 * WM; ++j) {
      const int token = wm * 32 * WM + j * 16 + c16;
      const int m = m0 + token, n = n0 + wn * 32 * WN + i * 16 + quad * 4;
      const float scale = ep.row_sumsq != nullptr ? scales[token] : 1.f;
      const float v[4] = {acc[i][j][0] * scale, acc[i][j][1] * scale, acc[i][j][2] * scale, acc[i][j][3] * scale};
      if constexpr (FIXED == kEpGeglu) {
        if (m < M && n < N) store_geglu4(ep, m, n, N, v);
      } else {
        finish4<(WM * WN < 10)>(ep, slice, slices, m, n, M, N, v);  // 256 x 320: the registers are full
      }
    }
}

// ---- tiled, 256 x 256, two groups of wavefronts in turn ------------------------------------------------
// The 256 x 256 tile by eight wavefronts of 128 tokens x 64 features (three quarters of the LDS reads per product of sixteen
// wavefronts of 64 x 64), two on every SIMD.  What gemm_direct_kernel loses beside its products is that all wavefronts wait, read and
// multiply at the same time; here the two groups take turns: while one multiplies, the other reads its next operands from
// LDS and asks for tiles from memory, and a barrier between the phases keeps them apart.
//  * A step (64 of k) is four phases of 16 products of 16 x 16 x 32: the tokens' halves X0, X1 (64 of a wavefront's 128) against the features'
//    halves W0, W1 (32 of 64) in the order X0 W0, X0 W1, X1 W1, X1 W0; before each, its group reads what that phase still lacks: X0, W1,
//    X1 and, in the last, W0 of the next step (into the registers of W1, so steps alternate between two sets).
//  * The four quarters of a slice lie in LDS apart (16 KB each, two slices: 128 KB).  As soon as both groups have read a quarter, the
//    same quarter of the slice two steps on is asked for into its place: every load has five quarters' time, a step and a quarter.
//  * wait counts: a quarter is two loads of a wavefront.  A quarter is waited for at the end of the reading phase before the one that
//    reads it, when five more (four for W0 of the next step) have been asked for since; the phase's barrier then answers for all wavefronts.
// Quarter q of a buffer: rows of 64 k (128 bytes), 16-byte pieces in the order piece ^ (row / 2) % 8, as in gemm_direct_kernel.
// Measured against gemm_direct_kernel with sixteen wavefronts of 64 x 64 on the same tile, weights from memory, microseconds (TFLOP/s), each
// with its results staged (stage_tile) here and stored from the accumulators there: 7B gate-up with its gating at 2,048 tokens 581 (958)
// to 505 (1,102), at 8,191 1,942 to 1,799 (1,236), at 1,048 299 to 280; 8,191 x 3,584 x 3,584 194 to 174 (1,210); 7B down at 8,191 984 to
// 927 (1,200), at 2,048 in two slices 265 to 238.  Without the staging, whole products were level with the old kernel
// (3,584 x 3,584 at 2,048: 78 there, 88 without and 70 with it).
// Bound by power: with products of 32 x 32 x 16 (see mfma.h) the same loop took, on one card in turn, 7B gate-up at 2,048 tokens 470 us (432
// here, 1,287 TFLOP/s), at 8,191 1,785 (1,647, 1,351), 7B down at 8,191 905 (838), at 2,048 in two slices 235 (215).  What is left of
// that: the tiles' way from memory into LDS is 15 % of the time, the operands' from LDS 7 % (each left out in a copy of the kernel).
constexpr int kPhaseQuarter = 128 * 128;             // bytes
constexpr int kPhaseBuffer = 4 * kPhaseQuarter;      // W0, W1, X0, X1
constexpr int kPhaseLds = staged_tile_bytes(256, 256);  // a little more than the two slices
static_assert(kPhaseLds >= 2 * kPhaseBuffer, "the slices fit");

__global__ __launch_bounds__(512, 2) void gemm_phased_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, GemmEpilogue ep,
                                                            QkvTarget, TileOrder order, int M, int N, int K) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float scales[256];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave / 4, wn = wave % 4;  // wavefronts w and w + 4 share a SIMD: one of each group
  const int c16 = lane % 16, quad = lane / 16;
  int slice, mt, nt;
  place_workgroup(order, blockIdx.x, slice, mt, nt);
  const int n0 = nt * 256, m0 = mt * 256;
  RowScaleLoads<1, 1> owed;
  if (ep.row_sumsq != nullptr) row_scales_issue(ep, owed, m0, 256, M);
  const int chunks = K / 8;
  const int slices = order.slices;
  const int k_slices = (K + 63) / 64;
  const int per = (k_slices + slices - 1) / slices;
  const int s_begin = slice * per;
  const int steps = min(k_slices, s_begin + per) - s_begin;

  const int w_rows = min(256, N - n0), x_rows = min(256, M - m0);
  const __amdgpu_buffer_rsrc_t w_buf = make_buffer(w + static_cast<int64_t>(n0) * K, static_cast<unsigned>(w_rows) * K * 2u);
  const __amdgpu_buffer_rsrc_t x_buf = make_buffer(x + static_cast<int64_t>(m0) * K, static_cast<unsigned>(x_rows) * K * 2u);
  // A quarter is 16 runs of 8 rows; this wavefront brings runs `wave` and `wave` + 8.  Row r of Wj: feature r / 32 * 64 + j * 32 +
  // r % 32 of the tile; row r of Xi: token r / 64 * 128 + i * 64 + r % 64 (64 rows on: 128 features or tokens on).
  const int row = 8 * wave + lane / 8;
  const int piece = (lane % 8) ^ ((4 * (wave % 2) + lane / 16) % 8);
  const unsigned w_off = static_cast<unsigned>(row / 32 * 64 + row % 32) * K * 2u + piece * 16u;
  const unsigned x_off = static_cast<unsigned>(row) * K * 2u + piece * 16u;
  auto fetch = [&](int step, int quarter) {  // quarter 0, 1: W0, W1; 2, 3: X0, X1
    const int s = s_begin + step;
    const unsigned past = step < steps && piece < chunks - s * 8 ? 0u : kOutOfBuffer;
    const unsigned half = quarter < 2 ? (quarter & 1) * 32u : (quarter & 1) * 64u;
    const unsigned off = (quarter < 2 ? w_off : x_off) + half * K * 2u + s * 128u;
    unsigned char* const dst = smem + (step & 1) * kPhaseBuffer + quarter * kPhaseQuarter + wave * 1024;
#pragma unroll
    for (int p = 0; p < 2; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(quarter < 2 ? w_buf : x_buf, (__attribute__((address_space(3))) void*)(dst + p * 8192), 16,
                                               (off + p * 256u * K) | past, 0, 0, 0);
  };

  f32x4_t acc[4][8];  // blocks of 16 features (half * 2 + block) and of 16 tokens (half * 4 + block)
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const bool idle = __builtin_amdgcn_readfirstlane(static_cast<int>(wm * 128 >= x_rows)) != 0;  // no tokens: keeps time only
  const int swz = c16 / 2;
  const int w_base = (wn * 32 + c16) * 128;
  const int x_base = 2 * kPhaseQuarter + (wm * 64 + c16) * 128;
  struct Weights {
    bf16x8_t v[2][2];  // 32 of k, block of 16 features
  };
  struct Tokens {
    bf16x8_t v[2][4];
  };
  auto read_weights = [&](Weights& t, int buf, int j) {
    if (idle) return;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        t.v[kk][b] = load_bf16x8(smem + buf * kPhaseBuffer + j * kPhaseQuarter + w_base + b * 16 * 128 + (((kk * 4 + quad) ^ swz) * 16));
  };
  auto read_tokens = [&](Tokens& t, int buf, int i) {
    if (idle) return;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        t.v[kk][b] = load_bf16x8(smem + buf * kPhaseBuffer + i * kPhaseQuarter + x_base + b * 16 * 128 + (((kk * 4 + quad) ^ swz) * 16));
  };
  // the end of a reading phase: operands are in registers, the quarter read next has landed (all but `pending` loads)
#define MLR_READ_DONE(pending)                                                                   \
  do {                                                                                           \
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(pending) : "memory");                    \
    __builtin_amdgcn_sched_barrier(0);                                                           \
    __builtin_amdgcn_s_barrier();                                                                \
    __builtin_amdgcn_sched_barrier(0);                                                           \
  } while (0)
  auto multiply = [&](const Weights& a, const Tokens& b, int j, int i) {
    if (!idle) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int f = 0; f < 2; ++f) {
            f32x4_t& sum = acc[j * 2 + turn_at(f, c, 2)][i * 4 + c];
            sum = mfma_16x16x32(a.v[kk][turn_at(f, c, 2)], b.v[kk][c], sum);
          }
      __builtin_amdgcn_s_setprio(0);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  fetch(0, 2);
  fetch(0, 0);
  fetch(0, 1);
  fetch(0, 3);
  fetch(1, 2);
  fetch(1, 0);
  fetch(1, 1);
  Weights wa, wb;
  Tokens tokens;
  MLR_READ_DONE(10);  // X0 and W0 of the first step
  read_weights(wa, 0, 0);
  if (wave >= 4) __builtin_amdgcn_s_barrier();  // the second group stays one phase behind
  __builtin_amdgcn_sched_barrier(0);
  // a step: w0 holds W0 of it and, at its end, w1 W0 of the next
  auto step_of = [&](int step, Weights& w0, Weights& w1) {
    const int buf = step & 1;
    fetch(step + 1, 3);
    read_tokens(tokens, buf, 0);
    MLR_READ_DONE(10);
    multiply(w0, tokens, 0, 0);
    fetch(step + 2, 2);
    read_weights(w1, buf, 1);
    MLR_READ_DONE(10);
    multiply(w1, tokens, 1, 0);
    fetch(step + 2, 0);
    read_tokens(tokens, buf, 1);
    MLR_READ_DONE(8);
    multiply(w1, tokens, 1, 1);
    fetch(step + 2, 1);
    read_weights(w1, buf ^ 1, 0);
    MLR_READ_DONE(12);
    multiply(w0, tokens, 0, 1);
  };
  int step = 0;
  for (; step + 1 < steps; step += 2) {
    step_of(step, wa, wb);
    step_of(step + 1, wb, wa);
  }
  if (step < steps) step_of(step, wa, wb);
#undef MLR_READ_DONE
  if (wave < 4) __builtin_amdgcn_s_barrier();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be on its way into LDS when the workgroup ends

  if (ep.row_sumsq != nullptr) row_scales_finish(ep, owed, m0, 256, M, K, scales);
  __syncthreads();
  if (stages_tile(ep, slices, N)) {
    if (ep.swiglu == kEpSwiglu)
      stage_tile<kEpSwiglu, 512, 256, 256>(ep, acc, smem, scales, wn * 64, wm * 128, m0, n0, M, N);
    else if (ep.swiglu == kEpGeglu)
      stage_tile<kEpGeglu, 512, 256, 256>(ep, acc, smem, scales, wn * 64, wm * 128, m0, n0, M, N);
    else
      stage_tile<kEpNone, 512, 256, 256>(ep, acc, smem, scales, wn * 64, wm * 128, m0, n0, M, N);
    return;
  }
  if (stages_sums(ep, N)) {
    stage_sums<512, 256, 256, staged_sums_rows(256, 256, 128, kPhaseLds)>(ep, acc, smem, scales, wn * 64, wm * 128, slice, m0, n0, M, N);
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int token = wm * 128 + i * 16 + c16;
      const float scale = ep.row_sumsq != nullptr ? scales[token] : 1.f;
      const float v[4] = {acc[j][i][0] * scale, acc[j][i][1] * scale, acc[j][i][2] * scale, acc[j][i][3] * scale};
      finish4(ep, slice, slices, m0 + token, n0 + wn * 64 + j * 16 + quad * 4, M, N, v);
    }
}

// ---- tiled, 128 x 128, two groups of wavefronts that share the slices of k ---------------------------------
// Eight wavefronts, four to a group; either group multiplies the whole tile (a wavefront 64 x 64), one the even slices of 64 k
// and one the odd, and they take turns as in gemm_phased_kernel: while one multiplies a slice from registers the other reads
// its next one from LDS.  A group has two LDS buffers of its own; a slice is asked for as soon as its buffer has been
// read, an iteration (two slices of the tile) ahead.  At the end each group hands the sums of half the features to the other.
// Bound, like the larger tile, by the LDS reads beside the products (64 x 64 a wavefront: as many cycles of one as of the other).  With
// products of 32 x 32 x 16 2,000 x 2,048 x 2,048 took 24.2 us (23.2 here), 1,048 x 3,584 x 3,584 36.1 (34.5).
// Measured against gemm_direct's 128 x 128 tile (two workgroups of four wavefronts a unit where there are as many), weights from
// memory, microseconds: 2,000 x 2,048 x 2,048 (256 tiles) 27.1 to 24.8, k = 4,096 49.7 to 41.8; 1,048 x 3,584 x 3,584 38.6 to 34.7;
// 768 x 4,608 x 3,584 41 to 32; in slices 1,024 x 1,536 x 8,960 46 to 42, 160 x 5,120 x 27,648 130 to 86.  See takes_turns for where it is used.
constexpr int kTurnSlice = 256 * 128;  // bytes: 64 k of 128 features, then of 128 tokens
constexpr int kTurnLds = 4 * kTurnSlice;
static_assert(kTurnLds >= 65536 + staged_tile_bytes(128, 128), "the sums that change hands, and the staged tile behind them, fit");

template <bool QKV>
__global__ __launch_bounds__(512, 2) void gemm_turns_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, GemmEpilogue ep,
                                                           QkvTarget qkv, TileOrder order, int M, int N, int K) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float scales[128];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int group = wave / 4, w4 = wave % 4;  // wavefronts w and w + 4 share a SIMD: one of each group
  const int wr = w4 / 2, wc = w4 % 2;
  const int c16 = lane % 16, quad = lane / 16;
  int slice, mt, nt;
  place_workgroup(order, blockIdx.x, slice, mt, nt);
  const int n0 = nt * 128, m0 = mt * 128;
  RowScaleLoads<1, 1> owed;
  if (ep.row_sumsq != nullptr) row_scales_issue(ep, owed, m0, 128, M);
  const int chunks = K / 8;
  const int slices = order.slices;
  const int k_slices = (K + 63) / 64;
  const int per = (k_slices + slices - 1) / slices;
  const int s_begin = slice * per;
  const int steps = min(k_slices, s_begin + per) - s_begin;
  const int x_rows = min(128, M - m0);
  const __amdgpu_buffer_rsrc_t w_buf = make_buffer(w + static_cast<int64_t>(n0) * K, static_cast<unsigned>(min(128, N - n0)) * K * 2u);
  const __amdgpu_buffer_rsrc_t x_buf = make_buffer(x + static_cast<int64_t>(m0) * K, static_cast<unsigned>(x_rows) * K * 2u);
  // a slice is 32 runs of 8 rows, 16 of weights and 16 of tokens; this wavefront brings every fourth to its group
  const int piece = (lane % 8) ^ ((4 * (w4 % 2) + lane / 16) % 8);  // 16-byte pieces in the order piece ^ (row / 2) % 8
  const unsigned row_off = static_cast<unsigned>(8 * w4 + lane / 8) * K * 2u + piece * 16u;
  auto fetch = [&](int it) {
    const int s = s_begin + 2 * it + group;
    const unsigned past = 2 * it + group < steps && piece < chunks - s * 8 ? 0u : kOutOfBuffer;
    unsigned char* const dst = smem + (group * 2 + (it & 1)) * kTurnSlice + w4 * 1024;
#pragma unroll
    for (int p = 0; p < 8; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(p < 4 ? w_buf : x_buf, (__attribute__((address_space(3))) void*)(dst + p * 4096), 16,
                                               (row_off + (p % 4) * 64u * K + s * 128u) | past, 0, 0, 0);
  };
  f32x4_t acc[4][4];  // blocks of 16 features, of 16 tokens
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const bool idle = __builtin_amdgcn_readfirstlane(static_cast<int>(wr * 64 >= x_rows)) != 0;  // no tokens: keeps time only
  const int swz = c16 / 2;
#define MLR_TURN()                        \
  do {                                    \
    __builtin_amdgcn_sched_barrier(0);    \
    __builtin_amdgcn_s_barrier();         \
    __builtin_amdgcn_sched_barrier(0);    \
  } while (0)
  fetch(0);
  fetch(1);
  asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  MLR_TURN();
  if (group == 1) __builtin_amdgcn_s_barrier();  // the second group stays one phase behind
  __builtin_amdgcn_sched_barrier(0);
  const int iterations = (steps + 1) / 2;
  for (int it = 0; it < iterations; ++it) {
    bf16x8_t wv[2][4], xv[2][4];
    if (!idle) {
      const unsigned char* const base = smem + (group * 2 + (it & 1)) * kTurnSlice;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          wv[kk][b] = load_bf16x8(base + (wc * 64 + b * 16 + c16) * 128 + (((kk * 4 + quad) ^ swz) * 16));
          xv[kk][b] = load_bf16x8(base + (128 + wr * 64 + b * 16 + c16) * 128 + (((kk * 4 + quad) ^ swz) * 16));
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the group has read its buffer once all of it is past the barrier
    MLR_TURN();
    fetch(it + 2);
    if (!idle) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            f32x4_t& sum = acc[turn_at(i, j, 4)][j];
            sum = mfma_16x16x32(wv[kk][turn_at(i, j, 4)], xv[kk][j], sum);
          }
      __builtin_amdgcn_s_setprio(0);
    }
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");  // all but the slice just asked for: the next one has landed
    MLR_TURN();
  }
#undef MLR_TURN
  if (group == 0) __builtin_amdgcn_s_barrier();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be on its way into LDS
  if (ep.row_sumsq != nullptr) row_scales_finish(ep, owed, m0, 128, M, K, scales);
  __syncthreads();
  // group g finishes feature block g of its wavefronts
  f32x4_t sum[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      *reinterpret_cast<f32x4_t*>(smem + ((wave * 2 + i) * 4 + j) * 1024 + lane * 16) = group == 0 ? acc[2 + i][j] : acc[i][j];
      sum[i][j] = group == 0 ? acc[i][j] : acc[2 + i][j];
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) sum[i][j] += *reinterpret_cast<const f32x4_t*>(smem + (((wave ^ 4) * 2 + i) * 4 + j) * 1024 + lane * 16);
  const int feature0 = wc * 64 + group * 32, token0 = wr * 64;
  if constexpr (QKV) {
    stage_qkv<512, 128, 128>(ep, qkv, sum, smem + 65536, scales, feature0, token0, m0, n0, M, N);
    return;
  }
  if (stages_tile(ep, slices, N)) {
    if (ep.swiglu == kEpSwiglu)
      stage_tile<kEpSwiglu, 512, 128, 128>(ep, sum, smem + 65536, scales, feature0, token0, m0, n0, M, N);
    else if (ep.swiglu == kEpGeglu)
      stage_tile<kEpGeglu, 512, 128, 128>(ep, sum, smem + 65536, scales, feature0, token0, m0, n0, M, N);
    else
      stage_tile<kEpNone, 512, 128, 128>(ep, sum, smem + 65536, scales, feature0, token0, m0, n0, M, N);
    return;
  }
  if (stages_sums(ep, N)) {
    stage_sums<512, 128, 128, staged_sums_rows(128, 128, 64, kTurnLds - 65536)>(ep, sum, smem + 65536, scales, feature0, token0, slice, m0, n0, M, N);
    return;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int token = token0 + j * 16 + c16;
      const float scale = ep.row_sumsq != nullptr ? scales[token] : 1.f;
      const float v[4] = {sum[i][j][0] * scale, sum[i][j][1] * scale, sum[i][j][2] * scale, sum[i][j][3] * scale};
      finish4(ep, slice, slices, m0 + token, n0 + feature0 + i * 16 + quad * 4, M, N, v);
    }
}

using DirectKernel = void (*)(const bf16*, const bf16*, GemmEpilogue, QkvTarget, TileOrder, int, int, int);
// `wave_rows`: rows of wavefronts in the tile (a last token tile that fills only the first is light)
static int launch_direct(DirectKernel kernel, int tile_tokens, int tile_features, int threads, int wave_rows, int lds_bytes,
                         bool& configured, const bf16* xb, const bf16* wb, const GemmEpilogue& ep, int m, int n, int k,
                         int slices, hipStream_t stream, const QkvTarget& qkv = QkvTarget{}) {
  const TileOrder order = make_tile_order(m, (n + tile_features - 1) / tile_features, slices, tile_tokens, wave_rows);
  const int64_t groups = static_cast<int64_t>(order.m_tiles) * order.n_tiles * slices;
  if (groups >= (1ll << 31)) {
    set_error("mlr_gemm_bf16: too many tiles for one launch");
    return -1;
  }
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) {
      set_error(std::string("mlr_gemm_bf16: cannot raise the LDS limit: ") + hipGetErrorString(e));
      return -1;
    }
    configured = true;
  }
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(groups)), dim3(threads), lds_bytes, stream, xb, wb, ep, qkv, order, m, n, k);
  return 0;
}

// ONCE: the tokens fit one tile, so every weight byte is read once; the kernel then loads the
// weights with the non-temporal hint (measured on matrices far larger than the caches, as a
// model's layers are to each other: 7B gate-up at 8 tokens 50.7 to 45.4 us, the output head 191
// to 168 us; a 7B decode step at batch 8 3.76 to 3.53 ms).
template <int WM, int WN, int GM, int GN, bool ONCE>
static int launch_tiled_as(const bf16* xb, const bf16* wb, const GemmEpilogue& ep, const TileOrder& order, int64_t groups,
                           int m, int n, int k, hipStream_t stream) {
  using Shape = TiledShape<WM, WN, GM, GN>;
  constexpr int kDepth = Shape::kDepth;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tiled_kernel<WM, WN, kDepth, GM, GN, false, ONCE>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, Shape::kLds);
    if (e != hipSuccess) {
      set_error(std::string("mlr_gemm_bf16: cannot raise the LDS limit: ") + hipGetErrorString(e));
      return -1;
    }
    configured = true;
  }
  gemm_tiled_kernel<WM, WN, kDepth, GM, GN, false, ONCE>
      <<<dim3(static_cast<unsigned>(groups)), Shape::kThreads, Shape::kLds, stream>>>(xb, wb, ep, QkvTarget{}, order, m, n, k);
  return 0;
}

template <int WM, int WN, int GM = 2, int GN = 2>
static int launch_tiled(const bf16* xb, const bf16* wb, const GemmEpilogue& ep, int m, int n, int k, int slices,
                        hipStream_t stream) {
  using Shape = TiledShape<WM, WN, GM, GN>;
  const TileOrder order = make_tile_order(m, (n + Shape::BN - 1) / Shape::BN, slices, Shape::BM, GM);
  const int64_t groups = static_cast<int64_t>(order.m_tiles) * order.n_tiles * slices;
  if (groups >= (1ll << 31)) {
    set_error("mlr_gemm_bf16: too many tiles for one launch");
    return -1;
  }
  if (order.m_tiles == 1) return launch_tiled_as<WM, WN, GM, GN, true>(xb, wb, ep, order, groups, m, n, k, stream);
  return launch_tiled_as<WM, WN, GM, GN, false>(xb, wb, ep, order, groups, m, n, k, stream);
}

// The fused query/key/value product on the tiled kernel: tiles of the rotated part first
// (pairs of 32-dim blocks), then tiles of consecutive rows for the rest.
template <int WM, int WN, int GM = 2, int GN = 2>
static int launch_tiled_qkv(const bf16* xb, const bf16* wb, GemmEpilogue ep, const QkvTarget& qkv, int m, int n, int k,
                            hipStream_t stream) {
  using Shape = TiledShape<WM, WN, GM, GN>;
  constexpr int kDepth = Shape::kDepth;
  static_assert(WN == 1 || WN == 2, "a rotated block finds its partner beside it or in the next wavefront");
  const int rot_pairs = qkv.cos != nullptr ? (qkv.heads + qkv.kv_heads) * (qkv.head_dim / 2) : 0;
  const int rot_tiles = (rot_pairs + Shape::BN / 2 - 1) / (Shape::BN / 2);
  const int rest_tiles = (n - 2 * rot_pairs + Shape::BN - 1) / Shape::BN;
  const TileOrder order = make_tile_order(m, rot_tiles + rest_tiles, 1, Shape::BM, GM);
  const int64_t groups = static_cast<int64_t>(order.m_tiles) * order.n_tiles;
  MLR_REQUIRE(groups < (1ll << 31), "too many tiles for one launch");
  static bool prepared = false;
  if (!prepared) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tiled_kernel<WM, WN, kDepth, GM, GN, true>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, Shape::kLds);
    if (e != hipSuccess) {
      set_error(std::string("mlr_qkv_rope_write_bf16: cannot raise the LDS limit: ") + hipGetErrorString(e));
      return -1;
    }
    prepared = true;
  }
  gemm_tiled_kernel<WM, WN, kDepth, GM, GN, true>
      <<<dim3(static_cast<unsigned>(groups)), Shape::kThreads, Shape::kLds, stream>>>(xb, wb, ep, qkv, order, m, n, k);
  MLR_LAUNCH_CHECK();
  return 0;
}

// K slices for a skinny product: enough workgroups to keep every compute unit
// streaming, as long as a slice keeps a few MFMA steps.  1 unless `allowed`.
static int choose_slices(int groups, int ksteps, int allowed, int enough = 256) {
  if (allowed <= 1) return 1;
  int slices = 1;
  while (slices < allowed && groups * slices < enough && ksteps / (slices * 2) >= 8) slices *= 2;
  return slices;
}

// Tiles of a shape under the 64 x 64 tiling.
static int tiles_64(int m, int n) { return ((n + 63) / 64) * ((m + 63) / 64); }

// Up to 16 tokens: the LDS-tiled kernel once its 64-feature tiles (times slices) fill seven
// eighths of the compute units, the 16-feature streaming kernel below that.
static bool few_tokens_tiled(int n, int slices) { return ((n + 63) / 64) * slices >= 224; }

// Up to 16 tokens through gemm_lines: features a workgroup (16 x blocks) and, where the consumer adds up partial sums, slices of k.  A
// product is done when the busiest compute unit has taken in its share, the tokens' rows of every workgroup included; a unit holds two
// workgroups of 16 or 32 features or one of 48 or 64, and starts the next when one is done.  Estimates (us): 44 KB/us a unit (as for the
// few-token tiles below), 3 for the launch and the first bytes, 1 or, with nobody beside it, 2.5 for every further round, 0.1 in the norm
// kernel for every slice that it adds.  83 products of 1 to 16 tokens that ran here below 20 MB or where the tiles would not fill the units (1.5 to 49 MB of weights, those
// cut along k with the norm behind them): the choice was 0.6 % off the best on average, 14 % at worst (2,048 x 11,008 at one token, 2 slices 15.0 us,
// 4 13.2).  Over 1,283 sums of the larger ones that lines_stream sends here it is 0.9 % off on average, 69 by more than 5 %, one by 37 % and no other by more than 18 %.
struct LinesPlan {
  int blocks, slices;
  float us;
};
static LinesPlan plan_lines(int m, int n, int k, int slices) {
  LinesPlan best{0, slices, 0.f};
  // From 20 MB on, once 32 features a workgroup make two of them a unit, these: the units share what memory gives, and two small workgroups
  // leave less of a gap at their ends than one large (32,768 x 3,584 at 8 tokens 35.9 us, 37.6 with 64 features; 1.5 to 5 % over nine shapes).
  const bool many = static_cast<int64_t>(n) * k * 2 >= (20ll << 20) && static_cast<int64_t>((n + 31) / 32) * slices >= 512;
  for (int blocks = many ? 2 : 1; blocks <= (many ? 2 : 4); ++blocks) {
    const int64_t groups = static_cast<int64_t>((n + blocks * 16 - 1) / (blocks * 16)) * slices;
    const int resident = blocks <= 2 ? 2 : 1;
    const float kb = (blocks * 16 + m) * (((k + 63) / 64 + slices - 1) / slices) * 0.128f;
    const float us = 3.f + (groups + 255) / 256 * kb / 44.f + ((groups - 1) / (256 * resident)) * (resident == 2 ? 1.f : 2.5f) + 0.1f * slices;
    if (best.blocks == 0 || us < best.us) best = {blocks, slices, us};
  }
  return best;
}

// Up to 16 tokens: whether gemm_lines takes the product also where the tiles would fill the compute units.  Below 20 MB always (2,048 x 4,096
// in 8 slices at 8 tokens, 17 MB: 7.4 us in tiles, 6.5).  Beyond, sums with their norm: at 8 tokens 14,336 x 768 9.3 us in tiles, 6.6 here;
// 3,584 x 3,584 12.0 and 10.9; 2,048 x 11,008 at 12 tokens 18.1 and 13.6; 16,384 x 1,536 15.4 and 10.5; 22,016 x 2,048 21.0 and 18.4; 3,584 x
// 18,944 29.0 and 26.4; 151,936 x 2,048 123 and 102; 152,064 x 3,584 167 and 158.  The tiles keep what they do better, by regions of some 7,000
// timings of 1 to 16 tokens, in which gemm_lines' time over the tiles' is, on average:
//  * rows that lie a multiple of 8 KB apart (and not of 32 KB, where both are slow: 0.9): from 4,096 rows on 1.01 to 1.09, up to 1.28 (8,064 x 8,192;
//    at k = 4,096 from 7,168 rows on), 1.03 to 1.05 beyond 2,048 rows if it is a multiple of 16 KB; 0.74 to 0.97 else.  28,672 x 4,096 43.9 us in tiles and 51.6.
//  * rows of which three make a multiple of 64 KB and up to 640 bytes: 1.07 to 1.1 for 4,096 to 8,192 rows (6,144 x 11,008 at 8 tokens 4.3 TB/s and
//    5.0 in tiles; x 11,136 6.1 and 5.9), and up to 1 KB for 2,049 to 4,095 rows of 32 KB and more: 1.07.
//  * many rows with a short k, whose workgroups end before their loads are all on their way (32,768 x 512 9.3 us in tiles and 10.5, 65,536 x
//    1,024 24.0 and 25.6, 151,936 x 896 45.8 and 49.8).
//  * more than 8 tokens, which every workgroup reads again, of more than 16,384 rows from k = 3,584 on: 1.03.
//  * rows that do not begin on a line of 128 bytes, from 128 MB on: 1.03 to 1.09 for 14,336 to 16,384 rows, 1.03 to 1.1 for up to 32,768 at more than 8 tokens or
//    beyond k = 8,192; 0.76 to 0.98 elsewhere.
//  * more than 8 tokens of 4,097 to 4,608 rows from k = 10,240 on, which make one full round of tiles of 160 features in 8 slices: 1.01 to 1.08.
//  * rows 4 KB apart from 196,608 of them on: 1.02 to 1.08.
//  * from 200 MB on, where memory's rate is the bound, more than 8 tokens (55,296 x 5,120 at 16 tokens 84 us and 91), and more than 4 of up to 65,536
//    rows, which tiles of up to 256 features stream in one round (at 8 tokens 55,296 x 5,120 83.8 both, 37,888 x 3,584 42.8 and 42.2; at one token,
//    where they cost as much as at 8, 43.4 and 41.5).
// What this makes of 3,503 drawn products (20 MB to 1.1 GB, k of 512 to 33,000, every alignment) whose route is gemm_lines or was: 2,862 times gemm_lines, 0.90 of the
// tiles' time on average, 60 of them more than 3 % slower and 32 more than 5 %, the worst 31 % (4 tokens of 7,392 x 16,320).
static bool lines_stream(int m, int n, int k) {
  const int64_t bytes = static_cast<int64_t>(n) * k * 2;
  if (bytes < (20ll << 20)) return true;
  if ((n >= 8192 && k % 4096 == 0) || (n >= 16384 && k < 1536)) return false;
  if (k % 4096 == 0 && k % 16384 != 0 && (n >= 7168 || (n >= 4096 && k > 4096) || (n > 2048 && k % 8192 == 0))) return false;
  const int three_rows = static_cast<int>(6ll * k % 65536);
  if (three_rows > 0 && ((three_rows <= 640 && n >= 4096 && n <= 8192) || (three_rows <= 1024 && n > 2048 && n < 4096 && k >= 16384))) return false;
  if (m > 8 && ((n > 16384 && k >= 3584) || (n > 4096 && n <= 4608 && k >= 10240))) return false;
  if (k % 64 != 0 && bytes >= (128ll << 20) && n >= 14336 && n <= 32768 && (n <= 16384 || m > 8 || k > 8192)) return false;
  if (k == 2048 && n >= 3 << 16) return false;
  if (bytes < (200ll << 20)) return true;
  return k >= 2048 && (m <= 4 || (m <= 8 && n > 65536));
}

// Up to 8 tokens of the fused query/key/value product: workgroups of 8 weight rows instead of 16 while that makes one round of them; beyond,
// gemm_lines makes one with more rows each.
static bool half_rows_fill_better(int blocks16) { return 2 * blocks16 <= 256; }

// Kernel and number of K slices for more than 64 tokens, when the consumer takes up to
// `max_slices` partial sums: the pair with the smallest estimated time.  The estimate counts
// rounds of workgroups over the 256 compute units.  A workgroup of a tiling spends `fixed` us
// outside its K loop and, per 64-wide step of K, `alone` us when it has its compute unit to itself
// or `busy` us times the workgroups resident beside each other (operand fetch and matrix cores
// do not overlap within a compute unit, so co-resident workgroups queue); steps are faster, by up to the share
// `eased`, while only a part of the compute units has work (less traffic into L2, a higher clock), and by the share `empty` of
// what the last tile of tokens has no rows for (its wavefronts without tokens read and multiply nothing).
// Sums in float32, of slices of k or whole, cost their kernel `wide` us more a tile (twice the bytes, which leave in turns) and their
// consumer, a norm that streams at 5.7 TB/s, 4 bytes per slice and element instead of 2.  A consumer that takes several slices gets
// float32 from one, too: how many there are is a matter of speed and must not decide what the sums are rounded to before they are
// added to the residual stream.  Constants fitted to 5,700 measured times (weights that rotate through more memory than the caches
// hold) of the products of a layer at six model sizes (hidden 896 to 5120), 65 to 8,191 tokens, around the edges of tiles too, those
// for the residual stream with the norm behind them.  What is fitted is the choice: of 815 products the chosen pair is 0.4 % off the best
// on average and 15 % at worst, 21 are off by more than 5 %.  (Without `empty`, and with the few-token tiles only where the 64 x 64 ones
// were chosen, it was 1.1 %, 64 by more than 5 %: 7B gate-up at 257 to 384 tokens 136 to 140 us in tiles of 128 x 128, 108 to 113 in
// one round of 256 x 320; 1.5B gate-up at 65 to 128 tokens 22 to 24, 20 to 22 in tiles of 64 x 160.  Fitted to three quarters of
// the matrices, the choice for the others is 0.7 to 1.0 % off.)  The kernels behind the tilings of 128 tokens and more have since moved on to products of 16 x 16 x 32,
// by 0 to 8 %, without a new fit: timed again, over 635 products of the layers of six model sizes at 65 to 8,191 tokens, sums with their norm, the
// choice is 0.7 % off the best on average, 31 are off by more than 5 %, and 21 % the worst (0.5B gate-up at 65 tokens: tiles of 64 x 96 11.6 us, of 64 x 64 9.6).
struct GemmPlan {
  int kernel, slices;
};
struct TilingCost {
  int kernel, tile_tokens, tile_features, resident;
  float alone, busy, fixed, eased, wide, empty;
};
// The narrower tiles of 256 tokens (gemm_direct; a step of k costs 7.2 ns per feature of the tile at 256
// features, 7.6 at 192, 8.4 at 160) are there for products whose 256 x 256 tiles leave compute units
// without work or make a round for a few tiles.  Weights from memory, 2,048 tokens: 7B query/key/value
// (4,608 features: 144 tiles, or 232 of 160 features) 92 to 80 us, 32B output projection (160 or 256
// tiles) 130 to 112, 1.5B gate-up 139 to 132; 7B gate-up at 512 tokens 199 to 165.  Over the four
// products of four model sizes at 256 to 4,096 tokens the chosen pairs add up to 0.6 % more than the
// best pairs.  (256 x 224 by fourteen wavefronts was level with 256 x 256 and is not built.)
// 256 x 320 by eight wavefronts of 64 x 160 (ten wavefronts have too few registers each) needs 0.7
// operand reads per product where the square tile needs 1, and makes one round where the others make
// two: 0.5B gate-up (248 tiles) 53 to 49 us, 7B gate-up at 512 tokens 168 to 135, 7B query/key/value at
// 4,096 tokens 159 to 134, 32B down at 4,096 tokens 1,084 to 938; level or behind where the square
// tiles already go round (7B gate-up at 2,048 tokens 533 against 517 on weights from memory).
constexpr TilingCost kTilingCosts[] = {{11, 64, 64, 8, 0.277f, 0.243f, 6.08f, 0.64f, 1.63f, 0.1f},
                                       {23, 128, 128, 2, 0.641f, 0.528f, 4.52f, 0.91f, 6.52f, 0.05f},
                                       {23, 128, 128, 1, 0.332f, 0.566f, 5.65f, 0.f, 4.11f, 0.03f},  // where takes_turns
                                       {45, 256, 256, 1, 1.225f, 1.576f, 9.07f, 0.59f, 9.34f, 0.12f},
                                       {46, 256, 192, 1, 1.226f, 1.453f, 5.5f, 0.45f, 6.9f, 0.13f},
                                       {47, 256, 160, 1, 0.85f, 1.327f, 5.45f, 0.34f, 8.51f, 0.01f},
                                       {48, 256, 320, 1, 1.419f, 2.21f, 9.82f, 0.22f, 13.99f, 0.32f}};
constexpr int kComputeUnits = 256;
// Up to 256 tokens of a matrix of 16 MB or more, tiles of 64 x 64 give way to the widths of choose_few_token_tiles (7B down at 128
// tokens in 4 slices: 50.6 us staged, 41.8 in tiles of 128 features; 32B down at 192 tokens 131 and 106).  Not for small matrices: the
// staged tiles, four workgroups to a compute unit, share the weights of neighbouring token tiles (1.5B query/key/value, 6 MB, at 192
// tokens: 7.4 us against 9.1).  On the scale of this estimate theirs is 0.87 of what it says, and 4.1 us with the norm behind.
constexpr float kFewTokenScale = 0.87f, kFewTokenNorm = 4.1f;
static int choose_few_token_tiles(int m, int n, int k, int slices, float* estimate = nullptr);
static bool few_token_tiles_pay(int m, int n, int k) { return m <= 256 && static_cast<int64_t>(n) * k * 2 >= (16ll << 20); }
// 128 x 128 tiles: gemm_turns where a tile has its compute unit to itself and eight steps of k or more, gemm_direct elsewhere.  650
// products cut into up to 4 slices, gemm_turns' time over gemm_direct's: up to 256 tiles, 24 steps or more 0.81 (0.58 to 0.91), 12 to 23
// steps 0.93, 8 to 11 0.95 to 0.98, 4 to 7 1.01; more tiles 1.13 to 1.41: two workgroups of gemm_direct on a unit fill each other's waits
// also at the tiles' beginnings and ends.
static bool takes_turns(int m, int n, int k, int slices) {
  const int64_t groups = static_cast<int64_t>((m + 127) / 128) * ((n + 127) / 128) * slices;
  const int ksteps = (k + kBK - 1) / kBK;
  return groups <= kComputeUnits && (ksteps + slices - 1) / slices >= 8;
}
static float tiled_time_us(const TilingCost& c, int m, int n, int k, int slices, bool sums) {
  const int64_t tiles = static_cast<int64_t>((m + c.tile_tokens - 1) / c.tile_tokens) * ((n + c.tile_features - 1) / c.tile_features);
  const int64_t groups = tiles * slices;
  const int ksteps = (k + kBK - 1) / kBK;
  auto step = [&](int resident, float fill) {
    return fmaxf(c.alone, resident * c.busy * (1.f - c.eased + c.eased * fill));
  };
  const int64_t capacity = static_cast<int64_t>(kComputeUnits) * c.resident;
  const int64_t full = groups / capacity, rest = groups % capacity;
  const float fixed = c.fixed + (sums ? c.wide : 0.f);
  const float rows = static_cast<float>((m + c.tile_tokens - 1) / c.tile_tokens) * c.tile_tokens;
  const float per = static_cast<float>((ksteps + slices - 1) / slices) * (1.f - c.empty * (1.f - m / rows));
  float t = full * (fixed + per * step(c.resident, 1.f));
  if (rest > 0) {
    const int resident = static_cast<int>((rest + kComputeUnits - 1) / kComputeUnits);
    t += fixed + per * step(resident, fminf(1.f, static_cast<float>(rest) / kComputeUnits));
  }
  return t;
}
// sums: the results are float32.
static GemmPlan plan_many_tokens(int m, int n, int k, int max_slices, bool sums) {
  GemmPlan best{11, 1};
  float best_time = 0.f;
  const int ksteps = (k + kBK - 1) / kBK;
  for (const TilingCost& c : kTilingCosts)
    for (int slices = 1; slices <= min(max_slices, 4); ++slices) {
      if (slices > 1 && ksteps / slices < 3) break;  // every slice keeps a few steps (0.5B output
                                                     // projection at 128 tokens, 14 steps: whole 8.0 us, in 4 slices 5.4)
      if (c.kernel == 23 && (c.resident == 1) != takes_turns(m, n, k, slices)) continue;
      int kernel = c.kernel;
      float t = 0.f;
      if (kernel == 11 && few_token_tiles_pay(m, n, k)) {
        kernel = choose_few_token_tiles(m, n, k, slices, &t);
        t = kFewTokenScale * t + (sums ? kFewTokenNorm : 0.f);
      } else {
        t = tiled_time_us(c, m, n, k, slices, sums);
      }
      if (sums) t += 4.f * slices * m * n / 5.7e6f;
      if (best_time == 0.f || t < best_time) best = {kernel, slices}, best_time = t;
    }
  return best;
}

// The kernel for a shape: 16 = up to 16 tokens gemm_lines (71 to 74: 16 to 64 features), else gemm_skinny_split, 11 / 22 / 44 = gemm_tiled with 64 x 64,
// 128 x 128 (four wavefronts each) and 256 x 256 (sixteen wavefronts) tiles, 23 = 128 x 128 by gemm_turns (24) or
// gemm_direct (25) as takes_turns has it,
// 45 = gemm_phased with 256 x 256 (eight wavefronts in two groups), 46 / 47 / 48 = gemm_direct with tiles of 256 tokens x 192 features (twelve
// wavefronts of 64 x 64), x 160 features (ten of 128 x 32) and x 320 features (eight of 64 x 160), 14 = gemm_tiled
// with tiles of 32 tokens x 64 features (two wavefronts): for up to 32 tokens it stages half the
// rows of the 64 x 64 tile and streams weights 5 to 15 % faster, 62 to 68 = gemm_direct with tiles of
// 64 tokens x 64, 96, ... 256 features for up to 64 tokens (see choose_few_token_tiles).
// A small matrix (an output projection of a narrow model) at 17 to 64 tokens: the tiled kernels have
// too few tiles of it to keep the compute units busy, the row-splitting kernel with its 16 features a
// workgroup has four times as many workgroups (0.5B output projection with the norm behind it, in a
// replayed graph: 32 tokens 9.0 us tiled in 2 slices, 6.4 row-splitting in 4; 64 tokens 9.4 and 7.3).
// Larger matrices read the tokens too often that way (0.5B gate-up at 64 tokens: 10 us tiled, 16).
static bool small_matrix(int n, int k) { return static_cast<int64_t>(n) * k * 2 <= (4ll << 20); }

// Up to 64 tokens through tiles: such a product streams its weights once and is done when the busiest
// compute unit has streamed its share, so what counts is how the tiles go round the 256 units and what
// a unit takes in.  Fitted to replayed graphs over weights that come from memory (the five products of
// seven model sizes at 8 to 64 tokens, 1,500 timings, rms error 9 %): a unit takes in 44 GB/s through the
// tiles of gemm_direct and 37 through the register-staged ones, tokens included (a tile of 64 tokens x
// 64 features reads as many token bytes as weight bytes, one of 256 features a fifth of that), all
// units together 6.1 TB/s of weights (23.8 GB/s each), a launch costs 3.7 us and a round of tiles that
// have their unit to themselves 2 us until their first bytes arrive (0.8 where two share a unit).
// The tiles of 64 tokens x 64 ... 256 features of gemm_direct (a wavefront per 32 x 32 block; as many
// slices of k in LDS as fit, 3 to 6, where the staged kernels have 2 on their way) are there so that some
// width makes one round that fills the units: 7B gate-up (37,888 rows) at 64 tokens 67 us in staged
// 64-feature tiles, 48.8 in 237 tiles of 160; 32B gate-up 130 to 92 (247 tiles of 224; at 8 tokens 101
// to 92, 6.2 TB/s); cut along k in 8: 7B down 31.8 to 28.4, 32B down 69.6 to 50.1; the 7B output head
// 244 to 212; 0.5B gate-up 10.3 to 8.9.  Over the sweep the chosen tilings add up to 1.4 % more than the
// best ones, and to 7 % less than the staged 64-feature tiles everywhere.
struct FewTokenTiling {
  int kernel, tokens, features;
  bool direct;
  float round_us;  // per round of tiles
};
constexpr FewTokenTiling kFewTokenTilings[] = {
    {62, 64, 64, true, 0.77f},  {63, 64, 96, true, 2.f},  {64, 64, 128, true, 2.f}, {65, 64, 160, true, 2.f}, {66, 64, 192, true, 2.f},
    {67, 64, 224, true, 2.f},   {68, 64, 256, true, 2.f}, {14, 32, 64, false, 0.f}, {11, 64, 64, false, 0.f}};
static float few_token_time_us(const FewTokenTiling& t, int m, int n, int k, int slices) {
  constexpr float kDirectIntake = 44.f, kStagedIntake = 37.f, kUnitShare = 23.8f, kLaunch = 3.7f;  // GB/s, GB/s, GB/s, us
  // more tokens than a tile: every tile of tokens streams the weights again, but only the first from memory
  const int token_tiles = (m + t.tokens - 1) / t.tokens;
  const int64_t groups = static_cast<int64_t>((n + t.features - 1) / t.features) * slices * token_tiles;
  const float tile_kb = static_cast<float>(t.features) * ((k + slices - 1) / slices) * 2.f / 1e3f;
  const float unit = (t.direct ? kDirectIntake : kStagedIntake) * t.features / (t.features + min(m, t.tokens));
  const float share = kUnitShare * token_tiles;
  const int64_t full = groups / kComputeUnits, rest = groups % kComputeUnits;
  float time = kLaunch + full * (tile_kb / fminf(unit, share) + t.round_us);
  if (rest > 0) time += tile_kb / fminf(unit, share * kComputeUnits / rest) + t.round_us;
  return time;
}
static int choose_few_token_tiles(int m, int n, int k, int slices, float* estimate) {
  int best = 0;
  float best_time = 0.f;
  // narrow tiles first (at a tie the one that fills more units), the staged ones last and only when
  // clearly ahead: where the estimate has them level the direct tile measured 10 to 20 % faster
  for (const FewTokenTiling& t : kFewTokenTilings) {
    if ((t.kernel == 14 && m > t.tokens) || (t.kernel == 11 && m <= 32)) continue;
    const float time = few_token_time_us(t, m, n, k, slices);
    if (best == 0 || time < (t.direct ? 0.99f : 0.97f) * best_time) best = t.kernel, best_time = time;
  }
  if (estimate != nullptr) *estimate = best_time;
  return best;
}

static int choose_kernel(int m, int n, int k, int slices, bool sums) {
  if (m <= 16 && (!few_tokens_tiled(n, slices) || lines_stream(m, n, k))) return 16;
  if (m <= 64 && small_matrix(n, k)) return 16;
  if (m <= 64) return choose_few_token_tiles(m, n, k, slices);
  const GemmPlan plan = plan_many_tokens(m, n, k, slices, sums);
  if (plan.slices == slices) return plan.kernel;
  return few_token_tiles_pay(m, n, k) ? choose_few_token_tiles(m, n, k, slices) : 11;  // more slices than the plan would make of it
}

static int gemm_bf16(const bf16* xb, const bf16* wb, const GemmEpilogue& ep, int m, int n, int k, int slices,
                     int kernel, hipStream_t stream) {
  switch (kernel) {
    case 16: {
      if (m > 64) {
        set_error("mlr_gemm_bf16: the streaming kernel takes up to 64 tokens");
        return -1;
      }
      dim3 grid((n + 15) / 16, slices);
      if (m <= 16) return gemm_bf16(xb, wb, ep, m, n, k, slices, 70 + plan_lines(m, n, k, slices).blocks, stream);
      if (m <= 32) gemm_skinny_split_kernel<4, false, 2><<<grid, 256, 0, stream>>>(xb, wb, ep, QkvTarget{}, m, n, k);
      else gemm_skinny_split_kernel<4, false, 4><<<grid, 256, 0, stream>>>(xb, wb, ep, QkvTarget{}, m, n, k);
      return 0;
    }
    case 71: return launch_lines<1>(xb, wb, ep, m, n, k, slices, stream);
    case 72: return launch_lines<2>(xb, wb, ep, m, n, k, slices, stream);
    case 73: return launch_lines<3>(xb, wb, ep, m, n, k, slices, stream);
    case 74: return launch_lines<4>(xb, wb, ep, m, n, k, slices, stream);
    case 11: return launch_tiled<1, 1>(xb, wb, ep, m, n, k, slices, stream);
    case 14: return launch_tiled<1, 1, 1, 2>(xb, wb, ep, m, n, k, slices, stream);  // 32 tokens x 64 features, two wavefronts
    case 22: return launch_tiled<2, 2>(xb, wb, ep, m, n, k, slices, stream);
    case 44: return launch_tiled<2, 2, 4, 4>(xb, wb, ep, m, n, k, slices, stream);
    case 45: {  // 256 x 256, eight wavefronts in two groups that take turns
      static bool configured = false;
      return launch_direct(gemm_phased_kernel, 256, 256, 512, 2, kPhaseLds, configured, xb, wb, ep, m, n, k, slices, stream);
    }
    // 64 tokens x 64 to 256 features, a wavefront per 32 x 32 block, as many slices of k in LDS as fit
    case 62: {
      static bool configured = false;
      return launch_direct(gemm_direct_kernel<1, 1, 2, 2, 4, true>, 64, 64, 256, 2, direct_lds_bytes(64, 64, 4, 4),
                           configured, xb, wb, ep, m, n, k, slices, stream);
    }
    case 63: {
      static bool configured = false;
      return launch_direct(gemm_direct_kernel<1, 1, 2, 3, 6, true>, 64, 96, 384, 2, direct_lds_bytes(64, 96, 6, 6),
                           configured, xb, wb, ep, m, n, k, slices, stream);
    }
    case 64: {
      static bool configured = false;
      return launch_direct(gemm_direct_kernel<1, 1, 2, 4, 6, true>, 64, 128, 512, 2, direct_lds_bytes(64, 128, 8, 6),
                           configured, xb, wb, ep, m, n, k, slices, stream);
    }
    case 65: {
      static bool configured = false;
      return launch_direct(gemm_direct_kernel<1, 1, 2, 5, 5, true>, 64, 160, 640, 2, direct_lds_bytes(64, 160, 10, 5),
                           configured, xb, wb, ep, m, n, k, slices, stream);
    }
    case 66: {
      static bool configured = false;
      return launch_direct(gemm_direct_kernel<1, 1, 2, 6, 4, true>, 64, 192, 768, 2, direct_lds_bytes(64, 192, 12, 4),
                           configured, xb, wb, ep, m, n, k, slices, stream);
    }
    case 67: {
      static bool configured = false;
      return launch_direct(gemm_direct_kernel<1, 1, 2, 7, 3, true>, 64, 224, 896, 2, direct_lds_bytes(64, 224, 14, 3),
                           configured, xb, wb, ep, m, n, k, slices, stream);
    }
    case 68: {
      static bool configured = false;
      return launch_direct(gemm_direct_kernel<1, 1, 2, 8, 3, true>, 64, 256, 1024, 2, direct_lds_bytes(64, 256, 16, 3),
                           configured, xb, wb, ep, m, n, k, slices, stream);
    }
    case 48: {  // 256 tokens x 320 features, eight wavefronts of 64 x 160
      if (ep.swiglu == kEpGeglu) {
        static bool configured_geglu = false;
        return launch_direct(gemm_direct_kernel<2, 5, 4, 2, 2, false, kEpGeglu>, 256, 320, 512, 4,
                             direct_lds_bytes(256, 320, 8, 2), configured_geglu, xb, wb, ep, m, n, k, slices, stream);
      }
      static bool configured = false;
      return launch_direct(gemm_direct_kernel<2, 5, 4, 2>, 256, 320, 512, 4, direct_lds_bytes(256, 320, 8, 2), configured,
                           xb, wb, ep, m, n, k, slices, stream);
    }
    case 46: {  // 256 tokens x 192 features, twelve wavefronts of 64 x 64
      static bool configured = false;
      return launch_direct(gemm_direct_kernel<2, 2, 4, 3>, 256, 192, 768, 4, direct_lds_bytes(256, 192, 12, 2), configured,
                           xb, wb, ep, m, n, k, slices, stream);
    }
    case 47: {  // 256 tokens x 160 features, ten wavefronts of 128 x 32
      static bool configured = false;
      return launch_direct(gemm_direct_kernel<4, 1, 2, 5>, 256, 160, 640, 2, direct_lds_bytes(256, 160, 10, 2), configured,
                           xb, wb, ep, m, n, k, slices, stream);
    }
    case 23: return gemm_bf16(xb, wb, ep, m, n, k, slices, takes_turns(m, n, k, slices) ? 24 : 25, stream);
    case 24: {  // 128 x 128, eight wavefronts in two groups that share the slices of k
      static bool configured = false;
      return launch_direct(gemm_turns_kernel<false>, 128, 128, 512, 2, kTurnLds, configured, xb, wb, ep, m, n, k, slices, stream);
    }
    case 25: {
      static bool configured = false;
      return launch_direct(gemm_direct_kernel<2, 2, 2, 2>, 128, 128, 256, 2, direct_lds_bytes(128, 128, 4, 2), configured,
                           xb, wb, ep, m, n, k, slices, stream);
    }
    default: set_error("mlr_gemm_bf16: kernel must be 0 (chosen by shape), 16, 14, 11, 22 to 25, 44 to 48, 62 to 68 or 71 to 74"); return -1;
  }
}

// Whether the query/key/value product may take tiles of 128 x 128 with the staged epilogue (stage_qkv).
static bool staged_qkv_fits(const QkvTarget& t) {
  return 128 % t.head_dim == 0 && (t.slots == nullptr || t.block_size % 8 == 0) && reinterpret_cast<uintptr_t>(t.q_out) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(t.key_pages) % 16 == 0 && reinterpret_cast<uintptr_t>(t.value_pages) % 16 == 0;
}
// And which, if any: gemm_turns (24) for a round of tiles that leaves few units without one (up to 79 tiles, or 127 of a long k, the 64 x 64
// tiles with their epilogue from registers, or the plain product and the rotation kernel, are as fast or faster), gemm_direct (25),
// two tiles a unit, up to 512.  Microseconds in a replayed graph, weights from memory, the best of the other two ways / this one: 896 x 1,152 at
// 768 tokens (54 tiles) 12.7 / 14.4, at 1,024 (72) 15.0 / 14.5, at 2,048 18.3 / 15.2, at 3,072 21.8 / 15.7, at 4,096 (288) 27.2 / 23.7, at
// 6,000 (423) 31.2 / 25.0, at 8,191 (576) 36.8 / 37.0; 2,048 x 3,072 at 512 (96) 25.3 / 25.2, at 1,048 28.4 / 23.8, at 2,000 (384) 46.9 / 42.0, at
// 3,072 (576) 59.3 / 64.0; 3,584 x 4,608 at 256 (72) 33.1 / 41.4, at 512 (144) 43.2 / 39.8, at 1,048 (324) 62.3 / 59.0, at 1,536 (432) 68.5 /
// 62.5, at 2,000 (576) 86 / 116; 5,120 x 7,168 at 256 (112) 51.1 / 59.6, at 512 (224) 63.8 / 58.2, at 1,048 (504) 98.8 / 90.3.
static int staged_qkv_kernel(int m, int64_t n, int k) {
  const int64_t tiles = ((m + 127) / 128) * ((n + 127) / 128);
  if (m <= 64 || k < 8 * kBK || tiles < (k <= 2048 ? 80 : 128) || tiles > 2 * kComputeUnits) return 0;
  return tiles <= kComputeUnits ? 24 : 25;
}

}  // namespace mlr

using namespace mlr;

extern "C" {

// How many K slices mlr_gemm_bf16 would use for this shape when the caller can take
// partial sums (at most `max_slices`); 1 means it writes the finished product.
int mlr_gemm_bf16_slices(int m, int n, int k, int max_slices) {
  if (k % 8 != 0) return 1;
  if (m > 64) return plan_many_tokens(m, n, k, max_slices, true).slices;
  if (m <= 16) {
    // Measured with the norm kernel that adds the slices up (its cost grows with their number).  What gemm_lines leaves goes through the
    // tiles, weights of 64 MB or more cut into 8 slices, others into 4 once that fills the compute units, into 8 where 4 would not fill
    // them twice.
    const int64_t bytes = static_cast<int64_t>(n) * k * 2;
    if (!lines_stream(m, n, k) && max_slices >= 4) {
      const bool eight = max_slices >= 8 && k >= 8 * 256;
      if (eight && bytes >= (64ll << 20) && few_tokens_tiled(n, 8)) return 8;
      if (eight && few_tokens_tiled(n, 4) && !few_tokens_tiled(n, 2)) return 8;
      if (k >= 4 * 256 && few_tokens_tiled(n, 4)) return 4;
    }
    // gemm_lines: at most 8 slices for the norm to add up, a step of k for each of a workgroup's wavefronts; 2 from 20 MB on where its rows go through
    // rmsnorm_any_kernel, one slice after the other (8 tokens of 10,240 x 2,816 in 4 slices 68 us with the norm, in 2 46).  From 20 MB on never whole if the
    // consumer takes 4 slices or more and k >= 1,024, as in the tiles: one slice would be rounded to bfloat16 before it is added (one token of
    // matrices of 20 to 40 MB pays for that with 1.1 us of 9).
    const bool large = bytes >= (20ll << 20);
    const int most = min(max_slices, large && n > 8192 ? 2 : 8);
    LinesPlan best = plan_lines(m, n, k, large && max_slices >= 4 && k >= 4 * 256 ? min(most, 4) : 1);
    for (int slices = 2; slices <= most && k >= slices * 256; slices *= 2) {
      const LinesPlan plan = plan_lines(m, n, k, slices);
      if (plan.us < best.us) best = plan;
    }
    return best.slices;
  }
  // 17 to 64 tokens of a small matrix: the row-splitting kernel (see choose_kernel) cut into 4 where
  // every slice keeps a few steps of k
  if (small_matrix(n, k)) return (k / 8 + 3) / 4 >= 16 ? min(4, max_slices) : 1;
  // 17 to 64 tokens: the small tiles keep few bytes in flight each, so two workgroups per compute
  // unit before the cutting stops (32B down at 32 tokens: 320 workgroups 65 us, 640 workgroups 56 us)
  return choose_slices(tiles_64(m, n), (k / 8 + 3) / 4, min(max_slices, 8), 512);
}

int mlr_gemm_bf16_kernel(int m, int n, int k, int slices) { return choose_kernel(m, n, k, slices, slices > 1); }

// y = x w^T (+ bias) in bfloat16 on the matrix cores; see mlr_gemm_simple for the
// argument meanings.  Requires k % 8 == 0 and 16-byte aligned x and w.  With
// `swiglu` the rows of w are (gate, gate, up, up) groups, there is no bias, n is
// a multiple of 4 and y is [m, n / 2].  With slices > 1 (the value of
// mlr_gemm_bf16_slices; not with swiglu) y is float32 [slices, m, n]: partial sums
// over slices of k, the bias in slice 0, for the consumer to add up.
// `swiglu` 2 and 3 are element-wise activations instead (squared ReLU, sigmoid; any n, after the
// bias), and `multiply` (bfloat16 [m, n], or null) is multiplied into the activated sums; with
// `multiply_rows` (int32 [m]) row i takes row multiply_rows[i] of `multiply` (a table [rows, n]).
// `swiglu` 5: rows (and bias) woven as for 1, y [m, n / 2] = g * sigmoid(glu_alpha g) * (u + 1) with
// g = min(gate, glu_limit), u = clamp(up, -glu_limit, glu_limit); 6: woven likewise, y = gelu(gate) * up (tanh form).
int mlr_gemm_bf16(const void* x, const void* w, const void* bias, int bias_is_f32, void* y, int out_is_f32,
                  int swiglu, int slices, int kernel, int m, int n, int k, const float* row_sumsq, int sumsq_parts,
                  float norm_eps, const void* multiply, const int* multiply_rows, float glu_limit, float glu_alpha,
                  hipStream_t stream) {
  MLR_REQUIRE(x && w && y, "null pointer");
  MLR_REQUIRE(swiglu >= kEpNone && swiglu <= kEpGeglu, "unknown epilogue");
  MLR_REQUIRE(swiglu != kEpClampedGlu || (n % 4 == 0 && multiply == nullptr && glu_limit > 0.f),
              "the clamped gating needs n % 4 == 0, a limit > 0 and no multiplier");
  MLR_REQUIRE(swiglu != kEpGeglu || (n % 4 == 0 && multiply == nullptr), "the GELU gating needs n % 4 == 0 and no multiplier");
  MLR_REQUIRE(multiply == nullptr || (swiglu != kEpSwiglu && slices == 1), "a multiplier goes with whole, unpaired sums");
  MLR_REQUIRE(slices == 1 || swiglu == kEpNone, "partial sums take no activation");
  MLR_REQUIRE(m > 0 && n > 0 && k > 0, "sizes must be > 0");
  MLR_REQUIRE(k % 8 == 0, "k must be a multiple of 8");
  MLR_REQUIRE(k <= (1 << 20), "k must not exceed 2^20 (32-bit byte offsets inside a tile)");
  MLR_REQUIRE(swiglu != kEpSwiglu || (n % 4 == 0 && bias == nullptr), "swiglu needs n % 4 == 0 and no bias");
  MLR_REQUIRE(slices >= 1 && slices <= 64, "slices must be within 1..64");
  MLR_REQUIRE(slices == 1 || (!swiglu && out_is_f32), "partial sums are float32, without SwiGLU");
  MLR_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0,
              "x and w must be 16-byte aligned");
  MLR_REQUIRE(row_sumsq == nullptr || (sumsq_parts > 0 && sumsq_parts <= (1 << 16) && norm_eps >= 0.f),
              "sums of squares come with their number per row (1..65536) and an eps >= 0");
  MLR_REQUIRE(multiply_rows == nullptr || multiply != nullptr, "row indices come with a multiplier");
  GemmEpilogue ep{bias, bias_is_f32, y, out_is_f32, swiglu, row_sumsq, sumsq_parts, norm_eps, multiply, glu_limit, glu_alpha,
                  multiply_rows};
  if (kernel == 0) kernel = choose_kernel(m, n, k, slices, out_is_f32 != 0);
  // the 256 x 320 tile has no room for a choice of activations and the multiplier in its epilogue (the GELU gating has an
  // instance of its own)
  if (kernel == 48 && ((swiglu >= kEpRelu2 && swiglu != kEpGeglu) || multiply != nullptr)) kernel = 45;
  if (gemm_bf16(static_cast<const bf16*>(x), static_cast<const bf16*>(w), ep, m, n, k, slices, kernel, stream) != 0)
    return -1;
  MLR_LAUNCH_CHECK();
  return 0;
}

// Whether mlr_qkv_rope_write_bf16 has tiles of 128 x 128 for a product of these sizes (block_size 0: no cache write), which make it
// the fastest way; beyond them the plain product with the rotation kernel behind it may be faster.
int mlr_qkv_bf16_staged(int m, int n, int k, int head_dim, int block_size) {
  return head_dim > 0 && 128 % head_dim == 0 && block_size % 8 == 0 && k % 8 == 0 && staged_qkv_kernel(m, n, k) != 0;
}

// The query/key/value product with everything that follows it before attention: bias, rotation of the query and key heads (cos, sin: [m, head_dim / 2] float32,
// or null for none), queries to q_out [m, heads * head_dim], keys and values into the slots
// of their pages (`write` 0: another layer owns the pages).  w is [(heads + 2 kv_heads) *
// head_dim, k]; head_dim a multiple of 16, k of 8.  kernel: 0 chooses (the streaming kernel up
// to 64 tokens unless it would read x too often, else a tiled one), or 16, 11, 22, 44, or 24 and 25 (tiles of 128 x 128 with a staged epilogue).
int mlr_qkv_rope_write_bf16(const void* x, const void* w, const void* bias, int bias_is_f32, const float* cos,
                            const float* sin, const int* slots, void* key_pages, void* value_pages, void* q_out,
                            int m, int k, int heads, int kv_heads, int head_dim, int block_size, int num_pages,
                            int write, int kernel, const float* row_sumsq, int sumsq_parts, float norm_eps,
                            hipStream_t stream) {
  MLR_REQUIRE(x && w && q_out, "null pointer");
  MLR_REQUIRE(row_sumsq == nullptr || (sumsq_parts > 0 && sumsq_parts <= (1 << 16) && norm_eps >= 0.f),
              "sums of squares come with their number per row (1..65536) and an eps >= 0");
  MLR_REQUIRE(m > 0, "no tokens");
  MLR_REQUIRE(k > 0 && k % 8 == 0 && k <= (1 << 20), "k must be a positive multiple of 8, at most 2^20");
  MLR_REQUIRE(heads > 0 && kv_heads > 0 && head_dim >= 16 && head_dim % 16 == 0, "head_dim must be a multiple of 16");
  MLR_REQUIRE((cos == nullptr) == (sin == nullptr), "cos and sin come together");
  MLR_REQUIRE(!write || (slots && key_pages && value_pages && block_size > 0 && num_pages > 0),
              "a cache write needs slots, pages and their sizes");
  MLR_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(q_out) % 8 == 0 && reinterpret_cast<uintptr_t>(key_pages) % 8 == 0 &&
                  reinterpret_cast<uintptr_t>(cos) % 16 == 0 && reinterpret_cast<uintptr_t>(sin) % 16 == 0,
              "operands must be 16-byte aligned");
  const int64_t n = static_cast<int64_t>(heads + 2 * kv_heads) * head_dim;
  MLR_REQUIRE(n / 16 < (1ll << 31), "too many rows for one launch");
  GemmEpilogue ep{bias, bias_is_f32, nullptr, 0, 0, row_sumsq, sumsq_parts, norm_eps};
  QkvTarget target{cos, sin, write ? slots : nullptr, static_cast<bf16*>(key_pages), static_cast<bf16*>(value_pages),
                   static_cast<bf16*>(q_out), heads, kv_heads, head_dim, block_size, num_pages};
  const bf16* xb = static_cast<const bf16*>(x);
  const bf16* wb = static_cast<const bf16*>(w);
  const bool stages = staged_qkv_fits(target);
  if (kernel == 0) {
    // Beyond 64 tokens tiles of 128 x 128 where staged_qkv_kernel has them, else the 64 x 64 tiles: with the epilogue from registers
    // (rotation, scattered cache stores) the larger tiles are slower than they are for the plain product.
    kernel = m <= 64 ? 16 : 11;
    if (kernel == 16 && m > 16 && (n / 16) * m * k * 2 > (32ll << 20)) kernel = 11;  // too many passes over x
    if (stages && staged_qkv_kernel(m, n, k) != 0) kernel = staged_qkv_kernel(m, n, k);
  }
  MLR_REQUIRE((kernel != 24 && kernel != 25) || stages, "the staged kernels take head sizes that divide 128, pages of a multiple of 8 tokens and 16-byte alignment");
  if (kernel == 24) {
    static bool configured = false;
    if (launch_direct(gemm_turns_kernel<true>, 128, 128, 512, 2, kTurnLds, configured, xb, wb, ep, m, static_cast<int>(n), k, 1, stream, target) != 0) return -1;
    MLR_LAUNCH_CHECK();
    return 0;
  }
  if (kernel == 25) {
    static bool configured = false;
    if (launch_direct(gemm_direct_kernel<2, 2, 2, 2, 2, false, -1, true>, 128, 128, 256, 2, direct_lds_bytes(128, 128, 4, 2), configured, xb, wb, ep, m,
                      static_cast<int>(n), k, 1, stream, target) != 0)
      return -1;
    MLR_LAUNCH_CHECK();
    return 0;
  }
  if (kernel == 8) {
    MLR_REQUIRE(m <= 8, "the 8-row kernel takes 1..8 tokens");
    gemm_skinny_qkv8_kernel<4><<<dim3(static_cast<unsigned>(n / 8)), 256, 0, stream>>>(xb, wb, ep, target, m, static_cast<int>(n), k);
    MLR_LAUNCH_CHECK();
    return 0;
  }
  if (kernel == 16) {
    MLR_REQUIRE(m <= 64, "the row-splitting kernel takes 1..64 tokens");
    const dim3 grid(static_cast<unsigned>(n / 16));
    if (m <= 8 && half_rows_fill_better(static_cast<int>(n / 16)))
      gemm_skinny_qkv8_kernel<4><<<dim3(static_cast<unsigned>(n / 8)), 256, 0, stream>>>(xb, wb, ep, target, m, static_cast<int>(n), k);
    else if (m <= 16) {
      const int rows = static_cast<int>(n);
      int status = 0;
      switch (plan_lines(m, rows, k, 1).blocks) {
        case 1: status = launch_lines<1, true>(xb, wb, ep, m, rows, k, 1, stream, target); break;
        case 2: status = launch_lines<2, true>(xb, wb, ep, m, rows, k, 1, stream, target); break;
        case 3: status = launch_lines<3, true>(xb, wb, ep, m, rows, k, 1, stream, target); break;
        default: status = launch_lines<4, true>(xb, wb, ep, m, rows, k, 1, stream, target); break;
      }
      if (status != 0) return -1;
    } else if (n * k * 2 <= (8ll << 20))
      // a small matrix: a workgroup per slab of 16 tokens reads a quarter of the tokens and the weights
      // again from L2, where one workgroup for all slabs is held up by the tokens it takes in (0.5B at
      // 64 tokens 8.4 to 6.8 us, at 48 7.7 to 5.2; 1.5B at 64 12.0 to 10.1; a 10 MB matrix: 14.6 to 16.1).
      // The same sums in the same order either way.
      gemm_skinny_split_kernel<4, true, 1><<<dim3(grid.x, 1, (m + 15) / 16), 256, 0, stream>>>(xb, wb, ep, target, m, static_cast<int>(n), k);
    else if (m <= 32)
      gemm_skinny_split_kernel<4, true, 2><<<grid, 256, 0, stream>>>(xb, wb, ep, target, m, static_cast<int>(n), k);
    else
      gemm_skinny_split_kernel<4, true, 4><<<grid, 256, 0, stream>>>(xb, wb, ep, target, m, static_cast<int>(n), k);
    MLR_LAUNCH_CHECK();
    return 0;
  }
  // the tiled kernels address the whole weight matrix, and one token's rows of x, with 31-bit offsets
  MLR_REQUIRE(n * k * 2 < (1ll << 31), "the weight matrix is too large for the tiled fused product");
  switch (kernel) {
    case 11: return launch_tiled_qkv<1, 1>(xb, wb, ep, target, m, static_cast<int>(n), k, stream);
    case 22: return launch_tiled_qkv<2, 2>(xb, wb, ep, target, m, static_cast<int>(n), k, stream);
    case 44: return launch_tiled_qkv<2, 2, 4, 4>(xb, wb, ep, target, m, static_cast<int>(n), k, stream);
    default: MLR_REQUIRE(false, "unknown kernel");
  }
  return 0;
}

}  // extern "C"
