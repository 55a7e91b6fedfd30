// float32 matrix products on the matrix cores: y[M, N] = x[M, K] * w[N, K]^T (+ bias), the product of the true
// 32-bit path.  The matrix cores multiply and add float32 as it is (v_mfma_f32_32x32x2_f32, 16x16x4_f32: no rounding of the
// inputs), at 256 operations a clock and compute unit, twice what the vector unit's multiply-adds give without packed instructions.
//
//  * gemm_f32_tiled: more than 64 tokens.  Bound by the matrix cores: a tile of 64 x 64 takes 1,024 clocks of them per
//    32-wide step of k and 16 KB of operands.  So what counts is that they never wait: blocks of 16 x 16 x 4, four independent sums a
//    wavefront, and two buffers of LDS a workgroup instead of three, so that five workgroups fit a compute unit; and that
//    all units are busy: tiles of 64 x 64, 64 features x 32 tokens or 32 x 32, the smaller ones also with two groups of wavefronts that
//    take the steps of k in turn (f32_time).  Tiles are loaded straight into LDS (rows of 32 floats are the 128 bytes of the bfloat16 kernels'
//    rows of 64, swizzled the same way), one step on its way.  Products whose consumer adds up partial sums are cut along k.
//    The order of a sum over k depends on the number of groups and of slices, and those on the number of tokens: the same token in
//    a step of another size may differ in its last bits (1,152 x 896 has two groups at 391 and 826 tokens, one at 512 and 1,024).
//  * gemm_f32_few: up to 64 tokens.  Bound by streaming w once: 16 weight rows a workgroup, whose eight wavefronts split k and
//    add their sums through LDS.
// Measured at 0.5B sizes and 826 tokens, against the plain kernel (gemm_simple.hip, 64 x 64 tiles of vector multiply-adds with
// 16-wide steps through single-buffered LDS), microseconds: gate-up (9,728 x 896) 228 to 116 (125 TFLOP/s; the matrix cores at 2.4 GHz
// would take 92), down (896 x 4,864) 659 to 63 in four slices, query/key/value (1,152 x 896) 117 to 19; at 8 tokens gate-up 94 to
// 12, down 363 to 17, the output head 353 to 127.
//
// K must be a multiple of 4 and the operands 16-byte aligned; other shapes take the plain kernel.
#include "api.h"
#include "common.h"
#include "gemm_epilogue.h"
#include "mfma.h"

#include <algorithm>
#include <cmath>

namespace mlr {

struct F32Epilogue {
  const float* bias;
  float* y;
  int kind;  // kEpNone .. kEpGeglu
  const float* multiply;
  const int* multiply_rows;
  float glu_limit, glu_alpha;
};

// Four consecutive features n .. n + 3 of token m, as the plain kernel finishes them.
__device__ __forceinline__ void finish4_f32(const F32Epilogue& ep, int slice, int slices, int m, int n, int M, int N, f32x4_t v) {
  if (m >= M || n >= N) return;
  const bool paired = ep.kind == kEpSwiglu || ep.kind == kEpClampedGlu || ep.kind == kEpGeglu;
  if (ep.bias != nullptr && slice == 0) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) v[e] += ep.bias[n + e];
  }
  if (paired) {  // n % 4 == 0 and N % 4 == 0: gate, gate, up, up
    float* dst = ep.y + static_cast<int64_t>(m) * (N / 2) + n / 2;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float g = v[j], u = v[j + 2];
      if (ep.kind == kEpSwiglu) {
        dst[j] = g / (1.0f + expf(-g)) * u;
      } else if (ep.kind == kEpGeglu) {
        dst[j] = 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))) * u;
      } else {
        g = fminf(g, ep.glu_limit);
        u = fminf(fmaxf(u, -ep.glu_limit), ep.glu_limit);
        dst[j] = g / (1.0f + expf(-ep.glu_alpha * g)) * (u + 1.0f);
      }
    }
    return;
  }
  const int64_t factor_row = ep.multiply_rows != nullptr ? ep.multiply_rows[m] : m;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (n + e >= N) continue;
    float r = v[e];
    if (ep.kind == kEpRelu2) {
      r = fmaxf(r, 0.f);
      r *= r;
    } else if (ep.kind == kEpSigmoid) {
      r = 1.0f / (1.0f + expf(-r));
    } else if (ep.kind == kEpGeluTanh) {
      r = 0.5f * r * (1.0f + tanhf(0.7978845608028654f * (r + 0.044715f * r * r * r)));
    }
    if (ep.multiply != nullptr) r *= ep.multiply[factor_row * N + n + e];
    v[e] = r;
  }
  float* dst = ep.y + (static_cast<int64_t>(slice) * M + m) * N + n;
  if (N % 4 == 0) {
    *reinterpret_cast<f32x4_t*>(dst) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) dst[e] = v[e];
  }
}

__device__ __forceinline__ f32x4_t load_f32x4(const void* p) { return *reinterpret_cast<const f32x4_t*>(p); }

// ---- more than 64 tokens ------------------------------------------------------------------------------
// Four wavefronts, each TU x TT blocks of 16 features x 16 tokens.  An operand read brings a lane 4 consecutive k of its row; product j
// of the four takes element j of every lane, so the lanes' quarters stand for k = 16 g + j, 4 + j, 8 + j and 12 + j: the same on both
// sides, and the order of k does not matter to a sum.
// Measured against blocks of 32 x 32 x 2 (one sum a wavefront) with three buffers, 64 x 64 tiles, microseconds: 826 x 9,728 x 896 122 to 115, 826 x 896 x
// 4,864 in four slices 64.6 to 61.7, 2,048 x 9,728 x 896 290 to 271; two buffers alone 120, 65.3 and 286, 16 x 16 x 4 alone 121, 63.3 and 282.
// Tiles of 128 x 64, 64 x 128 and 128 x 128 (fewer operand reads) were slower: 120, 144 and 181 instead of 117.
constexpr int kF32Step = 32;     // k per LDS slice
constexpr int kF32Buffers = 2;   // one multiplied, one on its way: with the other workgroups of the unit a step lasts longer than a trip to memory

template <int TU, int TT, int KG>
struct F32Tile {
  static constexpr int kRowsW = 32 * TU, kRowsX = 32 * TT;
  static constexpr int kBytes = (kRowsW + kRowsX) * kF32Step * 4;
  static constexpr int kLds = KG * kF32Buffers * kBytes;
};

// KG groups of four wavefronts take the steps of k in turn, each with buffers of its own, and add their sums in order at the end.
// (Not the kernel itself: a kernel's template whose loop bounds are constants of another template is not instantiated on the host.)
template <int TU, int TT, int KG>
__device__ __forceinline__ void f32_tile(const float* __restrict__ x, const float* __restrict__ w, const F32Epilogue& ep, int M, int N, int K, int slices) {
  using Tile = F32Tile<TU, TT, KG>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x % kWave;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int group = KG > 1 ? wave_all / 4 : 0, wave = wave_all % 4;
  const int wn = wave % 2, wm = wave / 2;
  const int r16 = lane % 16, q4 = lane / 16;
  const int n0 = blockIdx.x * Tile::kRowsW, m0 = blockIdx.y * Tile::kRowsX;
  const int slice = blockIdx.z;
  const int k_steps = (K + kF32Step - 1) / kF32Step;
  const int per = (k_steps + slices - 1) / slices;
  const int s_begin = slice * per, s_end = min(k_steps, s_begin + per);
  const int chunks = K / 4;  // 16-byte pieces of a row

  const int w_rows = min(Tile::kRowsW, N - n0), x_rows = min(Tile::kRowsX, M - m0);
  const __amdgpu_buffer_rsrc_t w_buf = make_buffer(w + static_cast<int64_t>(n0) * K, static_cast<unsigned>(w_rows) * K * 4u);
  const __amdgpu_buffer_rsrc_t x_buf = make_buffer(x + static_cast<int64_t>(m0) * K, static_cast<unsigned>(x_rows) * K * 4u);
  // a wavefront's load fills a run of 8 rows: lane l brings row l / 8, piece (l % 8) ^ key to slot l % 8, key = (row / 2) % 8
  // (LDS serves two rows of 128 bytes side by side); run p * 4 + wave: the first 4 TU runs are weight rows, the others token rows
  const int lane_row = lane / 8;
  const int lane_chunk = (lane % 8) ^ ((4 * (wave % 2) + lane_row / 2) % 8);  // runs p * 4 + wave: 8 rows each, the key repeats every 16
  const unsigned row_off = static_cast<unsigned>(8 * wave + lane_row) * K * 4u + lane_chunk * 16u;
  unsigned char* const mine = smem + group * kF32Buffers * Tile::kBytes;
  auto fetch = [&](int s, int buf) {
    const unsigned ok = s < s_end && lane_chunk < chunks - s * (kF32Step / 4) ? 0u : kOutOfBuffer;
#pragma unroll
    for (int p = 0; p < TU + TT; ++p) {
      __attribute__((address_space(3))) void* dst =
          (__attribute__((address_space(3))) void*)(mine + buf * Tile::kBytes + (p * 4 + wave) * 1024);
      const unsigned off = (row_off + (p < TU ? p : p - TU) * 32u * K * 4u + s * (kF32Step * 4u)) | ok;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(p < TU ? w_buf : x_buf, dst, 16, off, 0, 0, 0);
    }
  };

  // two sums of a block, of the steps' first and second halves: shorter chains, and a smaller error than one (5.4e-7 to 3.8e-7 with k = 896)
  f32x4_t acc[TU][TT], acc2[TU][TT];
#pragma unroll
  for (int u = 0; u < TU; ++u)
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[u][t] = acc2[u][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int swz = (r16 / 2) % 8;
  const int a_base = (wn * 16 * TU + r16) * (kF32Step * 4);
  const int b_base = (Tile::kRowsW + wm * 16 * TT + r16) * (kF32Step * 4);

  fetch(s_begin + group, 0);
  int buf = 0;
  for (int s = s_begin; s < s_end; s += KG) {
    // this slice has landed (this wavefront's share; the barrier answers for the others), and everybody has multiplied the one before
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fetch(s + group + KG, buf ^ 1);  // into the buffer of the slice before
    const unsigned char* base = mine + buf * Tile::kBytes;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int slot = ((g * 4 + q4) ^ swz) * 16;
      f32x4_t a[TU], b[TT];
#pragma unroll
      for (int u = 0; u < TU; ++u) a[u] = load_f32x4(base + a_base + u * 16 * 128 + slot);
#pragma unroll
      for (int t = 0; t < TT; ++t) b[t] = load_f32x4(base + b_base + t * 16 * 128 + slot);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int u = 0; u < TU; ++u)
#pragma unroll
          for (int t = 0; t < TT; ++t) {
            f32x4_t& sum = g == 0 ? acc[u][t] : acc2[u][t];
            sum = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][j], b[t][j], sum, 0, 0, 0);
          }
    }
    buf ^= 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past the end have landed before LDS is given back
#pragma unroll
  for (int u = 0; u < TU; ++u)
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[u][t] += acc2[u][t];

  if constexpr (KG > 1) {
    __syncthreads();
    f32x4_t* const sums = reinterpret_cast<f32x4_t*>(smem);
#pragma unroll
    for (int u = 0; u < TU; ++u)
#pragma unroll
      for (int t = 0; t < TT; ++t) sums[((wave_all * TU + u) * TT + t) * kWave + lane] = acc[u][t];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TU; ++u)
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        if ((u * TT + t) % KG != group) continue;
        f32x4_t v = sums[((wave * TU + u) * TT + t) * kWave + lane];
#pragma unroll
        for (int g = 1; g < KG; ++g) v += sums[(((g * 4 + wave) * TU + u) * TT + t) * kWave + lane];
        finish4_f32(ep, slice, slices, m0 + (wm * TT + t) * 16 + r16, n0 + (wn * TU + u) * 16 + q4 * 4, M, N, v);
      }
  } else {
#pragma unroll
    for (int u = 0; u < TU; ++u)
#pragma unroll
      for (int t = 0; t < TT; ++t)
        finish4_f32(ep, slice, slices, m0 + (wm * TT + t) * 16 + r16, n0 + (wn * TU + u) * 16 + q4 * 4, M, N, acc[u][t]);
  }
}

template <int TU, int TT, int KG>
__global__ __launch_bounds__(256 * KG) void gemm_f32_tiled_kernel(const float* __restrict__ x, const float* __restrict__ w, F32Epilogue ep,
                                                                  int M, int N, int K, int slices) {
  f32_tile<TU, TT, KG>(x, w, ep, M, N, K, slices);
}

template <int TU, int TT, int KG>
static void launch_f32(const float* x, const float* w, const F32Epilogue& ep, int m, int n, int k, int slices, hipStream_t stream) {
  using Tile = F32Tile<TU, TT, KG>;
  static_assert(Tile::kLds <= 65536, "more needs a function attribute");
  const dim3 grid((n + Tile::kRowsW - 1) / Tile::kRowsW, (m + Tile::kRowsX - 1) / Tile::kRowsX, slices);
  gemm_f32_tiled_kernel<TU, TT, KG><<<grid, 256 * KG, Tile::kLds, stream>>>(x, w, ep, m, n, k, slices);
}

// The tilings, and what a product takes in each (microseconds, an estimate): the busiest compute unit has `rounds` tiles and multiplies them
// beside one another, at `rate` of what the matrix cores do at 2.4 GHz; with few tiles there it waits for a step's operands instead (two groups of
// wavefronts half as often); and weights too large for the caches come from memory once for every row of tiles, with half the lines of a page
// open where tiles have 32 rows of them.  Constants fitted to 621 products (65 to 2,100 tokens, 64 to 20,000 features, k of 80 to 9,000): what the
// estimate chooses is 2.2 % over the best on average, 29 % at worst, 17 % of them by more than 5 %, and 22 % under 64 x 64 tiles everywhere; against the
// kernel of 32 x 32 x 2 blocks over 856 other products 0.76 of the time on average, 18 of them slower by more than 3 %: weights of 13 MB and more in 64 x 64 with a
// k under 500 (1,164 x 4,071 x 488 52.8 to 56.0), and in 64 x 32 of two to five rounds (556 x 4,014 x 7,972, the worst, 1.31; 536 x 4,630 x 4,724 1.08).  64 x 64,
// 64 x 32, 32 x 32 alone and with two groups, microseconds: 826 x 9,728 x 896 116, 121, 131, 138; 391 75, 65, 69, 75; 200 46, 41, 40, 42; 66 32, 22, 21,
// 21; 826 x 1,152 x 896 21, 20, 20, 20 (64 x 32 with two groups 19); 391 21, 14, 13, 13 (12); 200 21, 14, 13, 8.8 (12); 1,794 x 5,692 x 3,916 (weights of
// 89 MB) 657, 840, 845, 785.
struct F32Way {
  int tu, tt, kg;
  double rate;
};
constexpr F32Way kF32Ways[] = {{2, 2, 1, 0.89}, {2, 1, 1, 0.86}, {2, 1, 2, 0.84}, {1, 1, 1, 0.80}, {1, 1, 2, 0.71}};

static double f32_time(const F32Way& t, int m, int n, int k, int slices) {
  const int64_t m_tiles = (m + 32 * t.tt - 1) / (32 * t.tt), tiles = m_tiles * ((n + 32 * t.tu - 1) / (32 * t.tu)) * slices;
  const double rounds = static_cast<double>((tiles + 255) / 256);
  const int steps = ((k + kF32Step - 1) / kF32Step + slices - 1) / slices;
  const double alone = 0.427 * t.tu * t.tt / 4;
  const double busy = rounds * alone / t.rate, waits = t.kg == 1 ? alone + 0.143 : (alone + 0.143) / 2 + 0.038;
  const double weights = 4.0 * n * k;
  const double memory = weights > 24e6 ? m_tiles * weights / (t.tu == 1 ? 4.4e6 : 7.3e6) : 0.0;
  return 4.0 + std::max(steps * std::pow(std::pow(busy, 5) + std::pow(waits, 5), 0.2), memory);
}

// The tiling for a product in a given number of slices of k.
static int f32_way(int m, int n, int k, int slices) {
  int best = 0;
  double least = 1e30;
  for (int i = 0; i < static_cast<int>(sizeof(kF32Ways) / sizeof(kF32Ways[0])); ++i) {
    const F32Way& t = kF32Ways[i];
    if (i > 0 && (m + 32 * t.tt - 1) / (32 * t.tt) >= 65536) continue;
    const double time = f32_time(t, m, n, k, slices) * (i == 0 ? 0.96 : 1.0);  // near the line the largest tile is the safer choice
    if (time < least) least = time, best = i;
  }
  // Six workgroups of 64 x 32 fit a compute unit (24 KB each): a seventh begins when one of them has ended, which the estimate, all beside one another, does
  // not see.  With up to a round of those 64 x 64 (five to a unit, up to 1,280 at once) is faster.  32 x 32 x 2 blocks / 64 x 32 / 64 x 64, microseconds: 325 x
  // 9,511 x 1,360 100 / 110 / 93, 1,450 x 2,194 x 3,464 232 / 254 / 219, 386 x 7,598 x 6,460 419 / 449 / 395, 854 x 3,651 x 7,532 1.07 and 0.94 of
  // the first; one of 17 such products is slower so (804 x 3,789 x 3,512, 3 %).
  if (best == 1 && slices == 1) {
    const int64_t tiles = static_cast<int64_t>((m + 31) / 32) * ((n + 63) / 64);
    if (tiles > 6 * 256 && tiles <= 7 * 256) best = 0;
  }
  return best;
}

// ---- up to 64 tokens ----------------------------------------------------------------------------------
// MT: slabs of 16 tokens.  A lane holds weight row lane % 16 and, of every 16 k, the 4 from 4 (lane / 16) on; product j of four takes
// element j of every lane.  The sums of a lane are 4 consecutive features of one token.
constexpr int kFewWaves = 8;

template <int MT>
__global__ __launch_bounds__(kFewWaves * 64) void gemm_f32_few_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                     F32Epilogue ep, int M, int N, int K) {
  __shared__ f32x4_t sums[kFewWaves][MT][kWave];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int r16 = lane % 16, quarter = lane / 16;
  const int n0 = blockIdx.x * 16;
  const unsigned rows = static_cast<unsigned>(min(16, N - n0));
  const __amdgpu_buffer_rsrc_t w_buf = make_buffer(w + static_cast<int64_t>(n0) * K, rows * K * 4u);
  const __amdgpu_buffer_rsrc_t x_buf = make_buffer(x, static_cast<unsigned>(M) * K * 4u);
  f32x4_t acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // runs of 32 k go round the wavefronts, four at a time: a row's 128 bytes are one line of memory
  constexpr int kRuns = MT > 2 ? 2 : 4;
  const int all = (K + 31) / 32;
  for (int run0 = wave; run0 < all; run0 += kRuns * kFewWaves) {
    f32x4_t a[kRuns][2], b[kRuns][MT][2];
#pragma unroll
    for (int u = 0; u < kRuns; ++u)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int k = (run0 + u * kFewWaves) * 32 + half * 16 + quarter * 4;
        const unsigned out = k < K ? 0u : kOutOfBuffer;  // K is a multiple of 4
        a[u][half] = __builtin_bit_cast(
            f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_buf, ((static_cast<unsigned>(r16) * K + k) * 4u) | out, 0, 2));
#pragma unroll
        for (int t = 0; t < MT; ++t)
          b[u][t][half] = __builtin_bit_cast(
              f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(x_buf, ((static_cast<unsigned>(t * 16 + r16) * K + k) * 4u) | out, 0, 0));
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kRuns; ++u)
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = 0; t < MT; ++t)
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][half][j], b[u][t][half][j], acc[t], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) sums[wave][t][lane] = acc[t];
  __syncthreads();
  for (int t = wave; t < MT; t += kFewWaves) {
    f32x4_t v = sums[0][t][lane];
#pragma unroll
    for (int i = 1; i < kFewWaves; ++i) v += sums[i][t][lane];  // in the wavefronts' order
    finish4_f32(ep, 0, 1, t * 16 + r16, n0 + quarter * 4, M, N, v);
  }
}

}  // namespace mlr

using namespace mlr;

// How many partial sums (slices of k) a product is cut into, when its consumer takes up to `max_slices`: the number with
// the smallest estimate and the consumer's reading of a slice (0.8 us per million sums).  Never fewer than it takes for 512 workgroups of 64 x 64 in
// slices of at least 8 steps: fewer, longer sums are less exact.  Measured in 1, 2, 4 and 8 slices, the best tiling of each, microseconds: 826 x 896 x 4,864
// 88, 64, 64, 64; 826 x 896 x 896 16.3, 15.6, 16.5, 18; 2,048 x 896 x 4,864 155, 151, 139, 142; 200 x 896 x 896 (8 slices) 11, 7.6, 7.6, 7.5.
extern "C" int mlr_gemm_f32_slices(int m, int n, int k, int max_slices) {
  if (m <= 64) return 1;
  const int64_t tiles = static_cast<int64_t>((m + 63) / 64) * ((n + 63) / 64);
  const int steps = (k + kF32Step - 1) / kF32Step;
  int least = 1;
  while (least * 2 <= max_slices && tiles * least < 512 && steps / (least * 2) >= 8) least *= 2;
  int best = least;
  double time = 1e30;
  for (int slices = least; slices <= max_slices && (slices == least || steps / slices >= 6); slices *= 2) {
    const double t = f32_time(kF32Ways[f32_way(m, n, k, slices)], m, n, k, slices) + slices * 8e-7 * m * n;
    if (t < 0.95 * time) time = t, best = slices;
  }
  return best;
}

extern "C" int mlr_gemm_f32_tiling(int m, int n, int k, int slices) {
  const F32Way& t = kF32Ways[f32_way(m, n, k, std::max(1, slices))];
  return (t.tu * 10 + t.tt) * 10 + t.kg;
}

// y [M, N] (or [M, N / 2] for the pairings; [slices, M, N] with slices > 1) = x w^T.  `swiglu`: the epilogue, as for mlr_gemm_simple.
extern "C" int mlr_gemm_f32(const float* x, const float* w, const float* bias, float* y, int swiglu, int slices, int m, int n, int k,
                            const float* multiply, const int* multiply_rows, float glu_limit, float glu_alpha, hipStream_t stream) {
  MLR_REQUIRE(x && w && y, "null pointer");
  MLR_REQUIRE(m > 0 && n > 0 && k > 0 && k % 4 == 0, "sizes must be > 0 and k a multiple of 4");
  MLR_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0,
              "operands must be 16-byte aligned");
  MLR_REQUIRE(k <= (1 << 22), "k must be at most 2^22");  // 32-bit offsets into 64 rows, below the out-of-range mark
  MLR_REQUIRE(swiglu >= 0 && swiglu <= 6, "unknown epilogue");
  MLR_REQUIRE(swiglu != 1 || (n % 4 == 0 && bias == nullptr && multiply == nullptr), "swiglu needs n % 4 == 0, no bias and no multiplier");
  MLR_REQUIRE(swiglu != 5 || (n % 4 == 0 && multiply == nullptr && glu_limit > 0.f),
              "the clamped gating needs n % 4 == 0, a limit > 0 and no multiplier");
  MLR_REQUIRE(swiglu != 6 || (n % 4 == 0 && multiply == nullptr), "the GELU gating needs n % 4 == 0 and no multiplier");
  MLR_REQUIRE(slices >= 1 && slices < 65536 && (slices == 1 || (swiglu == 0 && multiply == nullptr && m > 64)),
              "slices of k are plain sums of more than 64 tokens");
  const F32Epilogue ep{bias, y, swiglu, multiply, multiply_rows, glu_limit, glu_alpha};
  if (m <= 64) {
    const dim3 grid((n + 15) / 16);
    if (m <= 16)
      gemm_f32_few_kernel<1><<<grid, kFewWaves * 64, 0, stream>>>(x, w, ep, m, n, k);
    else if (m <= 32)
      gemm_f32_few_kernel<2><<<grid, kFewWaves * 64, 0, stream>>>(x, w, ep, m, n, k);
    else
      gemm_f32_few_kernel<4><<<grid, kFewWaves * 64, 0, stream>>>(x, w, ep, m, n, k);
  } else {
    MLR_REQUIRE((m + 63) / 64 < 65536, "too many rows for one launch");
    switch (f32_way(m, n, k, slices)) {
      case 0: launch_f32<2, 2, 1>(x, w, ep, m, n, k, slices, stream); break;
      case 1: launch_f32<2, 1, 1>(x, w, ep, m, n, k, slices, stream); break;
      case 2: launch_f32<2, 1, 2>(x, w, ep, m, n, k, slices, stream); break;
      case 3: launch_f32<1, 1, 1>(x, w, ep, m, n, k, slices, stream); break;
      default: launch_f32<1, 1, 2>(x, w, ep, m, n, k, slices, stream);
    }
  }
  MLR_LAUNCH_CHECK();
  return 0;
}
