// float32 matrix products on the matrix cores: y[M, N] = x[M, K] * w[N, K]^T (+ bias), the product of the true
// 32-bit path.  The matrix cores multiply and add float32 as it is (v_mfma_f32_32x32x2_f32, 16x16x4_f32: no rounding of the
// inputs), at 256 operations a clock and compute unit, twice what the vector unit's multiply-adds give without packed instructions.
//
//  * gemm_f32_tiled: more than 64 tokens.  Bound by the matrix cores: a tile of 64 x 64 takes 1,024 clocks of them per
//    32-wide step of k and 16 KB of operands, far from what LDS and L2 give, so the small tile costs nothing and goes round
//    the compute units best.  Tiles are loaded straight into LDS (rows of 32 floats are the 128 bytes of the bfloat16 kernels'
//    rows of 64, swizzled the same way), two steps on their way.  Narrow products whose consumer adds up partial sums are
//    cut along k.
//  * gemm_f32_few: up to 64 tokens.  Bound by streaming w once: 16 weight rows a workgroup, whose eight wavefronts split k and
//    add their sums through LDS.
// Measured at 0.5B sizes and 826 tokens, against the plain kernel (gemm_simple.hip, 64 x 64 tiles of vector multiply-adds with
// 16-wide steps through single-buffered LDS), microseconds: gate-up (9,728 x 896) 228 to 122 (118 TFLOP/s; the matrix cores at 2.4 GHz
// would take 92), down (896 x 4,864) 659 to 66 in four slices, query/key/value (1,152 x 896) 117 to 21; at 8 tokens gate-up 94 to
// 12, down 363 to 17, the output head 353 to 127.
//
// K must be a multiple of 4 and the operands 16-byte aligned; other shapes take the plain kernel.
#include "api.h"
#include "common.h"
#include "gemm_epilogue.h"
#include "mfma.h"

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
// Four wavefronts, one block of 32 features x 32 tokens each.  An operand read brings a lane 4 consecutive k of its row; product j
// of the four takes element j of every lane, so the lanes' halves stand for k = 8 g + j and 8 g + 4 + j: the same on both
// sides, and the order of k does not matter to a sum.
constexpr int kF32Step = 32;     // k per LDS slice
constexpr int kF32Buffers = 3;   // slices in LDS: one multiplied, two on their way (48 KB: three workgroups a compute unit; with four buffers two
                                 // fit, and 826 x 9728 x 896 takes 129 us instead of 122)
constexpr int kF32Tile = 64;
constexpr int kF32BufferBytes = 2 * kF32Tile * kF32Step * 4;

__global__ __launch_bounds__(256) void gemm_f32_tiled_kernel(const float* __restrict__ x, const float* __restrict__ w, F32Epilogue ep,
                                                             int M, int N, int K, int slices) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wn = wave % 2, wm = wave / 2;
  const int r32 = lane % 32, h = lane / 32;
  const int n0 = blockIdx.x * kF32Tile, m0 = blockIdx.y * kF32Tile;
  const int slice = blockIdx.z;
  const int k_steps = (K + kF32Step - 1) / kF32Step;
  const int per = (k_steps + slices - 1) / slices;
  const int s_begin = slice * per, s_end = min(k_steps, s_begin + per);
  const int chunks = K / 4;  // 16-byte pieces of a row

  const int w_rows = min(kF32Tile, N - n0), x_rows = min(kF32Tile, M - m0);
  const __amdgpu_buffer_rsrc_t w_buf = make_buffer(w + static_cast<int64_t>(n0) * K, static_cast<unsigned>(w_rows) * K * 4u);
  const __amdgpu_buffer_rsrc_t x_buf = make_buffer(x + static_cast<int64_t>(m0) * K, static_cast<unsigned>(x_rows) * K * 4u);
  // a wavefront's load fills a run of 8 rows: lane l brings row l / 8, piece (l % 8) ^ key to slot l % 8, key = (row / 2) % 8
  // (LDS serves two rows of 128 bytes side by side); run p * 4 + wave: the first 8 runs are weight rows, the others token rows
  const int lane_row = lane / 8;
  const int lane_chunk = (lane % 8) ^ ((4 * (wave % 2) + lane_row / 2) % 8);  // runs p * 4 + wave: 8 rows each, the key repeats every 16
  const unsigned row_off = static_cast<unsigned>(8 * wave + lane_row) * K * 4u + lane_chunk * 16u;
  auto fetch = [&](int s, int buf) {
    const unsigned ok = s < s_end && lane_chunk < chunks - s * (kF32Step / 4) ? 0u : kOutOfBuffer;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      __attribute__((address_space(3))) void* dst =
          (__attribute__((address_space(3))) void*)(smem + buf * kF32BufferBytes + (p * 4 + wave) * 1024);
      const unsigned off = (row_off + (p % 2) * 32u * K * 4u + s * (kF32Step * 4u)) | ok;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(p < 2 ? w_buf : x_buf, dst, 16, off, 0, 0, 0);
    }
  };

  f32x16_t acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  const int swz = (r32 / 2) % 8;
  const int a_base = (wn * 32 + r32) * (kF32Step * 4);
  const int b_base = (kF32Tile + wm * 32 + r32) * (kF32Step * 4);

#pragma unroll
  for (int b = 0; b < kF32Buffers - 1; ++b) fetch(s_begin + b, b);
  int buf = 0;
  for (int s = s_begin; s < s_end; ++s) {
    // this slice has landed (this wavefront's share; the barrier answers for the others), and everybody has multiplied the one before
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kF32Buffers - 2) * 4) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fetch(s + kF32Buffers - 1, (buf + kF32Buffers - 1) % kF32Buffers);  // into the buffer of the slice before
    const unsigned char* base = smem + buf * kF32BufferBytes;
    f32x4_t a[4], b[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int slot = ((g * 2 + h) ^ swz) * 16;
      a[g] = load_f32x4(base + a_base + slot);
      b[g] = load_f32x4(base + b_base + slot);
    }
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g][j], b[g][j], acc, 0, 0, 0);
    buf = (buf + 1) % kF32Buffers;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past the end have landed before LDS is given back

  const int m = m0 + wm * 32 + r32;
#pragma unroll
  for (int g = 0; g < 4; ++g)
    finish4_f32(ep, slice, slices, m, n0 + wn * 32 + g * 8 + h * 4, M, N,
                f32x4_t{acc[g * 4], acc[g * 4 + 1], acc[g * 4 + 2], acc[g * 4 + 3]});
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

// How many partial sums (slices of k) a product is cut into, when its consumer takes up to `max_slices`: more than 64 tokens whose
// tiles leave compute units idle or give a few of them two.  A workgroup is one 64 x 64 tile; three fit a compute
// unit.  Tiles are cut until 512 run, and a slice keeps at least 8 steps of k.  Measured in 1, 2, 4 and 8 slices, microseconds: 826 x 896 x 4,864 (182
// tiles) 92, 80, 66, 72; 826 x 896 x 896 21.0, 20.7, 20.2, 23.4; 65 x 896 x 4,864 (28 tiles) 92, 48, 27, 17; 2,048 x 896 x 4,864
// (448 tiles) 157, 155, 145, 157.
extern "C" int mlr_gemm_f32_slices(int m, int n, int k, int max_slices) {
  if (m <= 64) return 1;
  const int64_t tiles = static_cast<int64_t>((m + kF32Tile - 1) / kF32Tile) * ((n + kF32Tile - 1) / kF32Tile);
  const int steps = (k + kF32Step - 1) / kF32Step;
  int slices = 1;
  while (slices * 2 <= max_slices && tiles * slices < 512 && steps / (slices * 2) >= 8) slices *= 2;
  return slices;
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
    const dim3 grid((n + kF32Tile - 1) / kF32Tile, (m + kF32Tile - 1) / kF32Tile, slices);
    MLR_REQUIRE(grid.y < 65536u, "too many rows for one launch");
    gemm_f32_tiled_kernel<<<grid, 256, kF32Buffers * kF32BufferBytes, stream>>>(x, w, ep, m, n, k, slices);
  }
  MLR_LAUNCH_CHECK();
  return 0;
}
