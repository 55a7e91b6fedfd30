// float32 paged attention of prompt portions on the matrix cores, for one head size (MLR_HEAD_DIM, up to 80 and multiples of 32 up to 128): the
// true 32-bit counterpart of the tiled kernel in attention_mfma.hip, with the same page layouts and the same lane
// layouts (scores transposed, S^T[key, query], so that probabilities go from one product to the next in registers).
//
// v_mfma_f32_16x16x4_f32: D[16x16] += A[16x4] B[4x16].  Lane l holds A[row l % 16][k l / 16], B[k l / 16][col l % 16],
// D[row (l / 16) * 4 + i][col l % 16].  The order of k is free as long as both sides agree, so a lane reads 4 consecutive k
// (16 bytes) and product i of four takes element i of every lane.
//
// Bound by the matrix cores (256 operations a clock and compute unit in float32): a 64-key tile of 64 queries at head size 64 is
// 4,096 clocks of them for 32 KB of keys and values, which one LDS buffer with the next tile on its way in registers keeps up
// with; and for short prompts by the chain of tiles that the last queries see.  A workgroup takes 64 queries of one head; one group of four
// wavefronts, 16 queries each, takes all key tiles, or two take them in turn and add up at the end, which halves that chain (groups_for).
// Measured at 0.5B sizes (14 query and 2 key/value heads of 64), prompts of 391, 268, 145 and 22 tokens in one step: 479 us with the
// plain kernel (a wavefront per token and head, attention_simple.hip), 36 with one group and pages looked up beside the loads, 31 with
// pages looked up a turn ahead, 27 with two groups.  Error against 64 bits: with one group as with pages looked up beside the loads, bit for bit; with two the
// same up to 64 tokens and 2 to 22 % less beyond (65 to 2,048 tokens, all head sizes here).
#include "common.h"
#include "mfma.h"

#ifndef MLR_HEAD_DIM
#error "compile with -DMLR_HEAD_DIM=<multiple of 16>"
#endif

#if MLR_HEAD_DIM <= 80 || (MLR_HEAD_DIM <= 128 && MLR_HEAD_DIM % 32 == 0)  // whole pieces for every thread, see below
namespace mlr {
namespace f32_attention {

constexpr int D = MLR_HEAD_DIM;
constexpr int kDimTiles = D / 16;
constexpr int kTileQ = 64;                 // queries of a workgroup
constexpr int kTileK = D > 80 ? 32 : 64;   // keys of a group in LDS at a time
constexpr int kSubTiles = kTileK / 16;
// rows padded to 32 bytes modulo 64: 16 rows x 4 pieces of 16 bytes are then read without bank conflicts
constexpr int kKLd = D + 8;
constexpr int kVLd = kTileK + 8;
constexpr int kPieces = kTileK * D / 4 / 256;  // 16-byte pieces of a thread, of the key and of the value tile
constexpr int kGroupFloats = kTileK * kKLd + D * kVLd;  // LDS of a group: its keys, then its values
static_assert(kGroupFloats >= (2 + D / 4) * 256, "what the second group hands over fits its tiles");
static_assert(kTileK * D / 4 % 256 == 0, "whole pieces for every thread");

// One token's attention by a wavefront, as paged_attention_simple_kernel has it: a lane scores a key and then owns dims.  For the few workgroups
// that meet values which are not finite (see sm_odd).
__device__ void attend_alone(const float* __restrict__ q, int64_t q_stride, const float* __restrict__ key_pages,
                             const float* __restrict__ value_pages, const int* __restrict__ table, int table_width, int t, int p, int head,
                             int heads, int kvh, int kv_heads, int block_size, int num_pages, float scale, int window, int chunk,
                             const float* __restrict__ sinks, float* __restrict__ out) {
  constexpr int kOwn = (D + kWave - 1) / kWave;  // dims of a lane
  const int lane = threadIdx.x % kWave;
  const float* qrow = q + t * q_stride + static_cast<int64_t>(head) * D;
  float m = -INFINITY, l = 0.f, acc[kOwn];
#pragma unroll
  for (int j = 0; j < kOwn; ++j) acc[j] = 0.f;
  bool gone = false;
  for (int k0 = first_visible_key(p, window, chunk); k0 <= p; k0 += kWave) {
    const int key = k0 + lane;
    int place = -1;  // the key's page
    float s = -INFINITY;
    if (key <= p) {
      const int page = key / block_size < table_width ? table[key / block_size] : -1;
      if (static_cast<unsigned>(page) < static_cast<unsigned>(num_pages)) {
        place = page;
        const float* row = key_pages + ((static_cast<int64_t>(page) * kv_heads + kvh) * block_size + key % block_size) * D;
        s = 0.f;
        for (int i = 0; i < D; ++i) s = fmaf(qrow[i] * scale, row[i], s);
      } else {
        gone = true;
      }
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float weight = place >= 0 ? expf(s - m_new) : 0.f;
    const float alpha = m == -INFINITY ? 0.f : expf(m - m_new);
    l = l * alpha + wave_sum(weight);
    m = m_new;
#pragma unroll
    for (int j = 0; j < kOwn; ++j) acc[j] *= alpha;
    for (int i = 0; i < min(kWave, p - k0 + 1); ++i) {
      const int page = __shfl(place, i, kWave);
      const float w = __shfl(weight, i, kWave);
      if (page < 0) continue;
      const float* column = value_pages + (static_cast<int64_t>(page) * kv_heads + kvh) * D * block_size + (k0 + i) % block_size;
#pragma unroll
      for (int j = 0; j < kOwn; ++j)
        if (lane + j * kWave < D) acc[j] = fmaf(w, column[static_cast<int64_t>(lane + j * kWave) * block_size], acc[j]);
    }
  }
  float keep = 1.0f;
  if (sinks != nullptr) {
    const float m_new = fmaxf(m, sinks[head]);
    keep = m == -INFINITY ? 0.f : expf(m - m_new);
    l = l * keep + expf(sinks[head] - m_new);
  }
  const float inv = __any(gone) ? __builtin_nanf("") : keep / l;
  float* orow = out + (static_cast<int64_t>(t) * heads + head) * D;
#pragma unroll
  for (int j = 0; j < kOwn; ++j)
    if (lane + j * kWave < D) orow[lane + j * kWave] = acc[j] * inv;
}

__device__ __attribute__((aligned(16))) const float kGoneKeys[4] = {__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf("")};

// GROUPS: of four wavefronts, which take the key tiles in turn (see groups_for)
template <int GROUPS>
__global__ __launch_bounds__(256 * GROUPS) void attn_prefill_f32_kernel(
    const float* __restrict__ q, int64_t q_stride, const float* __restrict__ key_pages, const float* __restrict__ value_pages,
    const int* __restrict__ block_table, int table_width, const int* __restrict__ tiles, const int* __restrict__ cu_q,
    const int* __restrict__ context_lens, float* __restrict__ out, int heads, int kv_heads, int block_size, int num_pages,
    float scale, int window, int chunk, const float* __restrict__ sinks) {
  extern __shared__ __attribute__((aligned(16))) float tile_lds[];
  __shared__ int sm_odd;  // a value that is not finite has come in a tile of keys that some query here does not see whole
  const int tile = blockIdx.x / heads;
  const int head = blockIdx.x - tile * heads;
  const int kvh = head / (heads / kv_heads);
  const int entry = tiles[2 * tile];
  const int q0 = tiles[2 * tile + 1];
  const int group = GROUPS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / 256);
  const int tid = threadIdx.x % 256;  // of the group
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);  // of the group: 16 queries
  float* const ks = tile_lds + group * kGroupFloats;
  float* const vs = ks + kTileK * kKLd;
  const int col = lane % 16, quarter = lane / 16;
  const int t_first = cu_q[entry];
  const int q_len = cu_q[entry + 1] - t_first;
  const int pos0 = context_lens[entry] - q_len;
  const int* table = block_table + static_cast<int64_t>(entry) * table_width;
  if (threadIdx.x == 0) sm_odd = 0;

  const int qi = q0 + wave * 16 + col;
  const bool q_ok = qi < q_len;
  const int pq = pos0 + qi;
  const int pq_first = first_visible_key(pq, window, chunk);
  f32x4_t qo[kDimTiles];
  const float* qrow = q + static_cast<int64_t>(t_first + (q_ok ? qi : 0)) * q_stride + static_cast<int64_t>(head) * D;
#pragma unroll
  for (int g = 0; g < kDimTiles; ++g) {
    qo[g] = *reinterpret_cast<const f32x4_t*>(qrow + g * 16 + quarter * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) qo[g][j] *= scale;
  }

  const int k_end = pos0 + min(q0 + kTileQ, q_len);           // one past the last key that a query here sees
  const int k_first = first_visible_key(pos0 + q0, window, chunk);  // the first one
  const int w_last = pos0 + min(q0 + wave * 16 + 15, q_len - 1);
  const int w_first = first_visible_key(pos0 + q0 + wave * 16, window, chunk);
  const int w_max_first = first_visible_key(pos0 + q0 + wave * 16 + 15, window, chunk);
  const bool wave_has_queries = q0 + wave * 16 < q_len;

  f32x4_t k_flight[kPieces], v_flight[kPieces];
  // The pages of a tile's pieces are looked up a turn ahead of their loads (looked up beside them they would be a trip to memory that
  // everything waits for).  4 keys of a value piece lie in one page, whose size is a multiple of 4, and are the same for all of a thread's.
  int k_page[kPieces], v_page = -1;
  bool v_hidden[4] = {true, true, true, true};
  static_assert(256 % (kTileK / 4) == 0, "a thread's value pieces are of the same keys");
  auto page_of = [&](int key) {  // -1: past the table
    const int logical = min(key, k_end - 1) / block_size;
    const int page = table[min(logical, table_width - 1)];
    return logical < table_width ? page : -1;
  };
  auto lookup = [&](int kt0) {
    if (kt0 >= k_end) return;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) k_page[i] = page_of(kt0 + (tid + i * 256) / (D / 4));
    v_page = page_of(kt0 + tid % (kTileK / 4) * 4);
  };
  // A page that is not there (or lies past the table) brings keys that are NaN: so is the sum of every query that sees one, and of no other
  auto fetch = [&](int kt0) {
    if (kt0 >= k_end) return;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int c = tid + i * 256;
      const int key = kt0 + c / (D / 4), dim = c % (D / 4) * 4;
      const bool in = static_cast<unsigned>(k_page[i]) < static_cast<unsigned>(num_pages);
      const int64_t base = static_cast<int64_t>(in ? k_page[i] : 0) * kv_heads + kvh;
      const float* piece = key_pages + (base * block_size + key % block_size) * D + dim;
      k_flight[i] = *reinterpret_cast<const f32x4_t*>(in ? piece : kGoneKeys);  // (a choice behind the load would wait for it here)
    }
    const int key = kt0 + tid % (kTileK / 4) * 4;
    const bool in = static_cast<unsigned>(v_page) < static_cast<unsigned>(num_pages);
    const int64_t base = static_cast<int64_t>(in ? v_page : 0) * kv_heads + kvh;
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int dim = (tid + i * 256) / (kTileK / 4);
      v_flight[i] = *reinterpret_cast<const f32x4_t*>(value_pages + (base * D + dim) * block_size + key % block_size);
    }
    // values that no query here may see are cleared where they are put down: what a page holds there may be anything, and 0 * NaN would
    // come through
#pragma unroll
    for (int e = 0; e < 4; ++e) v_hidden[e] = !in || key + e >= k_end || key + e < k_first;
  };
  auto stash = [&]() {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int c = tid + i * 256;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (v_hidden[e]) v_flight[i][e] = 0.f;
      *reinterpret_cast<f32x4_t*>(ks + c / (D / 4) * kKLd + c % (D / 4) * 4) = k_flight[i];
      *reinterpret_cast<f32x4_t*>(vs + c / (kTileK / 4) * kVLd + c % (kTileK / 4) * 4) = v_flight[i];
    }
  };

  float m_run = -INFINITY, l_run = 0.f;
  f32x4_t acc[kDimTiles];
#pragma unroll
  for (int dt = 0; dt < kDimTiles; ++dt) acc[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  auto all_finite = [&]() {  // of the values that this thread brought
    float zero = 0.f;
#pragma unroll
    for (int i = 0; i < kPieces; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) zero = fmaf(v_flight[i][e], 0.f, zero);
    return zero == 0.f;
  };

  const int k_begin = k_first / kTileK * kTileK;
  const int k_all_first = first_visible_key(pos0 + q0 + kTileQ - 1, window, chunk);  // from here on no query here is past its window
  bool odd = false;
  constexpr int kTurn = GROUPS * kTileK;
  lookup(k_begin + group * kTileK);
  fetch(k_begin + group * kTileK);
  lookup(k_begin + group * kTileK + kTurn);
  for (int kt0 = k_begin + group * kTileK; kt0 - group * kTileK < k_end; kt0 += kTurn) {
    __syncthreads();  // everybody has done with the tile before
    const bool any = kt0 < k_end;  // the last turn may have no tile for the second group
    if (any) stash();
    // A hidden key's weight is 0, but 0 times an infinity or NaN is NaN, and the products would hand it to queries that do not see the key.
    const bool all_seen = kt0 + kTileK - 1 <= pos0 + q0 && kt0 >= k_all_first;
    if (any && !all_seen && !all_finite()) sm_odd = 1;
    __syncthreads();
    if (sm_odd != 0) {
      odd = true;
      break;
    }
    fetch(kt0 + kTurn);  // on its way while this tile is computed
    lookup(kt0 + 2 * kTurn);
    if (!(any && wave_has_queries && kt0 <= w_last && kt0 + kTileK > w_first)) continue;
    f32x4_t s[kSubTiles];
#pragma unroll
    for (int sub = 0; sub < kSubTiles; ++sub) {
      s[sub] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int g = 0; g < kDimTiles; ++g) {
        const f32x4_t k = *reinterpret_cast<const f32x4_t*>(ks + (sub * 16 + col) * kKLd + g * 16 + quarter * 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) s[sub] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j], qo[g][j], s[sub], 0, 0, 0);
      }
    }
    if (!(kt0 + kTileK - 1 <= pos0 + q0 + wave * 16 && kt0 >= w_max_first)) {  // some query here does not see all of it
#pragma unroll
      for (int sub = 0; sub < kSubTiles; ++sub)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = kt0 + sub * 16 + quarter * 4 + i;
          if (!(key <= pq && key >= pq_first)) s[sub][i] = -INFINITY;
        }
    }
    float top = -INFINITY;
#pragma unroll
    for (int sub = 0; sub < kSubTiles; ++sub)
#pragma unroll
      for (int i = 0; i < 4; ++i) top = fmaxf(top, s[sub][i]);
    top = fmaxf(top, __shfl_xor(top, 16, kWave));
    top = fmaxf(top, __shfl_xor(top, 32, kWave));
    const float m_new = fmaxf(m_run, top);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;  // a query that has seen no key yet
    const float alpha = m_run == -INFINITY ? 0.f : expf(m_run - m_use);
    float sum = 0.f;
#pragma unroll
    for (int sub = 0; sub < kSubTiles; ++sub)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[sub][i] = expf(s[sub][i] - m_use);
        sum += s[sub][i];
      }
    l_run = l_run * alpha + sum;
    m_run = m_new;
#pragma unroll
    for (int dt = 0; dt < kDimTiles; ++dt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[dt][i] *= alpha;
#pragma unroll
      for (int sub = 0; sub < kSubTiles; ++sub) {
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(vs + (dt * 16 + col) * kVLd + sub * 16 + quarter * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[i], s[sub][i], acc[dt], 0, 0, 0);
      }
    }
  }
  if (odd) {  // the same for the whole workgroup: its queries one after the other, each over the keys it sees
    for (int u = group; u < 16 && q0 + wave * 16 + u < q_len; u += GROUPS)
      attend_alone(q, q_stride, key_pages, value_pages, table, table_width, t_first + q0 + wave * 16 + u, pos0 + q0 + wave * 16 + u, head,
                   heads, kvh, kv_heads, block_size, num_pages, scale, window, chunk, sinks, out);
    return;
  }
  if (GROUPS > 1 && k_begin + kTileK < k_end) {  // the second group's share to the first: [component][thread]
    static_assert(GROUPS <= 2, "one group hands over");
    __syncthreads();
    float* const given = tile_lds + kGroupFloats;
    if (group > 0) {
      given[tid] = m_run;
      given[256 + tid] = l_run;
#pragma unroll
      for (int dt = 0; dt < kDimTiles; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) given[(2 + dt * 4 + i) * 256 + tid] = acc[dt][i];
    }
    __syncthreads();
    if (group > 0) return;
    const float m_other = given[tid];
    const float m_new = fmaxf(m_run, m_other);
    const float mine = m_run == -INFINITY ? 0.f : expf(m_run - m_new), other = m_other == -INFINITY ? 0.f : expf(m_other - m_new);
    l_run = l_run * mine + given[256 + tid] * other;
#pragma unroll
    for (int dt = 0; dt < kDimTiles; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[dt][i] = acc[dt][i] * mine + given[(2 + dt * 4 + i) * 256 + tid] * other;
    m_run = m_new;
  }
  if (group > 0) return;
  float l = l_run;
  l += __shfl_xor(l, 16, kWave);
  l += __shfl_xor(l, 32, kWave);
  float keep = 1.0f;
  if (sinks != nullptr) {  // one more term exp(sink) of the denominator, with no key and no value
    const float sink = sinks[head];
    const float m_new = fmaxf(m_run, sink);
    keep = m_run == -INFINITY ? 0.f : expf(m_run - m_new);
    l = l * keep + expf(sink - m_new);
  }
  if (!q_ok) return;
  const float inv = keep / l;
  float* orow = out + (static_cast<int64_t>(t_first + qi) * heads + head) * D;
#pragma unroll
  for (int dt = 0; dt < kDimTiles; ++dt) {
    f32x4_t v = acc[dt];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= inv;
    *reinterpret_cast<f32x4_t*>(orow + dt * 16 + quarter * 4) = v;
  }
}

template <int GROUPS>
static int launch_groups(const float* q, int64_t q_stride, const float* key_pages, const float* value_pages, const int* block_table, int table_width,
                         const int* tiles, int num_tiles, const int* cu_q, const int* context_lens, float* out, int heads, int kv_heads,
                         int block_size, int num_pages, float scale, int window, int chunk, const float* sinks, hipStream_t stream) {
  constexpr int kLdsBytes = GROUPS * kGroupFloats * 4;
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(attn_prefill_f32_kernel<GROUPS>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
    if (e != hipSuccess) {
      set_error(std::string("mlr_attention_prefill_f32: cannot raise the LDS limit: ") + hipGetErrorString(e));
      return -1;
    }
    configured = true;
  }
  attn_prefill_f32_kernel<GROUPS><<<dim3(static_cast<unsigned>(num_tiles) * heads), 256 * GROUPS, kLdsBytes, stream>>>(
      q, q_stride, key_pages, value_pages, block_table, table_width, tiles, cu_q, context_lens, out, heads, kv_heads, block_size,
      num_pages, scale, window, chunk, sinks);
  return 0;
}

// One group of wavefronts or two.  A second halves a workgroup's chain of key tiles and takes the LDS of a second workgroup: 8 wavefronts a
// workgroup and two of them on a unit up to head size 64, where four of one group are; one beyond, where three or four are.  So two while every
// workgroup can have a unit to itself, and beyond that where the longest prompt (`longest` tiles of queries, 0: not known) makes chains that end
// long after the others: its first tiles are short and leave early, its last ones are the step's end.  Microseconds, with one group and pages looked
// up beside the loads (as it was) / one / two, 16 query heads unless stated: 64, 32 and so on in the first column are head sizes.
//   64 (14 heads)  391, 268, 145 and 22 tokens 35.6 / 31.0 / 27.1, 2,048 tokens 185 / 165 / 146, 32 prompts of 64 12.1 / 11.5 / 12.2
//   64 (28 heads)  2,048 tokens (896 workgroups) 255 / 238 / 224, 32 prompts of 64 21.5 / 20.4 / 24.5, 8 of 300 (1,120) 70.6 / 66.0 / 62.9
//   80             391 tokens 40.8 / 35.9 / 32.3, 32 prompts of 64 (512) 16.2 / 14.9 / 21.4, 8 of 130 (384) 26.3 / 24.3 / 28.3, 2,048 behind a
//                  window of 64 (512) 24.8 / 22.5 / 27.0
//   96             1,024 tokens (256) 122 / 105 / 86, 4,096 (1,024) 792 / 774 / 815, 1,536 (384) 203 / 183 / 166
//   128            64 tokens 12.7 / 11.5 / 12.1, 391 57.5 / 50.5 / 44.5, 2,048 (28 heads, 896) 484 / 445 / 475, 4,096 (1,792) 1,642 / 1,465 / 1,625,
//                  32 prompts of 64 (28 heads, 896) 38.4 / 34.2 / 49.5, 1,024, 512, 256, 128 and 64 tokens (496) 166 / 123 / 105
//   16             32 prompts of 64 6.1 / 6.3 / 6.6, 8 of 520 (1,152) 40.8 / 41.2 / 45.3, 391 tokens 16.0 / 15.8 / 13.4, 4 of 1,024 (1,024) 79.7 / 80.4 / 59.4
static int groups_for(int num_tiles, int longest, int heads, int window, int chunk) {
  constexpr int kUnits = 256;
  constexpr bool kTwoFit = D <= 64;  // two workgroups of two groups on a unit
  const int64_t workgroups = static_cast<int64_t>(num_tiles) * heads;
  if (workgroups <= kUnits) return 2;
  const int span = window > 0 ? window : chunk;
  const int chain = span > 0 ? min(longest, span / kTileQ + 1) : longest;
  if (workgroups <= 2 * kUnits) return chain >= (kTwoFit ? 3 : 6) ? 2 : 1;
  return kTwoFit && chain >= (D > 16 ? 8 : 12) ? 2 : 1;
}

}  // namespace f32_attention
}  // namespace mlr

using namespace mlr;

// How many groups of wavefronts mlr_attention_prefill_f32 has for these sizes.
extern "C" int mlr_attention_prefill_f32_groups(int num_tiles, int longest, int heads, int window, int chunk) {
  return f32_attention::groups_for(num_tiles, longest, heads, window, chunk);
}

// Attention of the query tiles in `tiles` ([num_tiles][2]: entry, first query; 64 queries per tile) in float32, with the arguments
// of mlr_attention_prefill; longest: the most tiles of one entry, or 0.  A page id out of range makes the rows of the tokens that see its keys NaN, as in the plain kernel.
extern "C" int mlr_attention_prefill_f32(const float* q, int64_t q_stride, const float* key_pages, const float* value_pages,
                                         const int* block_table, int table_width, const int* tiles, int num_tiles, const int* cu_q,
                                         const int* context_lens, float* out, int heads, int kv_heads, int block_size, int num_pages,
                                         float scale, int window, int chunk, const float* sinks, int longest, hipStream_t stream) {
  MLR_REQUIRE(q && key_pages && value_pages && block_table && tiles && cu_q && context_lens && out, "null pointer");
  MLR_REQUIRE(num_tiles > 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "bad sizes");
  MLR_REQUIRE(block_size > 0 && block_size % 4 == 0, "block_size must be a multiple of 4");
  MLR_REQUIRE(num_pages > 0 && table_width > 0, "page sizes must be > 0");
  MLR_REQUIRE(q_stride >= static_cast<int64_t>(heads) * MLR_HEAD_DIM && q_stride % 4 == 0, "q_stride must cover a row and keep 16-byte alignment");
  MLR_REQUIRE(reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(key_pages) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(value_pages) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0,
              "operands must be 16-byte aligned");
  MLR_REQUIRE(scale > 0.f && scale < INFINITY && window >= 0 && chunk >= 0 && !(window > 0 && chunk > 0), "bad scale, window or chunk");
  MLR_REQUIRE(longest >= 0, "the longest prompt's tiles must be >= 0 (0: not known)");
  MLR_REQUIRE(static_cast<int64_t>(num_tiles) * heads < (1ll << 31), "too many tiles for one launch");
  const auto launch = f32_attention::groups_for(num_tiles, longest, heads, window, chunk) == 1 ? f32_attention::launch_groups<1> : f32_attention::launch_groups<2>;
  if (launch(q, q_stride, key_pages, value_pages, block_table, table_width, tiles, num_tiles, cu_q, context_lens, out, heads, kv_heads, block_size,
             num_pages, scale, window, chunk, sinks, stream) != 0)
    return -1;
  MLR_LAUNCH_CHECK();
  return 0;
}
#endif
