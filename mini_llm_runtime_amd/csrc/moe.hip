// Routed experts: which experts a token uses and with what weight, the (token, choice) pairs
// sorted by expert into row tiles, and the two grouped products over those tiles.  Nothing here
// comes back to the host between the router's logits and the weighted expert outputs, so a step
// with routed experts can be recorded and replayed like any other.
//
// A pair is p = token * top + choice.  `sorted` lists the pairs expert by expert, `offsets[e]` is
// where expert e's run starts, and a tile is (expert, first row of `sorted`): up to `tile_rows`
// pairs of one expert, which share that expert's weights in a product.  The order of the pairs
// inside an expert's run is whatever the atomics made it; every output row is computed from its own
// input row alone, with the sums over k in a fixed order, so no value depends on that order or on
// what else is in the batch.
#include "api.h"
#include "common.h"
#include "mfma.h"

namespace mlr {

// ---- routing ---------------------------------------------------------------------------------

__device__ __forceinline__ void wave_argmax(float& v, int& i) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float ov = __shfl_xor(v, off, kWave);
    const int oi = __shfl_xor(i, off, kWave);
    if (ov > v || (ov == v && oi < i)) {
      v = ov;
      i = oi;
    }
  }
}

// One wavefront per token.  s = sigmoid(z) (score_kind 0), softmax(z) over all experts (1) or z itself (2: the weights
// are then the softmax over the chosen z, times the scale), c = s + correction;
// with `normalise` the chosen weights are divided by their sum (+ 1e-20) before the scale.  Block g of experts / groups
// consecutive experts scores top-2 sum of its c; c := -inf outside the `keep` highest blocks; then
// `top` rounds of arg-max over c (ties to the lower index), each winner e leaving ids = e and
// weights = s[e] * scale.
__global__ __launch_bounds__(kWave) void moe_route_kernel(const float* __restrict__ logits, int slices,
                                                          const float* __restrict__ correction,
                                                          int* __restrict__ ids, float* __restrict__ weights, int tokens,
                                                          int experts, int top, int groups, int keep, float scale,
                                                          int score_kind, int normalise) {
  extern __shared__ float route_lds[];
  float* c = route_lds;            // [experts]
  float* s = route_lds + experts;  // [experts]
  float* gs = s + experts;         // [groups]
  const int t = blockIdx.x;
  const int lane = threadIdx.x;
  const int per = experts / groups;
  auto logit = [&](int e) {
    float z = 0.f;
    for (int p = 0; p < slices; ++p) z += logits[(static_cast<int64_t>(p) * tokens + t) * experts + e];
    return z;
  };
  float z_max = 0.f, z_inv = 1.f;
  if (score_kind == 1) {
    float mx = -INFINITY;
    for (int e = lane; e < experts; e += kWave) mx = fmaxf(mx, logit(e));
    z_max = wave_max(mx);
    float sum = 0.f;
    for (int e = lane; e < experts; e += kWave) sum += expf(logit(e) - z_max);
    z_inv = 1.0f / wave_sum(sum);
  }
  for (int e = lane; e < experts; e += kWave) {
    const float z = logit(e);
    const float sv = score_kind == 2 ? z : (score_kind == 1 ? expf(z - z_max) * z_inv : 1.0f / (1.0f + expf(-z)));
    s[e] = sv;
    c[e] = sv + (correction != nullptr ? correction[e] : 0.f);
  }
  __syncthreads();
  if (groups > 1 && keep < groups) {
    for (int g = lane; g < groups; g += kWave) {
      float a = -INFINITY, b = -INFINITY;  // running top-2 of the block
      for (int e = g * per; e < (g + 1) * per; ++e) {
        const float v = c[e];
        if (v > a) {
          b = a;
          a = v;
        } else if (v > b) {
          b = v;
        }
      }
      gs[g] = per > 1 ? a + b : a;
    }
    __syncthreads();
    // the kept groups get +inf as their mark, one after the other
    for (int k = 0; k < keep; ++k) {
      float v = -INFINITY;
      int i = 0x7fffffff;
      for (int g = lane; g < groups; g += kWave) {
        const float x = gs[g];
        if (x != INFINITY && (x > v || (x == v && g < i))) {
          v = x;
          i = g;
        }
      }
      wave_argmax(v, i);
      if (lane == 0 && i < groups) gs[i] = INFINITY;
      __syncthreads();
    }
    for (int e = lane; e < experts; e += kWave)
      if (gs[e / per] != INFINITY) c[e] = -INFINITY;
    __syncthreads();
  }
  float chosen_sum = 0.f;
  float z_top = 0.f;  // the first chosen logit: the largest
  for (int k = 0; k < top; ++k) {
    float v = -INFINITY;
    int i = 0x7fffffff;
    for (int e = lane; e < experts; e += kWave) {
      const float x = c[e];
      if (x > v || (x == v && e < i)) {
        v = x;
        i = e;
      }
    }
    wave_argmax(v, i);
    if (i >= experts) i = 0;  // only if every score left is NaN or -inf: keep the id in range
    if (k == 0) z_top = s[i];
    const float w = score_kind == 2 ? expf(s[i] - z_top) : s[i];
    chosen_sum += w;
    if (lane == 0) {
      ids[static_cast<int64_t>(t) * top + k] = i;
      weights[static_cast<int64_t>(t) * top + k] = w * scale;
      c[i] = -INFINITY;
    }
    __syncthreads();
  }
  if (normalise) {
    const float inv = 1.0f / (chosen_sum + 1e-20f);
    for (int k = lane; k < top; k += kWave) weights[static_cast<int64_t>(t) * top + k] *= inv;
  }
}

// The same for up to 64 R experts, 64 groups and 64 choices: a lane keeps R experts in registers (expert r * 64 + lane), a round of
// arg-max is a maximum over the wavefront by lane moves and a vote for the lowest index, and only the groups' top-2 sums go through
// LDS.  The logits may come as `slices` partial sums [slices, tokens, experts], added up in order.
// Bound by latency: the plain kernel's rounds go through LDS six times each.  64 experts in 8 groups, 6 choices: 8 tokens 10.5 to 4.7
// us, 2,000 tokens 13.3 to 6.9.
//
// This is token t's part, by one wavefront: it returns what lane j < top wrote as the token's j-th expert.  lds: R * 64 floats of this
// wavefront's own.  Every wavefront of the workgroup calls it (it has a barrier).
template <int R>
__device__ __forceinline__ int route_by_lanes(const float* __restrict__ logits, int slices, const float* __restrict__ correction,
                                              int* __restrict__ ids, float* __restrict__ weights, int tokens, int experts, int top,
                                              int groups, int keep, float scale, int score_kind, int normalise, int t, float* lds) {
  const int lane = threadIdx.x % kWave;
  float z[R], s[R], c[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int e = r * kWave + lane;
    z[r] = 0.f;
    for (int p0 = 0; p0 < slices; p0 += 8) {  // eight on their way at once
      float part[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        part[u] = logits[(static_cast<int64_t>(min(p0 + u, slices - 1)) * tokens + t) * experts + min(e, experts - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u) z[r] += p0 + u < slices ? part[u] : 0.f;
    }
  }
  float z_max = 0.f, z_inv = 1.f;
  if (score_kind == 1) {
    float mx = -INFINITY, sum = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (r * kWave + lane < experts) mx = fmaxf(mx, z[r]);
    z_max = wave_max(mx);
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (r * kWave + lane < experts) sum += expf(z[r] - z_max);
    z_inv = 1.0f / wave_sum(sum);
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int e = r * kWave + lane;
    s[r] = score_kind == 2 ? z[r] : (score_kind == 1 ? expf(z[r] - z_max) * z_inv : 1.0f / (1.0f + expf(-z[r])));
    c[r] = s[r] + (correction != nullptr && e < experts ? correction[e] : 0.f);
  }
  // the lowest index among the largest of v[r] (index index(r), below `count`); NaN never wins; `count` if there is none
  auto arg_max = [&](const float(&v)[R], int count, float& best) {
    float mine = -INFINITY;
    int index = 0x7fffffff;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = r * kWave + lane;
      if (e < count && (v[r] > mine || (v[r] == mine && e < index))) {
        mine = v[r];
        index = e;
      }
    }
    best = wave_max(mine);
    int found = count;
#pragma unroll
    for (int r = R - 1; r >= 0; --r) {
      const unsigned long long lanes = __ballot(index == r * kWave + lane && mine == best);
      if (lanes != 0) found = r * kWave + __ffsll(lanes) - 1;
    }
    return found;
  };
  const int per = experts / groups;
  if (groups > 1 && keep < groups) {
#pragma unroll
    for (int r = 0; r < R; ++r) lds[r * kWave + lane] = c[r];
    __syncthreads();
    float gs[R];
#pragma unroll
    for (int r = 0; r < R; ++r) gs[r] = -INFINITY;
    if (lane < groups) {
      float a = -INFINITY, b = -INFINITY;  // running top-2 of the block
#pragma unroll 8
      for (int i = 0; i < per; ++i) {
        const float v = lds[lane * per + i];
        if (v > a) {
          b = a;
          a = v;
        } else if (v > b) {
          b = v;
        }
      }
      gs[0] = per > 1 ? a + b : a;
    }
    unsigned long long kept = 0;
    bool mine_kept = lane >= groups;  // groups that are kept already, or do not exist, are out of the choice
    for (int k = 0; k < keep; ++k) {
      const float v = mine_kept ? __builtin_nanf("") : gs[0];
      float one[R];
#pragma unroll
      for (int r = 0; r < R; ++r) one[r] = r == 0 ? v : __builtin_nanf("");
      float best;
      const int g = arg_max(one, groups, best);
      if (g >= groups) break;  // only NaN left
      kept |= 1ull << g;
      mine_kept = mine_kept || lane == g;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int e = r * kWave + lane;
      if (e < experts && !((kept >> (e / per)) & 1)) c[r] = -INFINITY;
    }
  }
  float chosen_sum = 0.f, z_top = 0.f, my_weight = 0.f;
  int my_id = 0;
  for (int k = 0; k < top; ++k) {
    float best;
    int i = arg_max(c, experts, best);
    if (i >= experts) i = 0;  // only if every score left is NaN: keep the id in range
    float si = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (i / kWave == r) si = lane_value(s[r], i % kWave);
      if (i == r * kWave + lane) c[r] = -INFINITY;
    }
    if (k == 0) z_top = si;
    const float w = score_kind == 2 ? expf(si - z_top) : si;
    chosen_sum += w;
    if (lane == k) {
      my_id = i;
      my_weight = w * scale;
    }
  }
  if (lane < top) {
    ids[static_cast<int64_t>(t) * top + lane] = my_id;
    weights[static_cast<int64_t>(t) * top + lane] = normalise ? my_weight * (1.0f / (chosen_sum + 1e-20f)) : my_weight;
  }
  return my_id;
}

template <int R>
__global__ __launch_bounds__(kWave) void moe_route_lanes_kernel(const float* __restrict__ logits, int slices,
                                                                const float* __restrict__ correction, int* __restrict__ ids,
                                                                float* __restrict__ weights, int tokens, int experts, int top,
                                                                int groups, int keep, float scale, int score_kind, int normalise) {
  __shared__ float lds[R * kWave];
  route_by_lanes<R>(logits, slices, correction, ids, weights, tokens, experts, top, groups, keep, scale, score_kind, normalise,
                    static_cast<int>(blockIdx.x), lds);
}

// Experts that hand their input on: where ids[t, j] >= first (such an expert has no matrices and the grouped
// products skip its pairs) out[j, t, :] = weights[t, j] * h[t, :].  One workgroup per pair.
template <typename T>
__global__ __launch_bounds__(256) void moe_identity_kernel(const T* __restrict__ h, const int* __restrict__ ids,
                                                           const float* __restrict__ weights, float* __restrict__ out,
                                                           int tokens, int top, int hidden, int first) {
  const int pair = blockIdx.x;
  if (ids[pair] < first) return;
  const int t = pair / top;
  const int j = pair - t * top;
  const float w = weights[pair];
  const T* src = h + static_cast<int64_t>(t) * hidden;
  float* dst = out + (static_cast<int64_t>(j) * tokens + t) * hidden;
  for (int i = threadIdx.x; i < hidden; i += 256) dst[i] = w * to_f32(src[i]);
}

// ---- pairs sorted by expert ------------------------------------------------------------------

// One workgroup.  counts -> offsets and tiles (the first wavefront) -> placement.  counts (cleared, behind a barrier) and start: LDS,
// [experts]; totals: LDS, the used tiles and the pairs with an expert here; count adds every pair of an expert with matrices to its expert's count, place writes where the pairs are once `start` is known.
// What the count returned is the pair's place among its expert's: who keeps it needs neither the ids nor the atomics a second time.
template <class Count, class Place>
__device__ __forceinline__ void align_pairs(int experts, int tile_rows, int max_tiles, int* counts, int* start, int* totals,
                                            int* __restrict__ sorted, int* __restrict__ offsets, int* __restrict__ tiles,
                                            const Count& count, const Place& place) {
  const int tid = threadIdx.x;
  count();
  __syncthreads();
  if (tid < kWave) {  // the first wavefront: where every expert's run and tiles start, 64 experts at a time
    int at = 0, nt = 0;
    for (int e0 = 0; e0 < experts; e0 += kWave) {
      const int e = e0 + tid;
      const int n = e < experts ? counts[e] : 0;
      const int mine = (n + tile_rows - 1) / tile_rows;
      int rows_upto = n, tiles_upto = mine;  // running sums over the lanes
#pragma unroll
      for (int off = 1; off < kWave; off *= 2) {
        const int r = __shfl_up(rows_upto, off, kWave), t = __shfl_up(tiles_upto, off, kWave);
        if (tid >= off) {
          rows_upto += r;
          tiles_upto += t;
        }
      }
      const int row0 = at + rows_upto - n;
      const int tile0 = nt + tiles_upto - mine;
      if (e < experts) {
        offsets[e] = row0;
        start[e] = row0;
        for (int i = 0; i < mine && tile0 + i < max_tiles; ++i) {
          tiles[2 * (tile0 + i)] = e;
          tiles[2 * (tile0 + i) + 1] = row0 + i * tile_rows;
        }
      }
      at += __shfl(rows_upto, kWave - 1, kWave);
      nt += __shfl(tiles_upto, kWave - 1, kWave);
    }
    if (tid == 0) {
      offsets[experts] = at;
      totals[0] = min(nt, max_tiles);
      totals[1] = at;
    }
  }
  __syncthreads();
  for (int i = totals[0] + tid; i < max_tiles; i += blockDim.x) {
    tiles[2 * i] = -1;  // a workgroup that finds this has nothing to do
    tiles[2 * i + 1] = totals[0];
  }
  place();
}

// KEPT: pairs that a thread keeps, their experts and places, in registers; they are put in order in LDS and leave in whole lines (a wavefront's
// 64 places are as many lines).  0: any number of pairs and experts, read and counted twice.
// In a replayed graph, 64 experts, 0 / 4 or 16, microseconds: 192 pairs 2.9 / 2.5, 1,024 3.7 / 2.7, 3,072
// 4.6 / 3.2, 6,144 5.9 / 4.8, 12,000 8.7 / 5.2, 16,384 10.7 / 6.1; 8 experts, 12,000 8.9 / 6.7; 256, 16,000 14.4 / 8.5.
constexpr int kKeptExperts = 2048;  // 16 KB of counts and starts beside up to 32 KB of pairs
template <int KEPT>
__global__ __launch_bounds__(1024) void moe_align_kernel(const int* __restrict__ ids, int pairs, int experts,
                                                         int tile_rows, int max_tiles, int* __restrict__ sorted,
                                                         int* __restrict__ offsets, int* __restrict__ tiles) {
  extern __shared__ int align_lds[];
  int* counts = align_lds;            // [experts]
  int* start = align_lds + experts;   // [experts]
  __shared__ int totals[2];
  const int tid = threadIdx.x;
  for (int e = tid; e < experts; e += blockDim.x) counts[e] = 0;
  __syncthreads();
  if constexpr (KEPT > 0) {
    unsigned short* in_order = reinterpret_cast<unsigned short*>(start + experts);  // [pairs]
    int held[KEPT > 0 ? KEPT : 1];  // place * 4,096 + expert, or -1
    align_pairs(
        experts, tile_rows, max_tiles, counts, start, totals, sorted, offsets, tiles,
        [&] {
#pragma unroll
          for (int u = 0; u < KEPT; ++u) held[u] = u * 1024 + tid < pairs ? ids[u * 1024 + tid] : -1;
#pragma unroll
          for (int u = 0; u < KEPT; ++u) {
            const int e = held[u];
            held[u] = e >= 0 && e < experts ? atomicAdd(&counts[e], 1) * 4096 + e : -1;
          }
        },
        [&] {
#pragma unroll
          for (int u = 0; u < KEPT; ++u)
            if (held[u] >= 0) in_order[start[held[u] % 4096] + held[u] / 4096] = static_cast<unsigned short>(u * 1024 + tid);
          __syncthreads();
          for (int i = tid; i < totals[1]; i += 1024) sorted[i] = in_order[i];
        });
  } else {
    // eight ids of a thread are asked for at once: one after the other each would be a trip to L2
    auto for_each_pair = [&](auto&& use) {
      for (int p0 = tid; p0 < pairs; p0 += 8 * 1024) {
        int e[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) e[u] = ids[min(p0 + u * 1024, pairs - 1)];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (p0 + u * 1024 < pairs && e[u] >= 0 && e[u] < experts) use(p0 + u * 1024, e[u]);
      }
    };
    align_pairs(
        experts, tile_rows, max_tiles, counts, start, totals, sorted, offsets, tiles,
        [&] { for_each_pair([&](int, int e) { atomicAdd(&counts[e], 1); }); },
        [&] {
          for (int e = tid; e < experts; e += blockDim.x) counts[e] = 0;
          __syncthreads();
          for_each_pair([&](int p, int e) { sorted[start[e] + atomicAdd(&counts[e], 1)] = p; });
        });
  }
}

// Both at once for up to 8 tokens: a workgroup with a wavefront for each.  A launch is most of what either costs: 64 experts in 8
// groups, 6 choices, in a replayed graph the two / this one: 1 token 6.9 / 5.0 us, 8 tokens 7.3 / 5.9, 16 7.3 / 7.5.
constexpr int kRouteAlignTokens = 8;
template <int R>
__global__ __launch_bounds__(kRouteAlignTokens* kWave) void moe_route_align_kernel(
    const float* __restrict__ logits, int slices, const float* __restrict__ correction, int* __restrict__ ids, float* __restrict__ weights,
    int tokens, int routed, int top, int groups, int keep, float scale, int score_kind, int normalise, int experts, int tile_rows, int max_tiles,
    int* __restrict__ sorted, int* __restrict__ offsets, int* __restrict__ tiles) {
  __shared__ float lds[kRouteAlignTokens][R * kWave];
  __shared__ int counts[R * kWave], start[R * kWave], totals[2];
  const int t = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  for (int e = threadIdx.x; e < R * kWave; e += blockDim.x) counts[e] = 0;
  const int id = route_by_lanes<R>(logits, slices, correction, ids, weights, tokens, routed, top, groups, keep, scale, score_kind, normalise, t, lds[t]);
  __syncthreads();
  const bool counted = lane < top && id < experts;
  int among = 0;
  align_pairs(
      experts, tile_rows, max_tiles, counts, start, totals, sorted, offsets, tiles,
      [&] {
        if (counted) among = atomicAdd(&counts[id], 1);
      },
      [&] {
        if (counted) sorted[start[id] + among] = t * top + lane;
      });
}

// ---- the clamped gating in a grouped product's epilogue ------------------------------------------------
// v: the sums of rows gate 2j, gate 2j + 1, up 2j, up 2j + 1 of an expert's first matrix, woven in pairs.  g * sigmoid(alpha
// g) * (u + 1) with g = min(gate, limit), u = clamp(up, -limit, limit).  PRECISE: the float32 engine's exponential.
template <bool PRECISE>
__device__ __forceinline__ float clamped_gate(float gate, float up, float limit, float alpha) {
  const float g = fminf(gate, limit);
  const float u = fminf(fmaxf(up, -limit), limit);
  const float e = PRECISE ? expf(-alpha * g) : __expf(-alpha * g);
  return g / (1.0f + e) * (u + 1.0f);
}

__device__ __forceinline__ void store_clamped_glu(bf16* dst, const float (&v)[4], float limit, float alpha) {
  *reinterpret_cast<uint32_t*>(dst) = pack_bf16x2(clamped_gate<false>(v[0], v[2], limit, alpha),
                                                  clamped_gate<false>(v[1], v[3], limit, alpha));
}

// ---- grouped products, plain 32-bit FMA arithmetic -----------------------------------------------
//
// UP:   act[row, n]  = f(sum_k h[token(row), k] * w[e, n, k])                  (rows in sorted order; with the
//       clamped gating (act 5) N woven rows make N / 2 activations)
// DOWN: out[choice(row), token(row), n] = weight[pair(row)] * sum_k act[row, k] * w[e, n, k]
// A workgroup owns 16 rows of one tile and 64 features; K in slices of 16 through LDS.

constexpr int kMoeRows = 16;
constexpr int kMoeCols = 64;
constexpr int kMoeK = 16;

template <typename T, bool UP>
__global__ __launch_bounds__(256) void moe_gemm_simple_kernel(const T* __restrict__ a, const T* __restrict__ w,
                                                              const int* __restrict__ sorted,
                                                              const int* __restrict__ offsets,
                                                              const int* __restrict__ tiles,
                                                              const float* __restrict__ pair_weights,
                                                              void* __restrict__ out, int tokens, int top, int N,
                                                              int K, int act, float glu_limit, float glu_alpha) {
  const int expert = tiles[2 * blockIdx.x];
  if (expert < 0) return;
  const int row0 = tiles[2 * blockIdx.x + 1];
  const int row_end = offsets[expert + 1];
  __shared__ float xs[kMoeK][kMoeRows + 1];
  __shared__ float ws[kMoeK][kMoeCols + 4];
  __shared__ int pair_of[kMoeRows];
  const int tid = threadIdx.x;
  if (tid < kMoeRows) pair_of[tid] = row0 + tid < row_end ? sorted[row0 + tid] : -1;
  __syncthreads();
  const int tm = tid / 16;  // row of the tile
  const int tn = tid % 16;  // features tn * 4 .. tn * 4 + 3
  const int n0 = blockIdx.y * kMoeCols;
  const T* wbase = w + static_cast<int64_t>(expert) * N * K;
  // the row of `a` this thread stages (one element per slice)
  const int lrow = tid / kMoeK;
  const int lk = tid % kMoeK;
  const int lpair = pair_of[lrow];
  const T* arow = nullptr;
  if (lpair >= 0) arow = UP ? a + static_cast<int64_t>(lpair / top) * K : a + static_cast<int64_t>(row0 + lrow) * K;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += kMoeK) {
    xs[lk][lrow] = (arow != nullptr && k0 + lk < K) ? to_f32(arow[k0 + lk]) : 0.f;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int idx = tid + it * 256;
      const int col = idx / kMoeK;
      const int kk = idx % kMoeK;
      const int gn = n0 + col;
      ws[kk][col] = (gn < N && k0 + kk < K) ? to_f32(wbase[static_cast<int64_t>(gn) * K + k0 + kk]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < kMoeK; ++kk) {
      const float x = xs[kk][tm];
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = fmaf(x, ws[kk][tn * 4 + j], acc[j]);
    }
    __syncthreads();
  }
  const int pair = pair_of[tm];
  if (pair < 0) return;
  const int token = pair / top;
  const int choice = pair - token * top;
  if (UP && act == 5) {
    const int gn = n0 + tn * 4;
    if (gn >= N) return;  // N is a multiple of 4 here
    T* dst = static_cast<T*>(out) + static_cast<int64_t>(row0 + tm) * (N / 2) + gn / 2;
    dst[0] = from_f32<T>(clamped_gate<true>(acc[0], acc[2], glu_limit, glu_alpha));
    dst[1] = from_f32<T>(clamped_gate<true>(acc[1], acc[3], glu_limit, glu_alpha));
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int gn = n0 + tn * 4 + j;
    if (gn >= N) continue;
    float v = acc[j];
    if (UP) {
      if (act == 2) {
        v = fmaxf(v, 0.f);
        v *= v;
      } else if (act == 3) {
        v = 1.0f / (1.0f + expf(-v));
      }
      static_cast<T*>(out)[static_cast<int64_t>(row0 + tm) * N + gn] = from_f32<T>(v);
    } else {
      static_cast<float*>(out)[(static_cast<int64_t>(choice) * tokens + token) * N + gn] = pair_weights[pair] * v;
    }
  }
}

// ---- grouped products in bfloat16 on the matrix cores ---------------------------------------------
//
// The same two products, two kernels.
//
// Streaming (tiles of 16 rows; decoding, where an expert sees a few rows): a workgroup of four
// wavefronts owns 16 rows of a tile (the columns of the 16 x 16 x 32 block; weights are the row
// operand, as in the other product kernels) and 64 features, 16 per wavefront.  A lane reads 8
// consecutive k of one weight row and of one input row per block, both straight from memory through
// range-checked buffer loads (rows past the tile's end, features past N and k past K read zeros, no
// branch around a load), eight blocks in flight before the first product: the kernel's time is the
// expert weights it streams, read once (non-temporal).
constexpr int kMoeDepth = 8;

// The offset that stands for no row of the input, and for k past its end: at or past the end of any input below 4 GB whose rows are whole
// pieces of 16 bytes.  (An expert's matrix stays below 2 GB, where kOutOfBuffer serves.)
constexpr unsigned kNoRow = 0xfffffff0u;

template <bool UP>
__global__ __launch_bounds__(256) void moe_gemm_mfma_kernel(const bf16* __restrict__ a, const bf16* __restrict__ w,
                                                            const int* __restrict__ sorted,
                                                            const int* __restrict__ offsets,
                                                            const int* __restrict__ tiles,
                                                            const float* __restrict__ pair_weights,
                                                            void* __restrict__ out, int tokens, int top, int N, int K,
                                                            int act, int a_rows, float glu_limit, float glu_alpha) {
  const int expert = tiles[2 * blockIdx.x];
  if (expert < 0) return;
  const int row0 = tiles[2 * blockIdx.x + 1];
  const int row_end = offsets[expert + 1];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int col = lane % 16;   // operand row: weight row / input row of the tile
  const int quad = lane / 16;  // which 8 of a block's 32 k
  const int n_base = (blockIdx.y * (blockDim.x / kWave) + wave) * 16;  // 16 features a wavefront
  if (n_base >= N) return;
  // the input row this lane loads (as the column operand), and the rows whose sums it ends up with
  const int in_row = row0 + col;
  const int in_pair = in_row < row_end ? sorted[in_row] : -1;
  const int a_row = in_pair < 0 ? -1 : (UP ? in_pair / top : in_row);
  const unsigned row_bytes = static_cast<unsigned>(K) * 2u;
  const __amdgpu_buffer_rsrc_t wbuf =
      make_buffer(w + static_cast<int64_t>(expert) * N * K, static_cast<unsigned>(N) * row_bytes);
  const __amdgpu_buffer_rsrc_t abuf = make_buffer(a, static_cast<unsigned>(a_rows) * row_bytes);
  const int wn = n_base + col;
  const unsigned w_off = wn < N ? static_cast<unsigned>(wn) * row_bytes : kOutOfBuffer;
  const unsigned a_off = a_row >= 0 ? static_cast<unsigned>(a_row) * row_bytes : kNoRow;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int kb = 0; kb < K; kb += 32 * kMoeDepth) {
    bf16x8_t wv[kMoeDepth], xv[kMoeDepth];
#pragma unroll
    for (int u = 0; u < kMoeDepth; ++u) {
      const int k = kb + u * 32 + quad * 8;
      const unsigned koff = static_cast<unsigned>(k) * 2u;
      const bool in = k < K;
      wv[u] = buffer_load_bf16x8_once(wbuf, in && w_off != kOutOfBuffer ? w_off + koff : kOutOfBuffer);
      xv[u] = buffer_load_bf16x8(abuf, in && a_off != kNoRow ? a_off + koff : kNoRow);
    }
#pragma unroll
    for (int u = 0; u < kMoeDepth; ++u) acc = mfma_16x16x32(wv[u], xv[u], acc);
  }
  // acc[i]: feature n_base + quad * 4 + i of tile row `col`
  if (in_pair < 0) return;
  const int token = in_pair / top;
  const int choice = in_pair - token * top;
  const int n = n_base + quad * 4;
  if (UP && act == 5) {
    const float v[4] = {acc[0], acc[1], acc[2], acc[3]};
    if (n < N) store_clamped_glu(static_cast<bf16*>(out) + static_cast<int64_t>(in_row) * (N / 2) + n / 2, v, glu_limit, glu_alpha);
  } else if (UP) {
    bf16* dst = static_cast<bf16*>(out) + static_cast<int64_t>(in_row) * N + n;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = acc[i];
      if (act == 2) {
        v = fmaxf(v, 0.f);
        v *= v;
      } else if (act == 3) {
        v = 1.0f / (1.0f + __expf(-v));
      }
      if (n + i < N) dst[i] = f32_to_bf16(v);
    }
  } else {
    const float pw = pair_weights[in_pair];
    float* dst = static_cast<float*>(out) + (static_cast<int64_t>(choice) * tokens + token) * N + n;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < N) dst[i] = pw * acc[i];
  }
}

// Streaming through LDS (tiles of 16 rows, as above): the same work with loads that cover whole lines.
// A workgroup owns 16 rows of a tile and 64 features; k in slices of STEP, loaded straight into four LDS buffers, three of them
// on their way.  Neighbouring lanes fetch the contiguous bytes that a slice holds of one weight row, one or two lines (the kernel above
// reads 64 bytes of 16 different rows per instruction, which streams a large matrix at little more than half the rate); the 16-byte pieces of a
// row lie in another order from row to row, so that the operand reads of sixteen rows fall on different banks.  Wavefront w multiplies
// features w * 16 .. + 16.
// STEP 128: 80 KB, two workgroups a compute unit with 48 KB of weights each on their way; 64: 40 KB, four with 24.  The first has
// the whole stream under way with few workgroups, the second loses less at the end of a round of many; see narrow_steps_pay.
// Bound by HBM and by how long a launch takes to begin and end: 8 tokens, 64 experts with 6 choices, matrices of 768 x 2,048: 13 experts chosen up
// 15.0 us, down 9.6, 34 (107 MB each) 21.9 and 23.2, 48 33 and 27; a plain product of 16 tokens takes 20 to 21 us for 100 MB.  (The input
// rows by a wavefront of their own, so that the weights never wait for their lookup: 0.5 us less each, nothing in a step.)
constexpr int kStCols = 64;
constexpr int kStBuffers = 4;
constexpr int stream_buffer_bytes(int step) { return (kStCols + kMoeRows) * step * 2; }
constexpr int stream_lds_bytes(int step) { return kStBuffers * stream_buffer_bytes(step); }

template <bool UP, int STEP>
__global__ __launch_bounds__(256) void moe_gemm_stream_kernel(const bf16* __restrict__ a, const bf16* __restrict__ w,
                                                              const int* __restrict__ sorted,
                                                              const int* __restrict__ offsets,
                                                              const int* __restrict__ tiles,
                                                              const float* __restrict__ pair_weights,
                                                              void* __restrict__ out, int tokens, int top, int N, int K,
                                                              int act, int a_rows, float glu_limit, float glu_alpha) {
  constexpr int kRowLanes = STEP / 8;             // lanes that bring a row's piece of a slice, 16 bytes each
  constexpr int kRunRows = kWave / kRowLanes;     // rows of a load (1 KB)
  constexpr int kWeightRuns = kStCols / kRunRows / 4, kInputRuns = kMoeRows / kRunRows;
  constexpr int kBuffer = stream_buffer_bytes(STEP);
  // Workgroups go to the eight dies in turn and the unused tiles lie at the end of the list: where a tile would be on the same die for every
  // run of features, each run starts at another tile (35 of 48 tiles used: five on some dies, four on others).
  const int tile = gridDim.x % 8 == 0 ? (blockIdx.x + blockIdx.y) % gridDim.x : blockIdx.x;
  const int expert = tiles[2 * tile];
  if (expert < 0) return;
  const int row0 = tiles[2 * tile + 1];
  const int row_end = offsets[expert + 1];
  extern __shared__ __attribute__((aligned(16))) unsigned char moe_lds[];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int n0 = blockIdx.y * kStCols;
  const unsigned row_bytes = static_cast<unsigned>(K) * 2u;
  const __amdgpu_buffer_rsrc_t wbuf =
      make_buffer(w + static_cast<int64_t>(expert) * N * K, static_cast<unsigned>(N) * row_bytes);
  const __amdgpu_buffer_rsrc_t abuf = make_buffer(a, static_cast<unsigned>(a_rows) * row_bytes);
  // This wavefront brings runs `wave`, `wave` + 4, ... of the weights and, where there are as many, run `wave` of the input tile; what
  // orders a row's pieces is the same for all of them, so is the piece that this lane brings
  auto order_of = [](int row) { return STEP == 128 ? row % 16 : row / 2 % 8; };
  const int my_row = kRunRows * wave + lane / kRowLanes;
  const int piece = (lane % kRowLanes) ^ order_of(my_row);
  unsigned w_off[4];  // loops over the runs go to 4 and break, see moe_gemm_tiled_kernel
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = n0 + i * 4 * kRunRows + my_row;
    w_off[i] = row < N ? static_cast<unsigned>(row) * row_bytes + piece * 16u : kOutOfBuffer;
  }
  const int my_pair = sorted[min(row0 + my_row, row_end - 1)];
  const int slices = (K + STEP - 1) / STEP;
  unsigned x_off = 0;
  auto fetch_weights = [&](int slice, int buf) {
    const unsigned koff = static_cast<unsigned>(slice) * STEP * 2u;
    const bool in = slice < slices && slice * STEP + piece * 8 < K;
    unsigned char* const dst = moe_lds + buf * kBuffer + wave * 1024;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i >= kWeightRuns) break;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wbuf, (__attribute__((address_space(3))) void*)(dst + i * 4096), 16,
                                               in && w_off[i] != kOutOfBuffer ? w_off[i] + koff : kOutOfBuffer, 0, 0, 2);
    }
  };
  auto fetch_rows = [&](int slice, int buf) {
    if (wave >= kInputRuns) return;
    const bool in = slice < slices && slice * STEP + piece * 8 < K && x_off != kNoRow;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        abuf, (__attribute__((address_space(3))) void*)(moe_lds + buf * kBuffer + kStCols * STEP * 2 + wave * 1024), 16,
        in ? x_off + static_cast<unsigned>(slice) * STEP * 2u : kNoRow, 0, 0, 0);
  };
  // the weights do not wait for the lookup of the rows
#pragma unroll
  for (int s = 0; s < kStBuffers - 1; ++s) fetch_weights(s, s);
  x_off = row0 + my_row < row_end ? static_cast<unsigned>(UP ? my_pair / top : row0 + my_row) * row_bytes + piece * 16u : kNoRow;
#pragma unroll
  for (int s = 0; s < kStBuffers - 1; ++s) fetch_rows(s, s);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // they were sent together and arrive together; from here on slices are waited for one by one
  const int col = lane % 16;
  const int quad = lane / 16;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < slices; ++s) {
    // this slice has landed (this wavefront's share; the barrier answers for the others), and everybody has multiplied the one before
    if (wave < kInputRuns)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kStBuffers - 2) * (kWeightRuns + 1)) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kStBuffers - 2) * kWeightRuns) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fetch_weights(s + kStBuffers - 1, (s + kStBuffers - 1) % kStBuffers);
    fetch_rows(s + kStBuffers - 1, (s + kStBuffers - 1) % kStBuffers);  // into the buffer of the slice before
    const unsigned char* const base = moe_lds + s % kStBuffers * kBuffer;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks >= STEP / 32) break;
      const int slot = ((ks * 4 + quad) ^ order_of(col)) * 16;
      acc = mfma_16x16x32(load_bf16x8(base + (wave * 16 + col) * STEP * 2 + slot), load_bf16x8(base + (kStCols + col) * STEP * 2 + slot), acc);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be on its way into LDS when the workgroup ends
  // acc[i]: feature n0 + wave * 16 + quad * 4 + i of tile row `col`
  const int pair = row0 + col < row_end ? sorted[row0 + col] : -1;
  if (pair < 0) return;
  const int token = pair / top;
  const int choice = pair - token * top;
  const int n = n0 + wave * 16 + quad * 4;
  if (UP && act == 5) {
    const float v[4] = {acc[0], acc[1], acc[2], acc[3]};
    if (n < N) store_clamped_glu(static_cast<bf16*>(out) + static_cast<int64_t>(row0 + col) * (N / 2) + n / 2, v, glu_limit, glu_alpha);
  } else if (UP) {
    bf16* dst = static_cast<bf16*>(out) + static_cast<int64_t>(row0 + col) * N + n;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = acc[i];
      if (act == 2) {
        v = fmaxf(v, 0.f);
        v *= v;
      } else if (act == 3) {
        v = 1.0f / (1.0f + __expf(-v));
      }
      if (n + i < N) dst[i] = f32_to_bf16(v);
    }
  } else {
    const float pw = pair_weights[pair];
    float* dst = static_cast<float*>(out) + (static_cast<int64_t>(choice) * tokens + token) * N + n;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < N) dst[i] = pw * acc[i];
  }
}

// Tiled (prompts, where an expert sees hundreds of rows): a workgroup owns a tile of 64 x RB rows and 128 features; k in slices of
// 64 loaded straight into two LDS buffers (a lane brings 16 bytes of the row that the tile's order names; pieces in the order
// piece ^ (row / 2) % 8).  Wavefront (wr, wc) of 2 x 2 owns rows wr * 32 RB .. + 32 RB and features wc * 64 .. + 64; the last
// quarter of a slice's products is kept for behind the barrier, where the next slice's first operands are on their way.  Finished
// tiles leave through LDS in whole lines: the down product's rows go to as many places as it has rows, 512 bytes each.
// Workgroup -> (tile, features): workgroups go to the eight dies in turn; a pair of neighbouring tiles (mostly one expert's) belongs to one
// die, or its features to a few of them where that would leave dies without work (order_tiles); a die takes their features one after the
// other, both tiles at a time, so that the rows and the expert's weights come from its L2.
// Bound by the operands' way through L2 and LDS (each 64 x RB + 128 rows of a slice make 64 RB x 128 products of it) and by tiles
// that are not full: 2,000 tokens, 64 experts with 6 choices (187 rows an expert in tiles of 128), 768 x 2,048: up 94.5 to 91.4 us,
// down 128 to 93 (400 TFLOP/s of the asked-for products, 550 with the padding).  Four buffers of 32 k instead: up the same, down 102.
struct TilePlace {
  int tile, column;  // column -1: none
};
// How the pairs of `used` tiles go to the dies: all of them one by one where that leaves no die with more than 1.15 times its share; else the
// whole rounds of eight, and the features of each pair of the rest to as many dies as make whole rounds of them, too.
// With one die for each pair / as here, both products with their gating, microseconds: 8 experts of 14,336 x 4,096 (4 pairs on 8 dies): 48 rows an
// expert 786 / 617, 97 900 / 692; 12 of 8,192 x 5,120: 97 798 / 646, 320 1,521 / 1,296; 32 of 2,880 x 2,880: 50 (33 tiles of 64) 280 / 251; 16 of
// 6,400 x 4,096: 64 503 / 409; 64 of 768 x 2,048, some four times as popular as others: 187 184 / 174.  Fewer dies read a pair's rows fewer
// times: that last one takes 204 where every pair beyond those of equal shares goes to all dies.  To look up how many tiles are used costs 0.5 us.
struct PairOrder {
  int first;   // pairs that have a die to themselves
  int spread;  // dies that share each of the others
};
__host__ __device__ inline PairOrder order_tiles(int used) {
  const int pairs = (used + 1) / 2, whole = (pairs + 7) / 8 * 8, rest = pairs % 8;
  if (whole * 100 <= pairs * 115) return {whole, 8};
  return {pairs / 8 * 8, 8 >> __builtin_ctz(rest)};
}
__host__ __device__ inline int features_of_a_die(int columns, int spread) { return (columns + spread - 1) / spread; }
__device__ __forceinline__ TilePlace place_tile(const int* __restrict__ tiles, int max_tiles, int columns) {
  // an unused tile names how many are used
  const PairOrder order = order_tiles(tiles[2 * max_tiles - 2] < 0 ? tiles[2 * max_tiles - 1] : max_tiles);
  const int firsts = order.first * 2 * columns;
  const bool shared = static_cast<int>(blockIdx.x) >= firsts;
  const int block = shared ? blockIdx.x - firsts : blockIdx.x, spread = shared ? order.spread : 1, pair0 = shared ? order.first : 0;
  const int each = features_of_a_die(columns, spread);
  const int local = block / 8, in_unit = local % (2 * each);
  const int unit = local / (2 * each) * 8 + block % 8;
  const int column = unit % spread * each + in_unit / 2;
  return {(pair0 + unit / spread) * 2 + in_unit % 2, column < columns ? column : -1};
}
// Workgroups that cover every number of used tiles.
static int64_t groups_of_tiles(int max_tiles, int columns) {
  int64_t most = 0;
  for (int used = max(1, max_tiles - 32); used <= max_tiles; ++used) {
    const PairOrder order = order_tiles(used);
    const int rest = max((used + 1) / 2 - order.first, 0);
    const int64_t groups = static_cast<int64_t>(order.first) * 2 * columns + static_cast<int64_t>(rest) * order.spread * 2 * features_of_a_die(columns, order.spread);
    most = groups > most ? groups : most;
  }
  return most;
}
constexpr int kBigCols = 128;
constexpr int kBigK = 64;
constexpr int big_rows(int rb) { return 64 * rb; }
constexpr int big_buffer_bytes(int rb) { return (kBigCols + big_rows(rb)) * kBigK * 2; }
constexpr int kBigRowF32 = kBigCols * 4 + 16, kBigRowBf16 = kBigCols * 2 + 16;  // staged rows, padded to other banks
constexpr int big_lds_bytes(int rb) {
  return big_rows(rb) * kBigRowF32 > 2 * big_buffer_bytes(rb) ? big_rows(rb) * kBigRowF32 : 2 * big_buffer_bytes(rb);
}

__device__ __forceinline__ u16x4_t activated4(float (&v)[4], int act) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (act == 2) {
      v[i] = fmaxf(v[i], 0.f);
      v[i] *= v[i];
    } else if (act == 3) {
      v[i] = 1.0f / (1.0f + __expf(-v[i]));
    }
  }
  return u16x4_t{f32_to_bf16(v[0]).bits, f32_to_bf16(v[1]).bits, f32_to_bf16(v[2]).bits, f32_to_bf16(v[3]).bits};
}

template <bool UP, int RB>
__global__ __launch_bounds__(256) void moe_gemm_tiled_kernel(const bf16* __restrict__ a, const bf16* __restrict__ w,
                                                             const int* __restrict__ sorted,
                                                             const int* __restrict__ offsets,
                                                             const int* __restrict__ tiles, int max_tiles,
                                                             const float* __restrict__ pair_weights,
                                                             void* __restrict__ out, int tokens, int top, int N, int K,
                                                             int act, int a_rows, float glu_limit, float glu_alpha) {
  constexpr int kRows = big_rows(RB);
  constexpr int kBuffer = big_buffer_bytes(RB);
  // runs of 8 rows, dealt out to four wavefronts: 4 of weights, then the input's (loops over them go to 8 and break: with a bound that
  // depends on the template's parameters the host pass left the kernel uninstantiated, without a message)
  constexpr int kLoads = (kBigCols + kRows) / 8 / 4;
  const TilePlace place = place_tile(tiles, max_tiles, (N + kBigCols - 1) / kBigCols);
  const int tile = place.tile;
  if (tile >= max_tiles || place.column < 0) return;
  const int expert = tiles[2 * tile];
  if (expert < 0) return;
  const int n0 = place.column * kBigCols;
  const int row0 = tiles[2 * tile + 1];
  const int rows = min(kRows, offsets[expert + 1] - row0);
  extern __shared__ __attribute__((aligned(16))) unsigned char moe_lds[];
  __shared__ int pair_of[kRows];
  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wr = wave / 2;
  const int wc = wave % 2;
  const unsigned row_bytes = static_cast<unsigned>(K) * 2u;
  const __amdgpu_buffer_rsrc_t wbuf = make_buffer(w + (static_cast<int64_t>(expert) * N + n0) * K, static_cast<unsigned>(min(kBigCols, N - n0)) * row_bytes);
  const __amdgpu_buffer_rsrc_t abuf = make_buffer(a, static_cast<unsigned>(a_rows) * row_bytes);
  // Which pairs this tile's rows are: all lookups are sent at once and without conditions, then the weights of the first two slices,
  // which do not depend on them (looked up one by one ahead of the first load, they took longer than a slice of products each).
  constexpr int kRowLoads = kLoads - 4;
  int pairs_of_lane[4];
#pragma unroll
  for (int p = 0; p < 4; ++p)
    if (p < kRowLoads) pairs_of_lane[p] = sorted[row0 + min(8 * (4 * p + wave) + lane / 8, rows - 1)];
  const int pair_of_thread = sorted[row0 + min(tid, rows - 1)];
  const int piece = (lane % 8) ^ ((4 * (wave % 2) + lane / 16) % 8);
  const int slices = (K + kBigK - 1) / kBigK;
  unsigned off[8];
  auto fetch = [&](int slice, int buf, bool weights) {
    const unsigned past = slice < slices && slice * kBigK + piece * 8 < K ? 0u : kOutOfBuffer;
    const unsigned koff = static_cast<unsigned>(slice) * kBigK * 2u;
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      if (p >= kLoads) break;
      if ((p < 4) != weights) continue;
      const unsigned at = p < 4 ? (off[p] + koff) | past : (past != 0u || off[p] == kNoRow ? kNoRow : off[p] + koff);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          p < 4 ? wbuf : abuf, (__attribute__((address_space(3))) void*)(moe_lds + buf * kBuffer + (4 * p + wave) * 1024), 16, at, 0, 0, 0);
    }
  };
#pragma unroll
  for (int p = 0; p < 4; ++p)  // rows past the last feature: past the resource
    off[p] = static_cast<unsigned>(8 * (4 * p + wave) + lane / 8) * row_bytes + piece * 16u;
  fetch(0, 0, true);
  fetch(1, 1, true);
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    if (p >= kRowLoads) break;
    const int at = 8 * (4 * p + wave) + lane / 8;
    off[4 + p] = at < rows ? static_cast<unsigned>(UP ? pairs_of_lane[p] / top : row0 + at) * row_bytes + piece * 16u : kNoRow;
  }
  if (tid < kRows) pair_of[tid] = tid < rows ? pair_of_thread : -1;
  f32x4_t acc[2 * RB][4];  // blocks of 16 rows, of 16 features
#pragma unroll
  for (int r = 0; r < 2 * RB; ++r)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[r][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int c16 = lane % 16;
  const int quad = lane / 16;  // which 8 of a block's 32 k
  const bool idle = __builtin_amdgcn_readfirstlane(static_cast<int>(wr * 32 * RB >= rows)) != 0;  // a tile with rows for the first wavefronts only
  const int swz = c16 / 2;
  // A slice's products come in quarters: 32 of k, all features, half the rows.
  struct Weights {
    bf16x8_t v[4];
  };
  struct Rows {
    bf16x8_t v[RB];
  };
  auto read_weights = [&](int buf, int kk) {
    Weights o;
    const unsigned char* const base = moe_lds + buf * kBuffer + (((kk * 4 + quad) ^ swz) * 16) + (wc * 64 + c16) * 128;
#pragma unroll
    for (int b = 0; b < 4; ++b) o.v[b] = load_bf16x8(base + b * 16 * 128);
    return o;
  };
  auto read_rows = [&](int buf, int kk, int half) {
    Rows o;
    const unsigned char* const base = moe_lds + buf * kBuffer + (((kk * 4 + quad) ^ swz) * 16) + (kBigCols + wr * 32 * RB + c16) * 128;
#pragma unroll
    for (int r = 0; r < RB; ++r) o.v[r] = load_bf16x8(base + (half * RB + r) * 16 * 128);
    return o;
  };
  auto multiply = [&](const Weights& u, const Rows& x, int half) {
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const int b = turn_at(f, r, 4);
        acc[half * RB + r][b] = mfma_16x16x32(u.v[b], x.v[r], acc[half * RB + r][b]);
      }
  };
  fetch(0, 0, false);
  fetch(1, 1, false);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kRowLoads) : "memory");
  __syncthreads();
  Weights u = read_weights(0, 0);
  Rows x = read_rows(0, 0, 0);
  int buf = 0;
  for (int s = 0; s < slices; ++s) {
    if (!idle) {
      const Rows second = read_rows(buf, 0, 1);
      multiply(u, x, 0);
      const Weights u1 = read_weights(buf, 1);
      const Rows third = read_rows(buf, 1, 0);
      multiply(u, second, 1);
      x = read_rows(buf, 1, 1);
      multiply(u1, third, 0);
      u = u1;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __syncthreads();
    fetch(s + 2, buf, true);
    fetch(s + 2, buf, false);
    buf ^= 1;
    if (!idle) {
      const Weights kept_u = u;
      const Rows kept = x;
      u = read_weights(buf, 0);
      x = read_rows(buf, 0, 0);
      multiply(kept_u, kept, 1);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();  // the slices are done with
  // acc[r][b][i]: feature n0 + wc * 64 + b * 16 + quad * 4 + i of tile row wr * 32 RB + r * 16 + c16.
  // N is a multiple of 8: four features are all inside or all outside.
  const bool paired = UP && act == 5;
  const bool staged = !UP || N % (paired ? 16 : 8) == 0;  // rows of results are multiples of 16 bytes
#pragma unroll
  for (int r = 0; r < 2 * RB; ++r) {
    const int row = wr * 32 * RB + r * 16 + c16;
    const int pair = pair_of[row];
    if (pair < 0) continue;
    const float pw = UP ? 1.f : pair_weights[pair];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int f = wc * 64 + b * 16 + quad * 4;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = acc[r][b][i];
      if constexpr (!UP) {
        *reinterpret_cast<f32x4_t*>(moe_lds + row * kBigRowF32 + f * 4) = f32x4_t{pw * v[0], pw * v[1], pw * v[2], pw * v[3]};
      } else if (paired) {
        bf16* const to = staged ? reinterpret_cast<bf16*>(moe_lds + row * kBigRowBf16) + f / 2
                                : static_cast<bf16*>(out) + static_cast<int64_t>(row0 + row) * (N / 2) + (n0 + f) / 2;
        if (staged || n0 + f < N) store_clamped_glu(to, v, glu_limit, glu_alpha);
      } else {
        *reinterpret_cast<u16x4_t*>(moe_lds + row * kBigRowBf16 + f * 2) = activated4(v, act);
      }
    }
  }
  if (!staged) return;
  __syncthreads();
  const int width = (paired ? N / 2 : N) * (UP ? 2 : 4);               // bytes of a row of results
  const int first = (paired ? n0 / 2 : n0) * (UP ? 2 : 4);             // where this tile's part of it starts
  const int pieces = (paired ? kBigCols / 2 : kBigCols) * (UP ? 2 : 4) / 16;  // 8, 16 or 32
  for (int p = tid; p < rows * pieces; p += 256) {
    const int row = p / pieces, at = (p - row * pieces) * 16;
    if (first + at >= width) continue;
    int64_t to = row0 + row;
    if constexpr (!UP) {
      const int pair = pair_of[row], token = pair / top;
      to = static_cast<int64_t>(pair - token * top) * tokens + token;
    }
    *reinterpret_cast<u32x4_t*>(static_cast<unsigned char*>(out) + to * width + first + at) =
        *reinterpret_cast<const u32x4_t*>(moe_lds + row * (UP ? kBigRowBf16 : kBigRowF32) + at);
  }
}

// Tiles of 256 rows and 256 features by eight wavefronts in two groups that take turns, one multiplying while the other reads its
// operands: the loop of gemm_phased_kernel (its comment explains the phases, the wait counts and the products' shape) over gathered rows.  What differs:
//  * quarter X0 holds the tile's rows 0 .. 127 and X1 the others, and a group takes 64 of each, so that the groups share the work of a
//    tile that is not full; blocks of 64 rows without rows are not multiplied (187 rows: three of four).
//  * the first slice's weights are asked for ahead of its rows, whose places have to be looked up first.
//  * the down product's rows are twice as wide as LDS has room for: they leave in two halves.
// An expert with up to 256 rows has its weights read once.  The workgroup -> (tile, features) map is the kernel's above.
// 2,000 tokens, 64 experts with 6 choices (187 rows an expert), 768 x 2,048, against the 128-row tiles: up 91.4 to 69.9 us (201 MB of
// weights alone take 31), down 93 to 91: its twelve slices are short beside the first loads and the 512 KB of results that a compute unit's
// two tiles leave, and with one workgroup there nothing runs meanwhile.
constexpr int kSqRows = 256, kSqCols = 256;
constexpr int kSqQuarter = 128 * 128;
constexpr int kSqBuffer = 4 * kSqQuarter;  // W0, W1, X0, X1: 64 k of 128 rows each
constexpr int kSqRowF32 = kSqCols * 4 + 16, kSqRowBf16 = kSqCols * 2 + 16;
constexpr int kSqLds = kSqRows * kSqRowBf16;
static_assert(kSqLds >= 2 * kSqBuffer && kSqLds >= kSqRows / 2 * kSqRowF32, "two slices, and half a tile of 32-bit results, fit");

template <bool UP>
__global__ __launch_bounds__(512, 2) void moe_gemm_phased_kernel(const bf16* __restrict__ a, const bf16* __restrict__ w,
                                                                const int* __restrict__ sorted, const int* __restrict__ offsets,
                                                                const int* __restrict__ tiles, int max_tiles,
                                                                const float* __restrict__ pair_weights, void* __restrict__ out,
                                                                int tokens, int top, int N, int K, int act, int a_rows,
                                                                float glu_limit, float glu_alpha) {
  extern __shared__ __attribute__((aligned(16))) unsigned char moe_lds[];
  __shared__ int pair_of[kSqRows];
  const TilePlace place = place_tile(tiles, max_tiles, (N + kSqCols - 1) / kSqCols);
  const int tile = place.tile;
  if (tile >= max_tiles || place.column < 0) return;
  const int expert = tiles[2 * tile];
  if (expert < 0) return;
  const int n0 = place.column * kSqCols;
  const int row0 = tiles[2 * tile + 1];
  const int rows = min(kSqRows, offsets[expert + 1] - row0);
  const int tid = threadIdx.x;
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave / 4, wn = wave % 4;  // wavefronts w and w + 4 share a SIMD: one of each group
  const int c16 = lane % 16, quad = lane / 16;
  const unsigned row_bytes = static_cast<unsigned>(K) * 2u;
  const __amdgpu_buffer_rsrc_t w_buf = make_buffer(w + (static_cast<int64_t>(expert) * N + n0) * K, static_cast<unsigned>(min(kSqCols, N - n0)) * row_bytes);
  const __amdgpu_buffer_rsrc_t x_buf = make_buffer(a, static_cast<unsigned>(a_rows) * row_bytes);
  const int steps = (K + 63) / 64;
  // A quarter is 16 runs of 8 rows; this wavefront brings runs `wave` and `wave` + 8.  Row r of Wj: feature r / 32 * 64 + j * 32 + r % 32.
  const int row = 8 * wave + lane / 8;
  const int piece = (lane % 8) ^ ((4 * (wave % 2) + lane / 16) % 8);
  const unsigned w_off = static_cast<unsigned>(row / 32 * 64 + row % 32) * row_bytes + piece * 16u;
  int looked_up[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int p = 0; p < 2; ++p) looked_up[i][p] = UP ? sorted[row0 + min(i * 128 + p * 64 + row, rows - 1)] : 0;
  const int pair_of_thread = sorted[row0 + min(tid, rows - 1)];
  auto fetch_weights = [&](int step, int j) {
    const unsigned past = step < steps && step * 64 + piece * 8 < K ? 0u : kOutOfBuffer;
    const unsigned off = w_off + j * 32u * row_bytes + step * 128u;
    unsigned char* const dst = moe_lds + (step & 1) * kSqBuffer + j * kSqQuarter + wave * 1024;
#pragma unroll
    for (int p = 0; p < 2; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_buf, (__attribute__((address_space(3))) void*)(dst + p * 8192), 16,
                                               (off + p * 128u * row_bytes) | past, 0, 0, 0);
  };
  fetch_weights(0, 0);
  fetch_weights(0, 1);
  unsigned x_off[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int at = i * 128 + p * 64 + row;
      x_off[i][p] = at < rows ? static_cast<unsigned>(UP ? looked_up[i][p] / top : row0 + at) * row_bytes + piece * 16u : kNoRow;
    }
  if (tid < kSqRows) pair_of[tid] = tid < rows ? pair_of_thread : -1;
  auto fetch_rows = [&](int step, int i) {
    const bool in = step < steps && step * 64 + piece * 8 < K;
    unsigned char* const dst = moe_lds + (step & 1) * kSqBuffer + (2 + i) * kSqQuarter + wave * 1024;
#pragma unroll
    for (int p = 0; p < 2; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_buf, (__attribute__((address_space(3))) void*)(dst + p * 8192), 16,
                                               in && x_off[i][p] != kNoRow ? x_off[i][p] + step * 128u : kNoRow, 0, 0, 0);
  };

  f32x4_t acc[4][8];  // blocks of 16 features (half * 2 + block) and of 16 rows (half * 4 + block)
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // whether this group has rows in each half
  bool any[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) any[i] = __builtin_amdgcn_readfirstlane(static_cast<int>(i * 128 + wm * 64 < rows)) != 0;
  const int swz = c16 / 2;
  const int w_base = (wn * 32 + c16) * 128;
  const int x_base = 2 * kSqQuarter + (wm * 64 + c16) * 128;
  struct Weights {
    bf16x8_t v[2][2];  // 32 of k, block of 16 features
  };
  struct Rows {
    bf16x8_t v[2][4];
  };
  auto read_weights = [&](Weights& t, int buf, int j) {
    if (!any[0]) return;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        t.v[kk][b] = load_bf16x8(moe_lds + buf * kSqBuffer + j * kSqQuarter + w_base + b * 16 * 128 + (((kk * 4 + quad) ^ swz) * 16));
  };
  auto read_rows = [&](Rows& t, int buf, int i) {
    if (!any[i]) return;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        t.v[kk][b] = load_bf16x8(moe_lds + buf * kSqBuffer + i * kSqQuarter + x_base + b * 16 * 128 + (((kk * 4 + quad) ^ swz) * 16));
  };
#define MLR_READ_DONE(pending)                                                                   \
  do {                                                                                           \
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(pending) : "memory");                    \
    __builtin_amdgcn_sched_barrier(0);                                                           \
    __builtin_amdgcn_s_barrier();                                                                \
    __builtin_amdgcn_sched_barrier(0);                                                           \
  } while (0)
  auto multiply = [&](const Weights& t, const Rows& b, int j, int i) {
    __builtin_amdgcn_s_setprio(1);
    if (any[i]) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int f = 0; f < 2; ++f) {
            f32x4_t& sum = acc[j * 2 + turn_at(f, c, 2)][i * 4 + c];
            sum = mfma_16x16x32(t.v[kk][turn_at(f, c, 2)], b.v[kk][c], sum);
          }
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  fetch_rows(0, 0);
  fetch_rows(0, 1);
  fetch_rows(1, 0);
  fetch_weights(1, 0);
  fetch_weights(1, 1);
  Weights wa, wb;
  Rows xr;
  MLR_READ_DONE(8);  // W0, W1 and X0 of the first step (X1 is the next, as in every later step)
  read_weights(wa, 0, 0);
  if (wave >= 4) __builtin_amdgcn_s_barrier();  // the second group stays one phase behind
  __builtin_amdgcn_sched_barrier(0);
  auto step_of = [&](int step, Weights& w0, Weights& w1) {
    const int buf = step & 1;
    fetch_rows(step + 1, 1);
    read_rows(xr, buf, 0);
    MLR_READ_DONE(10);
    multiply(w0, xr, 0, 0);
    fetch_rows(step + 2, 0);
    read_weights(w1, buf, 1);
    MLR_READ_DONE(10);
    multiply(w1, xr, 1, 0);
    fetch_weights(step + 2, 0);
    read_rows(xr, buf, 1);
    MLR_READ_DONE(8);
    multiply(w1, xr, 1, 1);
    fetch_weights(step + 2, 1);
    read_weights(w1, buf ^ 1, 0);
    MLR_READ_DONE(12);
    multiply(w0, xr, 0, 1);
  };
  int step = 0;
  for (; step + 1 < steps; step += 2) {
    step_of(step, wa, wb);
    step_of(step + 1, wb, wa);
  }
  if (step < steps) step_of(step, wa, wb);
#undef MLR_READ_DONE
  if (wave < 4) __builtin_amdgcn_s_barrier();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be on its way into LDS
  __syncthreads();

  // acc[j][i * 4 + c][e]: feature n0 + wn * 64 + j * 16 + quad * 4 + e of tile row i * 128 + wm * 64 + c * 16 + c16.
  // N is a multiple of 8: four features are all inside or all outside.
  const bool paired = UP && act == 5;
  const bool staged = !UP || N % (paired ? 16 : 8) == 0;  // rows of results are multiples of 16 bytes
  const int width = (paired ? N / 2 : N) * (UP ? 2 : 4);                         // bytes of a row of results
  const int first = (paired ? n0 / 2 : n0) * (UP ? 2 : 4);                       // where this tile's part of it starts
  const int pieces = (paired ? kSqCols / 2 : kSqCols) * (UP ? 2 : 4) / 16;       // 16, 32 or 64
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int half0 = UP ? 0 : i * 128;  // the first tile row that is in LDS
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int at = i * 128 + wm * 64 + c * 16 + c16;
      const int pair = pair_of[at];
      if (pair < 0) continue;
      const float pw = UP ? 1.f : pair_weights[pair];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int f = wn * 64 + j * 16 + quad * 4;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[j][i * 4 + c][e];
        if constexpr (!UP) {
          *reinterpret_cast<f32x4_t*>(moe_lds + (at - half0) * kSqRowF32 + f * 4) = f32x4_t{pw * v[0], pw * v[1], pw * v[2], pw * v[3]};
        } else if (paired) {
          bf16* const to = staged ? reinterpret_cast<bf16*>(moe_lds + at * kSqRowBf16) + f / 2
                                  : static_cast<bf16*>(out) + static_cast<int64_t>(row0 + at) * (N / 2) + (n0 + f) / 2;
          if (staged || n0 + f < N) store_clamped_glu(to, v, glu_limit, glu_alpha);
        } else {
          *reinterpret_cast<u16x4_t*>(moe_lds + at * kSqRowBf16 + f * 2) = activated4(v, act);
        }
      }
    }
    if (!staged || (UP && i == 0)) continue;
    __syncthreads();
    const int held = UP ? rows : min(128, rows - half0);
    for (int p = tid; p < held * pieces; p += 512) {
      const int at = p / pieces, byte = (p - at * pieces) * 16;
      if (first + byte >= width) continue;
      int64_t to = row0 + at;
      if constexpr (!UP) {
        const int pair = pair_of[half0 + at], token = pair / top;
        to = static_cast<int64_t>(pair - token * top) * tokens + token;
      }
      *reinterpret_cast<u32x4_t*>(static_cast<unsigned char*>(out) + to * width + first + byte) =
          *reinterpret_cast<const u32x4_t*>(moe_lds + at * (UP ? kSqRowBf16 : kSqRowF32) + byte);
    }
    if (!UP && i == 0) __syncthreads();  // the next half takes its place
  }
}

using MoeTiledKernel = void (*)(const bf16*, const bf16*, const int*, const int*, const int*, int, const float*, void*, int, int, int, int,
                                int, int, float, float);
struct MoeTiles {
  MoeTiledKernel kernel;
  int threads, cols, lds;
};
// Steps of 64 in moe_gemm_stream: where there are more pairs than experts, of matrices of 64 MB or more eight times as many.  Steps of 128 / 64, both
// products, microseconds: 64 experts of 768 x 2,048 with 6 choices: 2 tokens 25 / 26, 8 51 / 55, 13 69 / 64, 32 79 / 77, 64 87 / 80; 128 of it
// with 8: 2 26 / 28, 6 59 / 61, 16 98 / 93, 64 146 / 141; 32 of 2,880 x 2,880 with 4: 1 32 / 35, 8 130 / 125, 48 170 / 169; 16 of 6,400 x
// 4,096 with 2: 4 112 / 116, 10 209 / 205, 24 250 / 245; 8 of 14,336 x 4,096 (117 MB) with 2: 8 233 / 272, 13 259 / 299, 32 320 / 292,
// 48 377 / 360.  (A step through registers, three workgroups a unit: 64 experts at 13 tokens 64, at 64 82; 8 experts at 32 297.)
static bool narrow_steps_pay(int max_tiles, int64_t pairs, int64_t matrix_bytes) {
  if (max_tiles >= pairs) return false;  // mlr_moe_max_tiles: the pairs, or the full tiles and one for every expert
  return matrix_bytes < (64ll << 20) || pairs >= 8 * (max_tiles - pairs / kMoeRows);
}
static int launch_moe_tiled(const MoeTiles& t, bool& configured, const bf16* a, const bf16* w, const int* sorted, const int* offsets,
                            const int* tiles, const float* pair_weights, void* out, int max_tiles, int tokens, int top, int n, int k,
                            int act, int a_rows, float glu_limit, float glu_alpha, hipStream_t stream) {
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(t.kernel), hipFuncAttributeMaxDynamicSharedMemorySize, t.lds);
    if (e != hipSuccess) {
      set_error(std::string("mlr_moe_gemm: cannot raise the LDS limit: ") + hipGetErrorString(e));
      return -1;
    }
    configured = true;
  }
  const int64_t groups = groups_of_tiles(max_tiles, (n + t.cols - 1) / t.cols);
  if (groups >= (1ll << 31)) {
    set_error("mlr_moe_gemm: too many tiles for one launch");
    return -1;
  }
  hipLaunchKernelGGL(t.kernel, dim3(static_cast<unsigned>(groups)), dim3(t.threads), t.lds, stream, a, w, sorted, offsets, tiles, max_tiles,
                     pair_weights, out, tokens, top, n, k, act, a_rows, glu_limit, glu_alpha);
  return 0;
}

}  // namespace mlr

using namespace mlr;

extern "C" {

int mlr_moe_route(const float* logits, int slices, const float* correction, int* ids, float* weights, int tokens, int experts,
                  int top, int groups, int keep, float scale, int score_kind, int normalise, hipStream_t stream) {
  MLR_REQUIRE(logits && ids && weights, "null pointer");
  MLR_REQUIRE(slices >= 1, "logits come whole or in slices");
  MLR_REQUIRE(score_kind >= 0 && score_kind <= 2, "scores are sigmoids (0), a softmax (1) or the logits themselves (2)");
  MLR_REQUIRE(score_kind != 2 || correction == nullptr, "a softmax over the chosen logits has no correction");
  MLR_REQUIRE(tokens > 0 && experts > 0 && top > 0 && top <= experts, "sizes must be > 0 and top <= experts");
  MLR_REQUIRE(groups > 0 && experts % groups == 0 && keep > 0 && keep <= groups, "bad groups");
  MLR_REQUIRE(top <= keep * (experts / groups), "the kept groups hold fewer experts than a token uses");
  MLR_REQUIRE(experts <= 4096, "at most 4096 experts");
  const int norm = normalise || score_kind == 2;
  if (experts <= 4 * kWave && groups <= kWave && top <= kWave) {
    if (experts <= kWave)
      moe_route_lanes_kernel<1><<<tokens, kWave, 0, stream>>>(logits, slices, correction, ids, weights, tokens, experts, top, groups,
                                                              keep, scale, score_kind, norm);
    else
      moe_route_lanes_kernel<4><<<tokens, kWave, 0, stream>>>(logits, slices, correction, ids, weights, tokens, experts, top, groups,
                                                              keep, scale, score_kind, norm);
    MLR_LAUNCH_CHECK();
    return 0;
  }
  const size_t lds = (2 * static_cast<size_t>(experts) + groups) * sizeof(float);
  moe_route_kernel<<<tokens, kWave, lds, stream>>>(logits, slices, correction, ids, weights, tokens, experts, top, groups, keep,
                                                   scale, score_kind, norm);
  MLR_LAUNCH_CHECK();
  return 0;
}

// mlr_moe_route and mlr_moe_align (16 rows a tile) in one launch: up to 8 tokens, 256 router outputs, 64 groups and choices.  experts: how
// many of the `routed` router outputs have matrices (the first ones).
int mlr_moe_route_align_fits(int tokens, int routed, int top, int groups) {
  return tokens <= kRouteAlignTokens && routed <= 4 * kWave && groups <= kWave && top <= kWave;
}
int mlr_moe_route_align(const float* logits, int slices, const float* correction, int* ids, float* weights, int tokens, int routed, int top,
                        int groups, int keep, float scale, int score_kind, int normalise, int experts, int max_tiles, int* sorted, int* offsets,
                        int* tiles, hipStream_t stream) {
  MLR_REQUIRE(logits && ids && weights && sorted && offsets && tiles, "null pointer");
  MLR_REQUIRE(slices >= 1, "logits come whole or in slices");
  MLR_REQUIRE(score_kind >= 0 && score_kind <= 2, "scores are sigmoids (0), a softmax (1) or the logits themselves (2)");
  MLR_REQUIRE(score_kind != 2 || correction == nullptr, "a softmax over the chosen logits has no correction");
  MLR_REQUIRE(tokens > 0 && routed > 0 && top > 0 && top <= routed && experts > 0 && experts <= routed, "sizes must be > 0 and top <= experts");
  MLR_REQUIRE(groups > 0 && routed % groups == 0 && keep > 0 && keep <= groups, "bad groups");
  MLR_REQUIRE(top <= keep * (routed / groups), "the kept groups hold fewer experts than a token uses");
  MLR_REQUIRE(mlr_moe_route_align_fits(tokens, routed, top, groups), "too many tokens or experts for one launch");
  MLR_REQUIRE(max_tiles >= mlr_moe_max_tiles(tokens * top, experts, 0), "too few tiles for these pairs");
  const int norm = normalise || score_kind == 2;
  if (routed <= kWave)
    moe_route_align_kernel<1><<<1, tokens * kWave, 0, stream>>>(logits, slices, correction, ids, weights, tokens, routed, top, groups, keep, scale,
                                                                score_kind, norm, experts, kMoeRows, max_tiles, sorted, offsets, tiles);
  else
    moe_route_align_kernel<4><<<1, tokens * kWave, 0, stream>>>(logits, slices, correction, ids, weights, tokens, routed, top, groups, keep, scale,
                                                                score_kind, norm, experts, kMoeRows, max_tiles, sorted, offsets, tiles);
  MLR_LAUNCH_CHECK();
  return 0;
}

int mlr_moe_identity(const void* h, const int* ids, const float* weights, float* out, int dtype, int tokens, int top,
                     int hidden, int first, hipStream_t stream) {
  MLR_REQUIRE(h && ids && weights && out, "null pointer");
  MLR_REQUIRE(tokens > 0 && top > 0 && hidden > 0 && first >= 0, "sizes must be > 0");
  MLR_REQUIRE(dtype == kF32 || dtype == kBF16, "dtype must be 0 (float32) or 1 (bfloat16)");
  if (dtype == kF32)
    moe_identity_kernel<float><<<tokens * top, 256, 0, stream>>>(static_cast<const float*>(h), ids, weights, out, tokens,
                                                                 top, hidden, first);
  else
    moe_identity_kernel<bf16><<<tokens * top, 256, 0, stream>>>(static_cast<const bf16*>(h), ids, weights, out, tokens,
                                                                top, hidden, first);
  MLR_LAUNCH_CHECK();
  return 0;
}

// Rows of one tile of the grouped products: `big` 0 the kernels for few rows an expert (16), 1 to 3
// the tiled matrix-core kernels for many (64, 128 and 256).
int mlr_moe_tile_rows(int big) { return big == 3 ? kSqRows : (big ? big_rows(big) : kMoeRows); }

// The most tiles `pairs` pairs over `experts` experts can make.
int mlr_moe_max_tiles(int pairs, int experts, int big) {
  const int most = pairs / mlr_moe_tile_rows(big) + experts;  // full tiles, and at most one that is not per expert
  return most < pairs ? most : pairs;
}

int mlr_moe_align(const int* ids, int pairs, int experts, int big, int max_tiles, int* sorted, int* offsets, int* tiles,
                  hipStream_t stream) {
  MLR_REQUIRE(ids && sorted && offsets && tiles, "null pointer");
  MLR_REQUIRE(pairs > 0 && experts > 0 && experts <= 4096 && max_tiles > 0 && big >= 0 && big <= 3, "bad sizes");
  MLR_REQUIRE(max_tiles >= mlr_moe_max_tiles(pairs, experts, big), "too few tiles for these pairs");
  const int kept = experts > kKeptExperts || pairs > 16 * 1024 ? 0 : (pairs > 4 * 1024 ? 16 : 4);
  const auto kernel = kept == 16 ? moe_align_kernel<16> : (kept == 4 ? moe_align_kernel<4> : moe_align_kernel<0>);
  const size_t lds = 2 * static_cast<size_t>(experts) * sizeof(int) + (kept ? pairs * sizeof(unsigned short) : 0);
  hipLaunchKernelGGL(kernel, dim3(1), dim3(1024), lds, stream, ids, pairs, experts, mlr_moe_tile_rows(big),
                     max_tiles, sorted, offsets, tiles);
  MLR_LAUNCH_CHECK();
  return 0;
}

// One of the two grouped products (`up` 1: act = f(h w_up^T) for the sorted rows, `act` 0 none, 2
// squared ReLU, 3 sigmoid, 5 the clamped gating over rows woven in pairs, whose rows of `act` are n / 2 wide; `up` 0: out[choice, token] = weight * (act w_down^T), float32).  a and w
// in `dtype`; w is [experts, n, k].  `mfma` 1: the streaming matrix-core kernel (bfloat16, k % 8 == 0;
// tiles of 16 rows), 2 to 4: the tiled ones (tiles of 64, 128 and 256 rows, as mlr_moe_align made them
// with `big` 1 to 3; n % 8 == 0 too); 0: plain arithmetic (tiles of 16 rows).
int mlr_moe_gemm(const void* a, const void* w, const int* sorted, const int* offsets, const int* tiles,
                 const float* pair_weights, void* out, int up, int dtype, int mfma, int max_tiles, int tokens, int top,
                 int n, int k, int act, float glu_limit, float glu_alpha, hipStream_t stream) {
  MLR_REQUIRE(a && w && sorted && offsets && tiles && out, "null pointer");
  MLR_REQUIRE(up || pair_weights, "the down product needs the pairs' weights");
  MLR_REQUIRE(max_tiles > 0 && tokens > 0 && top > 0 && n > 0 && k > 0, "sizes must be > 0");
  MLR_REQUIRE(dtype == kF32 || dtype == kBF16, "dtype must be 0 (float32) or 1 (bfloat16)");
  MLR_REQUIRE(act == 0 || act == 2 || act == 3 || act == 5, "unknown activation");
  MLR_REQUIRE(act != 5 || (up && n % 4 == 0 && glu_limit > 0.f), "the clamped gating takes a first matrix of rows woven in pairs and a limit > 0");
  MLR_REQUIRE((n + kMoeCols - 1) / kMoeCols <= 65535, "too many features for one launch");
  const dim3 grid(max_tiles, (n + kMoeCols - 1) / kMoeCols);
  if (mfma) {
    MLR_REQUIRE(mfma >= 1 && mfma <= 4, "mfma must be within 0..4");
    MLR_REQUIRE(dtype == kBF16 && k % 8 == 0, "the matrix-core kernels take bfloat16 and k % 8 == 0");
    MLR_REQUIRE(mfma == 1 || n % 8 == 0, "the tiled kernel needs n % 8 == 0");
    MLR_REQUIRE(reinterpret_cast<uintptr_t>(a) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(out) % 16 == 0,
                "a, w and out must be 16-byte aligned");
    // rows of `a`: the tokens for the first product, the pairs for the second; both fit 32-bit offsets
    const int64_t a_rows = up ? tokens : static_cast<int64_t>(tokens) * top;
    MLR_REQUIRE(a_rows * k * 2 < (1ll << 32) && static_cast<int64_t>(n) * k * 2 < (1ll << 31),
                "the inputs or one expert's matrix are too large for 32-bit offsets");
    const bf16* ab = static_cast<const bf16*>(a);
    const bf16* wb = static_cast<const bf16*>(w);
    const int rows = static_cast<int>(a_rows);
    if (mfma >= 2) {
      static const MoeTiles kinds[3][2] = {
          {{moe_gemm_tiled_kernel<false, 1>, 256, kBigCols, big_lds_bytes(1)}, {moe_gemm_tiled_kernel<true, 1>, 256, kBigCols, big_lds_bytes(1)}},
          {{moe_gemm_tiled_kernel<false, 2>, 256, kBigCols, big_lds_bytes(2)}, {moe_gemm_tiled_kernel<true, 2>, 256, kBigCols, big_lds_bytes(2)}},
          {{moe_gemm_phased_kernel<false>, 512, kSqCols, kSqLds}, {moe_gemm_phased_kernel<true>, 512, kSqCols, kSqLds}}};
      static bool configured[3][2] = {};
      const int status = launch_moe_tiled(kinds[mfma - 2][up != 0], configured[mfma - 2][up != 0], ab, wb, sorted, offsets, tiles, pair_weights,
                                          out, max_tiles, tokens, top, n, k, act, rows, glu_limit, glu_alpha, stream);
      if (status != 0) return -1;
    } else if (static_cast<int64_t>(n) * k * 2 >= (1ll << 20)) {
      // an expert's matrix of a megabyte or more: whole lines through LDS
      using StreamKernel = void (*)(const bf16*, const bf16*, const int*, const int*, const int*, const float*, void*, int, int, int, int, int,
                                    int, float, float);
      static const StreamKernel kinds[2][2] = {{moe_gemm_stream_kernel<false, 128>, moe_gemm_stream_kernel<true, 128>},
                                               {moe_gemm_stream_kernel<false, 64>, moe_gemm_stream_kernel<true, 64>}};
      static bool configured[2][2] = {};
      const bool narrow = narrow_steps_pay(max_tiles, static_cast<int64_t>(tokens) * top, static_cast<int64_t>(n) * k * 2);
      const int lds = stream_lds_bytes(narrow ? 64 : 128);
      const StreamKernel kernel = kinds[narrow][up != 0];
      if (!configured[narrow][up != 0]) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        MLR_REQUIRE(e == hipSuccess, std::string("cannot raise the LDS limit: ") + hipGetErrorString(e));
        configured[narrow][up != 0] = true;
      }
      hipLaunchKernelGGL(kernel, dim3(max_tiles, (n + kStCols - 1) / kStCols), dim3(256), lds, stream, ab, wb, sorted, offsets, tiles,
                         pair_weights, out, tokens, top, n, k, act, rows, glu_limit, glu_alpha);
    } else {
      // four wavefronts (64 features) a workgroup, or two where that leaves the compute units with too
      // few workgroups to keep their loads in flight
      const int waves = static_cast<int64_t>(max_tiles) * ((n + 63) / 64) < 2048 ? 2 : 4;
      const dim3 small_grid(max_tiles, (n + waves * 16 - 1) / (waves * 16));
      if (up)
        moe_gemm_mfma_kernel<true><<<small_grid, waves * kWave, 0, stream>>>(ab, wb, sorted, offsets, tiles, pair_weights, out, tokens, top, n, k, act, rows, glu_limit, glu_alpha);
      else
        moe_gemm_mfma_kernel<false><<<small_grid, waves * kWave, 0, stream>>>(ab, wb, sorted, offsets, tiles, pair_weights, out, tokens, top, n, k, act, rows, glu_limit, glu_alpha);
    }
    MLR_LAUNCH_CHECK();
    return 0;
  }
#define MLR_MOE_SIMPLE(T, UP)                                                                                  \
  moe_gemm_simple_kernel<T, UP><<<grid, 256, 0, stream>>>(static_cast<const T*>(a), static_cast<const T*>(w), \
                                                          sorted, offsets, tiles, pair_weights, out, tokens, top, n, k, act, \
                                                          glu_limit, glu_alpha)
  if (dtype == kF32) {
    if (up)
      MLR_MOE_SIMPLE(float, true);
    else
      MLR_MOE_SIMPLE(float, false);
  } else {
    if (up)
      MLR_MOE_SIMPLE(bf16, true);
    else
      MLR_MOE_SIMPLE(bf16, false);
  }
#undef MLR_MOE_SIMPLE
  MLR_LAUNCH_CHECK();
  return 0;
}

}  // extern "C"
