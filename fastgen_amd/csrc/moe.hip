// A routed feed-forward (mixture of experts) on the device, without a look of the host at what went
// where, so that a step with it can be recorded:
//
//  route    per token (a workgroup): fp32 router logits (x W_r^T + b), the `top` largest, softmax over those
//  sort     the (token, choice) pairs ordered by expert, cut into tiles of at most TM rows of one expert
//  gate_up  per tile: act = silu(x W_gate^T) * (x W_up^T) with the expert's matrices, rows gathered by token
//  down     per tile: y[pair] = act W_down^T in fp32, one row per pair
//  combine  out[t] = plus[t] + sum_j weight[t][j] * y[t * top + j], in fp32, j ascending
//
// Experts from a number on may be identities: the router scores them like the others, but the sort makes no tiles of
// their pairs and combine takes the token's own row of x for their output.
//
// A tile's rows do not depend on one another: every output element is one dot product over k in an
// order fixed by k alone, so a token's result is the same whatever else the step holds and wherever
// the sort puts it.  The bf16 kernels run on the matrix cores (v_mfma_f32_16x16x32_bf16, the expert's
// matrix as the A operand: 16 of its rows x 32 k, a tile's rows of x as B), one wave per 16 output
// channels of a tile, its matrices streamed once for up to 16 * MB rows; the generic kernels (fp32 FMA,
// any dtype and size) are the true 32-bit path.
//
// The matrix-core kernels take the experts' matrices row by row or packed (ldw = 0): per expert blocks of 16 rows x
// 32 k in operand order, [expert][ceil(rows / 16)][ceil(k / 32)][64 lanes][8], zeros behind the last row and k.  A
// wave's load is then 1 KB of whole lines; from rows it is 16 halves of a line, and the other halves are asked for
// again a step later.  A model keeps its experts packed; matrices in rows and tiles of 64 rows, nowhere the better ones, are
// there for callers of the products that hand them over so.
#include "tile_product.h"

#include <type_traits>

// ------------------------------------------------------------------- route
// A workgroup one token, four or eight.  Logits: the WAVES waves take the experts in turns of EPW (a wave
// reads the rows of x once for its EPW experts, eight elements a lane and round, and an expert's row of the router once
// for its tokens; the lanes' partial sums are added by the wave in a fixed order, the same in every form), into LDS.  A
// turn is a chain of reads from the L2, so many waves of two experts each and, for one token, four rounds' reads together (12 tokens in a step, router
// not in the L2: 9.7 -> 8.7 us; several tokens are bound by their multiplications); several tokens, or the router would be read
// from the L2 once a token.  From there on a wave a token: the `top` largest (ties:
// the lower expert) by a wave-wide argmax repeated `top` times, and the softmax over them.  LDS, per token: n_experts +
// n_extra logits, then `top` chosen values, then n_experts scores, then n_groups ranks.
//
// A second way of scoring (`sigmoid_scores`): an expert's score is sigmoid(logit); the choice goes by the
// score plus `correction` (per expert, or null), inside the `keep_groups` best of `n_groups` groups of
// neighbouring experts (a group's rank: the sum of its two largest choice scores; the experts of the other
// groups cannot be chosen); the weights are the chosen experts' scores without the correction, divided by
// their sum (+ 1e-20) and multiplied by `weight_scale`.  A third way (`sigmoid_scores` = 2): the scores are the
// softmax of the logits over all experts; choice, groups and weights as with sigmoid scores.  `group_max`: a group
// ranks by its largest choice score alone.  `raw_weights`: the chosen scores are not divided by their sum.
//
// `n_extra`: the router matrix has that many rows more than there are experts; their logits (no bias) take no
// part in the choice and are stored as they are in `extra [n_tokens, n_extra]` (a gate of a shared expert, say).
struct RouteMode {
  int sigmoid_scores;
  const float* correction;
  int n_groups, keep_groups;
  float weight_scale;
  int n_extra;
  float* extra;
  int group_max, raw_weights;
};
// A value over the wave's lanes, in every one of them, without a trip through the LDS crossbar: rotations within rows of
// 16 lanes, then rows and halves exchanged between two registers.
template <class OP>
__device__ __forceinline__ uint32_t moe_over_wave(uint32_t v, OP op) {
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x121 /* row_ror:1 */, 0xf, 0xf, false));
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, false));
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false));
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false));
  const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = op(a[0], a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return op(b[0], b[1]);
}
__device__ __forceinline__ float moe_wave_sum(float v) {
  return __uint_as_float(moe_over_wave(__float_as_uint(v), [](uint32_t a, uint32_t b) {
    return __float_as_uint(__uint_as_float(a) + __uint_as_float(b)); }));
}
__device__ __forceinline__ float moe_wave_max(float v) {
  return __uint_as_float(moe_over_wave(__float_as_uint(v), [](uint32_t a, uint32_t b) {
    return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b))); }));
}
__device__ __forceinline__ int moe_wave_min(int v) {
  return (int)moe_over_wave((uint32_t)v, [](uint32_t a, uint32_t b) { return (uint32_t)min((int)a, (int)b); });
}

// What a wave's lanes wrote to LDS is there for the wave's other lanes.
__device__ __forceinline__ void moe_wave_sync() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

template <class T, int WAVES, int EPW, int TOK>
__global__ __launch_bounds__(64 * WAVES) void moe_route_kernel(
    const T* __restrict__ x, int ldx, const float* __restrict__ wr, const float* __restrict__ bias, int n_tokens,
    int dim, int n_experts, int top, int* __restrict__ choice, float* __restrict__ weight, const RouteMode mode) {
  static_assert(TOK <= WAVES, "a wave a token");
  extern __shared__ float lds[];
  const int n_rows = n_experts + mode.n_extra;  // rows of the router matrix
  const int per_token = n_rows + top + n_experts + mode.n_groups;
  const int lane = threadIdx.x % FG_WAVE, wave = threadIdx.x / FG_WAVE;
  const int t0 = blockIdx.x * TOK;
  const T* xr[TOK];
#pragma unroll
  for (int i = 0; i < TOK; ++i) xr[i] = x + (size_t)min(t0 + i, n_tokens - 1) * ldx;
  for (int e0 = wave * EPW; e0 < n_rows; e0 += WAVES * EPW) {
    float s[EPW][TOK];
#pragma unroll
    for (int j = 0; j < EPW; ++j)
#pragma unroll
      for (int i = 0; i < TOK; ++i) s[j][i] = 0.f;
    if (dim % 8 == 0 && ldx % 8 == 0) {
      constexpr int U = TOK == 1 ? 4 : 1, EIGHT = FG_WAVE * 8;  // rounds whose loads are in flight together
      typedef uint4 XRaw[sizeof(T) / 2];
      auto rounds = [&](int k0, auto in_flight) {
        constexpr int N = in_flight.value;
        XRaw xraw[N][TOK];
        float4 wraw[N][EPW][2];
#pragma unroll
        for (int u = 0; u < N; ++u) {
          const int k = k0 + u * EIGHT;
#pragma unroll
          for (int i = 0; i < TOK; ++i)
#pragma unroll
            for (int h = 0; h < (int)sizeof(T) / 2; ++h) xraw[u][i][h] = ((const uint4*)(xr[i] + k))[h];
#pragma unroll
          for (int j = 0; j < EPW; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) wraw[u][j][h] = ((const float4*)(wr + (size_t)min(e0 + j, n_rows - 1) * dim + k))[h];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < N; ++u) {
          float xv[TOK][8];
#pragma unroll
          for (int i = 0; i < TOK; ++i) load8<T>((const T*)&xraw[u][i], xv[i]);
#pragma unroll
          for (int j = 0; j < EPW; ++j) {
            float wv[8];
            load8<float>((const float*)&wraw[u][j], wv);
#pragma unroll
            for (int i = 0; i < TOK; ++i)
#pragma unroll
              for (int e = 0; e < 8; ++e) s[j][i] = fmaf(xv[i][e], wv[e], s[j][i]);
          }
        }
      };
      int k0 = 0;
      for (; k0 + U * EIGHT <= dim; k0 += U * EIGHT) rounds(k0 + lane * 8, std::integral_constant<int, U>());
      if constexpr (U > 1)
        for (; k0 + EIGHT <= dim; k0 += EIGHT) rounds(k0 + lane * 8, std::integral_constant<int, 1>());
      if (k0 + lane * 8 < dim) rounds(k0 + lane * 8, std::integral_constant<int, 1>());
    } else {
      for (int k = lane; k < dim; k += FG_WAVE) {
        float xv[TOK];
#pragma unroll
        for (int i = 0; i < TOK; ++i) xv[i] = to_f<T>(xr[i][k]);
#pragma unroll
        for (int j = 0; j < EPW; ++j) {
          const float wv = wr[(size_t)min(e0 + j, n_rows - 1) * dim + k];
#pragma unroll
          for (int i = 0; i < TOK; ++i) s[j][i] = fmaf(xv[i], wv, s[j][i]);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < EPW; ++j)
#pragma unroll
      for (int i = 0; i < TOK; ++i) {
        const float v = moe_wave_sum(s[j][i]);
        if (lane == 0 && e0 + j < n_rows) lds[i * per_token + e0 + j] = v + (bias && e0 + j < n_experts ? bias[e0 + j] : 0.f);
      }
  }
  __syncthreads();
  const size_t t = t0 + wave;
  if (wave >= TOK || t >= (size_t)n_tokens) return;  // whole waves; no block barrier below
  float* z = lds + wave * per_token;
  float* chosen = z + n_rows;
  float* score = chosen + top;
  for (int e = lane; e < mode.n_extra; e += FG_WAVE) mode.extra[t * mode.n_extra + e] = z[n_experts + e];
  if (mode.sigmoid_scores) {  // uniform
    float top_z = 0.f, all = 1.f;
    if (mode.sigmoid_scores == 2) {
      top_z = -INFINITY;
      for (int e = lane; e < n_experts; e += FG_WAVE) top_z = fmaxf(top_z, z[e]);
      top_z = moe_wave_max(top_z);
      all = 0.f;
      for (int e = lane; e < n_experts; e += FG_WAVE) all += expf(z[e] - top_z);
      all = moe_wave_sum(all);
    }
    for (int e = lane; e < n_experts; e += FG_WAVE) {
      const float sc = mode.sigmoid_scores == 2 ? expf(z[e] - top_z) / all : 1.f / (1.f + expf(-z[e]));
      score[e] = sc;
      z[e] = sc + (mode.correction ? mode.correction[e] : 0.f);
    }
    moe_wave_sync();
    if (mode.n_groups > 1 && mode.keep_groups < mode.n_groups) {  // uniform
      // a lane a group, in turns: the groups are ranked and the experts of those that lose are struck
      float* rank = score + n_experts;  // n_groups values
      const int per = n_experts / mode.n_groups;
      for (int g = lane; g < mode.n_groups; g += FG_WAVE) {
        float a = -INFINITY, b = -INFINITY;  // the two largest
        for (int i = 0; i < per; ++i) {
          const float v = z[g * per + i];
          if (v > a) { b = a; a = v; } else if (v > b) { b = v; }
        }
        rank[g] = per > 1 && !mode.group_max ? a + b : a;
      }
      moe_wave_sync();
      for (int g = lane; g < mode.n_groups; g += FG_WAVE) {
        // a group stays if fewer than keep_groups groups rank before it (ties: the lower group first)
        int before = 0;
        const float mine = rank[g];
        for (int o = 0; o < mode.n_groups; ++o) before += (rank[o] > mine || (rank[o] == mine && o < g)) ? 1 : 0;
        if (before >= mode.keep_groups)
          for (int i = 0; i < per; ++i) z[g * per + i] = -INFINITY;
      }
      moe_wave_sync();
    }
  }
  for (int j = 0; j < top; ++j) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < n_experts; e += FG_WAVE) {
      const float v = z[e];
      if (v > best || (v == best && e < at)) { best = v; at = e; }
    }
    const float all_best = moe_wave_max(best);
    at = moe_wave_min(best == all_best ? at : 0x7fffffff);  // of equal values the lowest expert
    best = all_best;
    if (lane == 0) {
      at = min(at, n_experts - 1);  // (only if every logit is NaN)
      z[at] = -INFINITY;
      chosen[j] = mode.sigmoid_scores ? score[at] : best;
      choice[t * top + j] = at;
    }
    moe_wave_sync();
  }
  if (lane == 0 && mode.sigmoid_scores) {
    float sum = 0.f;
    for (int j = 0; j < top; ++j) sum += chosen[j];
    for (int j = 0; j < top; ++j) weight[t * top + j] = (mode.raw_weights ? chosen[j] : chosen[j] / (sum + 1e-20f)) * mode.weight_scale;
  } else if (lane == 0) {
    const float m = chosen[0];  // the largest
    float sum = 0.f;
    for (int j = 0; j < top; ++j) sum += expf(chosen[j] - m);
    for (int j = 0; j < top; ++j) weight[t * top + j] = expf(chosen[j] - m) / sum;
  }
}

extern "C" int fg_moe_route_mode(const void* x, int ldx, int dtype, const float* wr, const float* bias, int n_tokens,
                                 int dim, int n_experts, int top, int* choice, float* weight, int sigmoid_scores,
                                 const float* correction, int n_groups, int keep_groups, float weight_scale,
                                 int n_extra, float* extra, int group_max, int raw_weights, hipStream_t stream) {
  if (n_tokens <= 0) return FG_OK;
  if (sigmoid_scores < 0 || sigmoid_scores > 2 || n_extra < 0 || (n_extra > 0 && !extra)) return FG_ERR_ARG;
  if (dim <= 0 || ldx < dim || n_experts <= 0 || top < 1 || top > n_experts) return FG_ERR_ARG;
  if (n_groups < 1 || n_experts % n_groups || keep_groups < 1 || keep_groups > n_groups ||
      top > keep_groups * (n_experts / n_groups) || (!sigmoid_scores && (correction || n_groups > 1)))
    return FG_ERR_ARG;
  const RouteMode mode = {sigmoid_scores, correction, n_groups, keep_groups, weight_scale, n_extra, extra, group_max, raw_weights};
  const size_t lds = (size_t)(2 * n_experts + n_extra + top + n_groups) * sizeof(float);  // a token's
  if (lds > 60000) return FG_ERR_ARG;
#define GO(T, WAVES, EPW, TOK)                                                                                        \
  moe_route_kernel<T, WAVES, EPW, TOK><<<(n_tokens + TOK - 1) / TOK, 64 * WAVES, TOK * lds, stream>>>(                 \
      (const T*)x, ldx, wr, bias, n_tokens, dim, n_experts, top, choice, weight, mode)
  // Tokens a workgroup: one while every token's workgroup has a place at once, then four, then eight, as their logits fit.
  // Waves: 16 of two rows a turn, or 8 where the router has no more than 16 rows, twice as many of which have a place.  bf16, router in the caches, us, 32
  // experts of 2048 with 4 waves of four rows before: 65 / 300 / 700 / 1024 / 1897 / 6000 tokens 6.6 / 9.8 / 10.2 / 11.1 / 13.9
  // / 36.5 against 10.0 / 10.7 / 12.4 / 15.6 / 17.0 / 38.3; 128 of 4096 25.7 / 41 / 48 / 55 / 74 / 206 against 49 / 52 / 61 / 74 /
  // 100 / 274; 16 of 1024 4.0 / 4.7 / 5.7 / 5.9 / 7.3 / 14.1 against 4.9 / 5.1 / 5.6 / 6.2 / 7.8 / 15.0 (512 tokens: one a
  // workgroup 5.1, four 5.5; 700: both 5.7).
  const bool few_rows = n_experts + n_extra <= 16;
  const int tok = n_tokens <= (few_rows ? 512 : 256) || 4 * lds > 60000 ? 1 : n_tokens <= 1280 || 8 * lds > 60000 ? 4 : 8;
#define FORMS(T)                                                   \
  do {                                                             \
    if (tok == 1 && few_rows) GO(T, 8, 2, 1);                      \
    else if (tok == 1) GO(T, 16, 2, 1);                            \
    else if (tok == 4 && few_rows) GO(T, 8, 2, 4);                 \
    else if (tok == 4) GO(T, 16, 2, 4);                            \
    else if (few_rows) GO(T, 8, 2, 8);                             \
    else GO(T, 16, 2, 8);                                          \
  } while (0)
  if (dtype == FG_F32) FORMS(float);
  else if (dtype == FG_BF16) FORMS(bf16_t);
  else return FG_ERR_ARG;
#undef FORMS
#undef GO
  return fg_launch_status();
}

extern "C" int fg_moe_route(const void* x, int ldx, int dtype, const float* wr, const float* bias, int n_tokens, int dim,
                            int n_experts, int top, int* choice, float* weight, hipStream_t stream) {
  return fg_moe_route_mode(x, ldx, dtype, wr, bias, n_tokens, dim, n_experts, top, choice, weight, 0, nullptr, 1, 1, 1.f,
                           0, nullptr, 0, 0, stream);
}

// -------------------------------------------------------------------- sort
// One workgroup.  sorted[pos] = pair (token * top + j) for the pairs in the order of their experts;
// tiles[i] = (expert, first pos, rows, 0) for i < max_tiles, rows = 0 for tiles that do not exist.  Experts from
// n_tiled on have no tiles.
// LDS: 3 * n_experts ints (count, first pos, first tile).
// Up to HELD pairs a thread are read once, all at the same time, and keep their number among their expert's from the count; more are read
// and numbered again.  As many as there are: eight held places for one pair a thread cost what they spare.  32 experts, us read twice and
// held, in eight places and in as many: 260 pairs 2.57, 3.03, 2.53, 1,000 2.93, 3.29, 2.73, 2,040 3.49, 3.52, 3.14, 4,000 4.62, 4.24, 3.95, 8,192 7.02, 5.83.
template <int SORT_THREADS, int HELD>
__global__ __launch_bounds__(SORT_THREADS) void moe_sort_kernel(
    const int* __restrict__ choice, int n_pairs, int n_experts, int n_tiled, int tile_rows, int max_tiles,
    int* __restrict__ sorted, int* __restrict__ tiles) {
  extern __shared__ int sm[];
  int* count = sm;
  int* first = sm + n_experts;
  int* first_tile = sm + 2 * n_experts;
  for (int e = threadIdx.x; e < n_experts; e += SORT_THREADS) count[e] = 0;
  const bool held = n_pairs <= HELD * SORT_THREADS;  // uniform
  int expert[HELD], number[HELD];
  if (held) {
#pragma unroll
    for (int i = 0; i < HELD; ++i) expert[i] = choice[min((int)threadIdx.x + i * SORT_THREADS, n_pairs - 1)];
#pragma unroll
    for (int i = 0; i < HELD; ++i) expert[i] = min(max(expert[i], 0), n_experts - 1);
  }
  __syncthreads();
  if (held) {
#pragma unroll
    for (int i = 0; i < HELD; ++i)
      if ((int)threadIdx.x + i * SORT_THREADS < n_pairs) number[i] = atomicAdd(&count[expert[i]], 1);
  } else {
    for (int p = threadIdx.x; p < n_pairs; p += SORT_THREADS) atomicAdd(&count[min(max(choice[p], 0), n_experts - 1)], 1);
  }
  __syncthreads();
  if (threadIdx.x < FG_WAVE) {  // exclusive sums of rows and of tiles, 64 experts a round
    const int lane = threadIdx.x;
    int rows_before = 0, tiles_before = 0;
    for (int base = 0; base < n_experts; base += FG_WAVE) {
      const int e = base + lane;
      const int c = e < n_experts ? count[e] : 0;
      const int nt = e < n_tiled ? (c + tile_rows - 1) / tile_rows : 0;
      int sc = c, st = nt;
#pragma unroll
      for (int d = 1; d < FG_WAVE; d <<= 1) {
        const int uc = __shfl_up(sc, d, FG_WAVE), ut = __shfl_up(st, d, FG_WAVE);
        if (lane >= d) { sc += uc; st += ut; }
      }
      if (e < n_experts) {
        first[e] = rows_before + sc - c;
        first_tile[e] = tiles_before + st - nt;
      }
      rows_before += __shfl(sc, FG_WAVE - 1, FG_WAVE);
      tiles_before += __shfl(st, FG_WAVE - 1, FG_WAVE);
    }
    // tiles that do not exist
    for (int i = tiles_before + lane; i < max_tiles; i += FG_WAVE) *(int4*)(tiles + 4 * (size_t)i) = make_int4(0, 0, 0, 0);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n_experts; e += SORT_THREADS) {
    const int c = count[e], f = first[e];
    for (int i = 0, r = 0; r < c && e < n_tiled; ++i, r += tile_rows) {
      const int at = first_tile[e] + i;
      if (at < max_tiles) *(int4*)(tiles + 4 * (size_t)at) = make_int4(e, f + r, min(tile_rows, c - r), 0);
    }
    count[e] = 0;  // now the cursor of the second pass
  }
  if (held) {
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      const int p = threadIdx.x + i * SORT_THREADS;
      if (p < n_pairs) sorted[first[expert[i]] + number[i]] = p;
    }
    return;
  }
  __syncthreads();
  for (int p = threadIdx.x; p < n_pairs; p += SORT_THREADS) {
    const int e = min(max(choice[p], 0), n_experts - 1);
    sorted[first[e] + atomicAdd(&count[e], 1)] = p;
  }
}

extern "C" int fg_moe_sort(const int* choice, int n_pairs, int n_experts, int n_tiled, int tile_rows, int max_tiles,
                           int* sorted, int* tiles, hipStream_t stream) {
  if (n_pairs <= 0) return FG_OK;
  if (n_experts <= 0 || n_tiled < 0 || n_tiled > n_experts || tile_rows <= 0 || max_tiles <= 0 || (size_t)3 * n_experts * sizeof(int) > 60000) return FG_ERR_ARG;
  const size_t lds = (size_t)3 * n_experts * sizeof(int);
#define SORT(THREADS, HELD) \
  moe_sort_kernel<THREADS, HELD><<<1, THREADS, lds, stream>>>(choice, n_pairs, n_experts, n_tiled, tile_rows, max_tiles, sorted, tiles)
  if (n_pairs <= 256 && n_experts <= 256) SORT(256, 1);
  else if (n_pairs <= 1024) SORT(1024, 1);
  else if (n_pairs <= 2048) SORT(1024, 2);
  else if (n_pairs <= 4096) SORT(1024, 4);
  else SORT(1024, 8);
#undef SORT
  return fg_launch_status();
}

// ------------------------------------------------------------ generic tiles
// fp32 FMA; a thread owns one (row, channel) and sums k ascending in partial sums of 16.
// Tiles of 16 rows; 256 threads: row = tid / 16, channel = blockIdx.y * 16 + tid % 16.
template <class T>
__device__ __forceinline__ float dot_ordered(const T* __restrict__ a, const T* __restrict__ b, int K) {
  float total = 0.f;
  for (int k0 = 0; k0 < K; k0 += 16) {
    float part = 0.f;
    const int k1 = min(K, k0 + 16);
    for (int k = k0; k < k1; ++k) part = fmaf(to_f<T>(a[k]), to_f<T>(b[k]), part);
    total += part;
  }
  return total;
}

template <class T>
__global__ __launch_bounds__(256) void moe_gate_up_generic_kernel(
    const T* __restrict__ x, int ldx, const T* __restrict__ wg, const T* __restrict__ wu, int ldw /* row stride of wg, wu */,
    const int* __restrict__ sorted, const int* __restrict__ tiles, int top, int dim, int hidden, T* __restrict__ act,
    int lda, const GatedAct fn) {
  const int4 tile = *(const int4*)(tiles + 4 * (size_t)blockIdx.x);
  const int r = threadIdx.x / 16, c = blockIdx.y * 16 + threadIdx.x % 16;
  if (r >= tile.z || c >= hidden) return;
  const int pos = tile.y + r;
  const T* xr = x + (size_t)(sorted[pos] / top) * ldx;
  const size_t wrow = ((size_t)tile.x * hidden + c) * ldw;
  const float g = dot_ordered<T>(xr, wg + wrow, dim), u = dot_ordered<T>(xr, wu + wrow, dim);
  act[(size_t)pos * lda + c] = from_f<T>(gated_act<false>(g, u, fn));
}

template <class T>
__global__ __launch_bounds__(256) void moe_down_generic_kernel(
    const T* __restrict__ act, int lda, const T* __restrict__ wd, int ldw, const int* __restrict__ sorted,
    const int* __restrict__ tiles, int dim, int hidden, float* __restrict__ y) {
  const int4 tile = *(const int4*)(tiles + 4 * (size_t)blockIdx.x);
  const int r = threadIdx.x / 16, c = blockIdx.y * 16 + threadIdx.x % 16;
  if (r >= tile.z || c >= dim) return;
  const int pos = tile.y + r;
  y[(size_t)sorted[pos] * dim + c] = dot_ordered<T>(act + (size_t)pos * lda, wd + ((size_t)tile.x * dim + c) * ldw, hidden);
}

// --------------------------------------------------------------- MFMA tiles
// One wave per (tile, 16 output channels); a tile has up to 16 * MB rows.  Lane 16 g + r holds, of the A
// operand, row r of the 16 matrix rows at k 8 g .. 8 g + 7, and of B the same k of the tile's row r.
__device__ __forceinline__ bf16x8 moe_zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.f;
  return z;
}
// What lies 32 s elements behind a lane's first chunk (k 8 g) of a row, or, if that is beyond k, a chunk that is there.
__device__ __forceinline__ int moe_k_at(int s, int K, int g) {
  return 32 * s + 8 * g < K ? 32 * s : (8 * g < K ? 0 : -8 * g);
}

// Where a lane finds its part of 16 matrix rows from `row` on at step s of 32 k: at base + s * stride elements.
template <bool PACKED>
struct MoeOperand {
  const bf16_t* base;
  __device__ __forceinline__ MoeOperand() {}
  __device__ __forceinline__ MoeOperand(const bf16_t* w, int ldw, int expert, int rows, int row, int K, int lane) {
    if constexpr (PACKED) {
      const int blocks = (rows + 15) / 16, steps = (K + 31) / 32;
      base = w + ((size_t)expert * blocks + min(row / 16, blocks - 1)) * steps * 512 + lane * 8;
    } else {
      base = w + ((size_t)expert * rows + min(row + lane % 16, rows - 1)) * ldw + 8 * (lane / 16);
    }
  }
  // (behind k: any readable place; what stands there is replaced by zeros before it is multiplied)
  __device__ __forceinline__ bf16x8 load(int s, int K, int g) const {
    if constexpr (PACKED) return *(const bf16x8*)(base + (size_t)(32 * s < K ? s : 0) * 512);
    else return *(const bf16x8*)(base + moe_k_at(s, K, g));
  }
};

// The products of up to 16 MB rows of x (B operands at px) with NM blocks of 16 matrix rows: a wave alone streams the
// matrices, U steps of 32 k a round, the next round's loads in flight while a round is multiplied.
template <int NM, int MB, bool PACKED>
__device__ __forceinline__ void moe_stream(const MoeOperand<PACKED> (&w)[NM], const bf16_t* const (&px)[MB], int K, int g,
                                           f32x4 (&acc)[NM][MB]) {
  constexpr int U = MB == 1 ? 4 : 2;
  bf16x8 a[2][U][NM], b[2][U][MB];
  auto load = [&](int s0, int set) {
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int m = 0; m < NM; ++m) a[set][i][m] = w[m].load(s0 + i, K, g);
#pragma unroll
    for (int i = 0; i < U; ++i)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) b[set][i][mb] = *(const bf16x8*)(px[mb] + moe_k_at(s0 + i, K, g));
  };
  // (where k ends inside the steps: zeros in both operands behind it, an infinity times a zero would be no number)
  auto multiply = [&](int s0, int set, auto ends) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const bool in = !ends.value || 32 * (s0 + i) + 8 * g < K;
      bf16x8 av[NM];
#pragma unroll
      for (int m = 0; m < NM; ++m) av[m] = in ? a[set][i][m] : moe_zero8();
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const bf16x8 bv = in ? b[set][i][mb] : moe_zero8();
#pragma unroll
        for (int m = 0; m < NM; ++m) acc[m][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], bv, acc[m][mb], 0, 0, 0);
      }
    }
  };
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[m][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (K + 31) / 32;
  load(0, 0);
  int s = 0;
  for (; 32 * (s + 2 * U) <= K; s += 2 * U) {
    load(s + U, 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(s, 0, std::false_type());
    load(s + 2 * U, 0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(s + U, 1, std::false_type());
  }
  if (s < steps) {
    load(s + U, 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(s, 0, std::true_type());
    multiply(s + U, 1, std::true_type());
  }
}

// Bound by the experts' matrices (12 tokens of 32 experts of 768 x 2048, top 4: 161 and 80 MB): 39 / 21 us from packed
// matrices, 54 / 24 from rows (and 50 / 23 with rounds of 8 steps whose loads all returned before the next were asked for);
// one token 16.5 / 8.2 us (23.7 / 9.3 from rows).
template <int MB, bool PACKED>
__global__ __launch_bounds__(256) void moe_gate_up_mfma_kernel(
    const bf16_t* __restrict__ x, int ldx, const bf16_t* __restrict__ wg, const bf16_t* __restrict__ wu, int ldw,
    const int* __restrict__ sorted, const int* __restrict__ tiles, int max_tiles, int top, int dim, int hidden,
    bf16_t* __restrict__ act, int lda, const GatedAct fn) {
  const int lane = threadIdx.x % FG_WAVE, wave = threadIdx.x / FG_WAVE;
  const int cblocks = (hidden + 15) / 16;
  const int item = blockIdx.x * 4 + wave;
  const int ti = item / cblocks, c0 = (item % cblocks) * 16;
  if (ti >= max_tiles) return;
  const int4 tile = *(const int4*)(tiles + 4 * (size_t)ti);
  if (tile.z <= 0) return;
  const int r16 = lane & 15, g = lane >> 4;
  // (rows beyond the matrix: clamped, not stored)
  const MoeOperand<PACKED> w[2] = {{wg, ldw, tile.x, hidden, c0, dim, lane}, {wu, ldw, tile.x, hidden, c0, dim, lane}};
  const bf16_t* px[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int r = min(mb * 16 + r16, tile.z - 1);
    px[mb] = x + (size_t)(sorted[tile.y + r] / top) * ldx + 8 * g;
  }
  f32x4 acc[2][MB];
  moe_stream<2, MB, PACKED>(w, px, dim, g, acc);
  // the lane holds, for the tile's row mb * 16 + r16, channels c0 + 4 g .. + 3
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int r = mb * 16 + r16, c = c0 + 4 * g;
    if (r >= tile.z || c >= hidden) continue;
    bf16x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[i] = (__bf16)gated_act<true>(acc[0][mb][i], acc[1][mb][i], fn);
    }
    bf16_t* dst = act + (size_t)(tile.y + r) * lda + c;
    if (c + 3 < hidden) {
      *(bf16x4*)dst = o;
    } else {
      for (int i = 0; c + i < hidden; ++i) dst[i] = o[i];
    }
  }
}

template <int MB, bool PACKED>
__global__ __launch_bounds__(256) void moe_down_mfma_kernel(
    const bf16_t* __restrict__ act, int lda, const bf16_t* __restrict__ wd, int ldw, const int* __restrict__ sorted,
    const int* __restrict__ tiles, int max_tiles, int dim, int hidden, float* __restrict__ y) {
  const int lane = threadIdx.x % FG_WAVE, wave = threadIdx.x / FG_WAVE;
  const int cblocks = (dim + 15) / 16;
  const int item = blockIdx.x * 4 + wave;
  const int ti = item / cblocks, c0 = (item % cblocks) * 16;
  if (ti >= max_tiles) return;
  const int4 tile = *(const int4*)(tiles + 4 * (size_t)ti);
  if (tile.z <= 0) return;
  const int r16 = lane & 15, g = lane >> 4;
  const MoeOperand<PACKED> w[1] = {{wd, ldw, tile.x, dim, c0, hidden, lane}};
  const bf16_t* pa[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) pa[mb] = act + (size_t)(tile.y + min(mb * 16 + r16, tile.z - 1)) * lda + 8 * g;
  f32x4 acc[1][MB];
  moe_stream<1, MB, PACKED>(w, pa, hidden, g, acc);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int r = mb * 16 + r16, c = c0 + 4 * g;
    if (r >= tile.z || c >= dim) continue;
    float* dst = y + (size_t)sorted[tile.y + r] * dim + c;
    if (c + 3 < dim && dim % 4 == 0) {
      *(f32x4*)dst = acc[0][mb];
    } else {
      for (int i = 0; c + i < dim; ++i) dst[i] = acc[0][mb][i];
    }
  }
}

// ------------------------------------------------------- large tiles
// Many rows an expert (prompt steps): a workgroup owns a tile of up to 128 WM rows of one expert and 256 rows of its
// matrix, a wave 128 x 64.  A compute unit takes in 64 bytes a clock from the vector memory path and reads 128 from LDS,
// and a wave's tile of 64 x 64 with both operands through LDS (the loop of gemm_tiled.hip) needs all of the one and one
// and a half times the other at the matrix cores' full rate.  So the rows of x, which the waves share, go through LDS
// and the rows of the matrix, which are a wave's own, from memory into its registers in operand order: 48 bytes a clock
// and 0.6 of LDS.  Rows of x are asked for two steps of 32 k ahead (registers, then one of two LDS buffers), rows of the
// matrix three; one barrier a step.  1897 tokens, 32 experts of 768 x 2048, top 4 (237 rows an expert, 48 + 24 GFLOP): 86 /
// 67 us, 116 / 83 with the matrices in rows, 150 / 87 with tiles of 64 x 64 a wave; 6000 tokens 182 / 142 us against 344 /
// 210, 0.83 / 0.53 PFLOP/s.  The tile's rows are gathered by token (gate_up) or are its sorted places (down);
// for gate_up the first half of a wave's blocks of 16 matrix rows are gate rows and the second half the up rows of the
// same channels, so that silu(gate) * up is applied to the accumulators.
#define MT_GATE_UP 0
#define MT_DOWN 1
#define MT_RUN 4

template <int WM, int NB, bool PACKED, int EPI>
__global__ __launch_bounds__(256 * WM, 2) void moe_tiled_kernel(
    const bf16_t* __restrict__ x, int ldx, const bf16_t* __restrict__ w0, const bf16_t* __restrict__ w1, int ldw,
    void* __restrict__ y, int ldy, const int* __restrict__ sorted, const int* __restrict__ tiles, int max_tiles, int top,
    int N /* columns of the result: hidden (gate_up), dim (down) */, int K, const GatedAct fn) {
  constexpr int XB = 8 * WM, BLOCK = 16 * 32;  // blocks of 16 rows of x; each lies in LDS as its lanes' operands
  constexpr int WAVE_N = EPI == MT_GATE_UP ? 8 * NB : 16 * NB, COLS = 4 * WAVE_N;  // columns of a wave, of the workgroup
  __shared__ __attribute__((aligned(16))) bf16_t xs[2][XB][BLOCK];
  // a run of MT_RUN tiles (an expert's mostly) and one block of columns stays on one die, whose L2 the matrix is read
  // into once
  const int cols = (N + COLS - 1) / COLS, place = blockIdx.x / 8, run = place / MT_RUN * 8 + blockIdx.x % 8;
  const int ti = run / cols * MT_RUN + place % MT_RUN;
  if (ti >= max_tiles) return;
  const int4 tile = *(const int4*)(tiles + 4 * (size_t)ti);
  if (tile.z <= 0) return;  // (the whole workgroup)
  const int lane = threadIdx.x % FG_WAVE, wave = threadIdx.x / FG_WAVE;
  const int r16 = lane & 15, g = lane >> 4;
  const int wm = wave / 4, wn = wave % 4;
  const int n_base = run % cols * COLS + wn * WAVE_N;
  const int n_steps = (K + 31) / 32;

  const bf16_t* xsrc[2];  // a wave brings two blocks of x a step
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int pos = tile.y + min(16 * (wave + 4 * WM * j) + r16, tile.z - 1);  // rows beyond the tile: its last row, not stored
    xsrc[j] = x + (size_t)(EPI == MT_GATE_UP ? sorted[pos] / top : pos) * ldx + 8 * g;
  }
  MoeOperand<PACKED> w[NB];  // gate_up: the first half gate rows, the second the up rows of the same channels
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
    w[nb] = EPI == MT_DOWN ? MoeOperand<PACKED>(w0, ldw, tile.x, N, n_base + 16 * nb, K, lane)
                           : MoeOperand<PACKED>(nb < NB / 2 ? w0 : w1, ldw, tile.x, N, n_base + 16 * (nb % (NB / 2)), K, lane);
  bf16x8 xr[2][2], wr[4][NB];
  f32x4 acc[8][NB];  // [row block mb][matrix block nb]
#pragma unroll
  for (int mb = 0; mb < 8; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};

  // what step s needs (a chunk beyond k is any readable one)
  auto load_x = [&](int s, bf16x8(&to)[2]) {
    const int at = moe_k_at(s, K, g);
#pragma unroll
    for (int j = 0; j < 2; ++j) to[j] = *(const bf16x8*)(xsrc[j] + at);
  };
  auto load_w = [&](int s, bf16x8(&to)[NB]) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) to[nb] = w[nb].load(s, K, g);
  };
  auto store_x = [&](int s, int buf, const bf16x8(&from)[2]) {
    const bool in = 32 * s + 8 * g < K;  // (asked here: behind the load it would wait for the load)
#pragma unroll
    for (int j = 0; j < 2; ++j) *(bf16x8*)(&xs[buf][wave + 4 * WM * j][lane * 8]) = in ? from[j] : moe_zero8();
  };
  load_x(0, xr[0]);
  load_w(0, wr[0]);
  load_x(1, xr[1]);
  load_w(1, wr[1]);
  load_w(2, wr[2]);
  store_x(0, 0, xr[0]);
  __syncthreads();
  // Four steps a round, so that the register sets have fixed names, in one block of code: with an exit between them
  // the compiler moves the loads behind it, to where their results are used.  The last round, if k ends inside it, is
  // code of its own, with zeros in both operands behind k (an infinity of the chunk read instead, times a zero of the
  // other operand, would be no number).
  auto round = [&](int i0, auto ends) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = i0 + u;
      load_x(i + 2, xr[u % 2]);
      load_w(i + 3, wr[(u + 3) % 4]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (ends.value) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) wr[u % 4][nb] = 32 * i + 8 * g < K ? wr[u % 4][nb] : moe_zero8();
      }
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        bf16x8 b[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) b[m] = *(const bf16x8*)(&xs[u % 2][8 * wm + 4 * half + m][lane * 8]);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int m = 0; m < 4; ++m)
            acc[4 * half + m][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[u % 4][nb], b[m], acc[4 * half + m][nb], 0, 0, 0);
      }
      store_x(i + 1, (u + 1) % 2, xr[(u + 1) % 2]);
      __syncthreads();
    }
  };
  int i0 = 0;
  for (; 32 * (i0 + 4) <= K; i0 += 4) round(i0, std::false_type());
  if (i0 < n_steps) round(i0, std::true_type());

  // acc[mb][nb][i]: the tile's row 128 wm + 16 mb + r16, row 4 g + i of the matrix block nb
#pragma unroll
  for (int mb = 0; mb < 8; ++mb) {
    const int ml = 128 * wm + 16 * mb + r16;
    if (ml >= tile.z) continue;
    const int pos = tile.y + ml;
    if constexpr (EPI == MT_DOWN) {
      float* row = (float*)y + (size_t)sorted[pos] * ldy;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int n = n_base + 16 * nb + 4 * g;
        if (n + 3 < N && (ldy & 3) == 0) {
          *(f32x4*)(row + n) = acc[mb][nb];
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (n + i < N) row[n + i] = acc[mb][nb][i];
        }
      }
    } else {
#pragma unroll
      for (int nb = 0; nb < NB / 2; ++nb) {
        const int n = n_base + 16 * nb + 4 * g;
        bf16x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (__bf16)gated_act<true>(acc[mb][nb][i], acc[mb][nb + NB / 2][i], fn);
        if (n < N) *(bf16x4*)((bf16_t*)y + (size_t)pos * ldy + n) = v;  // (N is a multiple of 8)
      }
    }
  }
}

template <int WM, int NB, int EPI>
static int launch_moe_tiled_as(const void* x, int ldx, const void* w0, const void* w1, int ldw, void* y, int ldy,
                               const int* sorted, const int* tiles, int max_tiles, int top, int N, int K, const GatedAct fn,
                               hipStream_t stream) {
  constexpr int COLS = (EPI == MT_GATE_UP ? 32 : 64) * NB;
  const long long runs = (long long)((max_tiles + MT_RUN - 1) / MT_RUN) * ((N + COLS - 1) / COLS);
  const long long grid = (runs + 7) / 8 * 8 * MT_RUN;
  if (grid > 2147483647LL) return FG_ERR_ARG;
  if (ldw == 0)
    moe_tiled_kernel<WM, NB, true, EPI><<<(unsigned)grid, 256 * WM, 0, stream>>>(
        (const bf16_t*)x, ldx, (const bf16_t*)w0, (const bf16_t*)w1, ldw, y, ldy, sorted, tiles, max_tiles, top, N, K, fn);
  else
    moe_tiled_kernel<WM, NB, false, EPI><<<(unsigned)grid, 256 * WM, 0, stream>>>(
        (const bf16_t*)x, ldx, (const bf16_t*)w0, (const bf16_t*)w1, ldw, y, ldy, sorted, tiles, max_tiles, top, N, K, fn);
  return fg_launch_status();
}

template <int WM, int EPI>
static int launch_moe_tiled(const void* x, int ldx, const void* w0, const void* w1, int ldw, void* y, int ldy,
                            const int* sorted, const int* tiles, int max_tiles, int top, int N, int K, const GatedAct fn,
                            hipStream_t stream) {
  // Narrow matrix tiles (a wave 128 x 32) while wide ones would leave a third of the compute units without a workgroup.
  // Measured (us, gate_up / down, packed, narrow against wide): 16 experts of 704 x 1024, top 2, 700 tokens (at most 26
  // tiles, 156 / 104 wide workgroups) 24 / 20 against 29 / 24, 1897 tokens (270 / 180) 35 / 31 against 31 / 27; 32 of 768 x
  // 2048, top 4, 700 tokens (318 / 424) 59 / 34 against 51 / 33.
  const long long wide = (long long)max_tiles * ((N + (EPI == MT_GATE_UP ? 127 : 255)) / (EPI == MT_GATE_UP ? 128 : 256));
  if (wide < 170)
    return launch_moe_tiled_as<WM, 2, EPI>(x, ldx, w0, w1, ldw, y, ldy, sorted, tiles, max_tiles, top, N, K, fn, stream);
  return launch_moe_tiled_as<WM, 4, EPI>(x, ldx, w0, w1, ldw, y, ldy, sorted, tiles, max_tiles, top, N, K, fn, stream);
}

// The same with packed matrices and k in multiples of 64: tile_product.h, 256 columns of the matrix a workgroup.  A tile of up to 64,
// of up to 128 rows is a product of that many, so an expert's last tile costs no more than it holds.  Bound by the matrices, which
// reach a die once, and by what a tile takes beside its product (14 us: the launch, its first loads, its last stores).  2,048
// tokens, 32 experts of 768 x 2048, top 4 (256 rows an expert; 201 and 101 MB of matrices, 48 + 24 GFLOP): 72 / 57 us with tiles of
// 256 rows, 79 / 61 of 128, 85 / 71 in the kernel above; 1,024 tokens 59 / 38 against 78 / 51; 4,096 117 / 97 against 148 / 106; 130
// tokens 40 / 22.5 against 47 / 26 with tiles of 32 rows and no LDS.
template <int MB, int NB, int NST, int WS, bool ONE_WAVE, int EPI>
__device__ __forceinline__ void moe_large_tile(bf16_t* lds, const bf16_t* x, unsigned x_bytes, int ldx, const bf16_t* w0,
                                               const bf16_t* w1, void* y, int ldy, const int* sorted, const int4 tile, int ct,
                                               int top, int N, int K, const GatedAct fn) {
#ifdef __HIP_DEVICE_COMPILE__
  typedef TileProduct<MB, NB, NST, WS, ONE_WAVE> Product;
  constexpr int WAVE_N = EPI == MT_GATE_UP ? 8 * NB : 16 * NB;
  const int lane = threadIdx.x % FG_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FG_WAVE);
  const int r16 = lane & 15, g = lane >> 4;
  const int n_base = (ct * 4 + wave) * WAVE_N, blocks = (N + 15) / 16, block = n_base / 16;
  TileOperands op;
  op.x = EPI == MT_GATE_UP ? (const void*)x : (const void*)(x + (size_t)tile.y * ldx);
  op.x_bytes = EPI == MT_GATE_UP ? x_bytes : 2u * (unsigned)((tile.z - 1) * ldx + K);
  op.w_row = (unsigned)K * 32u;
  const size_t expert = (size_t)tile.x * blocks * op.w_row;
  op.set_w(0, (const char*)w0 + expert, block, blocks, Product::HALF);
  if constexpr (EPI == MT_GATE_UP) op.set_w(1, (const char*)w1 + expert, block, blocks, NB - Product::HALF);
  else op.set_w(1, (const char*)w0 + expert, block + Product::HALF, blocks, NB - Product::HALF);
  unsigned xo[Product::XL];
#pragma unroll
  for (int j = 0; j < Product::XL; ++j) {
    const int row = Product::row_of(wave, j, lane);
    const int from = EPI == MT_GATE_UP ? sorted[tile.y + min(row, tile.z - 1)] / top : row;
    xo[j] = op.row_offset(row < tile.z, from, ldx, Product::chunk_of(lane));
  }
  f32x4 acc[MB][NB];
  Product::run(lds, op, xo, wave, lane, 0, K / 64, K / 64, acc);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int ml = 16 * mb + r16;
    const bool there = ml < tile.z;
    const int pos = tile.y + ml;
    if constexpr (EPI == MT_DOWN) {
      float* row = (float*)y + (size_t)(there ? sorted[pos] : 0) * ldy;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const f32x4 sum = Product::sums(acc[mb][nb]);
        const int n = n_base + 16 * nb + 4 * g;
        if (there && n + 3 < N && (ldy & 3) == 0) {
          *(f32x4*)(row + n) = sum;
        } else if (there) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (n + i < N) row[n + i] = sum[i];
        }
      }
    } else {
#pragma unroll
      for (int nb = 0; nb < NB / 2; ++nb) {
        const f32x4 gate = Product::sums(acc[mb][nb]), up = Product::sums(acc[mb][nb + NB / 2]);
        const int n = n_base + 16 * nb + 4 * g;
        bf16x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (__bf16)gated_act<true>(gate[i], up[i], fn);
        if (there && n < N) *(bf16x4*)((bf16_t*)y + (size_t)pos * ldy + n) = v;  // (N is a multiple of 8)
      }
    }
  }
#endif
}

// What workgroup `place` of die `die` does: a tile (rows 0: nothing) and a block of columns.
// Up to 64 tiles, which a wave sees at once: those of more than 128 rows come first and those of up to 64 last, so that no long one
// begins when the others end.  An expert's tiles, in runs of up to MT_RUN, and one block of columns are one die's, whose L2 that part of the
// matrix is read into once; runs and blocks of columns are dealt to the dies in turn, and a die's workgroups are counted
// without gaps (with places left free a quarter of the compute units got all of the work: 77 us against 40 for 130 tokens).
// Where no expert has a second tile there is nothing to share: a die takes one block of columns of MT_RUN experts in a row.  Gate and up with
// the columns of one expert dealt to the dies in turn / so, us, 8 rows an expert: 32 experts of 768 x 2048 46.2 / 40.0, 60 of 1,408 x 2048
// 144 / 128, 8 of 3,584 x 2048 51.7 / 47.3; 64 rows 48.3 / 45.1 of the first; two tiles an expert (128 rows) the other way round: 65 / 74.
// More tiles: a run of any MT_RUN tiles and one block of columns, so that nobody looks for its tile through all of them.
__device__ __forceinline__ int moe_lane(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ int4 moe_task(const int* tiles, int max_tiles, int cols, int die, int place, int& ct) {
  if (max_tiles > FG_WAVE) {
    const int run = place / MT_RUN * 8 + die, ti = run / cols * MT_RUN + place % MT_RUN;
    ct = run % cols;
    return ti < max_tiles ? *(const int4*)(tiles + 4 * (size_t)ti) : make_int4(0, 0, 0, 0);
  }
  const int lane = threadIdx.x % FG_WAVE;
  const int4 tile = lane < max_tiles ? *(const int4*)(tiles + 4 * (size_t)lane) : make_int4(0, 0, 0, 0);
  const bool there = tile.z > 0;
  const uint64_t upto = (2ull << lane) - 1, below = upto >> 1;
  const int before = __builtin_amdgcn_update_dpp(-1, tile.x, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
  const uint64_t firsts = __ballot(there && tile.x != before) & upto;  // experts' first tiles
  const int within = firsts ? lane - (63 - __clzll(firsts)) : 0;       // which of its expert's tiles
  if (__ballot(there && within > 0) == 0) {  // a tile an expert
    const int r = place / MT_RUN * 8 + die, at = r / cols * MT_RUN + place % MT_RUN;
    ct = r % cols;
    if (at >= __popcll(__ballot(there))) return make_int4(0, 0, 0, 0);  // (the tiles lie without gaps)
    return make_int4(moe_lane(tile.x, at), moe_lane(tile.y, at), moe_lane(tile.z, at), 0);
  }
  const int run = __popcll(__ballot(there && within % MT_RUN == 0) & upto) - 1;
  const int col0 = (die - run * cols) & 7, each = cols / 8;  // this tile's blocks of columns on this die: col0, col0 + 8, ..
  const bool one_more = col0 < cols % 8;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const bool in = there && (tile.z > 128 ? 0 : tile.z > 64 ? 1 : 2) == c;
    const uint64_t all = __ballot(in), more = __ballot(in && one_more);
    const int total = each * __popcll(all) + __popcll(more);
    if (place < total) {
      const int first = each * __popcll(all & below) + __popcll(more & below);
      const int at = __builtin_ctzll(__ballot(in && place >= first && place < first + each + (one_more ? 1 : 0)));
      ct = moe_lane(col0, at) + 8 * (place - moe_lane(first, at));
      return make_int4(moe_lane(tile.x, at), moe_lane(tile.y, at), moe_lane(tile.z, at), 0);
    }
    place -= total;
  }
  ct = 0;
  return make_int4(0, 0, 0, 0);
}

template <int MB, int NB, int NST, int WS, int OCC, int EPI>
__global__ __launch_bounds__(256, OCC) void moe_large_kernel(const bf16_t* x, unsigned x_bytes, int ldx, const bf16_t* w0,
                                                             const bf16_t* w1, void* y, int ldy, const int* sorted,
                                                             const int* tiles, int max_tiles, int top, int N, int K, const GatedAct fn) {
  constexpr int COLS = (EPI == MT_GATE_UP ? 32 : 64) * NB;
  extern __shared__ __attribute__((aligned(16))) bf16_t large_lds[];
  int ct;
  int4 tile = moe_task(tiles, max_tiles, (N + COLS - 1) / COLS, blockIdx.x % 8, blockIdx.x / 8, ct);
  if (tile.z <= 0) return;  // (the whole workgroup)
  tile = make_int4(__builtin_amdgcn_readfirstlane(tile.x), __builtin_amdgcn_readfirstlane(tile.y), __builtin_amdgcn_readfirstlane(tile.z), 0);
#define GO(ROWS) \
  moe_large_tile<ROWS, NB, NST, WS, OCC == 1, EPI>(large_lds, x, x_bytes, ldx, w0, w1, y, ldy, sorted, tile, ct, top, N, K, fn)
  if (tile.z <= 64) GO(4);
  else if (MB == 8 || tile.z <= 128) GO(8);
  else if constexpr (MB == 16) GO(16);
#undef GO
}

template <int MB, int NB, int NST, int WS, int OCC, int EPI>
static int launch_moe_large(const void* x, unsigned x_bytes, int ldx, const void* w0, const void* w1, void* y, int ldy,
                            const int* sorted, const int* tiles, int max_tiles, int n_experts, int top, int N, int K,
                            const GatedAct fn, hipStream_t stream) {
  constexpr int COLS = (EPI == MT_GATE_UP ? 32 : 64) * NB, lds = NST * MB * 2048;
  static_assert(OCC * lds <= 160 * 1024, "LDS of a compute unit");
  // (every expert's last run may be a part of one)
  const long long runs = (long long)(max_tiles / MT_RUN + (n_experts < max_tiles ? n_experts : max_tiles)) * ((N + COLS - 1) / COLS);
  const long long grid = (runs + 7) / 8 * 8 * MT_RUN;
  if (grid > 2147483647LL) return FG_ERR_ARG;
  static uint64_t raised = 0;  // devices that were asked for more than 64 KB of dynamic LDS, a bit each (asking twice does no harm)
  auto kernel = moe_large_kernel<MB, NB, NST, WS, OCC, EPI>;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return FG_ERR_LAUNCH;
  if (device >= 64 || !(__atomic_load_n(&raised, __ATOMIC_RELAXED) >> device & 1)) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return FG_ERR_LAUNCH;
    if (device < 64) __atomic_fetch_or(&raised, (uint64_t)1 << device, __ATOMIC_RELAXED);
  }
  kernel<<<(unsigned)grid, 256, lds, stream>>>((const bf16_t*)x, x_bytes, ldx, (const bf16_t*)w0, (const bf16_t*)w1, y, ldy, sorted, tiles,
                                               max_tiles, top, N, K, fn);
  return fg_launch_status();
}

// Whether wide tiles would leave a third of the compute units without a workgroup (see launch_moe_tiled).
static bool moe_few(int max_tiles, int N, int cols) { return (long long)max_tiles * ((N + cols - 1) / cols) < 170; }

// Whether the large tiles take it: packed matrices, k in steps of 64, 32-bit offsets within the rows of x and 64 rows of a matrix.
static bool moe_large_ok(const void* x, long long rows, int ldx, const void* w0, const void* w1, int ldw, int K, int tile_rows) {
  return ldw == 0 && K % 64 == 0 && (tile_rows == 128 || tile_rows == 256) && rows > 0 && rows * ldx * 2 <= 4000000000LL &&
         (long long)K * 128 <= 4000000000LL && !(((uintptr_t)x | (uintptr_t)w0 | (uintptr_t)w1) & 15);
}

// x [T, dim] rows gathered by token; wg, wu [E, hidden, ldw], act [n_pairs, lda] in the sorted order.
// mfma: bf16 with dim % 8 == 0, ldx % 8 == 0, ldw % 8 == 0 (16-byte loads); tile_rows = 16 * MB, MB in 1, 2, 4,
// or 128 / 256: the tiles that go through LDS.
// act_kind, limit, alpha: the gated activation (GatedAct in common.h).
// n_tokens, n_experts: the rows of x and the experts that tiles may name (0: not known, no large tiles).
extern "C" int fg_moe_gate_up_act(const void* x, int n_tokens, int n_experts, int ldx, const void* wg, const void* wu, int ldw, const int* sorted,
                                  const int* tiles, int max_tiles, int tile_rows, int top, int dim, int hidden, void* act,
                                  int lda, int dtype, int mfma, int act_kind, float limit, float alpha,
                                  hipStream_t stream) {
  if (max_tiles <= 0) return FG_OK;
  if (act_kind != FG_ACT_SILU && !(act_kind == FG_ACT_LIMITED && limit > 0.f)) return FG_ERR_ARG;
  const GatedAct fn = {act_kind, limit, alpha};
  if (dim <= 0 || hidden <= 0 || top <= 0 || ldx < dim || (ldw < dim && !(mfma && ldw == 0)) || lda < hidden) return FG_ERR_ARG;
  if (mfma) {
    if (dtype != FG_BF16 || dim % 8 || ldx % 8 || ldw % 8 || lda % 4) return FG_ERR_ARG;
    if (tile_rows == 128 || tile_rows == 256) {
      if (hidden % 8 || dim < 32) return FG_ERR_ARG;  // (a lane's stand-in load reads the row's first 32 k)
      if (n_experts > 0 && moe_large_ok(x, n_tokens, ldx, wg, wu, ldw, dim, tile_rows)) {
        const unsigned bytes = 2u * ((unsigned)(n_tokens - 1) * (unsigned)ldx + (unsigned)dim);
#define GO(MB, NB, NST, WS, OCC) \
  return launch_moe_large<MB, NB, NST, WS, OCC, MT_GATE_UP>(x, bytes, ldx, wg, wu, act, lda, sorted, tiles, max_tiles, n_experts, top, hidden, dim, fn, stream)
        if (tile_rows == 256) GO(16, 4, 5, 8, 1);
        if (moe_few(max_tiles, hidden, 128)) GO(8, 2, 5, 8, 2);
        GO(8, 4, 5, 4, 2);
#undef GO
      }
      return tile_rows == 128
                 ? launch_moe_tiled<1, MT_GATE_UP>(x, ldx, wg, wu, ldw, act, lda, sorted, tiles, max_tiles, top, hidden, dim, fn, stream)
                 : launch_moe_tiled<2, MT_GATE_UP>(x, ldx, wg, wu, ldw, act, lda, sorted, tiles, max_tiles, top, hidden, dim, fn, stream);
    }
    const long long items = (long long)max_tiles * ((hidden + 15) / 16);
    const unsigned blocks = (unsigned)((items + 3) / 4);
#define GO_AS(MB, PACKED)                                                                                         \
  moe_gate_up_mfma_kernel<MB, PACKED><<<blocks, 256, 0, stream>>>((const bf16_t*)x, ldx, (const bf16_t*)wg, (const bf16_t*)wu, \
                                                                  ldw, sorted, tiles, max_tiles, top, dim, hidden, (bf16_t*)act, lda, fn)
#define GO(MB)                    \
  do {                            \
    if (ldw == 0) GO_AS(MB, true); \
    else GO_AS(MB, false);        \
  } while (0)
    if (tile_rows == 16) GO(1);
    else if (tile_rows == 32) GO(2);
    else if (tile_rows == 64) GO(4);
    else return FG_ERR_ARG;
#undef GO
#undef GO_AS
    return fg_launch_status();
  }
  if (tile_rows != 16 || max_tiles > 2147483647 / 4) return FG_ERR_ARG;
  dim3 grid(max_tiles, (hidden + 15) / 16);
  if (grid.y > 65535) return FG_ERR_ARG;
  if (dtype == FG_F32)
    moe_gate_up_generic_kernel<float><<<grid, 256, 0, stream>>>((const float*)x, ldx, (const float*)wg, (const float*)wu,
                                                                ldw, sorted, tiles, top, dim, hidden, (float*)act, lda, fn);
  else if (dtype == FG_BF16)
    moe_gate_up_generic_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)x, ldx, (const bf16_t*)wg,
                                                                 (const bf16_t*)wu, ldw, sorted, tiles, top, dim, hidden,
                                                                 (bf16_t*)act, lda, fn);
  else
    return FG_ERR_ARG;
  return fg_launch_status();
}

extern "C" int fg_moe_gate_up(const void* x, int ldx, const void* wg, const void* wu, int ldw, const int* sorted,
                              const int* tiles, int max_tiles, int tile_rows, int top, int dim, int hidden, void* act,
                              int lda, int dtype, int mfma, hipStream_t stream) {
  return fg_moe_gate_up_act(x, 0, 0, ldx, wg, wu, ldw, sorted, tiles, max_tiles, tile_rows, top, dim, hidden, act, lda, dtype,
                            mfma, FG_ACT_SILU, 0.f, 1.f, stream);
}

// act [n_pairs, lda] in the sorted order; wd [E, dim, ldw]; y fp32 [n_pairs, dim], row = pair.
extern "C" int fg_moe_down(const void* act, int n_experts, int lda, const void* wd, int ldw, const int* sorted, const int* tiles,
                           int max_tiles, int tile_rows, int dim, int hidden, float* y, int dtype, int mfma,
                           hipStream_t stream) {
  if (max_tiles <= 0) return FG_OK;
  if (dim <= 0 || hidden <= 0 || lda < hidden || (ldw < hidden && !(mfma && ldw == 0))) return FG_ERR_ARG;
  if (mfma) {
    if (dtype != FG_BF16 || hidden % 8 || lda % 8 || ldw % 8) return FG_ERR_ARG;
    if ((tile_rows == 128 || tile_rows == 256) && hidden < 32) return FG_ERR_ARG;
    if (n_experts > 0 && moe_large_ok(act, tile_rows, lda, wd, nullptr, ldw, hidden, tile_rows)) {
#define GO(MB, NB, NST, WS, OCC)                                                                                               \
  return launch_moe_large<MB, NB, NST, WS, OCC, MT_DOWN>(act, 0, lda, wd, nullptr, y, dim, sorted, tiles, max_tiles, n_experts, 1, dim, hidden, \
                                                         GatedAct{0, 0.f, 1.f}, stream)
      if (tile_rows == 256) GO(16, 4, 5, 8, 1);
      if (moe_few(max_tiles, dim, 256)) GO(8, 2, 5, 8, 2);
      GO(8, 4, 5, 4, 2);
#undef GO
    }
    if (tile_rows == 128 || tile_rows == 256)
      return tile_rows == 128
                 ? launch_moe_tiled<1, MT_DOWN>(act, lda, wd, nullptr, ldw, y, dim, sorted, tiles, max_tiles, 1, dim, hidden, GatedAct{0, 0.f, 1.f}, stream)
                 : launch_moe_tiled<2, MT_DOWN>(act, lda, wd, nullptr, ldw, y, dim, sorted, tiles, max_tiles, 1, dim, hidden, GatedAct{0, 0.f, 1.f}, stream);
    const long long items = (long long)max_tiles * ((dim + 15) / 16);
    const unsigned blocks = (unsigned)((items + 3) / 4);
#define GO_AS(MB, PACKED)                                                                                            \
  moe_down_mfma_kernel<MB, PACKED><<<blocks, 256, 0, stream>>>((const bf16_t*)act, lda, (const bf16_t*)wd, ldw, sorted, \
                                                               tiles, max_tiles, dim, hidden, y)
#define GO(MB)                    \
  do {                            \
    if (ldw == 0) GO_AS(MB, true); \
    else GO_AS(MB, false);        \
  } while (0)
    if (tile_rows == 16) GO(1);
    else if (tile_rows == 32) GO(2);
    else if (tile_rows == 64) GO(4);
    else return FG_ERR_ARG;
#undef GO
#undef GO_AS
    return fg_launch_status();
  }
  if (tile_rows != 16) return FG_ERR_ARG;
  dim3 grid(max_tiles, (dim + 15) / 16);
  if (grid.y > 65535) return FG_ERR_ARG;
  if (dtype == FG_F32)
    moe_down_generic_kernel<float><<<grid, 256, 0, stream>>>((const float*)act, lda, (const float*)wd, ldw, sorted, tiles,
                                                             dim, hidden, y);
  else if (dtype == FG_BF16)
    moe_down_generic_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)act, lda, (const bf16_t*)wd, ldw, sorted,
                                                              tiles, dim, hidden, y);
  else
    return FG_ERR_ARG;
  return fg_launch_status();
}

// ----------------------------------------------------------------- combine
// out[t] = plus[t] + sum_j weight[t][j] * y[t * top + j]: the weighted sum first, j ascending, all fp32.
// plus: rows of the activation dtype, or (n_plus > 0) fp32 partial sums plus[p * plus_stride + t * ldp + d],
// whose sum, in order, is what is added.  plus_gate (fp32, one number a token at plus_gate[t * gate_stride]): the
// rows of plus are multiplied by its sigmoid before they are added.  choice [n_tokens, top] (or null): the output of an
// expert from n_tiled on is the token's row of x.
struct CombineIdentity {
  const int* choice; int n_tiled;
  const void* x; int ldx;
};
template <int VEC, class T> __device__ __forceinline__ void mc_load(const T* p, float (&v)[VEC]) {
  if constexpr (VEC == 4 && sizeof(T) == 4) {
    const float4 a = *(const float4*)p;
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) v[i] = to_f<T>(p[i]);
  }
}
// grid (n_tokens, ceil(dim / (256 VEC))): a thread VEC neighbouring columns, the outputs of four experts in flight
template <class TP, class TX, int VEC>
__global__ __launch_bounds__(256) void moe_combine_kernel(
    const float* __restrict__ y, const float* __restrict__ weight, const TP* __restrict__ plus, int ldp, int n_plus,
    size_t plus_stride, int top, int dim, float* __restrict__ out, const float* __restrict__ plus_gate, int gate_stride,
    const CombineIdentity id) {
  const int t = blockIdx.x, d = (blockIdx.y * 256 + threadIdx.x) * VEC;
  if (d >= dim) return;
  const float pg = plus_gate ? 1.f / (1.f + expf(-plus_gate[(size_t)t * gate_stride])) : 1.f;
  float own[VEC], s[VEC];
  if (id.choice) mc_load<VEC, TX>((const TX*)id.x + (size_t)t * id.ldx + d, own);
#pragma unroll
  for (int i = 0; i < VEC; ++i) s[i] = 0.f;
  for (int j0 = 0; j0 < top; j0 += 4) {
    float o[4][VEC], w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const size_t p = (size_t)t * top + min(j0 + j, top - 1);
      w[j] = j0 + j < top ? weight[p] : 0.f;
      if (id.choice && id.choice[p] >= id.n_tiled) {  // uniform
#pragma unroll
        for (int i = 0; i < VEC; ++i) o[j][i] = own[i];
      } else {
        mc_load<VEC, float>(y + p * dim + d, o[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j0 + j < top) {  // uniform
#pragma unroll
        for (int i = 0; i < VEC; ++i) s[i] = fmaf(w[j], o[j][i], s[i]);
      }
  }
  if (plus) {
    float m[VEC];
    mc_load<VEC, TP>(plus + (size_t)t * ldp + d, m);
    for (int p = 1; p < n_plus; ++p) {
      float more[VEC];
      mc_load<VEC, TP>(plus + p * plus_stride + (size_t)t * ldp + d, more);
#pragma unroll
      for (int i = 0; i < VEC; ++i) m[i] += more[i];
    }
#pragma unroll
    for (int i = 0; i < VEC; ++i) s[i] = (plus_gate ? m[i] * pg : m[i]) + s[i];
  }
  float* o = out + (size_t)t * dim + d;
  if constexpr (VEC == 4) *(float4*)o = make_float4(s[0], s[1], s[2], s[3]);
  else o[0] = s[0];
}

extern "C" int fg_moe_combine_identity(const float* y, const float* weight, const void* plus, int ldp, int plus_dtype,
                                       int n_plus, long long plus_stride, int n_tokens, int top, int dim, float* out,
                                       const float* plus_gate, int gate_stride, const int* choice, int n_tiled, const void* x,
                                       int ldx, int x_dtype, hipStream_t stream) {
  if (n_tokens <= 0) return FG_OK;
  if (plus_gate && (!plus || gate_stride < 1)) return FG_ERR_ARG;
  if (top <= 0 || dim <= 0 || (plus && (ldp < dim || n_plus < 1)) || (n_plus > 1 && plus_dtype != FG_F32)) return FG_ERR_ARG;
  if (choice && (!x || ldx < dim || n_tiled < 0)) return FG_ERR_ARG;
  const CombineIdentity id = {choice, n_tiled, x, ldx};
  if (x_dtype != FG_F32 && x_dtype != FG_BF16) return FG_ERR_ARG;
  // (16-byte loads of the fp32 operands)
  const bool vec = dim % 4 == 0 && !((uintptr_t)y & 15) && !((uintptr_t)out & 15) &&
                   (!plus || plus_dtype != FG_F32 || (ldp % 4 == 0 && plus_stride % 4 == 0 && !((uintptr_t)plus & 15))) &&
                   (!choice || x_dtype != FG_F32 || (ldx % 4 == 0 && !((uintptr_t)x & 15)));
  const dim3 grid(n_tokens, (dim + (vec ? 1023 : 255)) / (vec ? 1024 : 256));
  if (grid.y > 65535) return FG_ERR_ARG;
#define GO(TP, TX)                                                                                                         \
  do {                                                                                                                     \
    if (vec)                                                                                                               \
      moe_combine_kernel<TP, TX, 4><<<grid, 256, 0, stream>>>(y, weight, (const TP*)plus, ldp, n_plus, (size_t)plus_stride, \
                                                              top, dim, out, plus_gate, gate_stride, id);                  \
    else                                                                                                                   \
      moe_combine_kernel<TP, TX, 1><<<grid, 256, 0, stream>>>(y, weight, (const TP*)plus, ldp, n_plus, (size_t)plus_stride, \
                                                              top, dim, out, plus_gate, gate_stride, id);                  \
  } while (0)
  if (plus_dtype == FG_F32 && x_dtype == FG_F32) GO(float, float);
  else if (plus_dtype == FG_F32) GO(float, bf16_t);
  else if (plus_dtype == FG_BF16 && x_dtype == FG_BF16) GO(bf16_t, bf16_t);
  else if (plus_dtype == FG_BF16 && !choice) GO(bf16_t, float);
#undef GO
  else
    return FG_ERR_ARG;
  return fg_launch_status();
}

extern "C" int fg_moe_combine_gated(const float* y, const float* weight, const void* plus, int ldp, int plus_dtype,
                                    int n_plus, long long plus_stride, int n_tokens, int top, int dim, float* out,
                                    const float* plus_gate, int gate_stride, hipStream_t stream) {
  return fg_moe_combine_identity(y, weight, plus, ldp, plus_dtype, n_plus, plus_stride, n_tokens, top, dim, out, plus_gate,
                                 gate_stride, nullptr, 0, nullptr, 0, FG_F32, stream);
}

extern "C" int fg_moe_combine(const float* y, const float* weight, const void* plus, int ldp, int plus_dtype, int n_plus,
                              long long plus_stride, int n_tokens, int top, int dim, float* out, hipStream_t stream) {
  return fg_moe_combine_gated(y, weight, plus, ldp, plus_dtype, n_plus, plus_stride, n_tokens, top, dim, out, nullptr, 0,
                              stream);
}

// The combine inside the norm that follows it: h[t] += plus[t] + sum_j weight[t][j] * y[t * top + j], out = norm(h) * w, the
// same sums in the same order (the bits of the two kernels), for rows without identities and without a gate of plus.
// A workgroup a row, all of a row's loads
// in flight before anything is added; bound by them (1897 tokens of 2048, top 4: 19.5 us, 5.4 TB/s, against 15.2 + 13.8 for
// the kernels apart, whose sums went through memory; 12 tokens 5.4 against 4.8 + 4.6, and a launch less).
template <class TP, class TA, class TW, int NIT>
__global__ __launch_bounds__(256) void moe_combine_norm_kernel(
    const float* __restrict__ y, const float* __restrict__ weight, const TP* __restrict__ plus, int ldp, int n_plus,
    size_t plus_stride, int top, int dim, float* __restrict__ h, const TW* __restrict__ w, TA* __restrict__ out,
    float eps) {
  __shared__ float red[16];
  const size_t t = blockIdx.x;
  float* hrow = h + t * dim;
  int e[NIT], ec[NIT];  // a thread whose share lies behind the row reads its last 8 and stores nothing
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    e[it] = (threadIdx.x + it * 256) * 8;
    ec[it] = min(e[it], dim - 8);
  }
  float v[NIT][8], wv[NIT][8], m[NIT][8], s[NIT][8];
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    load8<float>(hrow + ec[it], v[it]);
    load8<TW>(w + ec[it], wv[it]);
    if (plus) load8<TP>(plus + t * ldp + ec[it], m[it]);
#pragma unroll
    for (int i = 0; i < 8; ++i) s[it][i] = 0.f;
  }
  constexpr int FLY = NIT == 1 ? 4 : 2;  // experts' rows in flight
  for (int j0 = 0; j0 < top; j0 += FLY) {
    float o[FLY][NIT][8], wj[FLY];
#pragma unroll
    for (int j = 0; j < FLY; ++j) {
      const size_t p = t * top + min(j0 + j, top - 1);
      wj[j] = weight[p];
#pragma unroll
      for (int it = 0; it < NIT; ++it) load8<float>(y + p * dim + ec[it], o[j][it]);
    }
#pragma unroll
    for (int j = 0; j < FLY; ++j)
      if (j0 + j < top) {  // uniform
#pragma unroll
        for (int it = 0; it < NIT; ++it)
#pragma unroll
          for (int i = 0; i < 8; ++i) s[it][i] = fmaf(wj[j], o[j][it][i], s[it][i]);
      }
  }
  if (plus) {
    for (int p = 1; p < n_plus; ++p) {
#pragma unroll
      for (int it = 0; it < NIT; ++it) {
        float more[8];
        load8<TP>(plus + p * plus_stride + t * ldp + ec[it], more);
#pragma unroll
        for (int i = 0; i < 8; ++i) m[it][i] += more[i];
      }
    }
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int i = 0; i < 8; ++i) s[it][i] = m[it][i] + s[it][i];
  }
  float ss = 0.f;
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[it][i] += s[it][i];
    if (e[it] < dim) {
      store8<float>(hrow + e[it], v[it]);
#pragma unroll
      for (int i = 0; i < 8; ++i) ss += v[it][i] * v[it][i];
    }
  }
  ss = block_sum(ss, red);
  const float rstd = rsqrtf(ss / (float)dim + eps);
  TA* orow = out + t * dim;
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    if (e[it] < dim) {
      float o[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = v[it][i] * rstd * wv[it][i];
      store8<TA>(orow + e[it], o);
    }
  }
}

extern "C" int fg_moe_combine_norm(const float* y, const float* weight, const void* plus, int ldp, int plus_dtype, int n_plus,
                                   long long plus_stride, int top, int dim, float* h, const void* w, int w_dtype,
                                   void* out, int out_dtype, int n_rows, float eps, hipStream_t stream) {
  if (n_rows <= 0) return FG_OK;
  if (top <= 0 || dim <= 0 || dim % 8 || dim > 4096 || (plus && (ldp < dim || ldp % 8 || n_plus < 1 || plus_stride % 8)) ||
      (n_plus > 1 && plus_dtype != FG_F32))
    return FG_ERR_ARG;
  if (((uintptr_t)y | (uintptr_t)plus | (uintptr_t)h | (uintptr_t)w | (uintptr_t)out) & 15) return FG_ERR_ARG;
#define GO_AS(TP, TA, TW, NIT)                                                                                          \
  moe_combine_norm_kernel<TP, TA, TW, NIT><<<n_rows, 256, 0, stream>>>(y, weight, (const TP*)plus, ldp, n_plus,         \
                                                                       (size_t)plus_stride, top, dim, h, (const TW*)w,  \
                                                                       (TA*)out, eps)
#define GO(TP, TA, TW)                        \
  do {                                        \
    if (dim <= 2048) GO_AS(TP, TA, TW, 1);    \
    else GO_AS(TP, TA, TW, 2);                \
  } while (0)
  const bool pf = plus_dtype == FG_F32, wf = w_dtype == FG_F32;
  if ((plus_dtype != FG_F32 && plus_dtype != FG_BF16) || (w_dtype != FG_F32 && w_dtype != FG_BF16)) return FG_ERR_ARG;
  if (out_dtype == FG_F32 && pf && wf) GO(float, float, float);
  else if (out_dtype == FG_BF16 && pf && wf) GO(float, bf16_t, float);
  else if (out_dtype == FG_BF16 && pf) GO(float, bf16_t, bf16_t);
  else if (out_dtype == FG_BF16 && wf) GO(bf16_t, bf16_t, float);
  else if (out_dtype == FG_BF16) GO(bf16_t, bf16_t, bf16_t);
#undef GO
#undef GO_AS
  else
    return FG_ERR_ARG;
  return fg_launch_status();
}
