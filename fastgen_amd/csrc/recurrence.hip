// A linear recurrence with a decay per key channel (gated linear attention), token by token:
//
//   a_t = sigmoid(z_t + b)^(1/tau)                       (per head and key channel, fp32; all tokens at once)
//   S_t = diag(a_t) S_(t-1) + k_t v_t^T                  (per head, [d, e] fp32, kept per request)
//   o_t = S_t^T (q_t * q_scale)
//
// The state lives in fp32 in a slot per request and is carried from step to step; a step brings a
// run of tokens per sequence (one when decoding).  Every token's arithmetic is the same whatever the
// step holds besides it: the tokens of a sequence are taken in order, each output element is one
// fixed chain of additions, so a prompt cut into portions or batched with others gives the same bits
// (long runs of tokens may instead be scanned chunk by chunk, see below: the same within rounding).
//
// grid (B sequences, H heads, ceil(e / 8)); one wave.  Lane l owns value channel 8 z + (l & 7) and the
// key channels rg * rpl .. rg * rpl + rpl - 1 with rg = l >> 3, rpl = ceil(d / 8): an eighth of a column
// of S in registers.  q, k and the decays of a run of tokens go through LDS.
#include "common.h"

// tokens staged at a time: as many as leave the kernel's registers unspilled
#define RC_TOKENS_FOR(RPL) ((RPL) <= 8 ? 16 : (RPL) <= 32 ? 8 : 4)

struct ScanArgs {
  const void* qkv; int row_stride, q_col, k_col, v_col;  // act dtype rows: q, k [H * d], v [H * e] at their columns
  const float* decay; int decay_stride;                  // fp32 [T, >= H * d]: a_t (fg_decay_from_logits)
  float q_scale;
  float* state;                                          // fp32 [n_slots, H, d, e]
  const int* slot_ids; const int* q_start;               // [B], [B + 1]
  float* out;                                            // fp32 [T, H * e]
  int H, d, e;
  int write_out, write_state;                            // what a sequence leaves: its tokens' outputs, its last state
};

// The loop over a sequence's tokens is a chain: what it costs is how many instructions one link takes
// (a wave issues one every few clocks) and what it waits for.  So the loads of a run of RC_TOKENS tokens
// (4, 8 or 16; decays, k, q: d of each a token, spread over the lanes; and each lane's own value channel) are all
// issued into registers before the run before it is computed, and reach LDS (q scaled) when that is
// done: memory latency passes behind the arithmetic.  The decays come ready from a kernel of their own
// (exponentials and logarithms of every token at once, not in this chain).  RPL >= ceil(d / 8); NJ =
// ceil(d / 64) is the number of staged elements a lane holds of each of the three, per token.
template <class TA, int RPL>
__global__ __launch_bounds__(FG_WAVE) void decay_scan_kernel(const ScanArgs a) {
  constexpr int NJ = RPL >= 8 ? RPL / 8 : 1;
  constexpr int RC_TOKENS = RC_TOKENS_FOR(RPL);
  // [RC_TOKENS][3][d + 32]: decay, k, q; key channel r lies at r + 4 (r / rpl), so that the eight parts
  // that the lane groups read at once start in different banks and every part is 16-byte aligned
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int lane = threadIdx.x;
  const int b = blockIdx.x, h = blockIdx.y;
  const int c = lane & 7, rg = lane >> 3;
  const int col = blockIdx.z * 8 + c;
  const bool col_ok = col < a.e;
  const int d = a.d, e = a.e;
  const int rpl = (d + 7) / 8;
  const int r0 = rg * rpl;
  const int ds = d + 32;              // a staged vector's stride
  const bool vec = rpl % 4 == 0 && d == 8 * rpl;  // uniform: the parts are read as float4
  const int t_begin = a.q_start[b], t_end = a.q_start[b + 1];
  float* S_mem = a.state + (((size_t)a.slot_ids[b] * a.H + h) * d) * e;
  float S[RPL];
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    const int r = r0 + i;
    S[i] = (i < rpl && r < d && col_ok) ? S_mem[(size_t)r * e + col] : 0.f;
  }
  const TA* qkv = (const TA*)a.qkv;
  // the key channels this lane stages (the same for every token): where they come from and where they go
  int src[NJ], dst[NJ];
  bool mine[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int r = lane + FG_WAVE * j;
    mine[j] = r < d;
    src[j] = h * d + min(r, d - 1);
    dst[j] = r + 4 * (r / rpl);
  }
  const int v_src = a.v_col + h * e + min(col, e - 1);
  float pa[RC_TOKENS][NJ], pk[RC_TOKENS][NJ], pq[RC_TOKENS][NJ], pv[RC_TOKENS];
  auto fetch = [&](int t0) {  // the run t0 .. t0 + n - 1 into registers: nothing waits here
    const int n = min(RC_TOKENS, t_end - t0);
#pragma unroll
    for (int tt = 0; tt < RC_TOKENS; ++tt) {
      const size_t t = (size_t)(t0 + min(tt, n - 1));  // (never conditional: beyond the run, its last token again)
      const TA* row = qkv + t * a.row_stride;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        pa[tt][j] = a.decay[t * a.decay_stride + src[j]];
        pk[tt][j] = to_f<TA>(row[a.k_col + src[j]]);
        pq[tt][j] = to_f<TA>(row[a.q_col + src[j]]);
      }
      pv[tt] = to_f<TA>(row[v_src]);
    }
  };
  if (t_begin < t_end) fetch(t_begin);
  for (int t0 = t_begin; t0 < t_end; t0 += RC_TOKENS) {
    const int n = min(RC_TOKENS, t_end - t0);
    __syncthreads();  // the run before has been read
    float v[RC_TOKENS];
#pragma unroll
    for (int tt = 0; tt < RC_TOKENS; ++tt) {
      v[tt] = pv[tt];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        if (mine[j]) {
          float* to = lds + (size_t)tt * 3 * ds + dst[j];
          to[0] = pa[tt][j];
          to[ds] = pk[tt][j];
          to[2 * ds] = pq[tt][j] * a.q_scale;
        }
      }
    }
    __syncthreads();
    if (t0 + RC_TOKENS < t_end) fetch(t0 + RC_TOKENS);  // in flight while this run is computed
    // One token after the other; the sums over the lane groups are taken for the whole run at once (the
    // lanes' exchange is the longest link of the chain: sixteen of them wait together).  Reading a token's
    // operands from LDS a token ahead into a second set of registers was measured slower (the registers spill).
    float acc[RC_TOKENS];
    const float* part0 = lds + r0 + 4 * rg;  // this lane group's part of a staged vector
    if (vec) {
#pragma unroll
      for (int tt = 0; tt < RC_TOKENS; ++tt) {
        const float* av = part0 + (size_t)tt * 3 * ds;
        // four sums side by side (channels u, u + 4, ..), added up at the end: no chain of dependent additions
        float part[4] = {0.f, 0.f, 0.f, 0.f};
        if (tt < n) {
#pragma unroll
          for (int i4 = 0; i4 < RPL / 4; ++i4) {
            if (4 * i4 < rpl) {
              const float4 a4 = ((const float4*)av)[i4], k4 = ((const float4*)(av + ds))[i4],
                           q4 = ((const float4*)(av + 2 * ds))[i4];
              const float aa[4] = {a4.x, a4.y, a4.z, a4.w}, kk[4] = {k4.x, k4.y, k4.z, k4.w}, qq[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                S[4 * i4 + u] = aa[u] * S[4 * i4 + u] + kk[u] * v[tt];
                part[u] += S[4 * i4 + u] * qq[u];
              }
            }
          }
        }
        acc[tt] = (part[0] + part[1]) + (part[2] + part[3]);
      }
    } else {
#pragma unroll
      for (int tt = 0; tt < RC_TOKENS; ++tt) {
        const float* av = part0 + (size_t)tt * 3 * ds;
        float sum = 0.f;
        if (tt < n) {
#pragma unroll
          for (int i = 0; i < RPL; ++i) {
            if (i < rpl && r0 + i < d) {
              S[i] = av[i] * S[i] + av[ds + i] * v[tt];
              sum += S[i] * av[2 * ds + i];
            }
          }
        }
        acc[tt] = sum;
      }
    }
    // the eight parts of a column: a butterfly whose order of additions is the same in every lane
#pragma unroll
    for (int m = 8; m < FG_WAVE; m <<= 1) {
      float other[RC_TOKENS];
#pragma unroll
      for (int tt = 0; tt < RC_TOKENS; ++tt) other[tt] = __shfl_xor(acc[tt], m, FG_WAVE);
#pragma unroll
      for (int tt = 0; tt < RC_TOKENS; ++tt) acc[tt] += other[tt];
    }
    if (rg == 0 && col_ok && a.write_out) {
#pragma unroll
      for (int tt = 0; tt < RC_TOKENS; ++tt)
        if (tt < n) a.out[(size_t)(t0 + tt) * ((size_t)a.H * e) + h * e + col] = acc[tt];
    }
  }
#pragma unroll
  for (int i = 0; i < RPL; ++i) {
    const int r = r0 + i;
    if (i < rpl && r < d && col_ok && a.write_state) S_mem[(size_t)r * e + col] = S[i];
  }
}

// out[t, c] = sigmoid(z[t, c] + bias[c])^(1/tau) for c < width, as exp(log sigmoid(.) / tau) with
// log sigmoid(x) = min(x, 0) - log1p(exp(-|x|)); fp32.
// LOG: its logarithm to the base 2.
template <bool LOG>
__global__ __launch_bounds__(256) void decay_from_logits_kernel(const float* __restrict__ z, int z_stride,
                                                                const float* __restrict__ bias, float inv_tau,
                                                                float* __restrict__ out, int width) {
  const size_t t = blockIdx.y;
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= width) return;
  const float x = z[t * z_stride + c] + (bias ? bias[c] : 0.f);
  const float l = (fminf(x, 0.f) - log1pf(expf(-fabsf(x)))) * inv_tau;
  out[t * width + c] = LOG ? l * 1.44269504088896340736f : expf(l);
}

extern "C" int fg_decay_from_logits(const float* z, int z_stride, const float* bias, float inv_tau, float* out,
                                    int n_rows, int width, int log2_of_it, hipStream_t stream) {
  if (n_rows <= 0) return FG_OK;
  if (width <= 0 || z_stride < width || !(inv_tau > 0.f) || !z || !out) return FG_ERR_ARG;
  for (int r0 = 0; r0 < n_rows; r0 += 65535) {
    const int nr = n_rows - r0 < 65535 ? n_rows - r0 : 65535;
    const dim3 grid((width + 255) / 256, nr);
    const float* from = z + (size_t)r0 * z_stride;
    float* to = out + (size_t)r0 * width;
    if (log2_of_it) decay_from_logits_kernel<true><<<grid, 256, 0, stream>>>(from, z_stride, bias, inv_tau, to, width);
    else decay_from_logits_kernel<false><<<grid, 256, 0, stream>>>(from, z_stride, bias, inv_tau, to, width);
  }
  return fg_launch_status();
}

// ------------------------------------------------------------ long prompts, chunk by chunk
// A long run of tokens is cut into chunks that are scanned side by side: first every chunk from a zero
// state (fg_decay_scan on the chunks as if they were sequences, states only), then, chunk after chunk of a
// sequence, the state each chunk starts from (below), then every chunk again from its true start, for
// the outputs.  Twice the arithmetic, as many times the waves as a sequence has chunks.
//
// prod[c, j] = the product of decay[t, j] over chunk c's tokens (chunk_start[c] .. chunk_start[c + 1] - 1).
__global__ __launch_bounds__(256) void decay_chunk_product_kernel(const float* __restrict__ decay, int decay_stride,
                                                                  const int* __restrict__ chunk_start,
                                                                  float* __restrict__ prod, int width) {
  const int c = blockIdx.y, j = blockIdx.x * 256 + threadIdx.x;
  if (j >= width) return;
  float p = 1.f;
  for (int t = chunk_start[c]; t < chunk_start[c + 1]; ++t) p *= decay[(size_t)t * decay_stride + j];
  prod[(size_t)c * width + j] = p;
}

// chunks [H, d, e] per chunk holds what each chunk adds to a zero state; it leaves with the state each chunk
// starts from: for sequence b's chunks c = seq_chunk[b] .. seq_chunk[b + 1] - 1 in order,
// start(c) = S; S = prod[c] * S + chunks[c], from S = state[slot_ids[b]], which takes the last S.
__global__ __launch_bounds__(256) void decay_chunk_states_kernel(float* __restrict__ chunks, const float* __restrict__ prod,
                                                                 float* __restrict__ state, const int* __restrict__ slot_ids,
                                                                 const int* __restrict__ seq_chunk, int H, int d, int e) {
  const int b = blockIdx.y;
  const size_t per = (size_t)H * d * e;
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;  // (head, key channel, value channel)
  if (i >= per) return;
  const size_t row = i / e;  // (head, key channel)
  float* S_mem = state + (size_t)slot_ids[b] * per + i;
  float S = *S_mem;
  constexpr int AHEAD = 8;  // chunks whose loads are in flight together
  const int c_end = seq_chunk[b + 1];
  for (int c = seq_chunk[b]; c < c_end; c += AHEAD) {
    float add[AHEAD], keep[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      const size_t cc = min(c + j, c_end - 1);
      add[j] = chunks[cc * per + i];
      keep[j] = prod[cc * H * d + row];
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
      if (c + j < c_end) {  // uniform
        chunks[(size_t)(c + j) * per + i] = S;
        S = keep[j] * S + add[j];
      }
    }
  }
  *S_mem = S;
}

extern "C" int fg_decay_chunk_product(const float* decay, int decay_stride, const int* chunk_start, float* prod,
                                      int n_chunks, int width, hipStream_t stream) {
  if (n_chunks <= 0) return FG_OK;
  if (width <= 0 || decay_stride < width || n_chunks > 65535 || !decay || !chunk_start || !prod) return FG_ERR_ARG;
  decay_chunk_product_kernel<<<dim3((width + 255) / 256, n_chunks), 256, 0, stream>>>(decay, decay_stride, chunk_start,
                                                                                      prod, width);
  return fg_launch_status();
}

extern "C" int fg_decay_chunk_states(float* chunks, const float* prod, float* state, const int* slot_ids,
                                     const int* seq_chunk, int n_seqs, int H, int d, int e, hipStream_t stream) {
  if (n_seqs <= 0) return FG_OK;
  const long long per = (long long)H * d * e;
  if (H <= 0 || d <= 0 || e <= 0 || n_seqs > 65535 || (per + 255) / 256 > 2147483647LL || !chunks || !prod || !state ||
      !slot_ids || !seq_chunk)
    return FG_ERR_ARG;
  decay_chunk_states_kernel<<<dim3((unsigned)((per + 255) / 256), n_seqs), 256, 0, stream>>>(chunks, prod, state, slot_ids,
                                                                                             seq_chunk, H, d, e);
  return fg_launch_status();
}

// ------------------------------------------- long prompts, 64 tokens at a time as matrix products
// The same in matrix products, for head sizes in multiples of 16 up to 128.  Chunks of 64 tokens, in blocks of 16.  With l
// the decays' logarithms to the base 2, P_t = 2^(the sum of l over t's block up to t, its own included), R_s = 2^(the sum
// over s's block behind s) and E_b = 2^(the sum over block b):
//   states   C = sum_s (k_s R_s E of the blocks behind) v_s^T, prod = 2^(the sum over the chunk)    (a chunk's own part)
//   fg_decay_chunk_states
//   outputs  o_t = (q_t P_t E of the blocks before)^T S0 + sum_s M[t, s] v_s;  for s in an earlier block
//            M = (q_t P_t) . (k_s R_s E of the blocks between), in t's own block
//            M = sum_r q_tr (k_sr a_(s+1)r .. a_tr), the key taken along from token to token.
// Sums of logarithms are added up only, never subtracted from one another (the difference of two long ones would keep
// few of its digits), so a weight is as exact as the decays that make it up, however strong other decays beside it are;
// no exponent is positive, and no decay needs a bound (2^x under 2^-126 is zero).  Products on v_mfma_f32_16x16x4_f32; an
// operand's k index runs as 16 j + 4 (lane / 16) + i over the four products i of a block j.  All of it in fp32, with at
// most 32 products in a chain (chains of 128: 1.3 to 1.45 times the error).  Error of the outputs against 64 bits (500
// tokens of 128 channels), products / token by token: decays near one 1.4 / 1.5e-7, lasting ones 1.8e-7 / 1.5e-6, 5 %
// of them strong 1.3 / 1.5e-7, half of them 1.1 / 1.05e-7, of every strength 1.04e-7 / 8.9e-8.  (With differences of
// sums in the place of R and of the own block's products: 1.9e-7, 2.9e-7, 1.1e-6, 2.3 to 8.9e-6, 3.5e-7.)
// 2000 tokens, 16 heads of 128 x 128: 23 + 14 + 47 us behind 16 us for the decays, against 137 + 137 (the scans of
// chunks of 128 token by token, twice) + 32 (the products of the decays) + 9 + 16 us.  A call of its own, in and out:
// 127 against 365 us; 8000 tokens 377 against 1210, 256 tokens 90 against 179, 4 times 300 tokens 118 against 338; float32
// operands 148 against 359, 483 against 1242, 90 against 177, 139 against 330.  The outputs' kernel is bound by what a
// workgroup does alone (its stages with a barrier between each), two workgroups a CU.
#define DC 64
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct ChunkArgs {
  const void* qkv; int row_stride, q_col, k_col, v_col;
  const float* logs;       // [T, H * d]
  float q_scale;
  const int* chunk_start;  // [n_chunks + 1]
  float* states;           // [n_chunks, H, d, e]: C, then S0
  float* prod;             // [n_chunks, H * d]
  float* out;              // [T, H * e]
  int H, d, e;
};

__device__ __forceinline__ f32x4 dc_mfma4(const f32x4 x, const f32x4 y, f32x4 acc) {
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y[i], acc, 0, 0, 0);
  return acc;
}
template <class T> __device__ __forceinline__ f32x4 dc_load4(const T* p);
template <> __device__ __forceinline__ f32x4 dc_load4<float>(const float* p) { return *(const f32x4*)p; }
template <> __device__ __forceinline__ f32x4 dc_load4<bf16_t>(const bf16_t* p) {
  const uint2 w = *(const uint2*)p;
  return f32x4{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u), __uint_as_float(w.y << 16),
               __uint_as_float(w.y & 0xffff0000u)};
}
__device__ __forceinline__ float dc_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// The logarithms of token u of block i / d, channel i % d, for the item i < 4 d; tokens behind the chunk's last: 0.
__device__ __forceinline__ void dc_logs(const ChunkArgs& a, int t0, int n, int h, int i, float (&l)[16]) {
  const int b = i / a.d, r = i % a.d;
#pragma unroll
  for (int u = 0; u < 16; ++u) l[u] = a.logs[(size_t)(t0 + min(16 * b + u, n - 1)) * a.H * a.d + h * a.d + r];
#pragma unroll
  for (int u = 0; u < 16; ++u) l[u] = 16 * b + u < n ? l[u] : 0.f;
}

// grid (n_chunks, H, ceil(e / 128)), 4 waves; wave w the state's rows of the blocks w, w + 4 of 16 key channels.
template <class TA, int NDM>
__global__ __launch_bounds__(256) void decay_chunk_sums_kernel(const ChunkArgs a) {
  constexpr int NT = (NDM + 3) / 4;
  __shared__ float R_s[DC][16 * NDM + 4];
  __shared__ float sum_s[4][16 * NDM];  // of each block's logarithms
  __shared__ float V_s[DC][128 + 4];
  const int lane = threadIdx.x % FG_WAVE, g = lane >> 4, r16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FG_WAVE);  // (so that what depends on it is a scalar branch)
  const int c = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * 128, nd = a.d / 16, cols = min(128, a.e - c0);
  const int t0 = a.chunk_start[c], n = a.chunk_start[c + 1] - t0;
  const TA* rows = (const TA*)a.qkv;
  float kt[NT][4][4];
#pragma unroll
  for (int m = 0; m < NT; ++m)
    if (wave + 4 * m < nd) {  // uniform in the wave
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          kt[m][j][i] = to_f<TA>(rows[(size_t)(t0 + min(16 * j + 4 * g + i, n - 1)) * a.row_stride + a.k_col + h * a.d + 16 * (wave + 4 * m) + r16]);
    }
  {
    const int col = threadIdx.x % 128, t_own = threadIdx.x / 128;  // two tokens at a time
    const TA* vp = rows + a.v_col + h * a.e + c0 + min(col, cols - 1);
#pragma unroll
    for (int u0 = 0; u0 < DC / 2; u0 += 16) {
      float v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = to_f<TA>(vp[(size_t)(t0 + min(2 * (u0 + u) + t_own, n - 1)) * a.row_stride]);
#pragma unroll
      for (int u = 0; u < 16; ++u) V_s[2 * (u0 + u) + t_own][col] = 2 * (u0 + u) + t_own < n ? v[u] : 0.f;
    }
  }
  for (int i = threadIdx.x; i < 4 * a.d; i += 256) {
    const int b = i / a.d, r = i % a.d;
    float l[16], behind = 0.f;
    dc_logs(a, t0, n, h, i, l);
#pragma unroll
    for (int u = 15; u >= 0; --u) {
      R_s[16 * b + u][r] = dc_exp2(behind);
      behind += l[u];
    }
    sum_s[b][r] = behind;
  }
  __syncthreads();
  if (blockIdx.z == 0)
    for (int r = threadIdx.x; r < a.d; r += 256)
      a.prod[((size_t)c * a.H + h) * a.d + r] = dc_exp2((sum_s[0][r] + sum_s[1][r]) + (sum_s[2][r] + sum_s[3][r]));
#pragma unroll
  for (int m = 0; m < NT; ++m)
    if (wave + 4 * m < nd) {
      const int r = 16 * (wave + 4 * m) + r16;
      const float after[4] = {dc_exp2((sum_s[1][r] + sum_s[2][r]) + sum_s[3][r]), dc_exp2(sum_s[2][r] + sum_s[3][r]),
                              dc_exp2(sum_s[3][r]), 1.f};
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int s = 16 * j + 4 * g + i;
          kt[m][j][i] = s < n ? kt[m][j][i] * (R_s[s][r] * after[j]) : 0.f;
        }
    }
  float* out = a.states + ((size_t)c * a.H + h) * a.d * a.e + c0;
  for (int cb = 0; 16 * cb < cols; ++cb) {
    f32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[j][i] = V_s[16 * j + 4 * g + i][16 * cb + r16];
#pragma unroll
    for (int m = 0; m < NT; ++m) {
      const int ti = wave + 4 * m;
      if (ti < nd) {
        f32x4 acc[2];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[j / 2] = dc_mfma4(f32x4{kt[m][j][0], kt[m][j][1], kt[m][j][2], kt[m][j][3]}, v[j],
                                j % 2 ? acc[j / 2] : f32x4{0.f, 0.f, 0.f, 0.f});
        if (16 * cb + r16 < cols) {
#pragma unroll
          for (int i = 0; i < 4; ++i) out[(size_t)(16 * ti + 4 * g + i) * a.e + 16 * cb + r16] = acc[0][i] + acc[1][i];
        }
      }
    }
  }
}

// grid (n_chunks, H, ceil(e / 128)), 4 waves: M by rows (wave w the tokens of block w), then each wave blocks of 16 value
// channels for all 64 tokens.  The decays' place in LDS is taken by q P, that by the queries against the state; that of
// the keys and queries by k R, and that by M.
template <class TA, int NDM>
__global__ __launch_bounds__(256, sizeof(TA) == 2 ? 2 : 1) void decay_chunk_outputs_kernel(const ChunkArgs a) {
  constexpr int D = 16 * NDM, LD = D + 4, LQ = D + 16 / (int)sizeof(TA), NI = (4 * D + 255) / 256;
  constexpr int ROWS = DC * LQ * (int)sizeof(TA), KR = DC * LD * 4, MS = DC * (DC + 4) * 4;
  static_assert(2 * ROWS >= KR && 2 * ROWS >= MS, "k R and M fit where the queries and keys were");
  __shared__ __attribute__((aligned(16))) float A_s[DC][LD];
  __shared__ __attribute__((aligned(16))) char qk[2 * ROWS];
  __shared__ __attribute__((aligned(16))) float E_s[4][D];
  TA(*Q_s)[LQ] = (TA(*)[LQ])qk;
  TA(*K_s)[LQ] = (TA(*)[LQ])(qk + ROWS);
  float(*R_s)[LD] = (float(*)[LD])qk;
  float(*M_s)[DC + 4] = (float(*)[DC + 4])qk;
  const int lane = threadIdx.x % FG_WAVE, g = lane >> 4, r16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FG_WAVE);  // (so that what depends on it is a scalar branch)
  const int c = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * 128, d = a.d, nd = d / 16, cols = min(128, a.e - c0);
  const int t0 = a.chunk_start[c], n = a.chunk_start[c + 1] - t0;
  const TA* rows = (const TA*)a.qkv;
  struct __attribute__((aligned(4 * sizeof(TA)))) Four { TA v[4]; };
  const bool vec = a.row_stride % 4 == 0 && a.q_col % 4 == 0 && a.k_col % 4 == 0 && (uintptr_t)rows % sizeof(Four) == 0;
  for (int i = threadIdx.x; i < DC * (d / 4); i += 256) {  // four elements at a time; tokens behind the last: zeros
    const int t = i / (d / 4), r = i % (d / 4) * 4;
    const TA* row = rows + (size_t)(t0 + min(t, n - 1)) * a.row_stride + h * d + r;
    Four q4, k4;
    if (vec) {  // uniform
      q4 = *(const Four*)(row + a.q_col);
      k4 = *(const Four*)(row + a.k_col);
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) q4.v[u] = row[a.q_col + u], k4.v[u] = row[a.k_col + u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      q4.v[u] = t < n ? q4.v[u] : from_f<TA>(0.f);
      k4.v[u] = t < n ? k4.v[u] : from_f<TA>(0.f);
    }
    *(Four*)&Q_s[t][r] = q4;
    *(Four*)&K_s[t][r] = k4;
  }
  float l[NI][16];
#pragma unroll
  for (int m = 0; m < NI; ++m) {
    const int i = threadIdx.x + 256 * m, b = i / d, r = i % d;
    if (i < 4 * d) {
      dc_logs(a, t0, n, h, i, l[m]);
      float sum = 0.f;
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        A_s[16 * b + u][r] = dc_exp2(l[m][u]);
        sum += l[m][u];
      }
      E_s[b][r] = dc_exp2(sum);
    }
  }
  __syncthreads();

  // M of the wave's own block: a lane takes key r16 along the tokens, for a quarter of the channels
  f32x4 own;
  {
    float sum[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) sum[t] = 0.f;
    for (int j = 0; j < nd; ++j) {
      const int r = 16 * j + 4 * g;
      const f32x4 kv = dc_load4<TA>(&K_s[16 * wave + r16][r]);
      f32x4 w = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        const f32x4 at = *(const f32x4*)&A_s[16 * wave + t][r], qv = dc_load4<TA>(&Q_s[16 * wave + t][r]);
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = t == r16 ? kv[i] : w[i] * at[i];
        sum[t] += (qv[0] * w[0] + qv[1] * w[1]) + (qv[2] * w[2] + qv[3] * w[3]);
      }
    }
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      sum[t] += __shfl_xor(sum[t], 16, FG_WAVE);
      sum[t] += __shfl_xor(sum[t], 32, FG_WAVE);
    }
    // this lane's four tokens 4 g + i (a token before the key sees nothing of it, whatever its decays are)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = g == 0 ? sum[i] : g == 1 ? sum[4 + i] : g == 2 ? sum[8 + i] : sum[12 + i];
      own[i] = r16 <= 4 * g + i ? x : 0.f;
    }
  }
  float qp[NI][16], kr[NI][16];
#pragma unroll
  for (int m = 0; m < NI; ++m) {
    const int i = threadIdx.x + 256 * m, b = i / d, r = i % d;
    if (i < 4 * d) {
      float sum = 0.f;
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        sum += l[m][u];
        qp[m][u] = to_f<TA>(Q_s[16 * b + u][r]) * dc_exp2(sum);
      }
      sum = 0.f;
#pragma unroll
      for (int u = 15; u >= 0; --u) {
        kr[m][u] = to_f<TA>(K_s[16 * b + u][r]) * dc_exp2(sum);
        sum += l[m][u];
      }
    }
  }
  __syncthreads();  // decays, queries and keys have been read
#pragma unroll
  for (int m = 0; m < NI; ++m) {
    const int i = threadIdx.x + 256 * m, b = i / d, r = i % d;
    if (i < 4 * d) {
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        A_s[16 * b + u][r] = qp[m][u];
        R_s[16 * b + u][r] = kr[m][u];
      }
    }
  }
  __syncthreads();
  f32x4 m[4], part[4];  // M of this wave's 16 tokens (4 g + i) with the keys 16 b + r16 of block b; 32 channels of it
#pragma unroll
  for (int b = 0; b < 4; ++b) m[b] = part[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
  for (int j = 0; j < nd; ++j) {
    const int r = 16 * j + 4 * g;
    const f32x4 qv = *(const f32x4*)&A_s[16 * wave + r16][r];
    f32x4 between = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
    for (int b = 2; b >= 0; --b) {
      if (b < wave) {  // uniform in the wave
        part[b] = dc_mfma4(qv, *(const f32x4*)&R_s[16 * b + r16][r] * between, part[b]);
        between *= *(const f32x4*)&E_s[b][r];
        if (j % 2 || j == nd - 1) {
          m[b] += part[b];
          part[b] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
  }
#pragma unroll
  for (int b = 0; b < 4; ++b)
    if (b == wave) m[b] = own;
  __syncthreads();  // q P and k R have been read
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // in a vector register by decree: where some of these sums lay in accumulator registers the compiler (of ROCm 7.2)
      // began to pair two stores, gave up over the two kinds of register, and left an offset divided by four behind
      float x = m[b][i];
      asm volatile("" : "+v"(x));
      M_s[16 * wave + 4 * g + i][16 * b + r16] = x;
    }
#pragma unroll
  for (int m = 0; m < NI; ++m) {
    const int i = threadIdx.x + 256 * m, b = i / d, r = i % d;
    if (i < 4 * d && b > 0) {
      float before = 1.f;
      for (int b2 = 0; b2 < b; ++b2) before *= E_s[b2][r];
#pragma unroll
      for (int u = 0; u < 16; ++u) A_s[16 * b + u][r] *= before;
    }
  }
  __syncthreads();
  const float* S0 = a.states + ((size_t)c * a.H + h) * d * a.e + c0;
  for (int cb = wave; 16 * cb < cols; cb += 4) {
    const int col = min(16 * cb + r16, cols - 1);
    f32x4 acc[4], part[4], v[4];
#pragma unroll
    for (int tb = 0; tb < 4; ++tb) acc[tb] = part[tb] = f32x4{0.f, 0.f, 0.f, 0.f};
    const TA* vp = rows + a.v_col + h * a.e + c0 + col;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[j][i] = to_f<TA>(vp[(size_t)(t0 + min(16 * j + 4 * g + i, n - 1)) * a.row_stride]);
    f32x4 s4[NDM];
#pragma unroll
    for (int j = 0; j < NDM; ++j)
      if (j < nd) {
        const float* sp = S0 + (size_t)(16 * j + 4 * g) * a.e + col;
#pragma unroll
        for (int i = 0; i < 4; ++i) s4[j][i] = sp[(size_t)i * a.e];
      }
#pragma unroll
    for (int j = 0; j < NDM; ++j)
      if (j < nd) {
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) {
          part[tb] = dc_mfma4(*(const f32x4*)&A_s[16 * tb + r16][16 * j + 4 * g], s4[j], part[tb]);
          if (j % 2 || j == nd - 1) {
            acc[tb] += part[tb];
            part[tb] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
      }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // an infinity or NaN among the values is added by hand: a weight of zero would not keep it from earlier tokens
      f32x4 whole;
      bool odd = false;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool fine = fabsf(v[j][i]) <= 3.402823466e38f;
        whole[i] = fine ? v[j][i] : 0.f;
        odd |= !fine;
      }
#pragma unroll
      for (int tb = j; tb < 4; ++tb) {
        part[tb] = dc_mfma4(*(const f32x4*)&M_s[16 * tb + r16][16 * j + 4 * g], whole, part[tb]);
        if (j % 2 || j == tb) {
          acc[tb] += part[tb];
          part[tb] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
      if (__any(odd)) {
        for (int u = 0; u < 16; ++u) {
          const int s = 16 * j + u;
          const float mine = u % 4 == 0 ? v[j][0] : u % 4 == 1 ? v[j][1] : u % 4 == 2 ? v[j][2] : v[j][3];
          const float x = __shfl(mine, 16 * (u / 4) + r16, FG_WAVE);  // token s's value in this lane's column
          if (fabsf(x) <= 3.402823466e38f) continue;
#pragma unroll
          for (int tb = 0; tb < 4; ++tb)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (16 * tb + 4 * g + i >= s) acc[tb][i] += M_s[16 * tb + 4 * g + i][s] * x;
        }
      }
    }
    if (16 * cb + r16 < cols) {
#pragma unroll
      for (int tb = 0; tb < 4; ++tb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = 16 * tb + 4 * g + i;
          if (t < n) a.out[(size_t)(t0 + t) * ((size_t)a.H * a.e) + h * a.e + c0 + col] = acc[tb][i] * a.q_scale;
        }
    }
  }
}

// Chunk by chunk as above: d a multiple of 16 up to 128, chunks of at most chunk_tokens = 64 tokens.  `state` [n_slots, H, d, e] is read and left at slot_ids.
extern "C" int fg_decay_chunk_scan(const ChunkArgs* args, const int* slot_ids, const int* seq_chunk, float* state,
                                   int n_chunks, int chunk_tokens, int n_seqs, int act_dtype, hipStream_t stream) {
  if (n_seqs <= 0 || n_chunks <= 0) return FG_OK;
  const ChunkArgs& a = *args;
  if (chunk_tokens != DC || a.H <= 0 || a.H > 65535 || a.d <= 0 || a.d % 16 || a.d > 128 || a.e <= 0 || (a.e + 127) / 128 > 65535 || !a.qkv ||
      !a.logs || !a.chunk_start || !a.states || !a.prod || !a.out)
    return FG_ERR_ARG;
  const dim3 grid(n_chunks, a.H, (a.e + 127) / 128);
#define GO(TA, NDM)                                                                                                     \
  do {                                                                                                                  \
    decay_chunk_sums_kernel<TA, NDM><<<grid, 256, 0, stream>>>(a);                                                      \
    const int st = fg_decay_chunk_states(a.states, a.prod, state, slot_ids, seq_chunk, n_seqs, a.H, a.d, a.e, stream);  \
    if (st != FG_OK) return st;                                                                                         \
    decay_chunk_outputs_kernel<TA, NDM><<<grid, 256, 0, stream>>>(a);                                                   \
  } while (0)
  if (act_dtype == FG_F32) {
    if (a.d <= 64) GO(float, 4);
    else GO(float, 8);
  } else if (act_dtype == FG_BF16) {
    if (a.d <= 64) GO(bf16_t, 4);
    else GO(bf16_t, 8);
  } else {
    return FG_ERR_ARG;
  }
#undef GO
  return fg_launch_status();
}

extern "C" int fg_decay_scan(const ScanArgs* args, int n_seqs, int act_dtype, hipStream_t stream) {
  if (n_seqs <= 0) return FG_OK;
  const ScanArgs& a = *args;
  if (a.H <= 0 || a.d <= 0 || a.d > 512 || a.e <= 0 || a.H > 65535 || (a.e + 7) / 8 > 65535 || !a.qkv || !a.decay ||
      !a.state || !a.slot_ids || !a.q_start || !a.out)
    return FG_ERR_ARG;
  dim3 grid(n_seqs, a.H, (a.e + 7) / 8);
  const int rpl = (a.d + 7) / 8;
#define GO(TA, RPL) \
  decay_scan_kernel<TA, RPL><<<grid, FG_WAVE, (size_t)RC_TOKENS_FOR(RPL) * 3 * (a.d + 32) * sizeof(float), stream>>>(a)
#define LAUNCH(TA)               \
  do {                           \
    if (rpl <= 4) GO(TA, 4);     \
    else if (rpl <= 8) GO(TA, 8);   \
    else if (rpl <= 16) GO(TA, 16); \
    else if (rpl <= 32) GO(TA, 32); \
    else GO(TA, 64);             \
  } while (0)
  if (act_dtype == FG_F32) LAUNCH(float);
  else if (act_dtype == FG_BF16) LAUNCH(bf16_t);
  else return FG_ERR_ARG;
#undef LAUNCH
#undef GO
  return fg_launch_status();
}
