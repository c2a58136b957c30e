// Paged causal attention over the cache, general form: any element type,
// any head size that is a multiple of 8 up to 512, any number of heads and
// groups, any page size that is a multiple of 8.  One wavefront computes one
// (query token, query head) from key 0 (or the window's first key) to the
// token's own position, in tiles of 64 keys that start at multiples of 64.
// The arithmetic for a (token, head) therefore depends on nothing but that
// token's keys: not on the batch, on how the prompt was cut, or on which
// pages hold the keys.  This is the fallback for shapes the matrix-core
// kernels refuse; the 32-bit path runs `attention_f32_kernel` (below) for up
// to 16 query heads a kv head, with the same guarantee.
//
// Semantics (fastgen/forward.py:176-258): query at position p of sequence b
// sees keys 0..p of b through block_table[b]; scores (q.k)*scale, softmax in
// fp32, o = P.V; query head h reads kv head h / (H/KV).  With window > 0 only
// keys p-window+1..p are seen.  With `dist` (r1, r2 per query head) a score loses r1 * ln(1 + r2 * n) for a key n
// tokens back.
#include "common.h"
#include "kv_layout.h"

#define ATT_WAVES 4
#define ATT_TILE 64
#define ATT_MAX_HD 512

template <class T> struct Vec8;
template <> struct Vec8<float> {
  float v[8];
  __device__ __forceinline__ void load(const float* p) {
    const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
};
template <> struct Vec8<bf16_t> {
  float v[8];
  __device__ __forceinline__ void load(const bf16_t* p) {
    const uint4 raw = *(const uint4*)p;
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(w[i] << 16);
      v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
};

template <class T>
__global__ __launch_bounds__(ATT_WAVES* FG_WAVE) void paged_attention_general_kernel(
    const T* __restrict__ q, int q_stride, T* __restrict__ out, int out_stride,
    const T* __restrict__ k_pages, const T* __restrict__ v_pages,
    const int* __restrict__ block_table, int bt_stride, const int* __restrict__ seq_of_token,
    const int* __restrict__ positions, int n_tokens, int n_heads, int n_kv, int hd,
    int page_size, float scale, int window, const float* __restrict__ sinks, const float* __restrict__ dist) {
  __shared__ float q_s[ATT_WAVES][ATT_MAX_HD];
  __shared__ float p_s[ATT_WAVES][ATT_TILE];
  const int lane = threadIdx.x % FG_WAVE, wave = threadIdx.x / FG_WAVE;
  const long long item = (long long)blockIdx.x * ATT_WAVES + wave;
  if (item >= (long long)n_tokens * n_heads) return;  // whole wave leaves; no block barrier below
  const int t = (int)(item / n_heads), h = (int)(item % n_heads);
  const int kvh = h / (n_heads / n_kv);
  const int seq = seq_of_token[t];
  const int pos = positions[t];
  const int* table = block_table + (size_t)seq * bt_stride;
  const int first = first_key(pos, window);
  const KvLayout lay(page_size, hd);
  const size_t head_elems = (size_t)page_size * hd;

  const T* qrow = q + (size_t)t * q_stride + (size_t)h * hd;
  float* qs = q_s[wave];
  float* ps = p_s[wave];
  for (int d = lane; d < hd; d += FG_WAVE) qs[d] = to_f<T>(qrow[d]);
  __builtin_amdgcn_wave_barrier();

  constexpr int MAXD = ATT_MAX_HD / FG_WAVE;  // head dims owned by a lane
  float o[MAXD];
#pragma unroll
  for (int i = 0; i < MAXD; ++i) o[i] = 0.f;
  float m = -INFINITY, l = 0.f;

  for (int kb = (first / ATT_TILE) * ATT_TILE; kb <= pos; kb += ATT_TILE) {
    // ---- scores: lane j owns key kb + j
    const int key = kb + lane;
    const bool valid = key >= first && key <= pos;
    float s = -INFINITY;
    if (valid) {
      const int page = table[key / page_size];
      const T* khead = k_pages + ((size_t)page * n_kv + kvh) * head_elems;
      const int kappa = key % page_size;
      float acc = 0.f;
      for (int d = 0; d < hd; d += 8) {
        Vec8<T> kv;
        kv.load(khead + lay.k_off(kappa, d));
#pragma unroll
        for (int e = 0; e < 8; ++e) acc += qs[d + e] * kv.v[e];
      }
      s = acc * scale;
      if (dist) s -= dist[2 * h] * log1pf(dist[2 * h + 1] * (float)(pos - key));
    }
    const float m_new = fmaxf(m, wave_max(s));
    const float p = valid ? expf(s - m_new) : 0.f;
    const float alpha = expf(m - m_new);  // m = -inf on the first tile: alpha = 0
    l = l * alpha + wave_sum(p);
    m = m_new;
    __builtin_amdgcn_wave_barrier();
    ps[lane] = p;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < MAXD; ++i) o[i] *= alpha;
    // ---- o += P.V: lane owns head dims lane, lane+64, ...; one stored chunk
    // of eight key slots at a time (one page; with the permuted order the
    // slots of chunk g of a 32-key group are keys 4g..4g+3 and 16+4g..16+4g+3)
    for (int q = 0; q < ATT_TILE / 8; ++q) {
      const int base = lay.permuted ? kb + 32 * (q / 4) + 4 * (q % 4) : kb + 8 * q;  // lowest key of the chunk
      const int stride_hi = lay.permuted ? 12 : 0;  // slots 4..7 are 16 keys on (4 + 12)
      if (base > pos) { if (lay.permuted) continue; else break; }
      if (base + 7 + stride_hi < first) continue;
      const int page = table[base / page_size];
      const T* vhead = v_pages + ((size_t)page * n_kv + kvh) * head_elems;
      const int kc = lay.v_slot(base % page_size) / 8;
#pragma unroll
      for (int i = 0; i < MAXD; ++i) {
        const int d = lane + i * FG_WAVE;
        if (d < hd) {
          Vec8<T> vv;
          vv.load(vhead + lay.v_chunk_off(kc, d));
          float acc = o[i];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int kk = base + e + (e >= 4 ? stride_hi : 0);
            // select, not multiply: a slot never written may hold NaN
            if (kk >= first && kk <= pos) acc += ps[kk - kb] * vv.v[e];
          }
          o[i] = acc;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  T* orow = out + (size_t)t * out_stride + (size_t)h * hd;
  // a sink: one more term exp(sinks[h]) in the softmax's denominator, which brings no value
  if (sinks) l += expf(sinks[h] - m);
  const float inv = 1.f / l;
#pragma unroll
  for (int i = 0; i < MAXD; ++i) {
    const int d = lane + i * FG_WAVE;
    if (d < hd) orow[d] = from_f<T>(o[i] * inv);
  }
}

// ------------------------------------------------------------------ float32
// The 32-bit path's attention on v_mfma_f32_16x16x4_f32 (fp32 products and sums).  A workgroup owns up to 16 rows:
// the query heads of one kv head for a few consecutive tokens of one sequence (blocks of 16 / group tokens, cut where
// the sequence changes; a workgroup a token is launched and all but a run's first leave, so that a prompt fills the
// rows and the decoded tokens of many sequences do not wait for one another).  Tiles of 64 keys start at multiples of
// 64; tile i belongs to wave i % 8 whatever the workgroup holds, a wave's tiles follow one another with a running
// maximum, the eight waves' results are merged in order: a (token, head)'s arithmetic depends on its own keys alone,
// so the bits are the same for a prompt, a decoded token and any cut.  S^T = K Q^T leaves a lane 4 keys of one row,
// which is how O^T += V^T P^T takes them: nothing moves between lanes but a row's maximum and sum.  Keys and values
// come straight from the pages, 1 KB (keys) and two halves of 2 KB (values) a load.
//
// Before: a wave a (token, head), a lane a key.  24 heads on 8 kv heads of 128, us before and now: a prompt of 400 /
// 2048 tokens 174 / 3628 -> 59 / 592 (a third of the fp32 matrix cores' rate), one token of 4 sequences of 500 keys
// 117 -> 30, of one of 4000 1243 -> 133 (the chain of a wave's 8 tiles), of 64 of 1000 455 -> 122, of 200 of 300 184 ->
// 188 (both bound by the pages' reads, 2.6 TB/s).
typedef float f32x4 __attribute__((ext_vector_type(4)));
#define AF_WAVES 8

// DB: head dims in blocks of 16, at least hd / 16 (hd is a multiple of 8).
template <int DB>
__global__ __launch_bounds__(AF_WAVES* FG_WAVE) void attention_f32_kernel(
    const float* __restrict__ q, int q_stride, float* __restrict__ out, int out_stride,
    const float* __restrict__ k_pages, const float* __restrict__ v_pages, const int* __restrict__ block_table,
    int bt_stride, const int* __restrict__ seq_of_token, const int* __restrict__ positions, int n_tokens, int n_heads,
    int n_kv, int hd, int page_size, float scale, int window, const float* __restrict__ sinks,
    const float* __restrict__ dist) {
  constexpr int MB = DB < 8 ? DB : 8;             // dim blocks merged at a time
  __shared__ f32x4 q_s[DB * 4][16];               // [4 dims][row]
  __shared__ f32x4 o_s[AF_WAVES][MB][FG_WAVE];
  __shared__ float m_s[AF_WAVES][16], l_s[AF_WAVES][16];
  const int tid = threadIdx.x, lane = tid % FG_WAVE, wave = tid / FG_WAVE;
  const int r = lane % 16, g = lane / 16;
  const int kvh = blockIdx.x % n_kv, group = n_heads / n_kv;
  // (the blocks' first tokens come first, a token's kv heads side by side: every die gets as many of them)
  const int full = 16 / group, blocks = (n_tokens + full - 1) / full, place = blockIdx.x / n_kv;
  const int t0 = place % blocks * full + place / blocks;
  if (t0 >= n_tokens) return;
  const int seq = seq_of_token[t0];
  if (t0 % full && seq_of_token[t0 - 1] == seq) return;  // an earlier workgroup's run holds this token
  int n_here = 1, p_lo = positions[t0], p_hi = p_lo;
  for (; t0 + n_here < n_tokens && (t0 + n_here) % full && seq_of_token[t0 + n_here] == seq; ++n_here) {
    const int p = positions[t0 + n_here];
    p_lo = min(p_lo, p);
    p_hi = max(p_hi, p);
  }
  const KvLayout lay(page_size, hd);
  const size_t head_elems = (size_t)page_size * hd;

  // this lane's row: a token of the block and one of its heads (rows behind the last repeat the last token)
  const int mine = min(r / group, n_here - 1);
  const bool live = r < n_here * group;
  const int head = kvh * group + r % group, pos = positions[t0 + mine], first = first_key(pos, window);
  const float d1 = dist ? dist[2 * head] : 0.f, d2 = dist ? dist[2 * head + 1] : 0.f;
  for (int i = tid; i < DB * 4 * 16 * 4; i += AF_WAVES * FG_WAVE) {  // element by element: q may lie anywhere
    const int d = i % (DB * 16), row = i / (DB * 16);
    const int t = t0 + min(row / group, n_here - 1), h = kvh * group + row % group;
    ((float*)&q_s[d / 4][row])[d % 4] = d < hd ? q[(size_t)t * q_stride + (size_t)h * hd + d] : 0.f;
  }
  __syncthreads();

  const int* table = block_table + (size_t)seq * bt_stride;
  const int lo = first_key(p_lo, window), hi = p_hi;  // the keys that some row of the run sees: their pages are held

  f32x4 acc[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  for (int tile = lo / ATT_TILE + ((wave - lo / ATT_TILE) & (AF_WAVES - 1)); tile * ATT_TILE <= hi; tile += AF_WAVES) {
    const int kb = tile * ATT_TILE;
    const float* kp[4];
    const float* vp[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {  // (keys that no row sees are read as the nearest one that some row does)
      const int key = min(max(kb + 16 * b + r, lo), hi);
      kp[b] = k_pages + ((size_t)table[key / page_size] * n_kv + kvh) * head_elems + lay.k_off(key % page_size, 0);
      const int four = min(max(kb + 16 * b + 4 * g, lo & ~3), hi & ~3), slot = lay.v_slot(four % page_size);
      vp[b] = v_pages + ((size_t)table[four / page_size] * n_kv + kvh) * head_elems + slot % 8 +
              lay.v_chunk_off(slot / 8, 0);
    }
    const size_t chunk = (size_t)8 << lay.kb_shift;  // from 8 head dims of a key to the next 8
    f32x4 s[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) s[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < DB; ++i) {
      const f32x4 qv = q_s[4 * i + g][r];
      f32x4 kv[4];
      const bool in = 16 * i + 4 * g < hd;
#pragma unroll
      for (int b = 0; b < 4; ++b)
        kv[b] = in ? *(const f32x4*)(kp[b] + chunk * (2 * i + g / 2) + g % 2 * 4) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int b = 0; b < 4; ++b) s[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[b][e], qv[e], s[b], 0, 0, 0);
    }
    float top = -INFINITY;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = kb + 16 * b + 4 * g + e;
        float v = s[b][e] * scale;
        if (dist) v -= d1 * log1pf(d2 * (float)(pos - key));
        s[b][e] = live && key >= first && key <= pos ? v : -INFINITY;
        top = fmaxf(top, s[b][e]);
      }
    top = fmaxf(top, __shfl_xor(top, 16, FG_WAVE));
    top = fmaxf(top, __shfl_xor(top, 32, FG_WAVE));
    const float m_new = fmaxf(m, top);
    // a row that has seen no key yet, or sees none in this tile, stays as it is
    const float alpha = m == m_new ? 1.f : expf(m - m_new);
    float sum = 0.f;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = kb + 16 * b + 4 * g + e;
        s[b][e] = live && key >= first && key <= pos ? expf(s[b][e] - m_new) : 0.f;
        sum += s[b][e];
      }
    sum += __shfl_xor(sum, 16, FG_WAVE);
    sum += __shfl_xor(sum, 32, FG_WAVE);
    l = l * alpha + sum;
    m = m_new;
    // whether some key of the tile is seen by one row of the run and not by another
    const bool mixed = kb + ATT_TILE - 1 > p_lo || kb < first_key(p_hi, window);
#pragma unroll
    for (int i = 0; i < DB; ++i) {
      acc[i] *= alpha;
      const int d = 16 * i + r;
      f32x4 vv[4];
      const size_t at = lay.v_chunk_off(0, d);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        vv[b] = d < hd ? *(const f32x4*)(vp[b] + at) : f32x4{0.f, 0.f, 0.f, 0.f};
        // what lies behind the keys was never written and may be anything
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = kb + 16 * b + 4 * g + e;
          if (key < lo || key > hi) vv[b][e] = 0.f;
        }
      }
      bool bad = false;
      if (mixed && p_lo != p_hi) {
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) bad |= !(fabsf(vv[b][e]) <= 3.402823466e38f);
      }
      if (!__any(bad)) {
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[b][e], s[b][e], acc[i], 0, 0, 0);
      } else {  // an infinity or NaN among the values: a weight of zero would not keep it from the rows before it
        for (int row = 0; row < 16; ++row) {
          const int p = __shfl(pos, row, FG_WAVE), f = __shfl(first, row, FG_WAVE);
          f32x4 one = acc[i];
#pragma unroll
          for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int key = kb + 16 * b + 4 * g + e;
              one = __builtin_amdgcn_mfma_f32_16x16x4f32(key >= f && key <= p ? vv[b][e] : 0.f, s[b][e], one, 0, 0, 0);
            }
          if (r == row) acc[i] = one;
        }
      }
    }
  }

  // ---- the waves' results, in order
  if (lane < 16) m_s[wave][r] = m, l_s[wave][r] = l;
  __syncthreads();
  float top = m_s[0][r];
#pragma unroll
  for (int w = 1; w < AF_WAVES; ++w) top = fmaxf(top, m_s[w][r]);
  const float factor = m == top ? 1.f : expf(m - top);
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < AF_WAVES; ++w) total += l_s[w][r] * (m_s[w][r] == top ? 1.f : expf(m_s[w][r] - top));
  // a sink: one more term exp(sinks[h]) in the softmax's denominator, which brings no value
  if (sinks) total += expf(sinks[head] - top);
  const float inv = 1.f / total;
#pragma unroll
  for (int i0 = 0; i0 < DB; i0 += MB) {
#pragma unroll
    for (int i = 0; i < MB; ++i) o_s[wave][i][lane] = acc[i0 + i] * factor;
    __syncthreads();
    if (wave < MB) {  // (a thread's lane stands for the same row and dims as above, its wave for the dim block)
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < AF_WAVES; ++w) o += o_s[w][wave][lane];
      const int d = 16 * (i0 + wave) + 4 * g;
      if (live) {
        float* at = out + (size_t)(t0 + mine) * out_stride + (size_t)head * hd + d;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < hd) at[e] = o[e] * inv;
      }
    }
    __syncthreads();
  }
}

extern "C" int fg_paged_attention_general_sink(
    const void* q, int q_stride, void* out, int out_stride, const void* k_pages,
    const void* v_pages, const int* block_table, int bt_stride, const int* seq_of_token,
    const int* positions, int n_tokens, int n_heads, int n_kv, int hd, int page_size,
    float scale, int window, const float* sinks, const float* dist, int dtype, hipStream_t stream) {
  if (n_tokens <= 0) return FG_OK;
  if (hd <= 0 || hd % 8 || hd > ATT_MAX_HD || page_size <= 0 || page_size % 8 || n_kv <= 0 ||
      n_heads <= 0 || n_heads % n_kv)
    return FG_ERR_ARG;
  const int group = n_heads / n_kv;
  if (dtype == FG_F32 && group <= 16) {
    const int full = 16 / group;
    const long long grid = (long long)((n_tokens + full - 1) / full * full) * n_kv;
    if (grid > 2147483647LL) return FG_ERR_ARG;
#define ATTENTION_F32(DB)                                                                                           \
  attention_f32_kernel<DB><<<(unsigned)grid, AF_WAVES * FG_WAVE, 0, stream>>>(                                                \
      (const float*)q, q_stride, (float*)out, out_stride, (const float*)k_pages, (const float*)v_pages, block_table, \
      bt_stride, seq_of_token, positions, n_tokens, n_heads, n_kv, hd, page_size, scale, window, sinks, dist)
    if (hd <= 64) ATTENTION_F32(4);
    else if (hd <= 128) ATTENTION_F32(8);
    else if (hd <= 256) ATTENTION_F32(16);
    else ATTENTION_F32(32);
#undef ATTENTION_F32
    return fg_launch_status();
  }
  const long long items = (long long)n_tokens * n_heads;
  const long long blocks = (items + ATT_WAVES - 1) / ATT_WAVES;
  if (blocks > 2147483647LL) return FG_ERR_ARG;
  dim3 grid((unsigned)blocks);
  if (dtype == FG_F32)
    paged_attention_general_kernel<float><<<grid, ATT_WAVES * FG_WAVE, 0, stream>>>(
        (const float*)q, q_stride, (float*)out, out_stride, (const float*)k_pages,
        (const float*)v_pages, block_table, bt_stride, seq_of_token, positions, n_tokens,
        n_heads, n_kv, hd, page_size, scale, window, sinks, dist);
  else if (dtype == FG_BF16)
    paged_attention_general_kernel<bf16_t><<<grid, ATT_WAVES * FG_WAVE, 0, stream>>>(
        (const bf16_t*)q, q_stride, (bf16_t*)out, out_stride, (const bf16_t*)k_pages,
        (const bf16_t*)v_pages, block_table, bt_stride, seq_of_token, positions, n_tokens,
        n_heads, n_kv, hd, page_size, scale, window, sinks, dist);
  else
    return FG_ERR_ARG;
  return fg_launch_status();
}

extern "C" int fg_paged_attention_general(
    const void* q, int q_stride, void* out, int out_stride, const void* k_pages,
    const void* v_pages, const int* block_table, int bt_stride, const int* seq_of_token,
    const int* positions, int n_tokens, int n_heads, int n_kv, int hd, int page_size,
    float scale, int window, int dtype, hipStream_t stream) {
  return fg_paged_attention_general_sink(q, q_stride, out, out_stride, k_pages, v_pages, block_table, bt_stride,
                                         seq_of_token, positions, n_tokens, n_heads, n_kv, hd, page_size, scale,
                                         window, nullptr, nullptr, dtype, stream);
}
