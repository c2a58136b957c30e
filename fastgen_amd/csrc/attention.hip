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
// The 32-bit path's attention on v_mfma_f32_16x16x4_f32 (fp32 products and sums).  A run is up to 16 rows: the query
// heads of one kv head for a few consecutive tokens of one sequence (blocks of 16 / group tokens, cut where the sequence
// changes; a workgroup a token is launched and all but a run's first leave, so that a prompt fills the rows and the
// decoded tokens of many sequences do not wait for one another).  Tiles of 64 keys start at multiples of 64; tile i
// belongs to part i % 8 whatever the run holds, a part's tiles follow one another with a running maximum, the eight
// parts' results are merged in order: a (token, head)'s arithmetic depends on its own keys alone, so the bits are the
// same for a prompt, a decoded token and any cut.  S^T = K Q^T leaves a lane 4 keys of one row, which is how
// O^T += V^T P^T takes them: nothing moves between lanes but a row's maximum and sum.  Keys and values come straight
// from the pages, 1 KB (keys) and two halves of 2 KB (values) a load.
//
// A workgroup's eight waves take the parts of its run.  Where many sequences have few keys each, most waves would have no
// tile and the others one, and a compute unit holds one such workgroup at a time (its registers).  So a run of at most 4
// rows and 8 tiles (a part has one tile at most) is, if there are many (`af_alone_from`), a single wave's: a workgroup
// takes eight runs, one a wave, which keeps the scores of its tiles in LDS until it knows the rows' maxima and then does
// what the eight waves' merge does, operation for operation: the same bits, so the choice is free to follow the load.
//
// A run of one tile (the first 64 places of a sequence) is where a workgroup of eight waves is most of it idle.  If there may
// be many, a kernel of its own takes them, a wave a run of up to 16 rows: it needs no sums but a block's, so its loads are
// 2 to 7 blocks of 16 dims ahead and several waves share a SIMD, and it leaves out the blocks of 16 keys behind the run's
// last, which bring zeros.  The same operations otherwise, the same bits.  us, (token, head) by (token, head) / without
// that kernel / with it, heads / kv heads x head size:
//                            32/8x128          32/32x128         16/16x64         16/1x80          16/4x256         8/8x512
//   64 prompts of 5      24 /  65 /  26    28 / 140 /  62    10 / 52 / 28    11 / 27 / 13    21 /  64 /  22    39 / 144 / 37
//   8 of 37              34 /  51 /  29    35 /  81 /  54    14 / 36 / 28    17 / 28 / 20    32 /  50 /  36    60 / 109 / 55
//   20 of 60            142 / 162 /  67   146 / 311 / 196    47 /103 / 71    61 / 66 / 29   134 / 127 /  62
//   300 decoded, 9 keys  35 /  43 /  29    37 / 130 /  96    14 / 45 / 42    13 / 27 / 13    29 /  35 /  25    49 / 171 / 66
// What is left to the first column is mostly the workgroups that find no run of theirs (9600 of 8 waves: 46 us).
//
// Bound by the latency of a tile's loads in each wave (the next block of 16 dims in flight while one is multiplied; more
// of them in flight cost the registers) and, for long sequences, by the pages' reads.  Before: a wave a (token, head), a
// lane a key (`paged_attention_general_kernel`).  us, before and now (heads / kv heads x head size):
//                                   24/8x128    32/32x128    16/16x64     16/4x256    16/16x256      8/8x512
//   a prompt of 400 tokens         181 /  58   230 /  94    94 /  38    251 /  64    267 /  68    415 /  79
//   a prompt of 2048 tokens       3682 / 516  4627 / 781  1295 / 267   4009 / 535   4394 / 608   5180 / 626
//   4 sequences of 500 keys        116 /  24   175 /  23    74 /  18    194 /  33    297 /  34    552 /  71
//   32 of 4000                    1589 / 296  1773 / 700  1024 / 201   2803 / 229   3050 / 688   5708 / 800
//   64 of 60, a wave a run          32 /  27    35 /  40    17 /  18     42 /  25*    45 /  38     75 /  83
//   64 of 60, a workgroup a run     32 /  30    35 / 108    17 /  41     42 /  25     45 /  86     75 / 102
//   200 of 100, a wave a run        61 /  45   177 / 168    41 /  52     84 /  62    155 / 150    206 / 217
//   200 of 300, a wave a run       180 / 101   430 / 409   123 / 116    274 / 141*   386 / 372    541 / 524
//   200 of 300, a workgroup a run  180 / 147   430 / 497   123 / 180    274 / 141    386 / 431    541 / 566
// (* too few runs: a workgroup each.)
typedef float f32x4 __attribute__((ext_vector_type(4)));
#define AF_WAVES 8
#define AF_ALONE_ROWS 4

// From how many runs on a wave alone takes a run of `tiles` tiles.  As measured, a wave a run / a workgroup a run: with 256
// runs of one tile 36 / 26 us (head size 256), with 512 25 / 30 (128); 512 runs of 4 tiles 66 / 36, 1024 of 4 125 / 120
// (256), 2048 of 4 107 / 139 (128); 800 of 5 145 / 144 (256), 1600 of 5 100 / 151 (128); 1600 of 8 152 / 179, 3200 of 8
// 581 / 571 (256).  Head sizes up to 64, where a workgroup's chain is shorter: 1024 of 4 45 / 45, 3200 of 5 116 / 180, 1600
// of 5 beside a prompt of 400 tokens 143 / 133.
__host__ __device__ constexpr int af_alone_from(int db, int tiles) { return db <= 4 ? 350 * tiles : 160 * (tiles + 1); }

struct AfArgs {
  const float* q; int q_stride;
  float* out; int out_stride;
  const float *k_pages, *v_pages;
  const int* block_table; int bt_stride;
  const int *seq_of_token, *positions;
  int n_tokens, n_heads, n_kv, hd, page_size;
  float scale; int window;
  const float *sinks, *dist;
  int few_runs;  // how many runs of few rows there may be: one a sequence and kv head
  int ones;      // whether runs of one tile are another kernel's
};

struct AfRun {
  int t0, n_here, seq, kvh, p_lo, p_hi;  // its tokens, and their lowest and highest position
  int lo;                                // keys lo .. p_hi are seen by some row: their pages are held
};
// A block's tokens, one a lane, and which of them start a run (bit i: token i).
struct AfBlock {
  int t0, n, seq, pos;
  unsigned starts;
};
__device__ __forceinline__ AfBlock af_block(const AfArgs& a, int block, int lane) {
  const int full = 16 / (a.n_heads / a.n_kv);
  AfBlock k;
  k.t0 = block * full;
  k.n = min(full, a.n_tokens - k.t0);
  const int t = k.t0 + min(lane, k.n - 1);
  k.seq = a.seq_of_token[t];
  k.pos = a.positions[t];
  const int before = __shfl_up(k.seq, 1, FG_WAVE);
  k.starts = (unsigned)__ballot(lane < k.n && (lane == 0 || before != k.seq));
  return k;
}
// Run j of a block for a kv head; false: there are not so many.  Uniform.
__device__ __forceinline__ bool af_run(const AfArgs& a, const AfBlock& k, int kvh, int j, AfRun& run) {
  unsigned rest = k.starts;
  for (; j > 0 && rest; --j) rest &= rest - 1;
  if (!rest) return false;
  const int at = __ffs(rest) - 1;
  rest &= rest - 1;
  const int end = rest ? __ffs(rest) - 1 : k.n;
  run.t0 = k.t0 + at, run.n_here = end - at, run.kvh = kvh;
  run.seq = __builtin_amdgcn_readlane(k.seq, at);
  run.p_lo = run.p_hi = __builtin_amdgcn_readlane(k.pos, at);
  for (int i = at + 1; i < end; ++i) {
    const int p = __builtin_amdgcn_readlane(k.pos, i);
    run.p_lo = min(run.p_lo, p);
    run.p_hi = max(run.p_hi, p);
  }
  run.lo = first_key(run.p_lo, a.window);
  return true;
}

// Who takes a run: a workgroup, or a wave that keeps its scores in LDS; or, where that is launched, a wave of the kernel
// for runs of one tile.
enum { AF_TOGETHER, AF_ALONE, AF_ONE };
// (at the largest head sizes the queries' room in LDS, and a wave's time for more keys, are too much)
__host__ __device__ constexpr int af_one_rows(int db) { return db <= 16 ? 16 : 8; }
__host__ __device__ constexpr int af_one_blocks(int db) { return db <= 16 ? 4 : 2; }  // of 16 keys
template <int DB>
__device__ __forceinline__ int af_kind(const AfArgs& a, const AfRun& run) {
  const int tiles = run.p_hi / ATT_TILE - run.lo / ATT_TILE + 1, rows = run.n_here * (a.n_heads / a.n_kv);
  if (a.ones && tiles == 1 && rows <= af_one_rows(DB) && run.p_hi % ATT_TILE / 16 < af_one_blocks(DB)) return AF_ONE;
  return rows <= AF_ALONE_ROWS && tiles <= AF_WAVES && a.few_runs >= af_alone_from(DB, tiles) ? AF_ALONE : AF_TOGETHER;
}

// Lane 16 g + r's row r: a token of the run and one of its heads (rows behind the last see no key and are not stored).
struct AfRow {
  int token, head, pos, first;
  bool live;
  float d1, d2;
};
__device__ __forceinline__ AfRow af_row(const AfArgs& a, const AfRun& run, int r) {
  const int group = a.n_heads / a.n_kv;
  AfRow row;
  row.token = run.t0 + min(r / group, run.n_here - 1);
  row.live = r < run.n_here * group;
  row.head = run.kvh * group + r % group;
  row.pos = a.positions[row.token];
  row.first = first_key(row.pos, a.window);
  row.d1 = a.dist ? a.dist[2 * row.head] : 0.f;
  row.d2 = a.dist ? a.dist[2 * row.head + 1] : 0.f;
  return row;
}
__device__ __forceinline__ bool af_sees(const AfRow& row, int key) { return row.live && key >= row.first && key <= row.pos; }

// Query rows first, first + step, .. (below `rows`) of the run into LDS, q_s[4 dims][N rows], by a wave, element by element:
// q may lie anywhere.
template <int DB, int N>
__device__ __forceinline__ void af_queries(const AfArgs& a, const AfRun& run, f32x4 (*q_s)[N], int first, int step, int rows,
                                           int lane) {
  const int group = a.n_heads / a.n_kv;
  for (int row = first; row < rows; row += step) {  // uniform in the wave
    const float* q = a.q + (size_t)(run.t0 + row / group) * a.q_stride + (size_t)(run.kvh * group + row % group) * a.hd;
    float x[DB / 4];
#pragma unroll
    for (int k = 0; k < DB / 4; ++k) x[k] = q[min(lane + k * FG_WAVE, a.hd - 1)];
#pragma unroll
    for (int k = 0; k < DB / 4; ++k) {
      const int d = lane + k * FG_WAVE;
      ((float*)&q_s[d / 4][row])[d % 4] = d < a.hd ? x[k] : 0.f;
    }
  }
}

// Scores of the tile's keys 16 b + 4 g + e with the lane's row (-infinity where the row does not see the key), and the
// row's highest.
template <int DB, int AHEAD, int N, int NB>
__device__ __forceinline__ float af_scores(const AfArgs& a, const AfRun& run, const AfRow& row, const KvLayout& lay, int tile,
                                           const f32x4 (*q_s)[N], int q_row, int r, int g, f32x4 (&s)[NB]) {
  const int kb = tile * ATT_TILE;
  const int* table = a.block_table + (size_t)run.seq * a.bt_stride;
  const float* kp[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {  // (keys that no row sees are read as the nearest one that some row does)
    const int key = min(max(kb + 16 * b + r, run.lo), run.p_hi);
    kp[b] = a.k_pages + ((size_t)table[key / a.page_size] * a.n_kv + run.kvh) * ((size_t)a.page_size * a.hd) +
            lay.k_off(key % a.page_size, 0);
    s[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const size_t chunk = (size_t)8 << lay.kb_shift;  // from 8 head dims of a key to the next 8
  // The next blocks of 16 dims are asked for before this one is multiplied, and never conditionally: behind the head's
  // dims its first ones, for zeros.
  f32x4 kv[AHEAD + 1][NB];
  auto load = [&](int i) {
    const size_t at = 16 * i + 4 * g < a.hd ? chunk * (2 * i + g / 2) + g % 2 * 4 : 0;
#pragma unroll
    for (int b = 0; b < NB; ++b) kv[i % (AHEAD + 1)][b] = *(const f32x4*)(kp[b] + at);
  };
#pragma unroll
  for (int i = 0; i < AHEAD && i < DB; ++i) load(i);
#pragma unroll
  for (int i = 0; i < DB; ++i) {
    if (i + AHEAD < DB) load(i + AHEAD);
    __builtin_amdgcn_sched_barrier(0);
    const f32x4 qv = q_s[4 * i + g][q_row];
    const bool in = 16 * i + 4 * g < a.hd;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int b = 0; b < NB; ++b)
        s[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? kv[i % (AHEAD + 1)][b][e] : 0.f, qv[e], s[b], 0, 0, 0);
  }
  float top = -INFINITY;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int key = kb + 16 * b + 4 * g + e;
      float v = s[b][e] * a.scale;
      if (a.dist) v -= row.d1 * log1pf(row.d2 * (float)(row.pos - key));
      asm("" : "+v"(v));  // rounded here in every use (a product fused with the maximum's subtraction would not be)
      s[b][e] = af_sees(row, key) ? v : -INFINITY;
      top = fmaxf(top, s[b][e]);
    }
  top = fmaxf(top, __shfl_xor(top, 16, FG_WAVE));
  return fmaxf(top, __shfl_xor(top, 32, FG_WAVE));
}

// The tile's weights in the place of its scores, and the row's sum of them.
template <int NB>
__device__ __forceinline__ float af_weights(const AfRow& row, int tile, float m, int g, f32x4 (&s)[NB]) {
  float sum = 0.f;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[b][e] = af_sees(row, tile * ATT_TILE + 16 * b + 4 * g + e) ? expf(s[b][e] - m) : 0.f;
      sum += s[b][e];
    }
  sum += __shfl_xor(sum, 16, FG_WAVE);
  return sum + __shfl_xor(sum, 32, FG_WAVE);
}

// done(i, start(i) + V^T P^T) for the blocks i of 16 head dims: lane 16 g + r gets dims 16 i + 4 g .. + 3 of row r.
template <int DB, int AHEAD, int NB, class Start, class Done>
__device__ __forceinline__ void af_values(const AfArgs& a, const AfRun& run, const AfRow& row, const KvLayout& lay, int tile,
                                          const f32x4 (&w)[NB], int r, int g, Start start, Done done) {
  const int kb = tile * ATT_TILE, lo = run.lo, hi = run.p_hi;
  const int* table = a.block_table + (size_t)run.seq * a.bt_stride;
  const float* vp[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int four = min(max(kb + 16 * b + 4 * g, lo & ~3), hi & ~3), slot = lay.v_slot(four % a.page_size);
    vp[b] = a.v_pages + ((size_t)table[four / a.page_size] * a.n_kv + run.kvh) * ((size_t)a.page_size * a.hd) + slot % 8 +
            lay.v_chunk_off(slot / 8, 0);
  }
  // whether some key of the tile is seen by one row of the run and not by another
  const bool mixed = run.p_lo != hi && (kb + ATT_TILE - 1 > run.p_lo || kb < first_key(hi, a.window));
  f32x4 vv[AHEAD + 1][NB];
  auto load = [&](int i) {
    const size_t at = lay.v_chunk_off(0, 16 * i + r < a.hd ? 16 * i + r : 0);
#pragma unroll
    for (int b = 0; b < NB; ++b) vv[i % (AHEAD + 1)][b] = *(const f32x4*)(vp[b] + at);
  };
#pragma unroll
  for (int i = 0; i < AHEAD && i < DB; ++i) load(i);
#pragma unroll
  for (int i = 0; i < DB; ++i) {
    if (i + AHEAD < DB) load(i + AHEAD);
    __builtin_amdgcn_sched_barrier(0);
    f32x4(&v)[NB] = vv[i % (AHEAD + 1)];
    // dims behind the head's, and keys that no row sees: their places may hold anything
    const bool in = 16 * i + r < a.hd;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = kb + 16 * b + 4 * g + e;
        v[b][e] = in && key >= lo && key <= hi ? v[b][e] : 0.f;
      }
    bool bad = false;
    if (mixed) {  // uniform
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) bad |= !(fabsf(v[b][e]) <= 3.402823466e38f);
    }
    f32x4 acc = start(i);
    if (!__any(bad)) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(v[b][e], w[b][e], acc, 0, 0, 0);
    } else {  // an infinity or NaN among the values: a weight of zero would not keep it from the rows before it
      for (int other = 0; other < 16; ++other) {
        const int p = __shfl(row.pos, other, FG_WAVE), f = __shfl(row.first, other, FG_WAVE);
        f32x4 one = acc;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int key = kb + 16 * b + 4 * g + e;
            one = __builtin_amdgcn_mfma_f32_16x16x4f32(key >= f && key <= p ? v[b][e] : 0.f, w[b][e], one, 0, 0, 0);
          }
        if (r == other) acc = one;
      }
    }
    done(i, acc);
  }
}

// A part's share of a row whose highest score is `top`.
__device__ __forceinline__ float af_factor(float m, float top) { return m == top ? 1.f : expf(m - top); }
__device__ __forceinline__ f32x4 af_scaled(const f32x4 x, float f) {  // rounded, whatever is added to it
  f32x4 y = x * f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float v = y[e];
    asm("" : "+v"(v));
    y[e] = v;
  }
  return y;
}
// A sink is one more term exp(sinks[h]) in the softmax's denominator, which brings no value.
__device__ __forceinline__ float af_inverse(const AfArgs& a, const AfRow& row, float total, float top) {
  if (a.sinks) total += expf(a.sinks[row.head] - top);
  return 1.f / total;
}
__device__ __forceinline__ void af_store(const AfArgs& a, const AfRow& row, int d, const f32x4 o, float inv) {
  if (!row.live) return;
  float* at = a.out + (size_t)row.token * a.out_stride + (size_t)row.head * a.hd + d;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (d + e < a.hd) at[e] = o[e] * inv;
}

// What a workgroup keeps in LDS for a run of its own, and what each of its waves does for one.
template <int DB>
struct AfShared {
  static constexpr int MB = DB < 8 ? DB : 8;  // dim blocks merged at a time
  f32x4 q_s[DB * 4][16];                      // [4 dims][row]
  f32x4 o_s[AF_WAVES][MB][FG_WAVE];
  float m_s[AF_WAVES][16], l_s[AF_WAVES][16];
};
template <int DB>
struct AfOne {
  f32x4 q_s[DB * 4][af_one_rows(DB)];
};
template <int DB>
struct AfAlone {
  f32x4 q_s[DB * 4][AF_ALONE_ROWS];
  f32x4 s_s[AF_WAVES][AF_ALONE_ROWS][ATT_TILE / 4];  // a part's scores
  float m_s[AF_WAVES][AF_ALONE_ROWS];
};

// A run by a workgroup; ends in a barrier.
template <int DB>
__device__ __forceinline__ void af_together(const AfArgs& a, const AfRun& run, AfShared<DB>& lds, int wave, int lane) {
  constexpr int MB = AfShared<DB>::MB;
  const int r = lane % 16, g = lane / 16;
  const KvLayout lay(a.page_size, a.hd);
  const AfRow row = af_row(a, run, r);
  af_queries<DB, 16>(a, run, lds.q_s, wave, AF_WAVES, run.n_here * (a.n_heads / a.n_kv), lane);
  __syncthreads();
  f32x4 acc[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const int t_lo = run.lo / ATT_TILE;
  for (int tile = t_lo + ((wave - t_lo) & (AF_WAVES - 1)); tile * ATT_TILE <= run.p_hi; tile += AF_WAVES) {
    f32x4 s[4];
    const float m_new = fmaxf(m, af_scores<DB, 1>(a, run, row, lay, tile, lds.q_s, r, r, g, s));
    // a row that has seen no key yet, or sees none in this tile, stays as it is
    const float alpha = af_factor(m, m_new);
    l = l * alpha + af_weights(row, tile, m_new, g, s);
    m = m_new;
    af_values<DB, 1>(a, run, row, lay, tile, s, r, g, [&](int i) { return acc[i] * alpha; },
                  [&](int i, const f32x4 x) { acc[i] = x; });
  }
  // ---- the parts' results, in order
  if (lane < 16) lds.m_s[wave][r] = m, lds.l_s[wave][r] = l;
  __syncthreads();
  float top = lds.m_s[0][r];
#pragma unroll
  for (int w = 1; w < AF_WAVES; ++w) top = fmaxf(top, lds.m_s[w][r]);
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < AF_WAVES; ++w) total = fmaf(lds.l_s[w][r], af_factor(lds.m_s[w][r], top), total);
  const float factor = af_factor(m, top), inv = af_inverse(a, row, total, top);
#pragma unroll
  for (int i0 = 0; i0 < DB; i0 += MB) {
#pragma unroll
    for (int i = 0; i < MB; ++i) lds.o_s[wave][i][lane] = acc[i0 + i] * factor;
    __syncthreads();
    if (wave < MB) {  // (a thread's lane stands for the same row and dims as above, its wave for the dim block)
      f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < AF_WAVES; ++w) o += lds.o_s[w][wave][lane];
      af_store(a, row, 16 * (i0 + wave) + 4 * g, o, inv);
    }
    __syncthreads();
  }
}

// A run of at most AF_ALONE_ROWS rows and AF_WAVES tiles by a wave: what `af_together` does, part after part.
template <int DB>
__device__ __forceinline__ void af_by_wave(const AfArgs& a, const AfRun& run, AfAlone<DB>& lds, int lane) {
  const int r = lane % 16, g = lane / 16, q_row = min(r, AF_ALONE_ROWS - 1);
  const bool keeps = r < AF_ALONE_ROWS;
  const KvLayout lay(a.page_size, a.hd);
  const AfRow row = af_row(a, run, r);
  af_queries<DB, AF_ALONE_ROWS>(a, run, lds.q_s, 0, 1, run.n_here * (a.n_heads / a.n_kv), lane);
  // (a wave's LDS operations are done in order; the fences keep the compiler to it)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const int t_lo = run.lo / ATT_TILE, t_hi = run.p_hi / ATT_TILE;
  float top = -INFINITY;
  for (int tile = t_lo; tile <= t_hi; ++tile) {
    f32x4 s[4];
    const float m = af_scores<DB, 1>(a, run, row, lay, tile, lds.q_s, q_row, r, g, s);
    top = fmaxf(top, m);
    if (keeps) {
#pragma unroll
      for (int b = 0; b < 4; ++b) lds.s_s[tile % AF_WAVES][r][4 * b + g] = s[b];
      if (g == 0) lds.m_s[tile % AF_WAVES][r] = m;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  f32x4 o[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float total = 0.f;
  for (int part = 0; part < AF_WAVES; ++part) {
    const int tile = t_lo + ((part - t_lo) & (AF_WAVES - 1));
    if (tile > t_hi) continue;
    f32x4 s[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) s[b] = lds.s_s[part][q_row][4 * b + g];
    const float m = lds.m_s[part][q_row], l = af_weights(row, tile, m, g, s), factor = af_factor(m, top);
    total = fmaf(l, factor, total);
    af_values<DB, 1>(a, run, row, lay, tile, s, r, g, [&](int) { return f32x4{0.f, 0.f, 0.f, 0.f}; },
                  [&](int i, const f32x4 x) { o[i] += af_scaled(x, factor); });
  }
  const float inv = af_inverse(a, row, total, top);
#pragma unroll
  for (int i = 0; i < DB; ++i) af_store(a, row, 16 * i + 4 * g, o[i], inv);
}

// A run of one tile and at most af_one_rows rows by a wave, the tile's first NB blocks of 16 keys: the others are behind
// every row's own place, so their weights are zeros, which change no sum.
template <int DB, int NB>
__device__ __forceinline__ void af_one_of(const AfArgs& a, const AfRun& run, const AfRow& row, const AfOne<DB>& lds, int r,
                                              int g) {
  constexpr int AHEAD = NB == 1 ? 7 : NB == 2 ? 3 : 2;  // (registers there are: a wave keeps no sums but a block's)
  const KvLayout lay(a.page_size, a.hd);
  const int tile = run.p_hi / ATT_TILE;
  f32x4 s[NB];
  const float top = af_scores<DB, AHEAD>(a, run, row, lay, tile, lds.q_s, min(r, af_one_rows(DB) - 1), r, g, s);
  const float inv = af_inverse(a, row, af_weights(row, tile, top, g, s), top);
  af_values<DB, AHEAD>(a, run, row, lay, tile, s, r, g, [&](int) { return f32x4{0.f, 0.f, 0.f, 0.f}; },
                       [&](int i, const f32x4 x) { af_store(a, row, 16 * i + 4 * g, f32x4{0.f, 0.f, 0.f, 0.f} + x, inv); });
}
template <int DB>
__device__ __forceinline__ void af_one(const AfArgs& a, const AfRun& run, AfOne<DB>& lds, int lane) {
  const int r = lane % 16, g = lane / 16, blocks = run.p_hi % ATT_TILE / 16 + 1;
  const AfRow row = af_row(a, run, r);
  af_queries<DB, af_one_rows(DB)>(a, run, lds.q_s, 0, 1, run.n_here * (a.n_heads / a.n_kv), lane);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (blocks == 1) return af_one_of<DB, 1>(a, run, row, lds, r, g);
  if (blocks == 2) return af_one_of<DB, 2>(a, run, row, lds, r, g);
  if constexpr (af_one_blocks(DB) > 2) af_one_of<DB, 4>(a, run, row, lds, r, g);
}

// The run at place `index` of a grid; false: none is.  Uniform.  (The blocks' first runs come first, a token's kv heads side
// by side: every die gets as many of them.)
__device__ __forceinline__ bool af_at(const AfArgs& a, int index, int lane, AfRun& run) {
  const int full = 16 / (a.n_heads / a.n_kv), blocks = (a.n_tokens + full - 1) / full, place = index / a.n_kv;
  return place < blocks * full && af_run(a, af_block(a, place % blocks, lane), index % a.n_kv, place / blocks, run);
}

// DB: head dims in blocks of 16, at least hd / 16 (hd is a multiple of 8).  ALONE: a wave alone takes what `af_kind` says.
template <int DB, bool ALONE>
__global__ __launch_bounds__(AF_WAVES* FG_WAVE) void attention_f32_kernel(const AfArgs a) {
  const int lane = threadIdx.x % FG_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FG_WAVE);
  AfRun run;
  if constexpr (!ALONE) {
    __shared__ AfShared<DB> lds;
    if (af_at(a, blockIdx.x, lane, run) && af_kind<DB>(a, run) != AF_ONE) af_together<DB>(a, run, lds, wave, lane);
  } else {
    __shared__ union {
      AfShared<DB> together;
      AfAlone<DB> alone[AF_WAVES];
    } lds;
    if (af_at(a, blockIdx.x, lane, run) && af_kind<DB>(a, run) == AF_TOGETHER) af_together<DB>(a, run, lds.together, wave, lane);
    // (the first eighth of the grid looks after the others' runs, not every eighth workgroup: those are all on one die)
    if (blockIdx.x < (gridDim.x + AF_WAVES - 1) / AF_WAVES && af_at(a, blockIdx.x * AF_WAVES + wave, lane, run) &&
        af_kind<DB>(a, run) == AF_ALONE)
      af_by_wave<DB>(a, run, lds.alone[wave], lane);
  }
}

// Runs of one tile and at most af_one_rows rows, a wave each.
template <int DB>
__global__ __launch_bounds__(4 * FG_WAVE) void attention_f32_one_kernel(const AfArgs a) {
  const int lane = threadIdx.x % FG_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FG_WAVE);
  __shared__ AfOne<DB> lds[4];
  AfRun run;
  if (af_at(a, blockIdx.x * 4 + wave, lane, run) && af_kind<DB>(a, run) == AF_ONE) af_one<DB>(a, run, lds[wave], lane);
}

extern "C" int fg_paged_attention_general_sink(
    const void* q, int q_stride, void* out, int out_stride, const void* k_pages,
    const void* v_pages, const int* block_table, int bt_stride, int n_seqs, const int* seq_of_token,
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
    // The kernel for runs of one tile where there may be many: among prompts, from 2048 (token, head)s in the first 16 places
    // of the sequences on (8 prompts of 37: 51 / 29 us without / with at 32 / 8 x 128, 50 / 36 at 16 / 4 x 256); with
    // decoded tokens alone from 4096 on (64 of 60 keys, 32/32 x 128: 34 / 40; 300 of 9: 130 / 96; 200 of 100, which are none
    // of them: 165 / 174).  Above head size 256, where a wave's run is long beside a workgroup's, among short sequences
    // alone (8 / 8 x 512, 64 prompts of 5: 145 / 36, 300 of 9: 172 / 66; with 10 prompts of 100 beside 30 of 700: 362 / 402).
    const bool decoded = n_tokens <= n_seqs, large = hd > 256;
    const int ones = min((long long)n_tokens, 16LL * n_seqs) * n_heads >= (decoded && !large ? 4096 : 2048) &&
                     (!large || n_tokens <= 16LL * n_seqs);
    const AfArgs a{(const float*)q, q_stride, (float*)out, out_stride, (const float*)k_pages, (const float*)v_pages, block_table,
                   bt_stride, seq_of_token, positions, n_tokens, n_heads, n_kv, hd, page_size, scale, window, sinks, dist,
                   (int)min((long long)min(n_seqs, n_tokens) * n_kv, 2147483647LL), ones};
    const bool alone = group <= AF_ALONE_ROWS && a.few_runs >= (hd <= 64 ? af_alone_from(4, 1) : af_alone_from(8, 1));
#define ATTENTION_F32(DB)                                                                                   \
  do {                                                                                                      \
    if (a.ones) attention_f32_one_kernel<DB><<<(unsigned)((grid + 3) / 4), 4 * FG_WAVE, 0, stream>>>(a);    \
    if (alone) attention_f32_kernel<DB, true><<<(unsigned)grid, AF_WAVES * FG_WAVE, 0, stream>>>(a);        \
    else attention_f32_kernel<DB, false><<<(unsigned)grid, AF_WAVES * FG_WAVE, 0, stream>>>(a);             \
  } while (0)
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
