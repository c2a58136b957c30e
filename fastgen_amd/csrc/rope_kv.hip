// Rotary position encoding of q and k and the write of k, v into the paged
// cache, in one launch (the reference issues four: fastgen/forward.py:449-460
// with kernels/rope.py and kernels/paged_memcpy.py).
//
// Rotation (kernels/rope.py:56-89): pair (x[2i], x[2i+1]) of a head, angle =
// float(pos) * freqs[i] in fp32, precise sin/cos,
//   x[2i] = a cos - b sin,  x[2i+1] = b cos + a sin,
// rounded once at the store.  Pairs beyond rotary_dim are left as they are.
//
// Cache layout, per cache layer: K pages [n_pages, KV, P*hd], V pages
// [n_pages, KV, hd*P], the elements inside a page ordered as kv_layout.h
// says (16-byte chunks placed for the matrix-core kernels; V transposed).  A
// token's place is slot = page*P + offset; a negative slot means "write
// nothing".
#include "common.h"
#include "kv_layout.h"

#define ROPE_THREADS 256

// cos and sin of float(pos) * freqs[i] for every token of the step, computed
// once and shared by all layers: table[(t * n_freqs + i) * 2 + {0, 1}].
__global__ __launch_bounds__(ROPE_THREADS) void rope_table_kernel(
    const int* __restrict__ positions, const float* __restrict__ freqs, float* __restrict__ table,
    int n_tokens, int n_freqs) {
  const int e = blockIdx.x * ROPE_THREADS + threadIdx.x;
  if (e >= n_tokens * n_freqs) return;
  const float ang = (float)positions[e / n_freqs] * freqs[e % n_freqs];
  table[2 * e] = cosf(ang);
  table[2 * e + 1] = sinf(ang);
}

extern "C" int fg_rope_table(const int* positions, const float* freqs, float* table, int n_tokens,
                             int n_freqs, hipStream_t stream) {
  if (n_tokens <= 0 || n_freqs <= 0) return FG_OK;
  const long long n = (long long)n_tokens * n_freqs;
  if (n > 2147483647LL) return FG_ERR_ARG;
  rope_table_kernel<<<(unsigned)((n + ROPE_THREADS - 1) / ROPE_THREADS), ROPE_THREADS, 0, stream>>>(
      positions, freqs, table, n_tokens, n_freqs);
  return fg_launch_status();
}

template <class T>
__global__ __launch_bounds__(ROPE_THREADS) void rope_kv_write_kernel(
    T* __restrict__ qkv, int row_stride, const int* __restrict__ positions,
    const float* __restrict__ freqs, const float* __restrict__ table, const int* __restrict__ slots,
    T* __restrict__ k_pages,
    T* __restrict__ v_pages, int n_heads, int n_kv, int hd, int rotary_dim, int page_size,
    int write_kv, int v_col) {
  const int t = blockIdx.x;
  T* row = qkv + (size_t)t * row_stride;
  const float pos = (float)positions[t];
  const int half = hd / 2;
  const int slot = write_kv ? slots[t] : -1;
  const int page = slot >= 0 ? slot / page_size : 0;
  const int off = slot >= 0 ? slot % page_size : 0;
  const KvLayout lay(page_size, hd);
  const size_t head_elems = (size_t)page_size * hd;

  // q heads then k heads: (n_heads + n_kv) * hd/2 pairs
  const int n_rot_heads = n_heads + (write_kv ? n_kv : 0);
  const int n_pairs = n_rot_heads * half;
  for (int p = threadIdx.x; p < n_pairs; p += ROPE_THREADS) {
    const int head = p / half, i = p % half;
    T* x = row + (size_t)head * hd + 2 * i;
    float a = to_f<T>(x[0]), b = to_f<T>(x[1]);
    if (2 * i < rotary_dim) {
      float s, c;
      if (table) {
        c = table[((size_t)t * (rotary_dim / 2) + i) * 2];
        s = table[((size_t)t * (rotary_dim / 2) + i) * 2 + 1];
      } else {
        const float ang = pos * freqs[i];
        s = sinf(ang);
        c = cosf(ang);
      }
      const float ra = a * c - b * s;
      const float rb = b * c + a * s;
      a = ra;
      b = rb;
    }
    if (head < n_heads) {
      x[0] = from_f<T>(a);
      x[1] = from_f<T>(b);
    } else if (slot >= 0) {
      const int kvh = head - n_heads;
      T* dst = k_pages + ((size_t)page * n_kv + kvh) * head_elems + lay.k_off(off, 2 * i);
      dst[0] = from_f<T>(a);
      dst[1] = from_f<T>(b);
    }
  }
  if (slot >= 0) {
    const T* v = row + v_col;
    for (int e = threadIdx.x; e < n_kv * hd; e += ROPE_THREADS) {
      const int kvh = e / hd, d = e % hd;
      v_pages[((size_t)page * n_kv + kvh) * head_elems + lay.v_off(off, d)] = v[e];
    }
  }
}

// The same with eight consecutive elements (four pairs) a thread; for
// hd % 8 == 0, rotary_dim % 8 == 0 and rows 16-byte aligned.
template <class T>
__global__ __launch_bounds__(ROPE_THREADS) void rope_kv_write_vec_kernel(
    T* __restrict__ qkv, int row_stride, const int* __restrict__ positions,
    const float* __restrict__ freqs, const float* __restrict__ table, const int* __restrict__ slots,
    T* __restrict__ k_pages,
    T* __restrict__ v_pages, int n_heads, int n_kv, int hd, int rotary_dim, int page_size,
    int write_kv, int v_col) {
  const int t = blockIdx.x;
  T* row = qkv + (size_t)t * row_stride;
  const float pos = (float)positions[t];
  const int slot = write_kv ? slots[t] : -1;
  const int page = slot >= 0 ? slot / page_size : 0;
  const int off = slot >= 0 ? slot % page_size : 0;
  const KvLayout lay(page_size, hd);
  const size_t head_elems = (size_t)page_size * hd;
  const int cph = hd / 8;  // chunks per head
  const int n_rot = (n_heads + (write_kv ? n_kv : 0)) * cph;
  for (int w = threadIdx.x; w < n_rot; w += ROPE_THREADS) {
    {
      const int head = w / cph, c = w % cph;
      if (head >= n_heads && slot < 0) continue;
      T* x = row + (size_t)head * hd + 8 * c;
      float v[8];
      load8<T>(x, v);
      if (8 * c < rotary_dim) {
        float cs4[8];  // cos, sin of the chunk's four pairs
        if (table) {
          load8<float>(table + ((size_t)t * (rotary_dim / 2) + 4 * c) * 2, cs4);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float ang = pos * freqs[4 * c + j];
            cs4[2 * j] = cosf(ang);
            cs4[2 * j + 1] = sinf(ang);
          }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float cs = cs4[2 * j], sn = cs4[2 * j + 1];
          const float a = v[2 * j], b = v[2 * j + 1];
          v[2 * j] = a * cs - b * sn;
          v[2 * j + 1] = b * cs + a * sn;
        }
      }
      if (head < n_heads)
        store8<T>(x, v);
      else
        store8<T>(k_pages + ((size_t)page * n_kv + (head - n_heads)) * head_elems + lay.k_off(off, 8 * c), v);
    }
  }
  if (slot >= 0) {
    // v: one element a thread, consecutive threads consecutive head dims: in the transposed page
    // these lie 16 bytes apart, so a wave's store stays within a few cache lines
    const T* v = row + v_col;
    for (int e = threadIdx.x; e < n_kv * hd; e += ROPE_THREADS) {
      const int kvh = e / hd, d = e % hd;
      v_pages[((size_t)page * n_kv + kvh) * head_elems + lay.v_off(off, d)] = v[e];
    }
  }
}

// qkv: [n_tokens, row_stride] with q heads, then k heads, then v heads in a
// row.  With write_kv == 0 only q is rotated (a mixer that reads another
// layer's cache).
// `table` (from fg_rope_table, for the same positions) replaces the sin/cos
// of `freqs` when given.  v_col: the column of a row at which the values begin:
// (n_heads + n_kv) * hd where they have a projection of their own, n_heads * hd
// where a token's value is its key before the rotation (the k columns of the row
// are never written: the rotated keys go to the pages only).
extern "C" int fg_rope_kv_write(void* qkv, int row_stride, const int* positions,
                                const float* freqs, const float* table, const int* slots, void* k_pages,
                                void* v_pages, int n_tokens, int n_heads, int n_kv, int hd,
                                int rotary_dim, int page_size, int write_kv, int v_col, int dtype,
                                hipStream_t stream) {
  if (n_tokens <= 0) return FG_OK;
  if (hd <= 0 || hd % 2 || rotary_dim < 0 || rotary_dim > hd || rotary_dim % 2 ||
      page_size <= 0 || n_heads <= 0 || n_kv < 0)
    return FG_ERR_ARG;
  if (write_kv && (hd % 8 || page_size % 8)) return FG_ERR_ARG;  // the page layout is in chunks of 8
  if (row_stride < (n_heads + (write_kv ? n_kv : 0)) * hd) return FG_ERR_ARG;
  if (write_kv && (v_col < n_heads * hd || v_col % 8 || row_stride < v_col + n_kv * hd)) return FG_ERR_ARG;
  const bool vec = hd % 8 == 0 && rotary_dim % 8 == 0 && row_stride % 8 == 0;
#define LAUNCH(T, KERNEL)                                                                         \
  KERNEL<T><<<n_tokens, ROPE_THREADS, 0, stream>>>((T*)qkv, row_stride, positions, freqs, table,  \
                                                   slots, (T*)k_pages, (T*)v_pages, n_heads, n_kv, \
                                                   hd, rotary_dim, page_size, write_kv, v_col)
  if (dtype == FG_F32) {
    if (vec) LAUNCH(float, rope_kv_write_vec_kernel); else LAUNCH(float, rope_kv_write_kernel);
  } else if (dtype == FG_BF16) {
    if (vec) LAUNCH(bf16_t, rope_kv_write_vec_kernel); else LAUNCH(bf16_t, rope_kv_write_kernel);
  } else {
    return FG_ERR_ARG;
  }
#undef LAUNCH
  return fg_launch_status();
}

// The same from a product's fp32 partial sums [n_parts, n_tokens, width]: they are added in order, rotated and rounded once; the
// queries go to q_out [n_tokens, n_heads * hd], keys and values into their pages.  With this behind it the q/k/v product of a
// decoding batch may cut k over workgroups, which it needs to fill the chip (6,144 outputs are 48 tiles of 128).
// Bound by latency: a thread's chunk of 8 columns, U parts in flight, and as many workgroups as 128 threads make of the columns, so that
// a few tokens are a few hundred waves.  64 tokens of 6,144 x 4,096: product and this kernel 18.6 us, the library's product with the
// kernel above 23.5.  value_from_key: there are no v columns, the values are the keys before the rotation.
#define ROPE_PARTS_THREADS 128
template <int U>
__global__ __launch_bounds__(ROPE_PARTS_THREADS) void rope_kv_parts_kernel(
    const float* __restrict__ parts, size_t part_elems, int n_parts, bf16_t* __restrict__ q_out, const float* __restrict__ table,
    const int* __restrict__ slots, bf16_t* __restrict__ k_pages, bf16_t* __restrict__ v_pages, int n_heads, int n_kv, int hd,
    int rotary_dim, int page_size, int value_from_key) {
  const int t = blockIdx.x;
  const int cph = hd / 8;  // chunks per head
  const int heads = n_heads + (value_from_key ? n_kv : 2 * n_kv);
  const int w = blockIdx.y * ROPE_PARTS_THREADS + threadIdx.x;
  if (w >= heads * cph) return;
  const int head = w / cph, c = w % cph;
  const int slot = slots[t];
  if (head >= n_heads && slot < 0) return;
  const float* src = parts + (size_t)t * heads * hd + 8 * w;
  float v[8] = {};
  for (int s = 0; s < n_parts; s += U) {
    float p[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u) load8<float>(src + (s + u) * part_elems, p[u]);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] += p[u][j];
  }
  const KvLayout lay(page_size, hd);
  const size_t head_elems = (size_t)page_size * hd;
  const int page = slot >= 0 ? slot / page_size : 0, off = slot >= 0 ? slot % page_size : 0;
  const int kvh = head < n_heads ? 0 : (head - n_heads) % n_kv;
  const size_t place = ((size_t)page * n_kv + kvh) * head_elems;
  const bool is_v = head >= n_heads + n_kv;
  if (is_v || (value_from_key && head >= n_heads)) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v_pages[place + lay.v_off(off, 8 * c + j)] = from_f<bf16_t>(v[j]);
  }
  if (is_v) return;
  if (8 * c < rotary_dim) {
    float cs4[8];  // cos, sin of the chunk's four pairs
    load8<float>(table + ((size_t)t * (rotary_dim / 2) + 4 * c) * 2, cs4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float cs = cs4[2 * j], sn = cs4[2 * j + 1];
      const float a = v[2 * j], b = v[2 * j + 1];
      v[2 * j] = a * cs - b * sn;
      v[2 * j + 1] = b * cs + a * sn;
    }
  }
  store8<bf16_t>(head < n_heads ? q_out + (size_t)t * n_heads * hd + 8 * w : k_pages + place + lay.k_off(off, 8 * c), v);
}

extern "C" int fg_rope_kv_parts(const float* parts, int n_parts, void* q_out, const float* table, const int* slots, void* k_pages,
                                void* v_pages, int n_tokens, int n_heads, int n_kv, int hd, int rotary_dim, int page_size,
                                int value_from_key, hipStream_t stream) {
  if (n_tokens <= 0) return FG_OK;
  if (n_parts <= 0 || hd <= 0 || hd % 8 || rotary_dim < 0 || rotary_dim > hd || rotary_dim % 8 || page_size <= 0 || page_size % 8 ||
      n_heads <= 0 || n_kv <= 0 || (rotary_dim && !table))
    return FG_ERR_ARG;
  const long long chunks = (long long)(n_heads + (value_from_key ? 1 : 2) * n_kv) * (hd / 8);
  const long long groups = (chunks + ROPE_PARTS_THREADS - 1) / ROPE_PARTS_THREADS;
  if (groups > 65535) return FG_ERR_ARG;
  const dim3 grid(n_tokens, (unsigned)groups);
#define LAUNCH(U)                                                                                                          \
  rope_kv_parts_kernel<U><<<grid, ROPE_PARTS_THREADS, 0, stream>>>(parts, (size_t)n_tokens * chunks * 8, n_parts,          \
      (bf16_t*)q_out, table, slots, (bf16_t*)k_pages, (bf16_t*)v_pages, n_heads, n_kv, hd, rotary_dim, page_size, value_from_key)
  if (n_parts % 4 == 0) LAUNCH(4);  // (the plan of the product before gives 2 to 4 parts)
  else if (n_parts % 2 == 0) LAUNCH(2);
  else LAUNCH(1);
#undef LAUNCH
  return fg_launch_status();
}
