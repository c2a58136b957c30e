// y = x W^T with W stored [out, in] row-major (fastgen/forward.py:433-440,
// 470, 488-496, 513: F.linear): the engine's own matrix products without a
// mode of reduced precision.
//
// float32 (the true 32-bit path) runs on v_mfma_f32_16x16x32_bf16, sixteen
// times the rate of v_mfma_f32_16x16x4_f32: every operand is the exact sum of
// three bf16 parts of 8 bits each (h = bf16(v), m = bf16(v - h), l = v - h - m;
// m and l scaled up, so that small operands keep all bits too), and a product of
// two is six instructions: h h, then h m + m h, then h l + l h + m m (Henry, Tang
// and Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for
// higher-precision computations", ARITH 2019, name the split).  m is up to
// 2^-8 of an operand's leading bit and l up to 2^-17, so the products left out
// (m l, l m; l l) are at most 2^-24 of the whole, half a unit of its last place,
// and of either sign.  Each of the three kinds is summed over the 32 k of an
// instruction from zero and added to the segment's sum by the vector units,
// rounded to nearest (the matrix core cuts off where it adds to its
// accumulator): 4 steps are a segment's sum, 8 segments a group's, the groups'
// sums the total, each ascending.  An output's order is fixed by K alone,
// whichever kernel takes the product, so a row's result does not depend on how
// many other rows the call holds.
//
// Error relative to the product in 64 bits (2-norms, units of 1e-7), in brackets
// that of the fp32 instructions with chains of 32 k; K = 128 / 1024 / 3072 / 14336:
//   random signs           0.57 / 0.79 / 0.87 / 1.08  (1.10 / 1.24 / 1.29 / 1.43)
//   magnitudes of those    0.43 / 0.52 / 0.43 / 0.62  (0.58 / 0.54 / 0.43 / 0.63)
//   uniform in [0, 1)      0.43 / 0.49 / 0.43 / 0.57  (0.57 / 0.50 / 0.44 / 0.57)
//   constant rows          0.25 / 0.64 / 0.47 / 1.07  (2.28 / 2.52 / 2.40 / 2.85)
//   e^N(0,2), one sign     0.91 / 1.67 / 0.92 / 0.90  (0.70 / 1.52 / 0.69 / 0.70)
//   the same, both signs   0.58 / 0.78 / 0.84 / 1.24  (0.68 / 0.85 / 1.11 / 1.21)
// The fifth line is where it is not the better one: inside an instruction eight
// products are cut off below the largest of them.  Magnitudes down to the
// smallest normal number change nothing; of an operand below it up to 3/4 of its
// last place is left out.  Infinities (and what rounds to one in
// bf16) have no such parts, and a part's product may be one where the whole one
// is not: an output that comes out as no number is computed again, one fp32 FMA
// a product (gf_again).
//
// Operands of bf16 with fp32 accumulation take the FMA kernel below, so that
// any shape has a product when the tuned kernels refuse it.
#include <type_traits>

#include "common.h"
#include "kv_layout.h"

#define GT_M 64
#define GT_N 64
#define GT_K 16
#define GT_THREADS 256

template <class TX, class TW, class TY>
__global__ __launch_bounds__(GT_THREADS) void gemm_nt_kernel(
    const TX* __restrict__ x, const TW* __restrict__ w, TY* __restrict__ y, int M, int N,
    int K, int ldx, int ldw, int ldy) {
  // tiles stored k-major so that the inner product reads consecutive floats
  __shared__ float xs[GT_K][GT_M + 4];
  __shared__ float ws[GT_K][GT_N + 4];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * GT_M, n0 = blockIdx.x * GT_N;
  const int tm = (tid / 16) * 4, tn = (tid % 16) * 4;
  float acc[4][4], mid[4][4];  // total; sum of up to 16 tiles' partial sums
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = mid[i][j] = 0.f;
  int tiles_in_mid = 0;

  // each thread loads 4 elements of each tile: row = tid / 4, k = (tid % 4) * 4 ..
  const int lr = tid / 4, lk = (tid % 4) * 4;
  for (int k0 = 0; k0 < K; k0 += GT_K) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = k0 + lk + e;
      const int m = m0 + lr, n = n0 + lr;
      xs[lk + e][lr] = (m < M && k < K) ? to_f<TX>(x[(size_t)m * ldx + k]) : 0.f;
      ws[lk + e][lr] = (n < N && k < K) ? to_f<TW>(w[(size_t)n * ldw + k]) : 0.f;
    }
    __syncthreads();
    float part[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) part[i][j] = 0.f;
#pragma unroll
    for (int k = 0; k < GT_K; ++k) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = xs[k][tm + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = ws[k][tn + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) part[i][j] = fmaf(a[i], b[j], part[i][j]);
    }
    const bool fold = ++tiles_in_mid == 16;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        mid[i][j] += part[i][j];
        if (fold) {
          acc[i][j] += mid[i][j];
          mid[i][j] = 0.f;
        }
      }
    if (fold) tiles_in_mid = 0;
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] += mid[i][j];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + tm + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tn + j;
      if (n < N) y[(size_t)m * ldy + n] = from_f<TY>(acc[i][j]);
    }
  }
}

// bf16 operands; y is `out_dtype` (fp32 output serves the LM head).
extern "C" int fg_gemm_nt(const void* x, const void* w, void* y, int M, int N, int K, int ldx,
                          int ldw, int ldy, int in_dtype, int out_dtype, hipStream_t stream) {
  if (M <= 0 || N <= 0) return FG_OK;
  if (K <= 0 || ldx < K || ldw < K || ldy < N) return FG_ERR_ARG;
  dim3 grid((N + GT_N - 1) / GT_N, (M + GT_M - 1) / GT_M);
  if (grid.y > 65535) return FG_ERR_ARG;
#define LAUNCH(TX, TY)                                                                      \
  gemm_nt_kernel<TX, TX, TY><<<grid, GT_THREADS, 0, stream>>>((const TX*)x, (const TX*)w,   \
                                                              (TY*)y, M, N, K, ldx, ldw, ldy)
  if (in_dtype == FG_BF16 && out_dtype == FG_BF16) LAUNCH(bf16_t, bf16_t);
  else if (in_dtype == FG_BF16 && out_dtype == FG_F32) LAUNCH(bf16_t, float);
  else return FG_ERR_ARG;
#undef LAUNCH
  return fg_launch_status();
}

// ------------------------------------------------------------------ float32
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define GF_SEG 128    // k of a segment: 4 steps
#define GF_GROUP 1024 // k of a group: 8 segments
#define GF_STEP 32    // k of a matrix instruction
#define GF_STEP_UP 256.f         // a part's scale against the part before it
#define GF_STEP_DOWN 0.00390625f

// Four elements of a row from k on, zeros behind K.  VEC: rows are 16-byte aligned and K is a multiple of 4.
template <bool VEC>
__device__ __forceinline__ f32x4 gf_load4(const float* __restrict__ row, int k, int K) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if constexpr (VEC) {
    if (k < K) v = *(const f32x4*)(row + k);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (k + e < K) v[e] = row[k + e];
  }
  return v;
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// The three parts of four numbers: v = part 0 + 2^-8 part 1 + 2^-16 part 2, exactly, whatever v is (down to the smallest
// number: the parts that are of 2^-9 and 2^-17 of it are kept 2^8 and 2^16 times as large, so that 8 bits with the
// smallest exponent of bf16 hold all of them).  The first two are rounded to nearest, so that what follows has either
// sign; the third is what is left, at most 7 bits.
__device__ __forceinline__ void gf_parts4(const f32x4 v, bf16x4* p0, bf16x4* p1, bf16x4* p2) {
  const unsigned top = 0xffff0000u;
  unsigned p[3][2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const f32x2 pair = {v[2 * e], v[2 * e + 1]};
    const unsigned h = __builtin_bit_cast(unsigned, __builtin_convertvector(pair, bf16x2));
    const float r0 = GF_STEP_UP * (pair[0] - __uint_as_float(h << 16)), r1 = GF_STEP_UP * (pair[1] - __uint_as_float(h & top));
    const unsigned m = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{r0, r1}), bf16x2));
    const float l0 = GF_STEP_UP * (r0 - __uint_as_float(m << 16)), l1 = GF_STEP_UP * (r1 - __uint_as_float(m & top));
    p[0][e] = h;
    p[1][e] = m;  // (a permutation of bytes takes the upper halves of two words)
    p[2][e] = __builtin_amdgcn_perm(__float_as_uint(l1), __float_as_uint(l0), 0x07060302u);
  }
  *p0 = __builtin_bit_cast(bf16x4, p[0]);
  *p1 = __builtin_bit_cast(bf16x4, p[1]);
  *p2 = __builtin_bit_cast(bf16x4, p[2]);
}

// An operand of the matrix instruction: lane 16 g + r holds of row r the k = 4 g .. 4 g + 3 and 16 + 4 g .. 19 + 4 g of
// a step (the instruction sums over k, so any order will do that is the same for W and x; a load of this one takes
// 64 bytes in a row).
struct GfParts {
  bf16x8 p[3];
};

__device__ __forceinline__ GfParts gf_parts(const f32x4 lo, const f32x4 hi) {
  bf16x4 a[3], b[3];
  gf_parts4(lo, &a[0], &a[1], &a[2]);
  gf_parts4(hi, &b[0], &b[1], &b[2]);
  GfParts s;
#pragma unroll
  for (int i = 0; i < 3; ++i) s.p[i] = __builtin_shufflevector(a[i], b[i], 0, 1, 2, 3, 4, 5, 6, 7);
  return s;
}

template <bool VEC>
__device__ __forceinline__ f32x4 gf_whole4(const float* p) {
  if constexpr (VEC) return *(const f32x4*)p;
  else return f32x4{p[0], p[1], p[2], p[3]};
}

#define GF_MFMA(A, B, C) __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B, C, 0, 0, 0)

// One step of one tile: the products of the parts by size, each kind from zero.  A: 16 rows of W, B: 16 rows of x; lane
// 16 g + r ends with outputs 4 g .. 4 g + 3 of x row r.
struct GfTerms {
  f32x4 whole, middle, small;
};

__device__ __forceinline__ GfTerms gf_step(const GfParts& w, const bf16x8 x0, const bf16x8 x1, const bf16x8 x2) {
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  GfTerms t;
  t.small = GF_MFMA(w.p[2], x0, zero);
  t.whole = GF_MFMA(w.p[0], x0, zero);
  t.middle = GF_MFMA(w.p[1], x0, zero);
  t.small = GF_MFMA(w.p[0], x2, t.small);
  t.middle = GF_MFMA(w.p[0], x1, t.middle);
  t.small = GF_MFMA(w.p[1], x1, t.small);
  return t;
}

// A step's products into its segment's sum, rounded to nearest (the matrix core cuts off where it adds).
__device__ __forceinline__ void gf_fold(f32x4& sum, const GfTerms& t) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    sum[i] += fmaf(fmaf(t.small[i], GF_STEP_DOWN, t.middle[i]), GF_STEP_DOWN, t.whole[i]);
  asm volatile("" : "+v"(sum));  // here, or the compiler keeps every step's terms up to the segment's end, in scratch memory
}

// An output whose sum is no number: the operands may hold an infinity, or a part's product have rounded up to one where
// the whole product is just below the largest number.
__device__ __forceinline__ bool gf_lost(float sum) { return !(fabsf(sum) <= 3.402823466e38f); }
__device__ __noinline__ float gf_again(const float* x, const float* w, int K) {
  float sum = 0.f;
  for (int k = 0; k < K && sum == sum; ++k) sum = fmaf(w[k], x[k], sum);
  return sum;
}

__device__ __forceinline__ f32x4 gf_read4(const float* p, int n, int N, bool wide) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (wide && n + 4 <= N) {
    v = *(const f32x4*)(p + n);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) v[e] = p[n + e];
  }
  return v;
}

__device__ __forceinline__ void gf_store4(float* __restrict__ y, int n, int N, bool wide, const f32x4 v) {
  if (wide && n + 4 <= N) {
    *(f32x4*)(y + n) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) y[n + e] = v[e];
  }
}

// What fg_silu_mul and fg_gelu_mul (rows.hip) give in fp32: the epilogue codes of the bf16 products.
#define GF_SILU 1
#define GF_GELU 4
__device__ __forceinline__ float gf_gated(float gate, float up, int act) {
  if (act == GF_GELU) return 0.5f * gate * (1.f + tanhf(0.7978845608028654f * (gate + 0.044715f * gate * gate * gate))) * up;
  return gate / (1.f + expf(-gate)) * up;
}

// 16 rows (decode, and outputs too few for tiles): bound by reading W.  A workgroup owns 16 outputs of 16 rows; a round is
// one group, a wave takes one of its segments, so 64 KB of W (every wave's next segment) are in flight a workgroup while
// the current ones are multiplied; the segments' sums meet in LDS and are added in order by one thread an output.
// N x K 3072 x 3072 / 16384 x 3072 / 3072 x 8192: 13 / 45 / 31 us at 4 rows (4.5 TB/s of W at the largest), 18 / 60 / 43 at
// 16 (in tiles 25 / 54 / 32); with the fp32 instructions 14 / 47 / 31 and 18 / 60 / 40.
// Two workgroups a compute unit (at most 128 registers): 441 workgroups of two groups 13 us, 15.7 with one.
// With `part` a workgroup takes one group of k (blockIdx.z) and stores its sum, as the kernel of tiles below: what few outputs need to
// have a workgroup for every compute unit.  With `act` the outputs are a gate and an up matrix interleaved in groups of eight, which
// are these 16, and silu(gate) * up is stored (the tanh form of GELU).
// A wave cuts its segment of x into parts once: with FEW (up to 8 rows), each number in one lane, through LDS into
// the operands' order; above, every lane the operand it needs.
template <bool FEW, bool VEC>
__global__ __launch_bounds__(512, 4) void gemm_f32_few_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                           float* __restrict__ y, float* __restrict__ part, int M, int N,
                                                           int K, int ldx, int ldw, int ldy, int act) {
  __shared__ f32x4 sums[2][8][FG_WAVE];
  __shared__ bf16x4 parts[FEW ? 8 : 1][4][3][4][8][2];  // [wave][step][part][g][row][half]
  const int tid = threadIdx.x, lane = tid % FG_WAVE, wave = tid / FG_WAVE;
  const int r = lane % 16, g = lane / 16, n0 = blockIdx.x * 16;
  x += (size_t)blockIdx.y * 16 * ldx;
  y += (size_t)blockIdx.y * 16 * ldy;
  if (part) part += ((size_t)blockIdx.z * M + blockIdx.y * 16) * N;
  M = min(M - (int)blockIdx.y * 16, 16);
  // rows behind the last repeat it: their outputs are not stored
  const float* wrow = w + (size_t)min(n0 + r, N - 1) * ldw;
  const float* xrow = x + (size_t)min(r, M - 1) * ldx;
  const int s_begin = part ? 8 * blockIdx.z : 0, n_seg = min((K + GF_SEG - 1) / GF_SEG, part ? s_begin + 8 : 0x7fffffff);
  f32x4 wv[8], next[8], xv[8];
  if (s_begin + wave < n_seg) {
#pragma unroll
    for (int i = 0; i < 8; ++i) next[i] = gf_load4<VEC>(wrow, (s_begin + wave) * GF_SEG + i * 16 + g * 4, K);
  }
  float total = 0.f;
  for (int s0 = s_begin, buf = 0; s0 < n_seg; s0 += 8, buf ^= 1) {
    const int seg = s0 + wave;
    if (seg < n_seg) {
      if constexpr (FEW) {
        const int c = lane % 32;  // four k of a row; the rows two apart
#pragma unroll
        for (int i = 0; i < 4; ++i)
          xv[i] = gf_load4<VEC>(x + (size_t)min(lane / 32 + 2 * i, M - 1) * ldx, seg * GF_SEG + c * 4, K);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) xv[i] = gf_load4<VEC>(xrow, seg * GF_SEG + i * 16 + g * 4, K);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) wv[i] = next[i];
      if (seg + 8 < n_seg) {
#pragma unroll
        for (int i = 0; i < 8; ++i) next[i] = gf_load4<VEC>(wrow, (seg + 8) * GF_SEG + i * 16 + g * 4, K);
      }
      if constexpr (FEW) {
        const int c = lane % 32;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = lane / 32 + 2 * i;
          bf16x4(*to)[4][8][2] = parts[wave][c / 8];
          if (2 * i < M) gf_parts4(xv[i], &to[0][c % 4][row][c / 4 % 2], &to[1][c % 4][row][c / 4 % 2],
                                   &to[2][c % 4][row][c / 4 % 2]);
        }
        // a wave reads only what it has written itself, but a lane what others have: behind their stores
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_wave_barrier();
      }
      f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        GfParts xp;
        if constexpr (FEW) {
#pragma unroll
          for (int p = 0; p < 3; ++p) xp.p[p] = *(const bf16x8*)&parts[wave][i][p][g][min(r, M - 1)][0];
        } else {
          xp = gf_parts(xv[2 * i], xv[2 * i + 1]);
        }
        gf_fold(sum, gf_step(gf_parts(wv[2 * i], wv[2 * i + 1]), xp.p[0], xp.p[1], xp.p[2]));
      }
      sums[buf][wave][lane] = sum;
    }
    __syncthreads();  // (a round's sums are read before the round after next writes them: one barrier between)
    if (tid < 256) {
      float mid = 0.f;
      const int here = min(8, n_seg - s0);
      for (int i = 0; i < here; ++i) mid += ((const float*)sums[buf][i])[tid];
      total += mid;
    }
  }
  // element tid of a wave's sums: lane tid / 4 = 16 g + r, output 4 g + tid % 4 of row r
  const int m = (tid / 4) % 16, n = n0 + (tid / 64) * 4 + tid % 4;
  const bool mine = tid < 256 && m < M && n < N;
  if (part) {
    if (mine) part[(size_t)m * N + n] = total;
    return;
  }
  if (mine && gf_lost(total)) total = gf_again(x + (size_t)m * ldx, w + (size_t)n * ldw, K);
  if (!act) {
    if (mine) y[(size_t)m * ldy + n] = total;
    return;
  }
  // the outputs are eight gates and the ups of their channels (N % 16 == 0)
  float* ups = (float*)sums;  // (behind a round's sums at the earliest: what is read there is read before the barrier)
  __syncthreads();
  if (tid >= 128 && tid < 256) ups[tid - 128] = total;
  __syncthreads();
  if (tid < 128 && m < M) y[(size_t)m * ldy + n0 / 2 + (tid / 64) * 4 + tid % 4] = gf_gated(total, ups[tid], act);
}

// Rows cut beforehand: [ceil(n / 16)][K / 32][3][64][8], a block's three parts of a step in operand order (K a multiple of 32; rows that are
// not there are zeros).  A wave takes a step of 16 rows.
__global__ __launch_bounds__(256) void gemm_f32_cut_kernel(const float* __restrict__ rows, int ld, int n, int K, bf16x8* __restrict__ out) {
  const int lane = threadIdx.x % FG_WAVE, steps = K / GF_STEP, step = blockIdx.y * 4 + threadIdx.x / FG_WAVE;
  const int row = blockIdx.x * 16 + lane % 16;
  if (step >= steps) return;
  f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
  if (row < n) {
    const float* from = rows + (size_t)row * ld + step * GF_STEP + lane / 16 * 4;
    lo = *(const f32x4*)from;
    hi = *(const f32x4*)(from + 16);
  }
  const GfParts c = gf_parts(lo, hi);
  bf16x8* to = out + ((size_t)blockIdx.x * steps + step) * 192 + lane;
#pragma unroll
  for (int p = 0; p < 3; ++p) to[64 * p] = c.p[p];
}

// Many rows: bound by the matrix cores at the clock they can hold.  NW waves own 16 MB rows x 16 NB NW outputs, each
// all the rows and 16 NB outputs: a wave takes its rows of W from memory into registers itself and reads every x from LDS, where the
// workgroup has put its three parts in the operands' order, 32 k at a time in two buffers.
// Operands as they are: a wave cuts W into parts once, and the two waves of a SIMD do it on either side of their matrix instructions
// (`late`), so that one's vector work runs beside the other's products.
// CUT, operands cut beforehand (xp, wp; K a multiple of 128): two fifths of the vector work are gone, and what is left, the sums, fits between
// the matrix instructions, two behind each.  Half as many bytes of W again, so not for a few rows.
// AHEAD: steps of W and x in flight, in registers; their loads stand
// under no condition (with one the compiler copies what it has just loaded, that is, waits for it: 1.7 us a step
// instead of 0.6 where the products take 0.1).  A group's sum is kept in LDS, which leaves the registers to the loads.
// With `part` a workgroup takes one group of k and stores its sum there ([groups][M][N]); else it adds each group's to
// y.  A die's workgroups are an eighth of the tiles, those that read the same rows of W one after the other.
//
// N x K 16384 x 3072 / 5120 x 3072 / 3072 x 8192, us: 400 rows 283 / 105 / 160, cut 237 / 89 / 129 (459 / 167 / 256 with the fp32
// instructions), 2000 rows 1300 / 412 / 641, cut 1103 / 344 / 543: 1.1 PFLOP/s of bf16, against 1.4 that
// a product of bf16 operands reaches; with the sums on the matrix core itself, cut off there, 12 % less.
// FAR: rows so far apart that a tile spans 4 GB, with offsets of 64 bits (of 32, a load is one register of offset behind
// a uniform base).
template <int MB, int NB, int NW, int AHEAD, bool VEC, bool FAR, bool CUT>
__global__ __launch_bounds__(64 * NW, 2) void gemm_f32_tiled_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const bf16x8* __restrict__ xp, const bf16x8* __restrict__ wp,
    float* __restrict__ y, float* __restrict__ part, int M, int N, int K, int ldx, int ldw, int ldy, int row_tiles, int col_tiles, int units,
    int wide) {
  // pieces of x that a thread brings a step: four k of a row, or eight of a part
  constexpr int TM = 16 * MB, TN = 16 * NB * NW, XV = ((CUT ? MB * 192 : TM * 8) + 64 * NW - 1) / (64 * NW);
  static_assert(4 % AHEAD == 0, "a segment's steps use the sets of registers in turn");
  __shared__ bf16x8 xs[2][CUT ? XV * 64 * NW : MB * 192];  // [block][part][lane]
  __shared__ f32x4 mids[NW][MB * NB][FG_WAVE];
  const int tile = blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8;  // (workgroup i runs on die i % 8)
  if (tile >= units * row_tiles) return;
  const int unit = tile / row_tiles, m0 = tile % row_tiles * TM, group = unit / col_tiles;
  const int tid = threadIdx.x, lane = tid % FG_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / FG_WAVE);
  const int r = lane % 16, g = lane / 16, n0 = (unit % col_tiles) * TN + wave * 16 * NB;
  const bool late = wave >= 4;
  const int k_begin = part ? group * GF_GROUP : 0, k_end = part ? min(K, k_begin + GF_GROUP) : K;
  const int k_full = k_begin + (k_end - k_begin) / GF_SEG * GF_SEG;  // whole segments
  // a lane's place behind the wave's (the tile's) first row; rows behind the last repeat it: their outputs are not stored
  const float *wb = w + (size_t)min(n0, N - 1) * ldw, *xb = x + (size_t)m0 * ldx;
  using Offset = std::conditional_t<FAR, size_t, unsigned>;
  Offset wo[NB], xo[XV];  // in bytes
  const int steps = K / GF_STEP, piece = tid % 8, row = tid / 8;  // of x as it is: the rows 8 NW apart
  const char *wc = nullptr, *xc = nullptr;
  if constexpr (CUT) {
    const int last = (N + 15) / 16 - 1, first = min(n0 / 16, last);
    wc = (const char*)(wp + (size_t)first * steps * 192);
    xc = (const char*)(xp + (size_t)(m0 / 16) * steps * 192);
#pragma unroll
    for (int j = 0; j < NB; ++j) wo[j] = 16 * ((unsigned)min(j, last - first) * steps * 192 + lane);
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int c = tid + 64 * NW * i, block = min(c / 192, min(MB, (M - m0 + 15) / 16) - 1);
      xo[i] = 16 * ((unsigned)block * steps * 192 + c % 192);
    }
  } else {
#pragma unroll
    for (int j = 0; j < NB; ++j) wo[j] = 4 * ((Offset)min(16 * j + r, max(N - 1 - n0, 0)) * ldw + 4 * g);
#pragma unroll
    for (int i = 0; i < XV; ++i) xo[i] = 4 * ((Offset)min(row + 8 * NW * i, M - 1 - m0) * ldx + 4 * piece);
  }

  f32x4 raw[CUT ? 1 : AHEAD][NB][2], xv[CUT ? 1 : AHEAD][XV], sum[MB][NB];
  bf16x8 xcut[CUT ? AHEAD : 1][XV];
  GfParts wpart[CUT ? AHEAD : 1][NB];
  // a whole step; what would be loaded ahead behind the last whole segment is its last step again
  auto load_w = [&](int set, int k) {
    k = min(k, k_full - GF_STEP);
    if constexpr (CUT) {
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int p = 0; p < 3; ++p) wpart[set][j].p[p] = *(const bf16x8*)(wc + (size_t)(k / GF_STEP) * 3072 + wo[j] + 1024 * p);
    } else {
      const char* at = (const char*)(wb + k);
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        raw[set][j][0] = gf_whole4<VEC>((const float*)(at + wo[j]));
        raw[set][j][1] = gf_whole4<VEC>((const float*)(at + wo[j]) + 16);
      }
    }
  };
  auto load_x = [&](int set, int k) {
    k = min(k, k_full - GF_STEP);
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      if constexpr (CUT) xcut[set][i] = *(const bf16x8*)(xc + (size_t)(k / GF_STEP) * 3072 + xo[i]);
      else xv[set][i] = gf_whole4<VEC>((const float*)((const char*)(xb + k) + xo[i]));
    }
  };
  auto store_x = [&](int set, int buf) {
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      if constexpr (CUT) {
        xs[buf][tid + 64 * NW * i] = xcut[set][i];
      } else {
        const int at = row + 8 * NW * i;
        if (TM % (8 * NW) == 0 || at < TM) {
          bf16x8* to = xs[buf] + at / 16 * 192 + (piece % 4) * 16 + at % 16;
          const int half = piece / 4;
          gf_parts4(xv[set][i], (bf16x4*)to + half, (bf16x4*)(to + 64) + half, (bf16x4*)(to + 128) + half);
        }
      }
    }
  };
  auto cut_w = [&](int set) {
#pragma unroll
    for (int j = 0; j < NB; ++j) wpart[0][j] = gf_parts(raw[set][j][0], raw[set][j][1]);
  };
  auto multiply = [&](int buf, int set) {
    GfTerms terms[2][NB];  // a row of blocks is added up behind the next one's products
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      bf16x8 b[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) b[p] = xs[buf][(3 * i + p) * 64 + lane];
#pragma unroll
      for (int j = 0; j < NB; ++j) terms[i % 2][j] = gf_step(wpart[set][j], b[0], b[1], b[2]);
      if (i > 0) {
#pragma unroll
        for (int j = 0; j < NB; ++j) gf_fold(sum[i - 1][j], terms[(i - 1) % 2][j]);
        if constexpr (CUT && MB > 5) {  // (in smaller tiles the compiler's own order is as good)
#pragma unroll
          for (int z = 0; z < 6 * NB; ++z) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // a matrix instruction
            __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);  // two vector instructions
          }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) gf_fold(sum[MB - 1][j], terms[(MB - 1) % 2][j]);
  };
  // the end of the segment from k0 on
  auto close = [&](int k0) {
    const int next = k0 + GF_SEG;
    const bool first = k0 % GF_GROUP == 0, last = next % GF_GROUP == 0 || next >= k_end;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int m = m0 + 16 * i + r;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        f32x4 mid = first ? f32x4{0.f, 0.f, 0.f, 0.f} : mids[wave][i * NB + j][lane];
        mid += sum[i][j];
        sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!last) {
          mids[wave][i * NB + j][lane] = mid;
        } else if (m < M) {
          const int n = n0 + 16 * j + 4 * g;
          if (part) {
            gf_store4(part + ((size_t)group * M + m) * N, n, N, wide, mid);
          } else {
            float* out = y + (size_t)m * ldy;
            if (k0 >= GF_GROUP) mid = gf_read4(out, n, N, wide) + mid;
            if (next >= k_end) {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (gf_lost(mid[e]) && n + e < N) mid[e] = gf_again(x + (size_t)m * ldx, w + (size_t)(n + e) * ldw, K);
            }
            gf_store4(out, n, N, wide, mid);
          }
        }
      }
    }
  };
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (k_begin < k_full) {
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
      load_x(a, k_begin + a * GF_STEP);
      load_w(a, k_begin + a * GF_STEP);
    }
    store_x(0, 0);
    if (!CUT && late) cut_w(0);
    __syncthreads();
    for (int k0 = k_begin; k0 < k_full; k0 += GF_SEG) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = k0 + q * GF_STEP, buf = q % 2;
        load_x(q % AHEAD, k + AHEAD * GF_STEP);
        if constexpr (CUT) {
          store_x((q + 1) % AHEAD, buf ^ 1);
          multiply(buf, q % AHEAD);
          load_w(q % AHEAD, k + AHEAD * GF_STEP);
        } else {
          if (!late) cut_w(q % AHEAD);
          load_w(q % AHEAD, k + AHEAD * GF_STEP);
          multiply(buf, 0);
          if (late) cut_w((q + 1) % AHEAD);
          store_x((q + 1) % AHEAD, buf ^ 1);
        }
        __syncthreads();
      }
      close(k0);
    }
  }
  if constexpr (!CUT) {
    if (k_full < k_end) {  // less than a segment at the end of the rows
      for (int k = k_full; k < k_end; k += GF_STEP) {
#pragma unroll
        for (int i = 0; i < XV; ++i) xv[0][i] = gf_load4<VEC>(xb + xo[i] / 4 - 4 * piece, k + 4 * piece, k_end);
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          raw[0][j][0] = gf_load4<VEC>(wb + wo[j] / 4 - 4 * g, k + 4 * g, k_end);
          raw[0][j][1] = gf_load4<VEC>(wb + wo[j] / 4 - 4 * g, k + 16 + 4 * g, k_end);
        }
        store_x(0, 0);
        cut_w(0);
        __syncthreads();
        multiply(0, 0);
        __syncthreads();
      }
      close(k_full);
    }
  }
}

// What a product leaves where every group of k has a workgroup of its own: fp32 [groups][M][N], to be added in order.  An
// output that comes out as no number is computed again from the operands.
struct GfSums {
  const float *part, *x, *w;
  int M, N, K, ldx, ldw, groups;
};

// Outputs n[v] .. n[v] + 3 of row m.  U: groups whose sums are in flight together: behind a product of few rows the kernels below are a
// chain of memory's latencies (3,072 outputs of 8 groups, 4 rows, with the norm: 8 us four by four, 4 at once).
template <int NV, int U>
__device__ __forceinline__ void gf_totals(const GfSums& s, int m, const int (&n)[NV], bool wide, f32x4 (&total)[NV]) {
#pragma unroll
  for (int v = 0; v < NV; ++v) total[v] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int g0 = 0; g0 < s.groups; g0 += U) {
    f32x4 p[U][NV];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int v = 0; v < NV; ++v) p[u][v] = gf_read4(s.part + ((size_t)min(g0 + u, s.groups - 1) * s.M + m) * s.N, n[v], s.N, wide);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (g0 + u < s.groups) {  // uniform
#pragma unroll
        for (int v = 0; v < NV; ++v) total[v] += p[u][v];
      }
  }
#pragma unroll
  for (int v = 0; v < NV; ++v)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (gf_lost(total[v][e]) && n[v] + e < s.N) total[v][e] = gf_again(s.x + (size_t)m * s.ldx, s.w + (size_t)(n[v] + e) * s.ldw, s.K);
}

__global__ __launch_bounds__(256) void gemm_f32_sum_kernel(const GfSums s, float* __restrict__ y, int ldy, int wide) {
  const int m = blockIdx.y, n = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (n >= s.N) return;
  const int at[1] = {n};
  f32x4 total[1];
  gf_totals<1, 4>(s, m, at, wide, total);
  gf_store4(y + (size_t)m * ldy, n, s.N, wide, total[0]);
}

// The sums of a gate and an up matrix interleaved in groups of eight, and the activation: four channels a thread.
// (N % 16 == 0, y [M][N / 2].)
__global__ __launch_bounds__(256) void gemm_f32_sum_act_kernel(const GfSums s, float* __restrict__ y, int act) {
  const int m = blockIdx.y, c = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (c >= s.N / 2) return;
  const int n[2] = {c / 8 * 16 + c % 8, c / 8 * 16 + c % 8 + 8};  // gates, ups
  f32x4 total[2], v;
  gf_totals<2, 4>(s, m, n, true, total);
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = gf_gated(total[0][e], total[1][e], act);
  *(f32x4*)(y + (size_t)m * (s.N / 2) + c) = v;
}

// The sums, added to the residual stream, and the norm behind: fg_add_rmsnorm (rows.hip) on the product's rows, in its order and with
// its bits.  A workgroup a row, eight elements a thread and round, in registers.  N % 8 == 0, N <= 2048 NIT.
template <int NIT>
__global__ __launch_bounds__(256) void gemm_f32_sum_norm_kernel(const GfSums s, float* __restrict__ h, const float* __restrict__ weight,
                                                                float* __restrict__ out, float eps) {
  __shared__ float red[16];
  const int m = blockIdx.x;
  float* hrow = h + (size_t)m * s.N;
  f32x4 v[2 * NIT], wv[2 * NIT], total[2 * NIT];
  int n[2 * NIT];  // (a thread whose share lies behind the row reads its last elements and stores nothing)
#pragma unroll
  for (int i = 0; i < 2 * NIT; ++i) {
    n[i] = min((int)(threadIdx.x + i / 2 * 256) * 8, s.N - 8) + 4 * (i % 2);
    v[i] = *(const f32x4*)(hrow + n[i]);
    wv[i] = *(const f32x4*)(weight + n[i]);
  }
  gf_totals<2 * NIT, NIT <= 2 ? 8 : 4>(s, m, n, true, total);
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 2 * NIT; ++i) {
    v[i] += total[i];
    if ((int)(threadIdx.x + i / 2 * 256) * 8 < s.N) {
      *(f32x4*)(hrow + n[i]) = v[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) ss += v[i][e] * v[i][e];
    }
  }
  ss = block_sum(ss, red);
  const float rstd = rsqrtf(ss / (float)s.N + eps);
#pragma unroll
  for (int i = 0; i < 2 * NIT; ++i) {
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = v[i][e] * rstd * wv[i][e];
    if ((int)(threadIdx.x + i / 2 * 256) * 8 < s.N) *(f32x4*)(out + (size_t)m * s.N + n[i]) = o;
  }
}

// The sums of a q/k/v product, rotated, keys and values into their pages: fg_rope_kv_write (rope_kv.hip) on the product's rows, the
// same bits, the queries to q_out [M][n_heads * hd].  A chunk of 8 columns a thread.
__global__ __launch_bounds__(128) void gemm_f32_sum_rope_kernel(const GfSums s, float* __restrict__ q_out, const float* __restrict__ table,
                                                                const int* __restrict__ slots, float* __restrict__ k_pages,
                                                                float* __restrict__ v_pages, int n_heads, int n_kv, int hd,
                                                                int rotary_dim, int page_size, int value_from_key) {
  const int t = blockIdx.x, cph = hd / 8, c8 = blockIdx.y * 128 + threadIdx.x;
  if (c8 * 8 >= s.N) return;
  const int head = c8 / cph, c = c8 % cph, slot = slots[t];
  if (head >= n_heads && slot < 0) return;
  const int n[2] = {8 * c8, 8 * c8 + 4};
  f32x4 total[2];
  gf_totals<2, 4>(s, t, n, true, total);
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = total[j / 4][j % 4];
  const KvLayout lay(page_size, hd);
  const size_t head_elems = (size_t)page_size * hd;
  const int page = slot >= 0 ? slot / page_size : 0, off = slot >= 0 ? slot % page_size : 0;
  const int kvh = head < n_heads ? 0 : (head - n_heads) % n_kv;
  const size_t place = ((size_t)page * n_kv + kvh) * head_elems;
  const bool is_v = head >= n_heads + n_kv;
  if (is_v || (value_from_key && head >= n_heads)) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v_pages[place + lay.v_off(off, 8 * c + j)] = v[j];
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
  store8<float>(head < n_heads ? q_out + (size_t)t * n_heads * hd + 8 * c8 : k_pages + place + lay.k_off(off, 8 * c), v);
}

struct GfCall {
  const float *x, *w;
  float *y, *part;
  int M, N, K, ldx, ldw, ldy, vec;
  hipStream_t stream;
  const bf16x8 *xp, *wp;  // the operands cut beforehand, or null
};

static int gf_wide(const GfCall& c) {
  return c.N % 4 == 0 && c.ldy % 4 == 0 && (uintptr_t)c.y % 16 == 0 && (uintptr_t)c.part % 16 == 0;
}

// The groups' sums to y, where there are any and somebody wants them added up.
static int gf_sum(const GfCall& c) {
  if (c.part && c.y) {
    const GfSums s = {c.part, c.x, c.w, c.M, c.N, c.K, c.ldx, c.ldw, (c.K + GF_GROUP - 1) / GF_GROUP};
    gemm_f32_sum_kernel<<<dim3((c.N + 1023) / 1024, c.M), 256, 0, c.stream>>>(s, c.y, c.ldy, gf_wide(c));
  }
  return fg_launch_status();
}

template <int MB, int NB, int NW, bool FAR = false, bool CUT = false>
static int gf_launch(const GfCall& c) {
  constexpr int AHEAD = MB <= 3 ? 4 : 2;
  const int groups = (c.K + GF_GROUP - 1) / GF_GROUP;
  const int wide = gf_wide(c);
  const int row_tiles = (c.M + 16 * MB - 1) / (16 * MB), col_tiles = (c.N + 16 * NB * NW - 1) / (16 * NB * NW);
  const long long units = (long long)col_tiles * (c.part ? groups : 1);
  const long long blocks = (units * row_tiles + 7) / 8 * 8;
  if (blocks > 2147483647LL || (c.part && c.M > 65535)) return FG_ERR_ARG;
#define TILED(VEC)                                                                                            \
  gemm_f32_tiled_kernel<MB, NB, NW, AHEAD, VEC, FAR, CUT><<<(unsigned)blocks, 64 * NW, 0, c.stream>>>(             \
      c.x, c.w, c.xp, c.wp, c.y, c.part, c.M, c.N, c.K, c.ldx, c.ldw, c.ldy, row_tiles, col_tiles, (int)units, wide)
  if constexpr (CUT) TILED(true);
  else if (c.vec) TILED(true);
  else TILED(false);
#undef TILED
  return gf_sum(c);
}

// mb, nw: the tile of the many-rows kernel, 16 mb rows (mb <= 5 with 4 waves, 7 with 8) and nw waves of 32 outputs
// (mb = 0: the kernel of 16 rows).
// part: null, or fp32 [ceil(K / 1024)][M][N] for a workgroup a group of k; with y null the sums stay there.
// act: 0, or (mb = 0 without part, N % 16 == 0) GF_SILU or GF_GELU: y is [M][N / 2].
extern "C" int fg_gemm_f32_act(const float* x, const float* w, float* y, float* part, int M, int N, int K, int ldx, int ldw, int ldy,
                               int mb, int nw, int act, hipStream_t stream) {
  if (M <= 0 || N <= 0) return FG_OK;
  if (K <= 0 || ldx < K || ldw < K || (y && ldy < (act ? N / 2 : N)) || (!y && !part)) return FG_ERR_ARG;
  if (act && ((act != GF_SILU && act != GF_GELU) || mb || part || N % 16)) return FG_ERR_ARG;
  const bool vec = K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0;
  if (mb == 0) {
    const int groups = (K + GF_GROUP - 1) / GF_GROUP;
    if (M > 16 * 65535 || (part && (M > 65535 || groups > 65535))) return FG_ERR_ARG;
    const dim3 blocks((N + 15) / 16, (M + 15) / 16, part ? groups : 1);
#define FEW_ROWS(FEW, VEC) gemm_f32_few_kernel<FEW, VEC><<<blocks, 512, 0, stream>>>(x, w, y, part, M, N, K, ldx, ldw, ldy, act)
    if (M <= 8) {
      if (vec) FEW_ROWS(true, true);
      else FEW_ROWS(true, false);
    } else {
      if (vec) FEW_ROWS(false, true);
      else FEW_ROWS(false, false);
    }
#undef FEW_ROWS
    return gf_sum({x, w, y, part, M, N, K, ldx, ldw, ldy, vec, stream, nullptr, nullptr});
  }
  const GfCall c = {x, w, y, part, M, N, K, ldx, ldw, ldy, vec, stream, nullptr, nullptr};
  if (mb < 1 || mb > 7 || (nw == 4 && mb > 5) || (nw != 4 && nw != 8)) return FG_ERR_ARG;
  // What the rows that a tile loads span, of x (8 a wave at a time) and of a wave's 32 of W: any strides are taken, beyond 32
  // bits of bytes by the smallest tile (every cut gives the same bits).
  const int loaded = (16 * mb + 8 * nw - 1) / (8 * nw) * 8 * nw;
  const long long span = max((long long)(min(loaded, M) - 1) * ldx, (long long)(min(32, N) - 1) * ldw);
  if (4 * (span + 32) > 0xffffffffLL) return gf_launch<1, 2, 8, true>(c);
#define CASE(MB)                                          \
  if (mb == MB && nw == 8) return gf_launch<MB, 2, 8>(c); \
  if (mb == MB && nw == 4) return gf_launch<MB < 6 ? MB : 5, 2, 4>(c);
  CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7)
#undef CASE
  return FG_ERR_ARG;
}

// Rows [n, K] in their three parts: out bf16 [ceil(n / 16)][K / 32][3][64][8].
extern "C" int fg_gemm_f32_cut(const float* rows, int ld, int n, int K, void* out, hipStream_t stream) {
  if (n <= 0) return FG_OK;
  if (K <= 0 || K % GF_STEP || ld < K || ld % 4 || ((uintptr_t)rows | (uintptr_t)out) % 16 || K / GF_STEP > 4 * 65535) return FG_ERR_ARG;
  gemm_f32_cut_kernel<<<dim3((n + 15) / 16, (K / GF_STEP + 3) / 4), 256, 0, stream>>>(rows, ld, n, K, (bf16x8*)out);
  return fg_launch_status();
}

// fg_gemm_f32_act's tiles (mb > 0, act 0) with the operands cut beforehand, xp and wp from fg_gemm_f32_cut; K a multiple of 128.
extern "C" int fg_gemm_f32_parts(const void* xp, const void* wp, const float* x, const float* w, float* y, float* part, int M, int N, int K,
                                 int ldx, int ldw, int ldy, int mb, int nw, hipStream_t stream) {
  if (M <= 0 || N <= 0) return FG_OK;
  if (!xp || !wp || ((uintptr_t)xp | (uintptr_t)wp) % 16 || K <= 0 || K % GF_SEG || K > 1 << 20 || ldx < K || ldw < K || (y && ldy < N) ||
      (!y && !part))
    return FG_ERR_ARG;
  if (mb < 1 || mb > 7 || (nw == 4 && mb > 5) || (nw != 4 && nw != 8)) return FG_ERR_ARG;
  const GfCall c = {x, w, y, part, M, N, K, ldx, ldw, ldy, 1, stream, (const bf16x8*)xp, (const bf16x8*)wp};
#define CASE(MB)                                                       \
  if (mb == MB && nw == 8) return gf_launch<MB, 2, 8, false, true>(c); \
  if (mb == MB && nw == 4) return gf_launch<MB < 6 ? MB : 5, 2, 4, false, true>(c);
  CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7)
#undef CASE
  return FG_ERR_ARG;
}

extern "C" int fg_gemm_f32(const float* x, const float* w, float* y, float* part, int M, int N, int K, int ldx,
                           int ldw, int ldy, int mb, int nw, hipStream_t stream) {
  return y || M <= 0 || N <= 0 ? fg_gemm_f32_act(x, w, y, part, M, N, K, ldx, ldw, ldy, mb, nw, 0, stream) : FG_ERR_ARG;
}

// The groups' sums `part` of x [M, K] and w [N, K] (what fg_gemm_f32_act left) and what comes behind the product.  All rows 16-byte aligned.
#define GF_SUMS const GfSums s = {part, x, w, M, N, K, ldx, ldw, (K + GF_GROUP - 1) / GF_GROUP}
static bool gf_sums_ok(const float* part, int M, int N, int K, const void* out) {
  return part && K > 0 && N % 8 == 0 && M <= 65535 && (uintptr_t)part % 16 == 0 && (uintptr_t)out % 16 == 0;
}

// silu(gate) * up (act GF_SILU) or the tanh form of GELU in its place (GF_GELU) of interleaved columns: y [M, N / 2].
extern "C" int fg_gemm_f32_sum_act(const float* part, const float* x, const float* w, float* y, int M, int N, int K, int ldx, int ldw,
                                   int act, hipStream_t stream) {
  if (M <= 0 || N <= 0) return FG_OK;
  if (!gf_sums_ok(part, M, N, K, y) || N % 16 || (act != GF_SILU && act != GF_GELU)) return FG_ERR_ARG;
  GF_SUMS;
  gemm_f32_sum_act_kernel<<<dim3((N / 2 + 1023) / 1024, M), 256, 0, stream>>>(s, y, act);
  return fg_launch_status();
}

// h [M, N] += the product, out = rmsnorm(h) * weight.  N <= 8192.
extern "C" int fg_gemm_f32_sum_norm(const float* part, const float* x, const float* w, float* h, const float* weight, float* out, int M,
                                    int N, int K, int ldx, int ldw, float eps, hipStream_t stream) {
  if (M <= 0 || N <= 0) return FG_OK;
  if (!gf_sums_ok(part, M, N, K, out) || N > 8192 || ((uintptr_t)h | (uintptr_t)weight) % 16) return FG_ERR_ARG;
  GF_SUMS;
  if (N <= 2048) gemm_f32_sum_norm_kernel<1><<<M, 256, 0, stream>>>(s, h, weight, out, eps);
  else if (N <= 4096) gemm_f32_sum_norm_kernel<2><<<M, 256, 0, stream>>>(s, h, weight, out, eps);
  else gemm_f32_sum_norm_kernel<4><<<M, 256, 0, stream>>>(s, h, weight, out, eps);
  return fg_launch_status();
}

// The rotated queries to q_out [M, n_heads * hd], keys and values into their pages (see fg_rope_kv_parts in rope_kv.hip).
extern "C" int fg_gemm_f32_sum_rope(const float* part, const float* x, const float* w, float* q_out, const float* table, const int* slots,
                                    float* k_pages, float* v_pages, int M, int N, int K, int ldx, int ldw, int n_heads, int n_kv, int hd,
                                    int rotary_dim, int page_size, int value_from_key, hipStream_t stream) {
  if (M <= 0 || N <= 0) return FG_OK;
  if (!gf_sums_ok(part, M, N, K, q_out) || hd <= 0 || hd % 8 || rotary_dim < 0 || rotary_dim > hd || rotary_dim % 8 || page_size <= 0 ||
      page_size % 8 || n_heads <= 0 || n_kv <= 0 || (rotary_dim && (!table || (uintptr_t)table % 16)) || (uintptr_t)k_pages % 16 ||
      N != (n_heads + (value_from_key ? 1 : 2) * n_kv) * hd)
    return FG_ERR_ARG;
  GF_SUMS;
  gemm_f32_sum_rope_kernel<<<dim3(M, (N / 8 + 127) / 128), 128, 0, stream>>>(s, q_out, table, slots, k_pages, v_pages, n_heads, n_kv, hd,
                                                                            rotary_dim, page_size, value_from_key);
  return fg_launch_status();
}
#undef GF_SUMS
