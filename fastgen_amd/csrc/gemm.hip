// y = x W^T with W stored [out, in] row-major (fastgen/forward.py:433-440,
// 470, 488-496, 513: F.linear): the engine's own matrix products without a
// mode of reduced precision.
//
// float32 (the true 32-bit path) runs on v_mfma_f32_16x16x4_f32, whose
// products and sums are fp32.  Every output element is summed in an order
// fixed by K alone, whichever kernel takes the product: 32 k in a chain of
// matrix instructions (instruction (s, j) adds the k = 16 s + 4 g + j of its
// four lane groups g, one after the other), 4 chains into a segment's sum, 8
// segments into a group's, the groups' into the total, each ascending.  A
// row's result therefore does not depend on how many other rows the call
// holds, and rounding grows with 32 + 4 + 8 + K/1024 additions (relative to
// the product in 64 bits, random operands of K = 3072 / 8192 / 14336: 1.3 /
// 1.4 / 1.4e-7; chains of 128 k: 2.1 / 2.2 / 2.2e-7).
//
// Operands of bf16 with fp32 accumulation take the FMA kernel below, so that
// any shape has a product when the tuned kernels refuse it.
#include "common.h"

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

#define GF_SEG 128    // k of a segment: 4 chains of matrix instructions
#define GF_GROUP 1024 // k of a group: 8 segments
#define GF_STEP 32    // k of a chain; what the tiled kernel holds in LDS at a time

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

// Four instructions: 16 k.  A: 16 rows of W, B: 16 rows of x; lane 16 g + r ends with outputs 4 g .. 4 g + 3 of x row r.
__device__ __forceinline__ f32x4 gf_mfma16(const f32x4 wv, const f32x4 xv, f32x4 acc) {
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j], xv[j], acc, 0, 0, 0);
  return acc;
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

// Up to 16 rows (decode): bound by reading W once.  A workgroup owns 16 outputs; a round is one group, a wave takes
// one of its segments, so 64 KB of W (every wave's next segment) are in flight a workgroup while the current ones
// are multiplied; the segments' sums meet in LDS and are added in order by one thread an output.  4 rows, N x K
// 3072 x 3072 / 16384 x 3072 / 3072 x 8192: 16 / 50 / 35 us, 2.4 / 4.0 / 2.9 TB/s of W (FMA with a thread an output: 490
// / 495 / 1250 us); at 16 rows the tiled kernel is level (31 / 54 / 38 against 20 / 61 / 45).
template <bool VEC>
__global__ __launch_bounds__(512) void gemm_f32_few_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                           float* __restrict__ y, int M, int N, int K, int ldx,
                                                           int ldw, int ldy) {
  __shared__ f32x4 sums[2][8][FG_WAVE];
  const int tid = threadIdx.x, lane = tid % FG_WAVE, wave = tid / FG_WAVE;
  const int r = lane % 16, g = lane / 16, n0 = blockIdx.x * 16;
  // rows behind the last repeat it: their outputs are not stored
  const float* wrow = w + (size_t)min(n0 + r, N - 1) * ldw;
  const float* xrow = x + (size_t)min(r, M - 1) * ldx;
  const int n_seg = (K + GF_SEG - 1) / GF_SEG;
  f32x4 wv[8], next[8], xv[8];
  if (wave < n_seg) {
#pragma unroll
    for (int i = 0; i < 8; ++i) next[i] = gf_load4<VEC>(wrow, wave * GF_SEG + i * 16 + g * 4, K);
  }
  float total = 0.f;
  for (int s0 = 0, buf = 0; s0 < n_seg; s0 += 8, buf ^= 1) {
    const int seg = s0 + wave;
    if (seg < n_seg) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        wv[i] = next[i];
        xv[i] = gf_load4<VEC>(xrow, seg * GF_SEG + i * 16 + g * 4, K);
      }
      if (seg + 8 < n_seg) {
#pragma unroll
        for (int i = 0; i < 8; ++i) next[i] = gf_load4<VEC>(wrow, (seg + 8) * GF_SEG + i * 16 + g * 4, K);
      }
      f32x4 acc[4], sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = gf_mfma16(wv[2 * i], xv[2 * i], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[i] = gf_mfma16(wv[2 * i + 1], xv[2 * i + 1], acc[i]);
        sum += acc[i];
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
  if (tid < 256) {
    const int m = (tid / 4) % 16, n = n0 + (tid / 64) * 4 + tid % 4;
    if (m < M && n < N) y[(size_t)m * ldy + n] = total;
  }
}

// Many rows: bound by the matrix cores (157 TFLOP/s of fp32).  Four waves own 32 MB rows x 32 NB outputs, both operands
// go through registers into LDS, 32 k at a time in two buffers, in pieces of 4 k a row, piece-major with two pieces
// of padding: a wave's operand reads are runs of 256 bytes, and 8 lanes load a whole line of a row (with 4 lanes a
// row, half lines and LDS stores as contiguous as the reads: 5 % slower).  With `part` a workgroup takes one group of
// k and stores its sum there ([groups][M][N]); the workgroups that read the same rows of W are neighbours on one die.
// 400 rows of 16384 x 3072: 440 us, 92 TFLOP/s (FMA: 1206 us); 2048 rows: 1883 us, 109 TFLOP/s, 1592 without the
// loads, so the rest is the matrix cores, the operand reads and the barrier of every 32 k.
template <int MB, int NB, bool VEC>
__global__ __launch_bounds__(256) void gemm_f32_tiled_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                             float* __restrict__ y, float* __restrict__ part, int M,
                                                             int N, int K, int ldx, int ldw, int ldy, int row_tiles,
                                                             int col_tiles, int units, int wide) {
  constexpr int TM = 32 * MB, TN = 32 * NB;
  __shared__ f32x4 xs[2][8][TM + 2], ws[2][8][TN + 2];
  const int unit = (blockIdx.x / 8 / row_tiles) * 8 + blockIdx.x % 8;
  if (unit >= units) return;
  const int m0 = (blockIdx.x / 8 % row_tiles) * TM, n0 = (unit % col_tiles) * TN, group = unit / col_tiles;
  const int tid = threadIdx.x, lane = tid % FG_WAVE, wave = tid / FG_WAVE;
  const int r = lane % 16, g = lane / 16;
  const int wm = (wave / 2) * 16 * MB, wn = (wave % 2) * 16 * NB;
  const int piece = tid % 8, row = tid / 8;
  const float* xr[MB];
  const float* wr[NB];
#pragma unroll
  for (int i = 0; i < MB; ++i) xr[i] = x + (size_t)min(m0 + row + 32 * i, M - 1) * ldx;
#pragma unroll
  for (int i = 0; i < NB; ++i) wr[i] = w + (size_t)min(n0 + row + 32 * i, N - 1) * ldw;
  const int k_begin = part ? group * GF_GROUP : 0, k_end = part ? min(K, k_begin + GF_GROUP) : K;

  f32x4 xv[MB], wv[NB], seg[MB][NB], mid[MB][NB], total[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) seg[i][j] = mid[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < MB; ++i) xs[0][piece][row + 32 * i] = gf_load4<VEC>(xr[i], k_begin + piece * 4, k_end);
#pragma unroll
  for (int i = 0; i < NB; ++i) ws[0][piece][row + 32 * i] = gf_load4<VEC>(wr[i], k_begin + piece * 4, k_end);
  __syncthreads();
  int buf = 0;
  for (int k0 = k_begin; k0 < k_end; k0 += GF_STEP, buf ^= 1) {
    const bool more = k0 + GF_STEP < k_end;
    if (more) {
#pragma unroll
      for (int i = 0; i < MB; ++i) xv[i] = gf_load4<VEC>(xr[i], k0 + GF_STEP + piece * 4, k_end);
#pragma unroll
      for (int i = 0; i < NB; ++i) wv[i] = gf_load4<VEC>(wr[i], k0 + GF_STEP + piece * 4, k_end);
    }
    f32x4 acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      f32x4 a[NB], b[MB];
#pragma unroll
      for (int j = 0; j < NB; ++j) a[j] = ws[buf][s * 4 + g][wn + 16 * j + r];
#pragma unroll
      for (int i = 0; i < MB; ++i) b[i] = xs[buf][s * 4 + g][wm + 16 * i + r];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][e], b[i][e], acc[i][j], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) seg[i][j] += acc[i][j];
    const int next_k = k0 + GF_STEP;
    if (next_k % GF_SEG == 0 || !more) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          mid[i][j] += seg[i][j];
          seg[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (next_k % GF_GROUP == 0 || !more) {
            total[i][j] += mid[i][j];
            mid[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
        }
    }
    if (more) {
#pragma unroll
      for (int i = 0; i < MB; ++i) xs[buf ^ 1][piece][row + 32 * i] = xv[i];
#pragma unroll
      for (int i = 0; i < NB; ++i) ws[buf ^ 1][piece][row + 32 * i] = wv[i];
    }
    __syncthreads();
  }
  float* out = part ? part + (size_t)group * M * N : y;
  const int ldo = part ? N : ldy;
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int m = m0 + wm + 16 * i + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < NB; ++j)
      gf_store4(out + (size_t)m * ldo, n0 + wn + 16 * j + 4 * g, N, wide, total[i][j]);
  }
}

// The groups' sums, added in order.
__global__ __launch_bounds__(256) void gemm_f32_sum_kernel(const float* __restrict__ part, float* __restrict__ y,
                                                           int M, int N, int ldy, int groups, int wide) {
  const int m = blockIdx.y, n = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (n >= N) return;
  f32x4 total = {0.f, 0.f, 0.f, 0.f};
  const float* p = part + (size_t)m * N + n;
  for (int g = 0; g < groups; ++g, p += (size_t)M * N) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (wide && n + 4 <= N) {
      v = *(const f32x4*)p;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) v[e] = p[e];
    }
    total += v;
  }
  gf_store4(y + (size_t)m * ldy, n, N, wide, total);
}

// mb, nb: the tile of the many-rows kernel in units of 32 rows and 32 outputs (mb = 0: up to 16 rows, no tile).
// part: null, or fp32 [ceil(K / 1024)][M][N] for a workgroup a group of k.
extern "C" int fg_gemm_f32(const float* x, const float* w, float* y, float* part, int M, int N, int K, int ldx,
                           int ldw, int ldy, int mb, int nb, hipStream_t stream) {
  if (M <= 0 || N <= 0) return FG_OK;
  if (K <= 0 || ldx < K || ldw < K || ldy < N) return FG_ERR_ARG;
  const bool vec = K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0;
  if (mb == 0) {
    if (M > 16 || part) return FG_ERR_ARG;
    const int blocks = (N + 15) / 16;
    if (vec) gemm_f32_few_kernel<true><<<blocks, 512, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy);
    else gemm_f32_few_kernel<false><<<blocks, 512, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy);
    return fg_launch_status();
  }
  const int groups = (K + GF_GROUP - 1) / GF_GROUP;
  const int wide = N % 4 == 0 && ldy % 4 == 0 && (uintptr_t)y % 16 == 0 && (uintptr_t)part % 16 == 0;
  const int row_tiles = (M + 32 * mb - 1) / (32 * mb), col_tiles = (N + 32 * nb - 1) / (32 * nb);
  const long long units = (long long)col_tiles * (part ? groups : 1);
  const long long blocks = (units + 7) / 8 * 8 * row_tiles;
  if (blocks > 2147483647LL || (part && M > 65535)) return FG_ERR_ARG;
#define TILED(MB, NB)                                                                                               \
  do {                                                                                                              \
    if (vec) gemm_f32_tiled_kernel<MB, NB, true><<<(unsigned)blocks, 256, 0, stream>>>(                             \
        x, w, y, part, M, N, K, ldx, ldw, ldy, row_tiles, col_tiles, (int)units, wide);                             \
    else gemm_f32_tiled_kernel<MB, NB, false><<<(unsigned)blocks, 256, 0, stream>>>(                                \
        x, w, y, part, M, N, K, ldx, ldw, ldy, row_tiles, col_tiles, (int)units, wide);                             \
  } while (0)
  if (mb == 1 && nb == 1) TILED(1, 1);
  else if (mb == 1 && nb == 2) TILED(1, 2);
  else if (mb == 2 && nb == 1) TILED(2, 1);
  else if (mb == 2 && nb == 2) TILED(2, 2);
  else return FG_ERR_ARG;
#undef TILED
  if (part) {
    gemm_f32_sum_kernel<<<dim3((N + 1023) / 1024, M), 256, 0, stream>>>(part, y, M, N, ldy, groups, wide);
  }
  return fg_launch_status();
}
