// y = x W^T for prompts: several hundred rows of x and more, bf16 operands, fp32 accumulation, W packed in operand order
// (gemm_skinny.hip).  The product itself is in tile_product.h; here are the shapes of its tiles, which tile a workgroup
// takes, and what becomes of the sums: bf16 or fp32 rows, or silu(gate) * up of a matrix whose rows are gate and up
// interleaved in groups of 8 (the tanh form of GELU in SiLU's place), so that the gate/up rows never go through memory.
//
// Up to 64 rows (a batch that decodes) it is bound by reading W, and what the tile brings is how W is read: a wave 1 KB at a time in whole
// lines, seven steps of 32 k ahead, and no barrier between W and the products.  28,672 x 4,096 with its activation at 64 rows 44.5 us = 5.3 TB/s
// (the wide kernel of gemm_skinny.hip 51), 4,096 x 14,336 in eight splits with the sums read back 26.3 (32), 4,096 x 4,096 12.1 (13.7),
// 3,072 x 8,192 15.7 (19.1), 2,048 x 2,048 6.6 (9.8).
//
// Where the tiles are few and k long, k is cut over workgroups (blockIdx.y) into fp32 partial sums that the norm kernel behind
// adds in order.  Sums run over k in ascending order (within a split), whatever the batch holds.
#include "tile_product.h"

#define EPI_STORE 0
#define EPI_SILU_MUL 1
#define EPI_GELU_MUL 4
#define EPI_IS_GATED(e) ((e) == EPI_SILU_MUL || (e) == EPI_GELU_MUL)
// gate * sigmoid(gate) * up; the tanh form of GELU is 0.5 (1 + tanh(u)) = sigmoid(2 u), which loses nothing where tanh is near -1
template <int EPI>
__device__ __forceinline__ float gl_gated(float gate, float up) {
  const float u = EPI == EPI_GELU_MUL ? 1.5957691216057308f * (gate + 0.044715f * gate * gate * gate) : gate;
  return gate / (1.f + __expf(-u)) * up;
}

// Four blocks of 16 columns of a row: lane 16 g + r holds columns 4 g .. 4 g + 3 of each, two columns a register, and gets all 16
// columns of block g (v[2 i], v[2 i + 1]: columns 4 i .. 4 i + 3), so that a row is stored 32 bytes a lane.
__device__ __forceinline__ void gl_turn(uint32_t (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // blocks 0, 1 with 2, 3: halves of the wave
    const auto a = __builtin_amdgcn_permlane32_swap(v[i], v[4 + i], false, false);
    v[i] = a[0];
    v[4 + i] = a[1];
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // then 0 with 1 and 2 with 3: rows of 16 lanes
    const int j = i < 2 ? i : i + 2;
    const auto a = __builtin_amdgcn_permlane16_swap(v[j], v[j + 2], false, false);
    v[j] = a[0];
    v[j + 2] = a[1];
  }
}
__device__ __forceinline__ uint32_t gl_pair(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 p = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, p);
}

// A tile: 16 MB rows from m0 on, 64 NB columns from 64 NB ct on.
template <int MB, int NB, int NST, int WS, bool ONE_WAVE, int EPI, class TY>
__device__ __forceinline__ void gemm_large_tile(bf16_t* lds, const bf16_t* x, int ldx, const bf16_t* w, TY* y, int ldy, int M, int N,
                                                int K, int m0, int ct, int first, int n_stages) {
#ifdef __HIP_DEVICE_COMPILE__
  typedef TileProduct<MB, NB, NST, WS, ONE_WAVE> Product;
  const int lane = threadIdx.x % FG_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FG_WAVE);
  const int r16 = lane & 15, g = lane >> 4;
  const int n0 = (ct * 4 + wave) * 16 * NB;
  TileOperands op;
  op.x = x + (size_t)m0 * ldx;
  op.x_bytes = 2u * (unsigned)((min(16 * MB, M - m0) - 1) * ldx + K);
  op.w_row = (unsigned)K * 32u;
  op.set_w(0, w, n0 / 16, (N + 15) / 16, Product::HALF);
  op.set_w(1, w, n0 / 16 + Product::HALF, (N + 15) / 16, NB - Product::HALF);
  unsigned xo[Product::XL];
#pragma unroll
  for (int j = 0; j < Product::XL; ++j) {
    const int row = Product::row_of(wave, j, lane);
    xo[j] = op.row_offset(m0 + row < M, row, ldx, Product::chunk_of(lane));
  }
  f32x4 acc[MB][NB];
  Product::run(lds, op, xo, wave, lane, first, n_stages, n_stages, acc);

#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int m = m0 + 16 * mb + r16;
    if constexpr (EPI_IS_GATED(EPI)) {
      // rows 0 .. 7 of a block are gates, 8 .. 15 the ups of the same channels, which the lanes 32 on hold: of two blocks the
      // lower half of the wave gets gate and up of the first one's channels, the upper half of the second one's
      uint32_t v[NB];
#pragma unroll
      for (int nb = 0; nb < NB; nb += 2) {
        const f32x4 one = Product::sums(acc[mb][nb]), two = Product::sums(acc[mb][nb + 1]);
        float a[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(one[e]), __float_as_uint(two[e]), false, false);
          a[e] = gl_gated<EPI>(__uint_as_float(both[0]), __uint_as_float(both[1]));
        }
        v[nb] = gl_pair(a[0], a[1]);
        v[nb + 1] = gl_pair(a[2], a[3]);
      }
      if constexpr (NB == 4) {
        // the lane's four channels of either pair of blocks against the other half row of lanes' : eight in a row
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const auto a = __builtin_amdgcn_permlane16_swap(v[i], v[2 + i], false, false);
          v[i] = a[0];
          v[2 + i] = a[1];
        }
        const int n = n0 / 2 + (g % 2) * 16 + (g / 2) * 8;
        if (m < M && n < N / 2) *(uint4*)((bf16_t*)y + (size_t)m * ldy + n) = make_uint4(v[0], v[1], v[2], v[3]);  // (N % 16 == 0, ldy % 8 == 0)
      } else {
        const int n = n0 / 2 + (g / 2) * 8 + (g % 2) * 4;
        if (m < M && n < N / 2) *(uint2*)((bf16_t*)y + (size_t)m * ldy + n) = make_uint2(v[0], v[1]);
      }
    } else if constexpr (NB == 4 && sizeof(TY) == 2) {
      uint32_t v[8];
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        const f32x4 sum = Product::sums(acc[mb][nb]);
        v[2 * nb] = gl_pair(sum[0], sum[1]);
        v[2 * nb + 1] = gl_pair(sum[2], sum[3]);
      }
      gl_turn(v);
      const int n = n0 + 16 * g;
      bf16_t* to = (bf16_t*)y + (size_t)m * ldy + n;
      if (m < M && n + 15 < N && ldy % 8 == 0) {
        *(uint4*)to = make_uint4(v[0], v[1], v[2], v[3]);
        *(uint4*)(to + 8) = make_uint4(v[4], v[5], v[6], v[7]);
      } else if (m < M) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (n + e < N) ((uint16_t*)to)[e] = (uint16_t)(v[e / 2] >> (e % 2 * 16));
      }
    } else {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const f32x4 sum = Product::sums(acc[mb][nb]);
        const int n = n0 + 16 * nb + 4 * g;
        if (m < M && n + 3 < N && (ldy & 3) == 0) {
          if constexpr (sizeof(TY) == 4) {
            *(f32x4*)((float*)y + (size_t)m * ldy + n) = sum;
          } else {
            *(uint2*)((bf16_t*)y + (size_t)m * ldy + n) = make_uint2(gl_pair(sum[0], sum[1]), gl_pair(sum[2], sum[3]));
          }
        } else if (m < M) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < N) y[(size_t)m * ldy + n + e] = from_f<TY>(sum[e]);
        }
      }
    }
  }
#endif
}

// Tiles of 256 rows: the first `whole` of them whole, the others in halves of 128 rows.  Where the last round of whole tiles would leave
// half of the compute units without one or more, halves take half of its time: 2,048 x 28,672 x 4,096 (896 tiles, three rounds and
// 128).
template <int MB, int NB, int NST, int WS, int OCC, int EPI, class TY>
__global__ __launch_bounds__(256, OCC) void gemm_large_kernel(const bf16_t* x, int ldx, const bf16_t* w, TY* y, int ldy,
                                                              long long part_stride, int M, int N, int K, int row_tiles,
                                                              int col_tiles, int whole, int split_stages) {
  extern __shared__ __attribute__((aligned(16))) bf16_t large_lds[];
  // A die (blockIdx % 8) takes a run of tiles, by bands of 2,048 rows, in a band column after column: its compute units
  // work on about as many rows of x as of W at a time, each of which its L2 reads once.
  constexpr int BAND = 2048 / (16 * MB);
  const int tiles = row_tiles * col_tiles, die = blockIdx.x % 8, place = blockIdx.x / 8, each = (whole + 7) / 8;
  int id = die * each + place, half = -1;
  if (place >= each) {
    const int halves = 2 * (tiles - whole), of_die = (halves + 7) / 8, h = die * of_die + place - each;
    if (place - each >= of_die || h >= halves) return;
    id = whole + h / 2;
    half = h % 2;
  } else if (id >= whole) {
    return;
  }
  const int band = id / (BAND * col_tiles), rows_here = min(BAND, row_tiles - band * BAND), at = id - band * BAND * col_tiles;
  const int ct = at / rows_here, m0 = (band * BAND + at % rows_here) * 16 * MB;
  const int first = blockIdx.y * split_stages, n_stages = min(split_stages, K / 64 - first);
  y += blockIdx.y * part_stride;
  if (MB != 16 || half < 0) {
    gemm_large_tile<MB, NB, NST, WS, OCC == 1, EPI, TY>(large_lds, x, ldx, w, y, ldy, M, N, K, m0, ct, first, n_stages);
  } else if constexpr (MB == 16) {
    if (m0 + 128 * half < M)
      gemm_large_tile<8, NB, NST, WS, OCC == 1, EPI, TY>(large_lds, x, ldx, w, y, ldy, M, N, K, m0 + 128 * half, ct, first, n_stages);
  }
}

template <int MB, int NB, int NST, int WS, int OCC, int EPI, class TY>
static int launch_large(const void* x, int ldx, const void* w, void* y, int ldy, long long part_stride, int splits, int M, int N,
                        int K, int whole_tiles, hipStream_t stream) {
  constexpr int lds = NST * MB * 2048;
  static_assert(OCC * lds <= 160 * 1024, "LDS of a compute unit");
  static uint64_t raised = 0;  // devices that were asked for more than 64 KB of dynamic LDS, a bit each (asking twice does no harm)
  auto kernel = gemm_large_kernel<MB, NB, NST, WS, OCC, EPI, TY>;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return FG_ERR_LAUNCH;
  if (device >= 64 || !(__atomic_load_n(&raised, __ATOMIC_RELAXED) >> device & 1)) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return FG_ERR_LAUNCH;
    if (device < 64) __atomic_fetch_or(&raised, (uint64_t)1 << device, __ATOMIC_RELAXED);
  }
  const long long rt = ((long long)M + 16 * MB - 1) / (16 * MB), ct = ((long long)N + 64 * NB - 1) / (64 * NB);
  if (rt * ct > 1 << 27) return FG_ERR_ARG;
  const int split_stages = (K / 64 + splits - 1) / splits;
  const long long whole = whole_tiles > 0 && MB == 16 && whole_tiles < rt * ct ? whole_tiles : rt * ct;
  const long long blocks = (whole + 7) / 8 * 8 + (2 * (rt * ct - whole) + 7) / 8 * 8;
  kernel<<<dim3((unsigned)blocks, splits), 256, lds, stream>>>((const bf16_t*)x, ldx, (const bf16_t*)w, (TY*)y, ldy, part_stride, M, N, K,
                                                               (int)rt, (int)ct, (int)whole, split_stages);
  return fg_launch_status();
}

// x [M, K] bf16 (K % 64 == 0, rows 16-byte aligned), w packed [N, K].  tile: 256256, 256192, 128256, 128192, 128128 or 64128 (rows and
// columns of a workgroup's tile).  epilogue 0: y [M, N] of out_dtype (splits > 1: fp32 [splits, M, N], part_stride elements
// apart, sums over ceil(K / 64 / splits) * 64 of k each; no split may be empty); 1 and 4: gate and up rows interleaved (N % 16 == 0), y [M, N / 2]
// bf16, one split.  whole_tiles: 0, or of the tiles of 256 rows those that are not cut into halves (a multiple of 8).
extern "C" int fg_gemm_large(const void* x, int ldx, const void* w, void* y, int ldy, long long part_stride, int splits, int M,
                             int N, int K, int out_dtype, int epilogue, int tile, int whole_tiles, hipStream_t stream) {
  if (M <= 0 || N <= 0) return FG_OK;
  if (whole_tiles < 0 || whole_tiles % 8) return FG_ERR_ARG;
  if (K <= 0 || K % 64 || ldx % 8 || ldx < K || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15)) return FG_ERR_ARG;
  // offsets within a tile's rows, and within 16 x 4 packed rows, are 32-bit
  if ((long long)ldx * 512 + 2ll * K > 4000000000LL || (long long)K * 32 * 4 > 4000000000LL) return FG_ERR_ARG;
  if (out_dtype != FG_BF16 && out_dtype != FG_F32) return FG_ERR_ARG;
  if (splits < 1 || splits > 64 || (splits > 1 && (out_dtype != FG_F32 || part_stride < (long long)M * ldy))) return FG_ERR_ARG;
  if ((long long)((K / 64 + splits - 1) / splits) * (splits - 1) >= K / 64) return FG_ERR_ARG;
  if (EPI_IS_GATED(epilogue) ? (N % 16 || ldy < N / 2 || ldy % 8 || out_dtype != FG_BF16 || splits != 1) : (epilogue != EPI_STORE || ldy < N))
    return FG_ERR_ARG;
#define GO(MB, NB, NST, WS, OCC, EPI, TY) \
  return launch_large<MB, NB, NST, WS, OCC, EPI, TY>(x, ldx, w, y, ldy, part_stride, splits, M, N, K, whole_tiles, stream)
#define STORE(...)                                                \
  do {                                                            \
    if (out_dtype == FG_BF16) GO(__VA_ARGS__, EPI_STORE, bf16_t); \
    GO(__VA_ARGS__, EPI_STORE, float);                            \
  } while (0)
#define PICK(...)                                                        \
  do {                                                                   \
    if (epilogue == EPI_SILU_MUL) GO(__VA_ARGS__, EPI_SILU_MUL, bf16_t); \
    if (epilogue == EPI_GELU_MUL) GO(__VA_ARGS__, EPI_GELU_MUL, bf16_t); \
    STORE(__VA_ARGS__);                                                  \
  } while (0)
  switch (tile) {
    case 256256: PICK(16, 4, 5, 4, 1);
    case 128256: PICK(8, 4, 5, 4, 2);
    case 128128: PICK(8, 2, 5, 8, 2);
    case 64128: PICK(4, 2, 5, 8, 3);
    case 256192: if (epilogue == EPI_STORE) STORE(16, 3, 5, 4, 1); return FG_ERR_ARG;
    case 128192: if (epilogue == EPI_STORE) STORE(8, 3, 5, 4, 2); return FG_ERR_ARG;
  }
#undef PICK
#undef STORE
#undef GO
  return FG_ERR_ARG;
}
