// The inner product of a large tile, for steps of many rows (prompts): 16 MB rows of x times 64 NB rows of a packed
// matrix, by four waves side by side along the columns, each 16 MB x 16 NB.  What it is built around:
//
//  * A compute unit's matrix cores take 256 x 256 x 32 products in 1,024 clocks.  Its vector memory path brings 64 bytes a
//    clock and its LDS gives 128, so a tile has to use what it loads often: the rows of x, which the waves share, go
//    through LDS, a wave's rows of the matrix are its own and go from memory into its registers in operand order (they
//    are packed so).  256 x 256: half of the one path and 0.6 of the other.
//  * One wave a SIMD at 256 x 256 (256 of its 512 registers are sums): what hides the latencies is the order of the
//    instructions.  Operands of x are read from LDS 6 blocks of 16 rows (24 matrix instructions) ahead, rows of the matrix
//    WS - 1 steps of 32 k ahead, stages of x NST - 2 stages of 64 k ahead (straight from memory into LDS), and every
//    other instruction stands alone between two matrix instructions, where it costs nothing.  The matrix instructions
//    are written as assembly because the compiler otherwise moves their sums between registers in the loop (308 moves
//    for 256 products).
//  * One barrier a stage.  A stage's place in the ring is written again two stages after it was read, so that the barrier
//    between is enough and nobody waits for reads in flight.
//  * A row of x in a stage is one cache line of 128 bytes, and the 16-byte chunk c of row r of 8 lies at place c ^ r, so
//    that eight lanes that read the same chunk of eight rows use all banks.
//
// 2,048 x 8,192 x 4,096 (256 workgroups of 256 x 256): 99 us = 1.38 PFLOP/s, the matrix cores busy 74 % of a wave's life
// (22 k of its 178 k clocks it waits at barriers and for its first loads); 14,336 of k 314 us = 1.53.  Without the order
// within a stage 329, and with eight waves of 128 x 64 and rows of x through registers 473 against 359 (28,672 x 4,096, gated).
//
// Rows of x beyond the tile and stages beyond the k range are loads behind the end of their buffer: zeros, and no access.  Whether and
// how a load's scalar offset takes part in that check must not matter for where it reads: a row that is not there has a lane's offset
// (TP_NOWHERE) that is behind any buffer and stays so with the scalar offset added, a stage that is not there has a size of 0,
// and a block of the matrix that is not there is the last one that is: its sums are not stored.
#pragma once

#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// A lane's offset behind the end of any buffer (they have up to 4,000,000,000 bytes, of which a row's 2 K are at most 62,500,000): the
// load gives zeros.
#define TP_NOWHERE 0xf0000000u

struct TileOperands {
  const void* x;     // first byte that an offset of a row counts from
  unsigned x_bytes;  // readable there
  const void* w[2];  // packed rows of the wave's first (NB + 1) / 2 blocks of 16, and of the others
  unsigned w_bytes[2];
  unsigned w_row;    // bytes of 16 packed rows
  unsigned w_step[2];  // from a part's first block to its second: 0 where there is none

  // w[part]: `most` blocks from block `block` on of a matrix of `blocks`, those that are there.
  __host__ __device__ __forceinline__ void set_w(int part, const void* matrix, int block, int blocks, int most) {
    const int there = max(0, min(most, blocks - block));
    w[part] = (const char*)matrix + (there ? (size_t)block * w_row : 0);
    w_bytes[part] = there * w_row;
    w_step[part] = there > 1 ? w_row : 0;
  }
  __host__ __device__ __forceinline__ unsigned row_offset(bool there, int row, int ldx, unsigned chunk) const {
    return there ? 2u * (unsigned)row * (unsigned)ldx + chunk : TP_NOWHERE;
  }
};

// What a load's buffer holds, and the scalar part of its offset.
struct TileLoad {
  unsigned bytes, at;
};

template <int MB, int NB, int NST, int WS, bool ONE_WAVE>
struct TileProduct {
  static constexpr int XL = MB / 2;                  // loads of x a wave issues a stage: 8 rows x 64 k each
  static constexpr int STAGE = MB * 1024;            // elements of a stage: 16 MB rows x 64 k
  static constexpr int RB = MB < 8 ? MB : 8;         // operands of x in registers
  static constexpr int AHEAD = MB < 8 ? MB - 1 : 6;  // blocks of 16 rows that they are read ahead
  static constexpr int LA = NST - 2;                 // stages asked for ahead
  static constexpr int U = WS / 2;                   // stages a round of the loop
  static constexpr int HALF = (NB + 1) / 2;
  static_assert(MB % RB == 0 && MB % 4 == 0 && NB <= 4 && WS % 2 == 0 && NST >= 4, "tile");

  // The loads of stage s of the range's n_stages, and of block nb and step t of 32 k.  (HALF is at most 2.)
  __host__ __device__ static __forceinline__ TileLoad x_load(const TileOperands& op, int s, int first, int n_stages) {
    return {s < n_stages ? op.x_bytes : 0u, 128u * (unsigned)(first + s)};
  }
  __host__ __device__ static __forceinline__ TileLoad w_load(const TileOperands& op, int nb, int t, int first, int n_stages) {
    const int part = nb < HALF ? 0 : 1;
    return {t < 2 * n_stages ? op.w_bytes[part] : 0u,
            (nb - part * HALF) * op.w_step[part] + 1024u * (unsigned)(2 * first + t)};
  }

#ifdef __HIP_DEVICE_COMPILE__
  template <int N>
  __device__ static __forceinline__ void wait_vmcnt() {
    constexpr int n = N < 63 ? N : 63;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
    asm volatile("" ::: "memory");
  }
  __device__ static __forceinline__ void barrier() {  // (__syncthreads would wait for every load in flight)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  __device__ static __forceinline__ void mfma(f32x4& c, const bf16x8& a, const bf16x8& b) {
    if constexpr (ONE_WAVE) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  }
  // A block of sums where arithmetic can use it (from the accumulation registers one block at a time: the compiler would
  // move all of them at once, to registers that are not there).
  __device__ static __forceinline__ f32x4 sums(const f32x4& c) {
    if constexpr (!ONE_WAVE) return c;
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float f;
      asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(f) : "a"(c[e]));
      v[e] = f;
    }
    return v;
  }
  // The row of the tile whose chunk lane `lane` of wave `wave` brings with its load j, and that chunk's bytes behind the
  // row's begin in a stage.
  __device__ static __forceinline__ int row_of(int wave, int j, int lane) { return 8 * (wave + 4 * j) + lane / 8; }
  __device__ static __forceinline__ unsigned chunk_of(int lane) { return 16u * ((lane % 8) ^ (lane / 8)); }

  // acc[mb][nb][i] = sum over stages first .. first + n_stages - 1 of 64 k: row 16 mb + lane % 16 of x, row 16 nb + 4 (lane /
  // 16) + i of the wave's rows of the matrix.  ring: NST stages of LDS; xo: byte offsets of the lane's chunks (row_of,
  // chunk_of) at k 0; wave: 0 .. 3.  n_loop >= n_stages: the same for every wave of the workgroup, for they share the
  // barriers; what lies behind n_stages is zeros.
  __device__ static __forceinline__ void run(bf16_t* ring, const TileOperands& op, const unsigned (&xo)[XL], int wave,
                                             int lane, int first, int n_stages, int n_loop, f32x4 (&acc)[MB][NB]) {
    bf16x8 wr[WS][NB], b[RB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto load_x = [&](int s, int slot, int j) {
      const TileLoad load = x_load(op, s, first, n_stages);
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)op.x, 0, load.bytes, 0x20000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(ring + slot * STAGE + (wave + 4 * j) * 512),
                                               16, xo[j], load.at, 0, 0);
    };
    const unsigned wo = lane * 16;
    auto load_w = [&](int t, int set, int nb) {
      const TileLoad load = w_load(op, nb, t, first, n_stages);
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)op.w[nb < HALF ? 0 : 1], 0, load.bytes, 0x20000);
      wr[set][nb] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, wo, load.at, 0));
    };
    const int r16 = lane & 15, g = lane >> 4, row8 = r16 % 8;
    int off[2];  // this lane's place in a block of 16 rows, for the first and the second 32 k of a stage
#pragma unroll
    for (int h = 0; h < 2; ++h) off[h] = (r16 / 8) * 512 + row8 * 64 + ((4 * h + g) ^ row8) * 8;
    auto read_x = [&](const bf16_t* st, int h, int m) { b[m % RB] = *(const bf16x8*)(st + off[h] + m * 1024); };

#pragma unroll
    for (int s = 0; s < LA; ++s)
#pragma unroll
      for (int j = 0; j < XL; ++j) load_x(s, s, j);
    // the count below is of loads behind these: all of x before the first of the matrix
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < WS - 1; ++t)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) load_w(t, t, nb);
    wait_vmcnt<(LA - 2) * XL + (WS - 1) * NB>();  // stages 0 and 1 of this wave have landed, and behind the barrier everyone's
    barrier();
    int slot = 0;
    const bf16_t* st = ring;
#pragma unroll
    for (int m = 0; m < AHEAD; ++m) read_x(st, 0, m);
    for (int s0 = 0; s0 < n_loop; s0 += U) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int s = s0 + u;
        const int in = slot + LA >= NST ? slot + LA - NST : slot + LA, next = slot + 1 == NST ? 0 : slot + 1;
        const bf16_t* nst = ring + next * STAGE;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int t = 2 * u + h;
#pragma unroll
          for (int m = 0; m < MB; ++m) {
            if (h == 1 && m == MB - AHEAD) {
              // this wave's part of stage s + 1 has landed: it was asked for LA - 1 stages ago, and since then at least the
              // loads of LA - 2 whole stages, this stage's of x and its first of the matrix
              wait_vmcnt<(LA - 1) * (XL + 2 * NB) - NB>();
              barrier();
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
              mfma(acc[m][nb], wr[t][nb], b[m % RB]);
              __builtin_amdgcn_sched_barrier(0);
              if (nb == 0) {
                const int q = m + AHEAD;
                if (q < MB) read_x(st, h, q);
                else if (h == 0) read_x(st, 1, q - MB);
                else read_x(nst, 0, q - MB);
                __builtin_amdgcn_sched_barrier(0);
              }
              if (nb == NB / 2 && h == 0 && m < XL) {
                load_x(s + LA, in, m);
                __builtin_amdgcn_sched_barrier(0);
              }
              if (nb == NB - 1) {
#pragma unroll
                for (int n = 0; n < NB; ++n)
                  if ((n * MB + MB / 2) / NB == m) load_w(2 * s + h + WS - 1, (t + WS - 1) % WS, n);
                __builtin_amdgcn_sched_barrier(0);
              }
            }
          }
        }
        slot = next;
        st = nst;
      }
    }
    // loads past the end have landed before the LDS is given up, and the last sums are there to be read (the compiler does
    // not know how long an instruction in assembly takes)
    wait_vmcnt<0>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
#endif
};
