// True 32-bit matrix product: y[m][n] = sum_k x[m][k] * W[n][k], W row-major [N][K].
//
// Every output is ONE fused multiply-add chain over k = 0..K-1 starting from 0.0f, the
// order of the reference's scalar definition (src/kernels.cpp:236-244).  The tiling only
// decides which outputs share a pass over k (64x64 outputs per workgroup, 4x4 per thread,
// k staged through LDS 16 at a time); it never splits K, so a row's bits do not depend on
// the number of rows.  bfloat16 weights are widened exactly (src/kernels.cpp:77-81).
#include "common.h"
#include "api.h"

#define F32_BM 64
#define F32_BN 64
#define F32_BK 16

template <typename WT>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ x, const WT* __restrict__ w,
                                                       float* __restrict__ y, int M, int N, int K, int ldx,
                                                       int ldy, int accumulate) {
  __shared__ float xs[F32_BK][F32_BM + 4];
  __shared__ float ws[F32_BK][F32_BN + 4];
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const int m0 = blockIdx.y * F32_BM, n0 = blockIdx.x * F32_BN;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.0f;

  const int lr = tid >> 2;         // 0..63: row of the tile this thread loads
  const int lk = (tid & 3) * 4;    // 0,4,8,12: first of its four k
  for (int k0 = 0; k0 < K; k0 += F32_BK) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k = k0 + lk + q;
      const int m = m0 + lr, n = n0 + lr;
      xs[lk + q][lr] = (m < M && k < K) ? x[(size_t)m * ldx + k] : 0.0f;
      float wv = 0.0f;
      if (n < N && k < K) {
        if constexpr (sizeof(WT) == 2) wv = bf16_to_f32(w[(size_t)n * K + k]);
        else wv = w[(size_t)n * K + k];
      }
      ws[lk + q][lr] = wv;
    }
    __syncthreads();
    const int kend = (K - k0) < F32_BK ? (K - k0) : F32_BK;
    for (int kk = 0; kk < kend; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = xs[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = ws[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      float* o = y + (size_t)m * ldy + n;
      *o = accumulate ? (*o + acc[i][j]) : acc[i][j];
    }
  }
}

// Prompt portions: the same chains in tiles of 128x128 outputs, 8x8 per thread (as 2x2 blocks of 4x4, 64 rows
// or columns apart, so that every LDS read is 16 bytes and free of bank conflicts), k staged through LDS 16 at a
// time in two buffers (the next stage's loads fly while this one is worked on; one barrier a stage).
// K a multiple of 16, rows 16-byte aligned.
#define F32T_BM 128
#define F32T_BN 128
#define F32T_BK 16
#define F32T_STR 132            // floats from k to k in LDS

template <typename WT>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(const float* __restrict__ x, const WT* __restrict__ w,
                                                            float* __restrict__ y, int M, int N, int K, int ldx,
                                                            int ldy, int accumulate) {
  __shared__ __attribute__((aligned(16))) float xs[2][F32T_BK][F32T_STR];
  __shared__ __attribute__((aligned(16))) float ws[2][F32T_BK][F32T_STR];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int m0 = blockIdx.y * F32T_BM, n0 = blockIdx.x * F32T_BN;
  // loads of a stage: x rows lm and lm + 64, elements 4*lq..; W row wr, elements 8*wh.. (rows past the end are
  // clamped: what they bring is never stored)
  const int lm = tid >> 2, lq = tid & 3, wr = tid >> 1, wh = tid & 1;
  const float* xp0 = x + (size_t)min(m0 + lm, M - 1) * ldx + 4 * lq;
  const float* xp1 = x + (size_t)min(m0 + lm + 64, M - 1) * ldx + 4 * lq;
  const WT* wp = w + (size_t)min(n0 + wr, N - 1) * K + 8 * wh;
  f32x4 xr0, xr1;
  u32x4 wq0, wq1;                                          // bfloat16: 8 elements in wq0; 32-bit: 4 and 4
  auto load_stage = [&](int k0) {
    xr0 = *reinterpret_cast<const f32x4*>(xp0 + k0);
    xr1 = *reinterpret_cast<const f32x4*>(xp1 + k0);
    wq0 = *reinterpret_cast<const u32x4*>(wp + k0);
    if constexpr (sizeof(WT) == 4) wq1 = *reinterpret_cast<const u32x4*>(wp + k0 + 4);
  };
  auto store_stage = [&](int b) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      xs[b][4 * lq + i][lm] = xr0[i];
      xs[b][4 * lq + i][lm + 64] = xr1[i];
    }
    if constexpr (sizeof(WT) == 2) {                       // bfloat16 -> 32-bit: the bits, shifted (exact)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ws[b][8 * wh + 2 * i][wr] = __uint_as_float(wq0[i] << 16);
        ws[b][8 * wh + 2 * i + 1][wr] = __uint_as_float(wq0[i] & 0xffff0000u);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ws[b][8 * wh + i][wr] = __uint_as_float(wq0[i]);
        ws[b][8 * wh + 4 + i][wr] = __uint_as_float(wq1[i]);
      }
    }
  };
  float acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = 0.0f;
  load_stage(0);
  store_stage(0);
  __syncthreads();
  int b = 0;
  for (int k0 = 0; k0 < K; k0 += F32T_BK) {
    const bool more = k0 + F32T_BK < K;
    if (more) load_stage(k0 + F32T_BK);
#pragma unroll
    for (int kk = 0; kk < F32T_BK; ++kk) {
      const f32x4 a0 = *reinterpret_cast<const f32x4*>(&xs[b][kk][4 * ty]);
      const f32x4 a1 = *reinterpret_cast<const f32x4*>(&xs[b][kk][64 + 4 * ty]);
      const f32x4 b0 = *reinterpret_cast<const f32x4*>(&ws[b][kk][4 * tx]);
      const f32x4 b1 = *reinterpret_cast<const f32x4*>(&ws[b][kk][64 + 4 * tx]);
      const float av[8] = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
      const float bv[8] = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = fmaf(av[i], bv[j], acc[i][j]);
    }
    if (more) store_stage(b ^ 1);
    __syncthreads();
    b ^= 1;
  }
  const bool vec = (ldy & 3) == 0 && ((uintptr_t)y & 15) == 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int m = m0 + (i < 4 ? 4 * ty + i : 64 + 4 * ty + i - 4);
    if (m >= M) continue;
#pragma unroll
    for (int jh = 0; jh < 2; ++jh) {
      const int n = n0 + 64 * jh + 4 * tx;
      float* o = y + (size_t)m * ldy + n;
      if (vec && n + 3 < N) {
        f32x4 v = {acc[i][4 * jh], acc[i][4 * jh + 1], acc[i][4 * jh + 2], acc[i][4 * jh + 3]};
        if (accumulate) {
          const f32x4 old = *reinterpret_cast<const f32x4*>(o);
          v = (f32x4){old[0] + v[0], old[1] + v[1], old[2] + v[2], old[3] + v[3]};
        }
        *reinterpret_cast<f32x4*>(o) = v;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (n + j < N) o[j] = accumulate ? (o[j] + acc[i][4 * jh + j]) : acc[i][4 * jh + j];
      }
    }
  }
}

// Up to 64 rows (decoded tokens): the same chains, one per thread and block of 16 rows.  A workgroup owns 16 columns and all rows,
// thread (m, n) the output of row m and column 16 * blockIdx.x + n; its 256 threads together bring 256 elements
// of k of the 16 rows of W and of the rows of x into LDS at a time (16-byte loads; the next stage's loads fly
// while this one is worked on), widened to 32-bit there, and every thread then walks the stage in k order with
// one 16-byte read of its row of W and one of its row of x per four multiply-adds.  Few columns a workgroup,
// so that a product with few outputs still has loads in flight from many compute units.
// K a multiple of 8 (of 4 for 32-bit weights), rows 16-byte aligned.
#define F32R_NB 16

// MR blocks of 16 rows (up to 64 rows): thread (m, n) then runs the chains of rows m, m + 16, ... of its column,
// and a stage is 128 elements of k instead of 256 (the rows of x take LDS).
template <typename WT, int MR>
__global__ __launch_bounds__(256) void gemm_f32_rows_kernel(const float* __restrict__ x, const WT* __restrict__ w,
                                                            float* __restrict__ y, int M, int N, int K, int ldx,
                                                            int ldy, int accumulate) {
  constexpr int F32R_KB = MR == 1 ? 256 : 128;            // elements of k a stage
  constexpr int F32R_STRIDE = F32R_KB + 4;                 // floats from row to row in LDS: 16-byte reads of 16 rows hit 64 different banks
  constexpr int WC = sizeof(WT) == 2 ? 8 : 4;             // elements of W in a 16-byte chunk
  constexpr int WPR = F32R_KB / WC;                        // chunks in a stage's row of W
  constexpr int WJ = F32R_NB * WPR / 256;                  // chunks of W a thread and stage
  constexpr int XJ = 16 * MR * (F32R_KB / 4) / 256;        // chunks of x a thread and stage (16 * MR rows)
  extern __shared__ __attribute__((aligned(16))) float rows_lds[];   // [2][W: 16 rows | x: 16 rows] of F32R_STRIDE
  const int tid = threadIdx.x, n = tid & 15, m = tid >> 4;
  const int n0 = blockIdx.x * F32R_NB;
  // Two stages' loads are in flight while one is worked on: register sets A and B take the even and the odd stages
  // in turn.  Every load is unconditional and inside the operands (rows past N or M and k past K are clamped: what
  // they bring is never used), so that a wait for one set's loads need not be a wait for the other's.
  u32x4 wa[WJ], wb[WJ];
  f32x4 xa[XJ], xb[XJ];
  auto load_stage = [&](int k0, u32x4 (&wreg)[WJ], f32x4 (&xreg)[XJ]) {
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
      const int c = tid + 256 * j, row = min(n0 + c / WPR, N - 1), k = min(k0 + (c % WPR) * WC, K - WC);
      wreg[j] = *reinterpret_cast<const u32x4*>(w + (size_t)row * K + k);
    }
#pragma unroll
    for (int j = 0; j < XJ; ++j) {
      const int c = tid + 256 * j, row = min(c / (F32R_KB / 4), M - 1), k = min(k0 + (c % (F32R_KB / 4)) * 4, K - 4);
      xreg[j] = *reinterpret_cast<const f32x4*>(x + (size_t)row * ldx + k);
    }
  };
  auto store_stage = [&](float* buf, const u32x4 (&wreg)[WJ], const f32x4 (&xreg)[XJ]) {
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
      const int c = tid + 256 * j, row = c / WPR, kk = (c % WPR) * WC;
      float* dst = buf + row * F32R_STRIDE + kk;
      if constexpr (sizeof(WT) == 2) {                     // bfloat16 -> 32-bit: the bits, shifted (exact)
        *reinterpret_cast<u32x4*>(dst) = (u32x4){wreg[j][0] << 16, wreg[j][0] & 0xffff0000u, wreg[j][1] << 16, wreg[j][1] & 0xffff0000u};
        *reinterpret_cast<u32x4*>(dst + 4) = (u32x4){wreg[j][2] << 16, wreg[j][2] & 0xffff0000u, wreg[j][3] << 16, wreg[j][3] & 0xffff0000u};
      } else {
        *reinterpret_cast<u32x4*>(dst) = wreg[j];
      }
    }
#pragma unroll
    for (int j = 0; j < XJ; ++j) {
      const int c = tid + 256 * j, row = c / (F32R_KB / 4), kk = (c % (F32R_KB / 4)) * 4;
      *reinterpret_cast<f32x4*>(buf + (F32R_NB + row) * F32R_STRIDE + kk) = xreg[j];
    }
  };
  constexpr int BUF = (1 + MR) * 16 * F32R_STRIDE;         // floats of one buffer
  float acc = 0.0f;
  float accs[MR];                                          // (MR > 1)
#pragma unroll
  for (int r = 0; r < MR; ++r) accs[r] = 0.0f;
  auto work = [&](const float* buf, int k0) {              // the stage's steps of every chain, k ascending
    const int kend = (K - k0) < F32R_KB ? (K - k0) : F32R_KB;
    if (m >= M || kend <= 0) return;
    const float* wr = buf + n * F32R_STRIDE;
    const float* xr = buf + (F32R_NB + m) * F32R_STRIDE;
    if constexpr (MR > 1) {
#pragma unroll 4
      for (int kk = 0; kk < kend; kk += 4) {
        const f32x4 wv = *reinterpret_cast<const f32x4*>(wr + kk);
#pragma unroll
        for (int r = 0; r < MR; ++r) {
          const f32x4 xv = *reinterpret_cast<const f32x4*>(xr + 16 * r * F32R_STRIDE + kk);   // (rows past M: finite, never stored)
          accs[r] = fmaf(xv[0], wv[0], accs[r]);
          accs[r] = fmaf(xv[1], wv[1], accs[r]);
          accs[r] = fmaf(xv[2], wv[2], accs[r]);
          accs[r] = fmaf(xv[3], wv[3], accs[r]);
        }
      }
      return;
    }
    if (kend == F32R_KB) {
      // a whole stage: blocks of 32 steps, the operands of the next block read from LDS while this block's steps
      // run (the wave has little company on its SIMD: what hides its read latency is its own chain)
      constexpr int BLK = 8, NBLK = F32R_KB / 4 / BLK;
      f32x4 wv[2][BLK], xv[2][BLK];
#pragma unroll
      for (int i = 0; i < BLK; ++i) {
        wv[0][i] = *reinterpret_cast<const f32x4*>(wr + 4 * i);
        xv[0][i] = *reinterpret_cast<const f32x4*>(xr + 4 * i);
      }
#pragma unroll
      for (int blk = 0; blk < NBLK; ++blk) {
        if (blk + 1 < NBLK) {
#pragma unroll
          for (int i = 0; i < BLK; ++i) {
            wv[(blk + 1) & 1][i] = *reinterpret_cast<const f32x4*>(wr + 4 * (BLK * (blk + 1) + i));
            xv[(blk + 1) & 1][i] = *reinterpret_cast<const f32x4*>(xr + 4 * (BLK * (blk + 1) + i));
          }
        }
#pragma unroll
        for (int i = 0; i < BLK; ++i) {
          acc = fmaf(xv[blk & 1][i][0], wv[blk & 1][i][0], acc);
          acc = fmaf(xv[blk & 1][i][1], wv[blk & 1][i][1], acc);
          acc = fmaf(xv[blk & 1][i][2], wv[blk & 1][i][2], acc);
          acc = fmaf(xv[blk & 1][i][3], wv[blk & 1][i][3], acc);
        }
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 2 * BLK, 0);
#pragma unroll
      for (int blk = 0; blk + 1 < NBLK; ++blk) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * BLK, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4 * BLK, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x002, 4 * BLK, 0);
      return;
    }
#pragma unroll 8
    for (int kk = 0; kk < kend; kk += 4) {               // (unrolled: the reads of the steps ahead are under way)
      const f32x4 wv = *reinterpret_cast<const f32x4*>(wr + kk);
      const f32x4 xv = *reinterpret_cast<const f32x4*>(xr + kk);
      acc = fmaf(xv[0], wv[0], acc);
      acc = fmaf(xv[1], wv[1], acc);
      acc = fmaf(xv[2], wv[2], acc);
      acc = fmaf(xv[3], wv[3], acc);
    }
  };
  float* buf0 = rows_lds;
  float* buf1 = rows_lds + BUF;
  load_stage(0, wa, xa);
  load_stage(F32R_KB, wb, xb);
  store_stage(buf0, wa, xa);
  __syncthreads();
  for (int k0 = 0; k0 < K; k0 += 2 * F32R_KB) {
    load_stage(k0 + 2 * F32R_KB, wa, xa);
    work(buf0, k0);
    store_stage(buf1, wb, xb);
    __syncthreads();
    load_stage(k0 + 3 * F32R_KB, wb, xb);
    work(buf1, k0 + F32R_KB);
    store_stage(buf0, wa, xa);
    __syncthreads();
  }
  if (n0 + n >= N) return;
#pragma unroll
  for (int r = 0; r < MR; ++r) {
    const int mr = m + 16 * r;
    if (mr >= M) continue;
    float* o = y + (size_t)mr * ldy + n0 + n;
    const float v = MR == 1 ? acc : accs[r];
    *o = accumulate ? (*o + v) : v;
  }
}

// ------------------------------------------------------------------------------ a wave a row, the row four elements a register

// Few rows of many columns (f32_by_chains): a wave is a row and 64 columns, lane l the chain of (row, column n0 + l); weights and
// rows travel from memory straight into an LDS ring (buffer loads with LDS as destination: 8 rows of W, 128 bytes each, or 4 rows of x, 256
// bytes each, an instruction; whole cache lines, the 16-byte chunks of a row of W permuted against bank conflicts; a ring of
// stages, waits by counting loads).  The weights stay packed there: a lane reads its column's 16-byte chunks and widens them in
// registers.  x[row][k] is the same number for every lane of the wave; read as such from LDS it costs what any read costs.  Here lane
// l reads the 16 bytes at element 4 * (l % 4) of a run of sixteen, so that a register holds four elements of the row,
// the same four in every quad of lanes, and the multiply-add picks its element with the quad permutation of its
// first operand (v_fmac_f32 with quad_perm [i,i,i,i]: the same fused multiply-add, the operand routed on the way
// in): sixteen elements a read instead of four.
// A workgroup is 64 columns and all rows (a chain wave a row, sharing the ring).  A block is 64 bytes of a row of W
// (four 16-byte chunks: 32 bfloat16 or 16 32-bit elements), a stage two blocks; the next block's operands are read
// from LDS while this block's chains run.  (A chain is bound by its own links: a multiply-add that waits for the one
// before it issues every 3.8 ns, and 5.3 ns with one other vector instruction a link, such as the widening of a
// bfloat16 weight, wherever that instruction stands.)
#define F32C_W (64 * 128)                                             // 64 rows of W, 128 bytes each
#define F32C_X (8 * 256)                                              // 8 rows of x, up to 64 elements each
#define F32C_STAGE (F32C_W + F32C_X)

template <int KB>
struct ChainBlock {
  f32x4 x[KB / 16];                                                   // register j of x[a]: element 16 a + 4 (lane % 4) + j of the block
  u32x4 w[4];
};

template <typename WT>
__device__ __forceinline__ void chain_read(ChainBlock<64 / (int)sizeof(WT)>& b, const unsigned char* stage, int half, int my, int swz,
                                           const unsigned char* xs) {
  constexpr int KB = 64 / (int)sizeof(WT);
#pragma unroll
  for (int a = 0; a < KB / 16; ++a) b.x[a] = *reinterpret_cast<const f32x4*>(xs + (half * KB + 16 * a) * 4);
#pragma unroll
  for (int j = 0; j < 4; ++j) b.w[j] = *reinterpret_cast<const u32x4*>(stage + my + (((4 * half + j) ^ swz) * 16));
}

// acc = fma(x of quad lane I, w, acc): v_fmac_f32 with its first operand routed through the quad permutation
// [I,I,I,I] (written out: the compiler keeps a move of its own in front of the multiply-add otherwise, which costs
// what the multiply-add costs).  The operand comes from an LDS read, never from a vector instruction just before
// (which would want two idle states in between).
template <int I>
__device__ __forceinline__ float fma_quad(float xq, float w, float acc) {
  static_assert(I >= 0 && I < 4, "a quad has four lanes");
  if constexpr (I == 0) asm("v_fmac_f32_dpp %0, %1, %2 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(xq), "v"(w));
  else if constexpr (I == 1) asm("v_fmac_f32_dpp %0, %1, %2 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(xq), "v"(w));
  else if constexpr (I == 2) asm("v_fmac_f32_dpp %0, %1, %2 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(xq), "v"(w));
  else asm("v_fmac_f32_dpp %0, %1, %2 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(xq), "v"(w));
  return acc;
}

// element k of the block: register k % 4 of x[k / 16], quad lane (k / 4) % 4
template <int K16>
__device__ __forceinline__ float chain_step(float acc, const f32x4& x, float w) {
  constexpr int I = (K16 >> 2) & 3, J = K16 & 3;
  return fma_quad<I>(x[J], w, acc);
}

// Element e of 16-byte chunk ``c`` as a 32-bit float (bfloat16: the bits, shifted: exact).
template <typename WT, int E>
__device__ __forceinline__ float chain_weight(const u32x4& c) {
  if constexpr (sizeof(WT) == 2) return __uint_as_float((E & 1) ? (c[E >> 1] & 0xffff0000u) : (c[E >> 1] << 16));
  else return __uint_as_float(c[E]);
}

// The block's chains.  A multiply-add that depends on the one before it can issue every other slot, and one whose
// weight was widened in the slot before it waits for that as well: so chunk j + 1 is widened between the multiply-adds
// of chunk j (``f`` comes in with the block's chunk 0 widened, and leaves with chunk 0 of the next block).
template <typename WT>
__device__ __forceinline__ float chain_run(float acc, const ChainBlock<64 / (int)sizeof(WT)>& b, const ChainBlock<64 / (int)sizeof(WT)>& nxt,
                                           float (&f)[16 / (int)sizeof(WT)]) {
  constexpr int EPC = 16 / (int)sizeof(WT);                           // elements a chunk
  float g[EPC];
#define BW_CHAIN_STEP(J, E, FROM, TO, SRC)                                                \
  TO[E] = chain_weight<WT, E>(SRC);                                                       \
  acc = chain_step<(EPC * J + E) & 15>(acc, b.x[(EPC * J + E) >> 4], FROM[E]);
#define BW_CHAIN_CHUNK(J, FROM, TO, SRC)                                                  \
  BW_CHAIN_STEP(J, 0, FROM, TO, SRC) BW_CHAIN_STEP(J, 1, FROM, TO, SRC) BW_CHAIN_STEP(J, 2, FROM, TO, SRC) BW_CHAIN_STEP(J, 3, FROM, TO, SRC) \
  if constexpr (EPC == 8) {                                                               \
    BW_CHAIN_STEP(J, (EPC == 8 ? 4 : 0), FROM, TO, SRC) BW_CHAIN_STEP(J, (EPC == 8 ? 5 : 1), FROM, TO, SRC)                                   \
    BW_CHAIN_STEP(J, (EPC == 8 ? 6 : 2), FROM, TO, SRC) BW_CHAIN_STEP(J, (EPC == 8 ? 7 : 3), FROM, TO, SRC)                                   \
  }
  BW_CHAIN_CHUNK(0, f, g, b.w[1])
  BW_CHAIN_CHUNK(1, g, f, b.w[2])
  BW_CHAIN_CHUNK(2, f, g, b.w[3])
  BW_CHAIN_CHUNK(3, g, f, nxt.w[0])
#undef BW_CHAIN_CHUNK
#undef BW_CHAIN_STEP
  return acc;
}

template <typename WT>
__device__ __forceinline__ void chain_first(const ChainBlock<64 / (int)sizeof(WT)>& b, float (&f)[16 / (int)sizeof(WT)]) {
  f[0] = chain_weight<WT, 0>(b.w[0]);
  f[1] = chain_weight<WT, 1>(b.w[0]);
  f[2] = chain_weight<WT, 2>(b.w[0]);
  f[3] = chain_weight<WT, 3>(b.w[0]);
  if constexpr (sizeof(WT) == 2) {
    f[4] = chain_weight<WT, 4>(b.w[0]);
    f[5] = chain_weight<WT, 5>(b.w[0]);
    f[6] = chain_weight<WT, 6>(b.w[0]);
    f[7] = chain_weight<WT, 7>(b.w[0]);
  }
}

// The loads are not the chain waves' business.  A buffer load with LDS as destination holds the wave that issues it
// for some hundred clocks (ten of them a stage were more than the stage's chains), so a workgroup has two waves more
// that do nothing else: they ask for the stages, wait for them and meet the chain waves at the stage's barrier.  A
// loader issues five loads a stage: the ten are the eight blocks of 8 rows of W and two blocks of 4 rows of x,
// dealt in turn (loads for rows the workgroup does not have go outside the descriptor: no traffic, zeros into a
// spare KB behind the ring, so that both loaders count alike).
#define F32C_LOADERS 2
#define F32C_LPL 5                                                    // loads a loader and stage

template <int STAGES>
__device__ __forceinline__ void chain_issue(unsigned char* lds, __amdgpu_buffer_rsrc_t rs_w, __amdgpu_buffer_rsrc_t rs_x, const int* voff,
                                            int loader, int step, int steps, int x_step) {
  typedef __attribute__((address_space(3))) void* lds_ptr;
  unsigned char* dst = lds + (step % STAGES) * F32C_STAGE;
  const bool real = step < steps;                                     // scalar
#pragma unroll
  for (int t = 0; t < F32C_LPL; ++t) {
    const int q = loader + F32C_LOADERS * t;                          // 0..7: W; 8, 9: x
    if (q < 8) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_w, (lds_ptr)(dst + q * 1024), 16, real ? voff[t] : 0x7ffffff0, step * 128, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_x, (lds_ptr)(dst + F32C_W + (q - 8) * 1024), 16, real ? voff[t] : 0x7ffffff0,
                                                  step * x_step, 0, 0);
  }
}

template <typename WT, int STAGES>
__global__ __launch_bounds__(64 * (8 + F32C_LOADERS)) void gemm_f32_chain_kernel(const float* __restrict__ x, const WT* __restrict__ w,
                                                                                 float* __restrict__ y, int M, int N, int K, int ldx,
                                                                                 int ldy, int accumulate) {
  constexpr int KB = 64 / (int)sizeof(WT);                            // elements of k a block
  extern __shared__ __attribute__((aligned(16))) unsigned char chain_lds[];   // [stages][W: 64 rows of 128 B | x: 8 rows of 256 B]
  const int wave = wave_index(), lane = threadIdx.x & 63, rw = (int)(blockDim.x >> 6) - F32C_LOADERS;
  const int n0 = blockIdx.x * 64;
  const int m0 = blockIdx.y * rw;                                     // the workgroup's first row
  const int steps = K / (2 * KB);
  if (wave >= rw) {
    // ---- a loader
    const int loader = wave - rw;
    const int w_rows = min(64, N - n0), x_rows = min(rw, M - m0);
    const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)n0 * K), 0,
                                                                          (int)((size_t)w_rows * K * sizeof(WT)), 0x00020000);
    const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)(x + (size_t)m0 * ldx), 0,
                                                                          (int)((((size_t)x_rows - 1) * ldx + K) * 4), 0x00020000);
    // W: lane l of a load fetches row l / 8 of its 8 rows, chunk (l % 8) ^ (row within 16 >> 1) of the row's 128 bytes;
    // x: lane l fetches row 4 (q - 8) + l / 16 of the workgroup's, chunk l % 16 of the stage's elements (with 32-bit
    // weights a stage is 32 elements: the chunks past them lie outside)
    int voff[F32C_LPL];
#pragma unroll
    for (int t = 0; t < F32C_LPL; ++t) {
      const int q = loader + F32C_LOADERS * t;
      if (q < 8) {
        const int r = 8 * q + (lane >> 3);
        voff[t] = (int)((r * K) * (int)sizeof(WT) + 16 * ((lane & 7) ^ ((r & 15) >> 1)));
      } else {
        const int xrow = 4 * (q - 8) + (lane >> 4), xchunk = lane & 15;
        voff[t] = (xrow < x_rows && 4 * xchunk < 2 * KB) ? (xrow * ldx + 4 * xchunk) * 4 : 0x7ffffff0;
      }
    }
#pragma unroll
    for (int st = 0; st < STAGES - 1; ++st) chain_issue<STAGES>(chain_lds, rs_w, rs_x, voff, loader, st, steps, 2 * KB * 4);
    for (int step = 0; step < steps; ++step) {
      // this stage and the next have landed (the next stage's first block is read during this one's second); behind
      // the barrier every chain wave is done with the stage before, which the new loads overwrite
      __builtin_amdgcn_s_waitcnt(vmcnt_only(F32C_LPL * (STAGES - 3)));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      chain_issue<STAGES>(chain_lds, rs_w, rs_x, voff, loader, step + STAGES - 1, steps, 2 * KB * 4);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));                        // the padding loads too, before the wave ends
    return;
  }
  // ---- a chain wave: row m0 + wave
  const int row = m0 + wave;
  // this lane's row of the tile: chunk j lies in slot j ^ (row within 16 >> 1); its four elements of the wave's row
  const int my = (lane >> 3) * 1024 + (lane & 7) * 128, swz = (lane & 15) >> 1;
  const int mine = F32C_W + wave * 256 + (lane & 3) * 16;
  ChainBlock<KB> even, odd;
  float f[16 / (int)sizeof(WT)];                                      // a chunk of W, widened
  float acc = 0.0f;
  for (int step = 0; step < steps; ++step) {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const unsigned char* stage = chain_lds + (step % STAGES) * F32C_STAGE;
    const unsigned char* next = chain_lds + ((step + 1) % STAGES) * F32C_STAGE;
    if (step == 0) {
      chain_read<WT>(even, stage, 0, my, swz, stage + mine);
      chain_first<WT>(even, f);
    }
    __builtin_amdgcn_sched_barrier(0);
    chain_read<WT>(odd, stage, 1, my, swz, stage + mine);
    __builtin_amdgcn_sched_barrier(0);
    acc = chain_run<WT>(acc, even, odd, f);
    __builtin_amdgcn_sched_barrier(0);
    chain_read<WT>(even, next, 0, my, swz, next + mine);              // (past the last stage: whatever the ring holds, unused)
    __builtin_amdgcn_sched_barrier(0);
    acc = chain_run<WT>(acc, odd, even, f);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  }
  const int n = n0 + lane;
  if (n >= N || row >= M) return;
  float* o = y + (size_t)row * ldy + n;
  *o = accumulate ? (*o + acc) : acc;
}

#define F32C_STAGES 7
#define F32C_MAX_ROWS 8
#define F32C_MIN_BLOCKS 256                                           // blocks of 64 columns

// Which products of up to eight rows and at least as many blocks of 64 columns as there are compute units go by chains and not on the
// matrix cores (gemm_f32_matrix.h).  A workgroup of chains is two to a compute unit, its loaders ask for little at a time and its waves
// start at once; a tile with 32-bit weights has a compute unit to itself, so columns cost a round of the chip for every 16,384 of them.
// Tiles / chains, us (K: 64, 256, 1024, 2048):
//   32-bit weights, 2 rows, 16,321 columns  3.9/3.3  6.2/5.6  12.6/13.0 29.4/30.5     28,000 columns  6.0/3.9  9.8/7.9  26.9/25.5 48.7/44.3
//                   4 rows, 24,000          6.0/4.0  9.6/7.9  25.5/24.0 46.8/42.3     8 rows, 65,000  11.5/7.2 18.5/15.5 43.6/42.8 99/105
//   bfloat16        2 rows, 24,000          4.4/3.8  6.8/6.5  14.9/15.1 24.2/23.6     4 rows, 100,000 10.7/9.7 17.3/16.7 42.6/42.2 91/91
// Of 1,350 products of two to eight rows (16,321 to 128,256 columns, K of 64 to 8192) the rule leaves 1.004 times the time of the better
// kernel, 1.11 times at most; tiles for all of them left 1.08 and 1.86.  One row: by chains whatever K (16,384 columns, K = 2048, bfloat16
// weights, 14.4 and 15.0 to 15.8 us; a head of 49,152 columns 36.6 and 37.4).
static bool f32_by_chains(int M, int N, int K, bool bf16) {
  const int blocks = (N + 63) / 64;
  if (M > F32C_MAX_ROWS || blocks < F32C_MIN_BLOCKS || K % (bf16 ? 64 : 32) != 0) return false;
  if (M == 1) return true;
  if (bf16) return M == 2 ? K <= 512 || (blocks >= 1024 && K <= 1536) : M <= 4 && K <= 128;
  if (K <= 256) return true;
  // (no whole stages of 64: the other way is tiles of 64 x 64, whatever the rows; 8 rows of 39,549 columns, K = 1824, 59 and 53 us, 65,000 82 and 88)
  if (K % 64 != 0 && K > 1024 && (blocks == 256 || (blocks >= 600 && blocks % 256 <= 230))) return true;
  if (M > 4) return blocks >= 600 && K <= 1024;
  // (more than 1,024 steps of k: where the tiles' last round is not a full one)
  return blocks > 256 && (K <= 1024 || (blocks % 256 >= 1 && blocks % 256 <= 230));
}

extern "C" int bw_gemm_f32_by_chains(int M, int N, int K, int w_is_bf16) { return f32_by_chains(M, N, K, w_is_bf16 != 0); }

template <typename WT>
static void launch_chain(const float* x, const WT* w, float* y, int M, int N, int K, int ldx, int ldy, int accumulate, hipStream_t s) {
  constexpr int lds_bytes = F32C_STAGES * F32C_STAGE + 1024;
  static_assert(F32C_LPL * (F32C_STAGES - 3) < 64, "the wait count has six bits");
  static_assert(F32C_LPL * F32C_LOADERS == 10, "eight loads of W and two of x a stage");
  static bool allowed = false;                       // 64 KB of dynamic LDS and more has to be asked for once
  if (!allowed) {
    (void)hipFuncSetAttribute((const void*)gemm_f32_chain_kernel<WT, F32C_STAGES>, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    allowed = true;
  }
  int rw = 1;
  while (rw < M) rw *= 2;                            // (1, 2, 4 or 8 chain waves)
  hipLaunchKernelGGL((gemm_f32_chain_kernel<WT, F32C_STAGES>), dim3((N + 63) / 64, 1), dim3(64 * (rw + F32C_LOADERS)), lds_bytes, s, x, w, y,
                     M, N, K, ldx, ldy, accumulate);
}

#include "gemm_f32_matrix.h"

// ------------------------------------------------------------------------------ which kernel a product gets

// Which tiles a prompt's product gets, rows x columns: clocks a step of k a round of the compute units, as measured with bfloat16
// weights (100 and 200 rows, K = 2048 and 8192: 15.8, 31 and 58 ns), times the rounds.  With 32-bit weights, which need no widening,
// every tile takes 1.02 to 1.06 times as long (their loads are twice as wide), so the same rule holds.
struct F32PromptTile {
  int rows, columns;
};

static F32PromptTile f32_prompt_tile(int M, int N) {
  auto cost = [&](int bm, int bn, int clocks) {
    return (long long)clocks * ((((long long)(M + bm - 1) / bm) * ((N + bn - 1) / bn) + 255) / 256);
  };
  const long long big = cost(128, 128, 137), one = cost(64, 64, 37), two = cost(128, 64, 73);
  if (one < big && one <= two) return {64, 64};
  if (two < big) return {128, 64};
  return {128, 128};
}

extern "C" int bw_gemm_f32_prompt_tile(int M, int N, int* rows, int* columns) {
  if (M <= 0 || N <= 0) return -2;
  const F32PromptTile t = f32_prompt_tile(M, N);
  *rows = t.rows;
  *columns = t.columns;
  return 0;
}

// (GATED: N counts the outputs; the tiles are chosen by the rows of the stacked weight)
template <typename WT, bool GATED = false>
static void launch_f32_prompt(const float* x, const WT* w, float* y, int M, int N, int K, int ldx, int ldy, int accumulate, hipStream_t s) {
  const F32PromptTile tile = f32_prompt_tile(M, GATED ? 2 * N : N);
  if (tile.rows == 64) {
    // more than two workgroups a compute unit: without loading waves three of them fit (450 rows, 6144 x 2048: 96 us against 117);
    // with no more than that their own loads cost the working waves more (2048 x 8192: 145 us against 133)
    const long long wgs = ((M + 63) / 64) * (long long)(((GATED ? 2 * N : N) + 63) / 64);
    if (wgs > 512) return launch_f32_tiles<WT, 4, 1, 1, 4, 32, 4, 0, GATED>(x, w, y, M, N, K, ldx, ldy, accumulate, s);
    return launch_f32_tiles<WT, 4, 1, 1, 4, 32, 4, 4, GATED>(x, w, y, M, N, K, ldx, ldy, accumulate, s);
  }
  if (tile.columns == 64) return launch_f32_tiles<WT, 8, 1, 1, 4, 32, 4, 2, GATED>(x, w, y, M, N, K, ldx, ldy, accumulate, s);
  launch_f32_tiles<WT, 8, 2, 1, 4, 32, 4, 2, GATED>(x, w, y, M, N, K, ldx, ldy, accumulate, s);
}

// Up to 64 rows, K a multiple of 64 (of 32 where the tiles of 64 x 64 take it); us with bfloat16 weights and K = 2048:
//   as strips while those of 32 columns are one workgroup a compute unit at most (8 rows of 6144 columns 10.9, as tiles 14.8; 32 rows
//   of 2048 columns 11.1 and 14.7; beyond that LDS bounds them: 32 rows of 6144 columns 20.6 and 14.9);
//   up to 16 rows as tiles of 16 x 64 (16384 columns 15.8; strips 20);
//   more rows as tiles of 32 x 32 (16384 columns 23, 6144 15 to 22), from 33 rows and 256 blocks of 64 columns on as tiles of 64 x 64
//   (64 rows of 16384 columns 41 and 37; of 6144 columns 22 and 36).
enum { F32_STRIPS, F32_TILES_16, F32_TILES_32, F32_TILES_64 };

static int f32_few_rows_kernel(int M, int N, int K) {
  if (K % 64 != 0) return F32_TILES_64;
  if ((M + 15) / 16 * ((long long)(N + 31) / 32) <= 256) return F32_STRIPS;
  if (M <= 16) return F32_TILES_16;
  return M > 32 && (N + 63) / 64 >= 256 ? F32_TILES_64 : F32_TILES_32;
}

template <typename WT, bool GATED = false>
static void launch_f32_few_rows(const float* x, const WT* w, float* y, int M, int N, int K, int ldx, int ldy, int accumulate, hipStream_t s) {
  switch (f32_few_rows_kernel(M, GATED ? 2 * N : N, K)) {
    case F32_STRIPS: if constexpr (!GATED) return launch_f32_strips<WT, 2, 9>(x, w, y, M, N, K, ldx, ldy, accumulate, s);
    case F32_TILES_16: return launch_f32_tiles<WT, 1, 1, 1, 4, 64, sizeof(WT) == 2 ? 6 : 5, 2, GATED>(x, w, y, M, N, K, ldx, ldy, accumulate, s);
    case F32_TILES_32: return launch_f32_tiles<WT, 1, 1, 2, 2, 64, 4, 0, GATED>(x, w, y, M, N, K, ldx, ldy, accumulate, s);
    default: return launch_f32_tiles<WT, 4, 1, 1, 4, 32, 4, 4, GATED>(x, w, y, M, N, K, ldx, ldy, accumulate, s);
  }
}

template <typename WT, int MR>
static void launch_rows_mr(const float* x, const WT* w, float* y, int M, int N, int K, int ldx, int ldy, int accumulate,
                           hipStream_t s) {
  constexpr int lds_bytes = 2 * (1 + MR) * 16 * ((MR == 1 ? 256 : 128) + 4) * (int)sizeof(float);
  static bool allowed = false;                       // more than 64 KB of dynamic LDS has to be asked for once
  if (!allowed) {
    (void)hipFuncSetAttribute((const void*)gemm_f32_rows_kernel<WT, MR>, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    allowed = true;
  }
  hipLaunchKernelGGL((gemm_f32_rows_kernel<WT, MR>), dim3((N + F32R_NB - 1) / F32R_NB), dim3(256), lds_bytes, s, x, w, y, M, N, K,
                     ldx, ldy, accumulate);
}

template <typename WT>
static void launch_rows(const float* x, const WT* w, float* y, int M, int N, int K, int ldx, int ldy, int accumulate,
                        hipStream_t s) {
  if (M <= 16) launch_rows_mr<WT, 1>(x, w, y, M, N, K, ldx, ldy, accumulate, s);
  else if (M <= 32) launch_rows_mr<WT, 2>(x, w, y, M, N, K, ldx, ldy, accumulate, s);
  else launch_rows_mr<WT, 4>(x, w, y, M, N, K, ldx, ldy, accumulate, s);
}

extern "C" int bw_gemm_f32(const float* x, const void* w, int w_is_bf16, float* y, int M, int N, int K, int ldx,
                           int ldy, int accumulate, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || ldx < K || ldy < N) return -2;
  dim3 grid((N + F32_BN - 1) / F32_BN, (M + F32_BM - 1) / F32_BM), block(256);
  hipStream_t s = (hipStream_t)stream;
  // which kernel runs depends on the shape alone, and both run the same chains
  const int wc = w_is_bf16 ? 8 : 4;
  // offsets within a tile's rows of x and columns of W must fit the buffer descriptors' 31 bits
  const bool vectors = ldx % 4 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0;
  const int tile_rows = M > 64 ? 128 : (M < 64 ? M : 64), tile_columns = M > 64 ? 128 : 64;
  const bool fits = vectors && (size_t)tile_rows * ldx * 4 < ((size_t)1 << 31) && (size_t)tile_columns * K * 4 < ((size_t)1 << 31);
  // up to eight rows, many columns, K in whole stages: a chain a lane, the row four elements a register, loader waves
  if (fits && f32_by_chains(M, N, K, w_is_bf16 != 0)) {
    if (w_is_bf16) launch_chain<bf16_t>(x, (const bf16_t*)w, y, M, N, K, ldx, ldy, accumulate, s);
    else launch_chain<float>(x, (const float*)w, y, M, N, K, ldx, ldy, accumulate, s);
    return BW_LAUNCH_CHECK();
  }
  // up to 64 rows, K in whole stages: the chains run on the matrix cores (K % 64 == 32: for so many outputs only that the chains of
  // the vector units, which take 16 rows by 16 columns a workgroup, are slower)
  if (fits && M <= 64 && (K % 64 == 0 || (K % 32 == 0 && (M > 16 || (N + 63) / 64 >= 256)))) {
    if (w_is_bf16) launch_f32_few_rows<bf16_t>(x, (const bf16_t*)w, y, M, N, K, ldx, ldy, accumulate, s);
    else launch_f32_few_rows<float>(x, (const float*)w, y, M, N, K, ldx, ldy, accumulate, s);
    return BW_LAUNCH_CHECK();
  }
  if (M <= 64 && K % wc == 0 && vectors) {
    if (w_is_bf16) launch_rows<bf16_t>(x, (const bf16_t*)w, y, M, N, K, ldx, ldy, accumulate, s);
    else launch_rows<float>(x, (const float*)w, y, M, N, K, ldx, ldy, accumulate, s);
    return BW_LAUNCH_CHECK();
  }
  // prompt portions, K in whole stages: tiles on the matrix cores (the same chains)
  if (fits && M > 64 && K % 32 == 0) {
    if (w_is_bf16) launch_f32_prompt<bf16_t>(x, (const bf16_t*)w, y, M, N, K, ldx, ldy, accumulate, s);
    else launch_f32_prompt<float>(x, (const float*)w, y, M, N, K, ldx, ldy, accumulate, s);
    return BW_LAUNCH_CHECK();
  }
  if (M > 64 && K % F32T_BK == 0 && vectors) {
    dim3 tgrid((N + F32T_BN - 1) / F32T_BN, (M + F32T_BM - 1) / F32T_BM);
    if (w_is_bf16)
      hipLaunchKernelGGL(gemm_f32_tile_kernel<bf16_t>, tgrid, block, 0, s, x, (const bf16_t*)w, y, M, N, K, ldx, ldy, accumulate);
    else
      hipLaunchKernelGGL(gemm_f32_tile_kernel<float>, tgrid, block, 0, s, x, (const float*)w, y, M, N, K, ldx, ldy, accumulate);
    return BW_LAUNCH_CHECK();
  }
  if (w_is_bf16)
    hipLaunchKernelGGL(gemm_f32_kernel<bf16_t>, grid, block, 0, s, x, (const bf16_t*)w, y, M, N, K, ldx, ldy, accumulate);
  else
    hipLaunchKernelGGL(gemm_f32_kernel<float>, grid, block, 0, s, x, (const float*)w, y, M, N, K, ldx, ldy, accumulate);
  return BW_LAUNCH_CHECK();
}

// Up to eight rows of more than 8,192 outputs: more than one gated tile for every compute unit, and the product as it goes without
// the epilogue can be so much faster that two kernels are.  Tiles with the epilogue / two kernels, us, outputs x K:
//   32-bit weights, one row   8200 x 64 6.1/5.5, x 1024 20.3/17.8, x 4096 68/51; 16384 x 512 15.1/15.8, x 1024 42/31; 50000 x 64 18.7/11.0
//                   8 rows    8200 x 64 6.5/6.0, x 256 9.6/10.2; 16384 x 256 11.0/11.4; 32768 x 512 36.6/30.0
//   bfloat16, one row         8200 x 512 9.0/8.9, x 1024 13.8/12.4, x 4096 43/29; 14336 x 1024 14.6/16.1, x 2048 23.8/23.7
// Of 804 such products this leaves 1.007 times the time of the better way (tiles for all 1.043; 1.69 times at most, and now 1.27).
// One row of 8,192 outputs, K = 2048: 16.3 us in tiles and 17.2; with 32-bit weights 30.0 and 32.3.
static bool f32_gated_apart(int M, int outputs, int K, bool bf16) {
  if (M > 8 || outputs <= 8192) return false;
  if (bf16) return M == 1 && K >= 1024 && (outputs < 11000 || (K >= 2048 && K <= 4096 && outputs < 16000));
  if (M <= 4) return K <= 2048 || (K <= 4096 && outputs < 10000);
  return K <= 64 || (K <= 256 && outputs >= 18000) || (K <= 1024 && outputs >= 24000);
}

// Whether the product goes in tiles with the activation in their epilogue.
static bool f32_gated_in_tiles(const float* x, const void* w, bool bf16, int M, int outputs, int K, int ldx) {
  const size_t limit = (size_t)0x7ff00000;             // (a tile's descriptor spans the whole weight)
  if (ldx % 4 != 0 || ((uintptr_t)x & 15) != 0 || ((uintptr_t)w & 15) != 0) return false;
  if ((size_t)(M < 128 ? M : 128) * ldx * 4 >= limit || (size_t)2 * outputs * K * (bf16 ? 2 : 4) >= limit) return false;
  if (M > 64) return K % 32 == 0;
  return K % 64 == 0 && !f32_gated_apart(M, outputs, K, bf16) && f32_few_rows_kernel(M, 2 * outputs, K) != F32_STRIPS;
}

extern "C" int bw_gemm_f32_swiglu_in_tiles(const float* x, const void* w, int w_is_bf16, int M, int outputs, int K, int ldx) {
  return M > 0 && outputs > 0 && K > 0 && ldx >= K && f32_gated_in_tiles(x, w, w_is_bf16 != 0, M, outputs, K, ldx);
}

// h = silu(x Wg^T) * (x Wu^T), w = [Wg; Wu] (outputs rows each).  Where the product goes in tiles its epilogue computes h; otherwise
// the sums go to gate_up and swiglu_f32_kernel behind it.  The same operations on the same sums.
extern "C" int bw_gemm_f32_swiglu(const float* x, const void* w, int w_is_bf16, float* gate_up, float* h, int M, int outputs, int K, int ldx,
                                  void* stream) {
  if (M <= 0 || outputs <= 0) return 0;
  if (K <= 0 || ldx < K) return -2;
  hipStream_t s = (hipStream_t)stream;
  if (!f32_gated_in_tiles(x, w, w_is_bf16 != 0, M, outputs, K, ldx)) {
    const int rc = bw_gemm_f32(x, w, w_is_bf16, gate_up, M, 2 * outputs, K, ldx, 2 * outputs, 0, stream);
    return rc != 0 ? rc : bw_swiglu_f32(gate_up, h, M, outputs, stream);
  }
  if (M > 64) {
    if (w_is_bf16) launch_f32_prompt<bf16_t, true>(x, (const bf16_t*)w, h, M, outputs, K, ldx, outputs, 0, s);
    else launch_f32_prompt<float, true>(x, (const float*)w, h, M, outputs, K, ldx, outputs, 0, s);
  } else {
    if (w_is_bf16) launch_f32_few_rows<bf16_t, true>(x, (const bf16_t*)w, h, M, outputs, K, ldx, outputs, 0, s);
    else launch_f32_few_rows<float, true>(x, (const float*)w, h, M, outputs, K, ldx, outputs, 0, s);
  }
  return BW_LAUNCH_CHECK();
}

// Whether bw_gemm_f32_qkv_rope takes the stacked product: up to 64 rows that go as strips, whole tiles of 16 pairs.
extern "C" int bw_gemm_f32_rope_in_strips(const float* x, const void* w, int w_is_bf16, int M, int all_heads, int head_dim, int K, int ldx) {
  const long long N = (long long)all_heads * head_dim;
  if (M <= 0 || M > 64 || all_heads <= 0 || head_dim <= 0 || head_dim % 32 || K <= 0 || K % 64 || ldx < K || N > (1 << 28)) return 0;
  const size_t limit = (size_t)1 << 31;                // (a tile's descriptors: 16 rows of x, a head's columns of W)
  if (ldx % 4 || (((uintptr_t)x | (uintptr_t)w) & 15) || (size_t)64 * ldx * 4 >= limit || (size_t)head_dim * K * 4 >= limit) return 0;
  return !f32_by_chains(M, (int)N, K, w_is_bf16 != 0) && f32_few_rows_kernel(M, (int)N, K) == F32_STRIPS;
}

// y = x W^T with q and k rotated and k and v in their page slots: the bits of bw_gemm_f32 followed by bw_rope_kvwrite on 32-bit
// caches, in one kernel; -7: not this shape (bw_gemm_f32_rope_in_strips).
extern "C" int bw_gemm_f32_qkv_rope(const float* x, const void* w, int w_is_bf16, float* y, int M, int K, int ldx, int ldy, const int32_t* positions,
                                    const int32_t* row_seq, const int32_t* block_table, int table_stride, const float* cos_table,
                                    const float* sin_table, float* k_cache, float* v_cache, int heads, int kv_heads, int head_dim, int page_size,
                                    int write_cache, void* stream) {
  if (M <= 0) return 0;
  const int all_heads = heads + 2 * kv_heads, N = all_heads * head_dim;
  if (page_size <= 0 || ldy < N || kv_heads <= 0 || heads <= 0) return -2;
  if (!bw_gemm_f32_rope_in_strips(x, w, w_is_bf16, M, all_heads, head_dim, K, ldx)) return -7;
  const F32RopeArgs ra{positions, row_seq, block_table, cos_table, sin_table, k_cache, v_cache,
                       heads, kv_heads, head_dim, page_size, page_size & (page_size - 1) ? -1 : __builtin_ctz((unsigned)page_size), table_stride, write_cache};
  hipStream_t s = (hipStream_t)stream;
  if (w_is_bf16) launch_f32_strips<bf16_t, 2, 9, true>(x, (const bf16_t*)w, y, M, N, K, ldx, ldy, 0, s, ra);
  else launch_f32_strips<float, 2, 9, true>(x, (const float*)w, y, M, N, K, ldx, ldy, 0, s, ra);
  return BW_LAUNCH_CHECK();
}
