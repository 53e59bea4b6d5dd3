// 32-bit matrix products on the matrix cores (included by gemm_f32.hip).
//
// v_mfma_f32_16x16x4_f32 computes D[i][j] = fma(A[i][3], B[3][j], fma(A[i][2], B[2][j], fma(A[i][1], B[1][j], fma(A[i][0], B[0][j],
// D[i][j])))): four steps of k one after the other, k ascending, each a multiply-add with a single rounding, denormal numbers,
// infinities and signed zeros included (held against chains of fmaf over seven kinds of operands, and against std::fma by the
// tests).  A chain of such instructions is therefore the scalar chain of the definition.  An instruction takes 13.7 ns (32 clocks)
// whether or not it waits for the one before it, 3.4 ns a step of k for 256 outputs, where the vector unit takes 3.8 ns a step of 64.
// While it runs, vector instructions do not, not even another wave's (2.3 ns each), and an LDS instruction of the same wave costs
// about 4 ns.  So what is left to save beside the matrix instructions are operand reads and the widening of bfloat16 weights.
//
// Operands: lane l holds row (of x; A) or column (of W; B) l % 16 and element 4 i + l / 16 of instruction i.
#pragma once

// ------------------------------------------------------------------------------ tiles

// Workgroups of WR x WC working waves, each with RB x CB blocks of 16 x 16 outputs, and LW waves that only load (none: every wave
// loads its share).  x and W (as it is in memory) travel straight into a ring of ST stages of KB steps of k; a lane reads its
// elements one at a time, and bfloat16 ones are widened in registers: RB matrix instructions for every shift.  (Sixteen rows' elements
// are in distinct ones of 64 banks, but two rows each share one of 32, and every such read is replayed once: SQ_LDS_BANK_CONFLICT is half
// of SQ_LDS_IDX_ACTIVE in all tiles.  In those of 128 x 128 that is under matrix instructions that are at work all the time; in those
// of 16 x 64, 8 rows of 16384 x 2048, LDS is at work for 8 of 17 us, half of that replays.)
// The row blocks are shared out evenly over the row tiles (450 rows are 29 blocks: four tiles of seven or eight, not three of eight
// and one of five), and a block without rows costs nothing.
// Against the kernels before it (one step of k an instruction: 16x16x1, 32x32x1 and 4x4x1), bfloat16 weights, us:
//   rows   16384 x 2048   6144 x 2048   2048 x 8192   2048 x 2048      (columns x K)
//    452    334 -> 247      119 -> 97     190 -> 134     54 -> 39
//   2048   1183 -> 997      440 -> 374    575 -> 481    150 -> 127       (138 to 143 TFLOP/s)
//     32     89 -> 23        45 -> 15
//     16     39 -> 17        23 -> 14
// Tried: W and x widened and put in the order of the operands by the loading waves, so that a working wave reads 16 bytes for four
// instructions (10 % slower: the LDS writes and shifts of the loading waves cost the SIMDs more); two waves a SIMD of half the rows (the
// same); stages of 64 for the tiles (10 % slower).
template <typename WT, int RB, int CB, int WR, int WC, int KB, int ST, int LW>
struct F32KShape {
  static constexpr int WAVES = WR * WC, ROWS = 16 * RB * WR, COLS = 16 * CB * WC;
  static constexpr int XROW = KB * 4, WROW = KB * (int)sizeof(WT);            // bytes of a stage's row of x and of W
  static constexpr int XBYTES = ROWS * XROW, STAGE = XBYTES + COLS * WROW;
  static constexpr int XL = XBYTES / 1024, WL = COLS * WROW / 1024;           // loads of 1 KB a stage
  static constexpr int LOADERS = LW > 0 ? LW : WAVES;                         // waves that load
  static constexpr int XW = XL / LOADERS, WW = WL / LOADERS, LPW = XW + WW;   // loads of one of them
  static constexpr int LDS = ST * STAGE;
  static constexpr int KG = KB / 8;                                           // instructions' worth of k in half a stage
  static_assert(XL % LOADERS == 0 && WL % LOADERS == 0, "every loading wave counts alike");
  static_assert(ST >= 4 && LPW * (ST - 2) < 64, "the wait count has six bits");
  static_assert(LDS <= BW_LDS_LIMIT, "the ring has to fit");
};

// Which 16-byte chunk of a row of BYTES lies in slot 0: sixteen rows' equal chunks (of bfloat16: halves of chunks) then lie in
// different ones of 64 banks.
template <int BYTES>
__device__ __forceinline__ int f32k_swizzle(int row) {
  if constexpr (BYTES == 64) return (row >> 2) & 3;
  else if constexpr (BYTES == 128) return (row >> 1) & 7;
  else return row & 15;
}

// (The device functions are for the device pass only: they pass buffer descriptors, a type that the host pass does not know.)
#if defined(__HIP_DEVICE_COMPILE__)
template <typename S>
__device__ __forceinline__ void f32k_issue(unsigned char* ring, __amdgpu_buffer_rsrc_t rs_x, __amdgpu_buffer_rsrc_t rs_w, const int* voff_x,
                                           const int* voff_w, int loader, int slot, int step, int steps) {
  typedef __attribute__((address_space(3))) void* lds_ptr;
  unsigned char* dst = ring + slot * S::STAGE;
  const bool real = step < steps;                                             // scalar (past K: outside the descriptors, zeros)
#pragma unroll
  for (int t = 0; t < S::XW; ++t)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_x, (lds_ptr)(dst + (loader + t * S::LOADERS) * 1024), 16, real ? voff_x[t] : 0x7ffffff0,
                                             step * S::XROW, 0, 0);
#pragma unroll
  for (int t = 0; t < S::WW; ++t)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_w, (lds_ptr)(dst + S::XBYTES + (loader + t * S::LOADERS) * 1024), 16,
                                             real ? voff_w[t] : 0x7ffffff0, step * S::WROW, 0, 0);
}

// The operands of half a stage.
template <typename S, int RBL, int CB>
struct F32KHalf {
  float x[RBL][S::KG];
  uint32_t w[CB][S::KG];
};

template <typename S, typename WT, int RBL, int CB, int HALF>
__device__ __forceinline__ void f32k_read(const unsigned char* stage, const int* xa, const int* wa, F32KHalf<S, RBL, CB>& h) {
#pragma unroll
  for (int i = 0; i < S::KG; ++i) {
    const int c = HALF * S::KG + i;
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      if constexpr (sizeof(WT) == 2) h.w[b][i] = *reinterpret_cast<const uint16_t*>(stage + wa[c >> 1] + 8 * (c & 1) + b * 16 * S::WROW);
      else h.w[b][i] = *reinterpret_cast<const uint32_t*>(stage + wa[c] + b * 16 * S::WROW);
    }
#pragma unroll
    for (int b = 0; b < RBL; ++b) h.x[b][i] = *reinterpret_cast<const float*>(stage + xa[c] + b * 16 * S::XROW);
  }
}

template <typename S, typename WT, int RBL, int CB>
__device__ __forceinline__ void f32k_run(const F32KHalf<S, RBL, CB>& h, f32x4 (&acc)[RBL][CB]) {
  float wv[CB][S::KG];                                                         // bfloat16 -> 32-bit: the bits, shifted (exact)
#pragma unroll
  for (int i = 0; i < S::KG; ++i)
#pragma unroll
    for (int b = 0; b < CB; ++b) wv[b][i] = __uint_as_float(sizeof(WT) == 2 ? h.w[b][i] << 16 : h.w[b][i]);
#pragma unroll
  for (int i = 0; i < S::KG; ++i)                                              // k ascending
#pragma unroll
    for (int b = 0; b < CB; ++b)
#pragma unroll
      for (int r = 0; r < RBL; ++r) acc[r][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(h.x[r][i], wv[b][i], acc[r][b], 0, 0, 0);
}

// The order of a run: a matrix instruction, then a share of the reads of the run to come.
template <int MFMAS, int READS, int AT = 0>
__device__ __forceinline__ void f32_order() {
  if constexpr (AT < MFMAS) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    constexpr int n = (READS * (AT + 1)) / MFMAS - (READS * AT) / MFMAS;
    if constexpr (n > 0) __builtin_amdgcn_sched_group_barrier(0x100, n, 0);
    f32_order<MFMAS, READS, AT + 1>();
  }
}

// register i, lane l: row 4 * (l / 16) + i of the block, column l % 16
template <int RBL, int CB>
__device__ __forceinline__ void f32_write(const f32x4 (&acc)[RBL][CB], float* y, int ldy, int m0, int n0, int M, int N, int accumulate) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < RBL; ++r)
#pragma unroll
    for (int b = 0; b < CB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + 16 * r + 4 * (lane >> 4) + i, n = n0 + 16 * b + (lane & 15);
        if (m < M && n < N) {
          float* o = y + (size_t)m * ldy + n;
          *o = accumulate ? (*o + acc[r][b][i]) : acc[r][b][i];
        }
      }
}

// Gated: gate and up of an output meet in one wave (f32k_weight_row): as its two column blocks, or as the halves of one, whose lanes
// then exchange half of their rows.  h = g * (1/(1+exp(-g))) * u, as swiglu_f32_kernel has it.
__device__ __forceinline__ float f32_swiglu(float g, float u) { return g * (1.0f / (1.0f + bw_expf(-g))) * u; }

template <int RBL, int CB>
__device__ __forceinline__ void f32_write_gated(const f32x4 (&acc)[RBL][CB], float* h, int ldh, int m0, int n0, int M, int N) {
  const int lane = threadIdx.x & 63;
  if constexpr (CB == 2) {
    const int n = n0 + (lane & 15);
#pragma unroll
    for (int r = 0; r < RBL; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + 16 * r + 4 * (lane >> 4) + i;
        const float v = f32_swiglu(acc[r][0][i], acc[r][1][i]);
        if (m < M && n < N) h[(size_t)m * ldh + n] = v;
      }
  } else {
    const bool up = lane & 8;
    const int n = n0 + (lane & 7);
#pragma unroll
    for (int r = 0; r < RBL; ++r)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float got = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(up ? acc[r][0][i] : acc[r][0][2 + i]), 0x128, 0xf, 0xf, true));
        const int m = m0 + 16 * r + 4 * (lane >> 4) + i + (up ? 2 : 0);
        const float v = f32_swiglu(up ? got : acc[r][0][i], up ? acc[r][0][2 + i] : got);
        if (m < M && n < N) h[(size_t)m * ldh + n] = v;
      }
  }
}

template <typename S, typename WT, int RBL, int CB, int ST, int LW, bool GATED>
__device__ __forceinline__ void f32k_tile(unsigned char* ring, __amdgpu_buffer_rsrc_t rs_x, __amdgpu_buffer_rsrc_t rs_w, const int* voff_x,
                                          const int* voff_w, int loader, const int* xa, const int* wa, int steps, float* y, int ldy, int m0, int n0,
                                          int M, int N, int accumulate) {
  constexpr int R = RBL > 0 ? RBL : 1;                                         // (RBL = 0: a wave without rows, which loads its share)
  f32x4 acc[R][CB];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int b = 0; b < CB; ++b) acc[r][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
  F32KHalf<S, R, CB> h0, h1;
  if constexpr (RBL > 0) f32k_read<S, WT, R, CB, 0>(ring, xa, wa, h0);
  for (int base = 0; base < steps; base += ST) {
#pragma unroll
    for (int u = 0; u < ST; ++u) {
      const int step = base + u;
      if (step >= steps) break;                                                // scalar
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (RBL > 0) {
        f32k_read<S, WT, R, CB, 1>(ring + u * S::STAGE, xa, wa, h1);
        f32k_run<S, WT, R, CB>(h0, acc);
        f32_order<R * CB * S::KG, (R + CB) * S::KG>();
      }
      __builtin_amdgcn_sched_barrier(0);
      // a loading wave's share of the next stage has landed (past K: zeros, unused); behind the barrier everyone's has, and
      // everyone is done with the stage before this one, whose place the stage asked for next takes
      if constexpr (LW == 0) __builtin_amdgcn_s_waitcnt(vmcnt_only(S::LPW * (ST - 3)));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if constexpr (LW == 0) f32k_issue<S>(ring, rs_x, rs_w, voff_x, voff_w, loader, (u + ST - 1) % ST, step + ST - 1, steps);
      if constexpr (RBL > 0) {
        f32k_read<S, WT, R, CB, 0>(ring + (u + 1) % ST * S::STAGE, xa, wa, h0);
        f32k_run<S, WT, R, CB>(h1, acc);
        f32_order<R * CB * S::KG, (R + CB) * S::KG>();
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (LW == 0) __builtin_amdgcn_s_waitcnt(vmcnt_only(0));             // the padding loads too, before the waves end
  if constexpr (RBL > 0) {
    if constexpr (GATED) f32_write_gated<R, CB>(acc, y, ldy, m0, n0, M, N);
    else f32_write<R, CB>(acc, y, ldy, m0, n0, M, N, accumulate);
  }
}

// Which row of the stacked weight [gate; up] is a gated tile's column c: blocks of 16 in turn, or halves of a block of 16.
// (Past the last output: the last one's again.)
template <int CB>
__device__ __forceinline__ int f32k_weight_row(int c, int first, int outputs) {
  constexpr int H = 8 * CB;
  const int row = min(first + c / (2 * H) * H + c % H, outputs - 1);
  return c & H ? row + outputs : row;
}
#endif

// GATED: w is [gate; up], N counts the outputs, and y takes silu(gate) * up.  8 rows, 8192 outputs of K = 2048, bfloat16 weights: the sums to
// memory and a kernel behind them 18.1 us, so 16.0; 64 rows 40.2 and 37.9, 2048 rows 1035 and 1025; 4104 outputs of K = 512, 8 rows,
// 10.0 and 6.2.
template <typename WT, int RB, int CB, int WR, int WC, int KB, int ST, int LW, bool GATED>
__global__ __launch_bounds__(64 * (WR * WC + LW)) void gemm_f32_tiles_kernel(const float* __restrict__ x, const WT* __restrict__ w,
                                                                            float* __restrict__ y, int M, int N, int K, int ldx, int ldy,
                                                                            int accumulate, int row_tiles) {
#if defined(__HIP_DEVICE_COMPILE__)
  using S = F32KShape<WT, RB, CB, WR, WC, KB, ST, LW>;
  extern __shared__ __attribute__((aligned(16))) unsigned char f32k_ring[];
  const int wave = wave_index(), lane = threadIdx.x & 63;
  // the row tiles of a column tile run one after the other on one die: its weights come from memory once (where the workgroups divide
  // by the dies; other grids are dealt as they come, and a column tile's weights go to several dies)
  int bid = blockIdx.x;
  if (gridDim.x % 8 == 0) bid = (bid % 8) * (gridDim.x / 8) + bid / 8;
  const int blocks = (M + 15) / 16, tile = bid % row_tiles;
  const int first = (int)((long long)blocks * tile / row_tiles), last = (int)((long long)blocks * (tile + 1) / row_tiles);
  const int m0 = 16 * first, n0 = (bid / row_tiles) * (GATED ? S::COLS / 2 : S::COLS);
  const int x_rows = min(16 * (last - first), M - m0), w_rows = GATED ? 2 * N : min(S::COLS, N - n0);
  const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(x + (size_t)m0 * ldx), 0, (int)((((size_t)x_rows - 1) * ldx + K) * sizeof(float)), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_w =
      __builtin_amdgcn_make_buffer_rsrc((void*)(w + (GATED ? 0 : (size_t)n0 * K)), 0, (int)((size_t)w_rows * K * sizeof(WT)), 0x00020000);
  // loads: 1 KB an instruction, whole rows of a stage, lane l the 16 bytes at 16 l; which chunk of its row a lane asks for is permuted
  // (rows past the operand are clamped to its last: their outputs are never stored)
  const int loader = LW > 0 ? wave - S::WAVES : wave;                          // (negative: a wave that does not load)
  int voff_x[S::XW], voff_w[S::WW];
#pragma unroll
  for (int t = 0; t < S::XW; ++t) {
    constexpr int CH = S::XROW / 16;                                           // chunks a row
    const int row = (loader + t * S::LOADERS) * (64 / CH) + lane / CH, chunk = (lane % CH) ^ f32k_swizzle<S::XROW>(row);
    voff_x[t] = (min(row, x_rows - 1) * ldx + 4 * chunk) * 4;
  }
#pragma unroll
  for (int t = 0; t < S::WW; ++t) {
    constexpr int CH = S::WROW / 16;
    const int row = (loader + t * S::LOADERS) * (64 / CH) + lane / CH, chunk = (lane % CH) ^ f32k_swizzle<S::WROW>(row);
    int w_row = min(row, w_rows - 1);
    if constexpr (GATED) w_row = f32k_weight_row<CB>(row, n0, N);
    voff_w[t] = w_row * K * (int)sizeof(WT) + 16 * chunk;
  }
  const int steps = K / KB;
  if (LW == 0 || wave >= S::WAVES) {
#pragma unroll
    for (int st = 0; st < ST - 1; ++st) f32k_issue<S>(f32k_ring, rs_x, rs_w, voff_x, voff_w, loader, st, st, steps);
    __builtin_amdgcn_s_waitcnt(vmcnt_only(S::LPW * (ST - 2)));                 // this wave's share of stage 0 has landed
  }
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if (LW > 0 && wave >= S::WAVES) {
    int slot = ST - 1;
    for (int step = 0; step < steps; ++step) {
      __builtin_amdgcn_s_waitcnt(vmcnt_only(S::LPW * (ST - 3)));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      f32k_issue<S>(f32k_ring, rs_x, rs_w, voff_x, voff_w, loader, slot, step + ST - 1, steps);
      slot = slot == ST - 1 ? 0 : slot + 1;
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    return;
  }
  const int wr = wave / WC, wc = wave % WC, row = lane & 15, g = lane >> 4;
  int xa[KB / 4], wa[KB * (int)sizeof(WT) / 16];
#pragma unroll
  for (int c = 0; c < KB / 4; ++c) xa[c] = (wr * 16 * RB + row) * S::XROW + ((c ^ f32k_swizzle<S::XROW>(row)) * 16) + 4 * g;
#pragma unroll
  for (int c = 0; c < KB * (int)sizeof(WT) / 16; ++c)
    wa[c] = S::XBYTES + (wc * 16 * CB + row) * S::WROW + ((c ^ f32k_swizzle<S::WROW>(row)) * 16) + (int)sizeof(WT) * g;
  const int live = min(RB, last - first - wr * RB);                            // scalar: this wave's row blocks
  const int mw = m0 + wr * 16 * RB, nw = n0 + wc * (GATED ? 8 : 16) * CB;
#define BW_F32K_TILE(L) \
  return f32k_tile<S, WT, L, CB, ST, LW, GATED>(f32k_ring, rs_x, rs_w, voff_x, voff_w, loader, xa, wa, steps, y, ldy, mw, nw, M, N, accumulate)
  // (tiles of eight blocks are for more than 64 rows: evenly shared, four at least)
  if constexpr (RB == 8) {
    static_assert(WR == 1, "every wave has all rows");
    if (live == 8) BW_F32K_TILE(8);
    if (live == 7) BW_F32K_TILE(7);
    if (live == 6) BW_F32K_TILE(6);
    if (live == 5) BW_F32K_TILE(5);
    BW_F32K_TILE(4);
  } else if constexpr (RB == 4) {
    static_assert(WR == 1, "every wave has all rows");
    if (live == 4) BW_F32K_TILE(4);
    if (live == 3) BW_F32K_TILE(3);
    if (live == 2) BW_F32K_TILE(2);
    BW_F32K_TILE(1);
  } else {
    static_assert(RB == 1, "one block a wave");
    if (live >= 1) BW_F32K_TILE(1);
    BW_F32K_TILE(0);
  }
#undef BW_F32K_TILE
#endif
}

template <typename WT, int RB, int CB, int WR, int WC, int KB, int ST, int LW, bool GATED = false>
static void launch_f32_tiles(const float* x, const WT* w, float* y, int M, int N, int K, int ldx, int ldy, int accumulate, hipStream_t s) {
  using S = F32KShape<WT, RB, CB, WR, WC, KB, ST, LW>;
  static bool allowed = false;                       // more than 64 KB of dynamic LDS has to be asked for once
  if (S::LDS > 48 * 1024 && !allowed) {
    (void)hipFuncSetAttribute((const void*)gemm_f32_tiles_kernel<WT, RB, CB, WR, WC, KB, ST, LW, GATED>, hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS);
    allowed = true;
  }
  const int row_tiles = ((M + 15) / 16 + RB * WR - 1) / (RB * WR);
  hipLaunchKernelGGL((gemm_f32_tiles_kernel<WT, RB, CB, WR, WC, KB, ST, LW, GATED>), dim3(row_tiles * (((GATED ? 2 : 1) * N + S::COLS - 1) / S::COLS)),
                     dim3(64 * (S::WAVES + LW)), S::LDS, s, x, w, y, M, N, K, ldx, ldy, accumulate, row_tiles);
}

// ------------------------------------------------------------------------------ few rows, few columns

// Where a product has fewer blocks of 16 x 16 outputs than the chip has SIMDs, its time is that of one chain, and what counts is that
// nothing but matrix instructions stands in the chain's wave.  A workgroup is WC waves with a block of outputs each and two that
// bring the operands: they load a few stages ahead into registers, widen bfloat16 weights and put both operands into LDS in the
// order in which the instructions want them, so that a working wave reads 16 bytes of each for four instructions and issues no
// vector instruction at all.  Three stages of 64 steps of k lie in LDS: the one worked on, the next one (whose first operands are
// read before the barrier between them) and the one that is being written.
// A row's block of 16 k is 64 bytes: chunk g holds elements g, 4 + g, 8 + g and 12 + g, at a place that keeps sixteen lanes served
// together (0-3, 12-15, 20-27 of a half wave, and the others) in distinct banks, and the writers', too.
// Bfloat16 weights, 8 rows, us: 2048 x 2048 12.8 -> 10.3 (a chain's instructions alone are 7.0), 2048 x 8192 43.3 -> 32.6 (28), 6144 x 2048
// 17.1 -> 12.2; 64 rows, 2048 x 8192 240 -> 38.6.  With four working waves a compute unit LDS is what bounds (16384 x 2048 20.7, and 17.0 in
// tiles of 16 x 64 as they are above): not for as many columns.
template <typename WT, int WC, int D>
struct F32SShape {
  static constexpr int KB = 64, LW = 2, COLS = 16 * WC;
  static constexpr int RUNS = KB / 8, BLOCKS = KB / 16;                       // of a row of a stage: runs of 8 k, blocks of 16
  static constexpr int XBLOCK = 16 * 64, WBLOCK = COLS * 64;                  // bytes of a block of all rows, of all columns
  static constexpr int XBYTES = BLOCKS * XBLOCK, STAGE = XBYTES + BLOCKS * WBLOCK, LDS = 3 * STAGE;
  static constexpr int XW = 16 * RUNS / 64 / LW, WW = COLS * RUNS / 64 / LW;  // a loading wave's runs a stage, 64 at a time
  static_assert(XW * LW * 64 == 16 * RUNS && WW * LW * 64 == COLS * RUNS, "every loading wave counts alike");
  static_assert(D % 3 == 0, "whole turns of the three stages");
};

// Where chunk g (elements g, 4 + g, 8 + g and 12 + g) of a row's block lies in the row's 64 bytes.
__device__ __forceinline__ int f32s_chunk(int g, int row, int block) {
  return ((((g & 1) ^ (block & 1)) << 1) | ((g >> 1) ^ ((row >> 3) & 1))) * 16;
}

#if defined(__HIP_DEVICE_COMPILE__)
// What a loading wave has of one stage.
template <typename S, typename WT>
struct F32SRegs {
  u32x4 x[S::XW][2], w[S::WW][sizeof(WT) == 2 ? 1 : 2];
};

template <typename S, typename WT>
__device__ __forceinline__ void f32s_load(__amdgpu_buffer_rsrc_t rs_x, __amdgpu_buffer_rsrc_t rs_w, const int* voff_x, const int* voff_w, int step,
                                          int steps, F32SRegs<S, WT>& r) {
  const bool real = step < steps;                                             // scalar (past K: outside the descriptors, zeros)
#pragma unroll
  for (int t = 0; t < S::XW; ++t)
#pragma unroll
    for (int h = 0; h < 2; ++h) r.x[t][h] = __builtin_amdgcn_raw_buffer_load_b128(rs_x, real ? voff_x[t] + 16 * h : 0x7ffffff0, step * S::KB * 4, 0);
#pragma unroll
  for (int t = 0; t < S::WW; ++t)
#pragma unroll
    for (int h = 0; h < (sizeof(WT) == 2 ? 1 : 2); ++h)
      r.w[t][h] = __builtin_amdgcn_raw_buffer_load_b128(rs_w, real ? voff_w[t] + 16 * h : 0x7ffffff0, step * S::KB * (int)sizeof(WT), 0);
}

template <typename S, typename WT>
__device__ __forceinline__ void f32s_store(unsigned char* stage, const int (*at_x)[4], const int (*at_w)[4], const F32SRegs<S, WT>& r) {
#pragma unroll
  for (int t = 0; t < S::XW; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) *reinterpret_cast<u32x2*>(stage + at_x[t][g]) = (u32x2){r.x[t][0][g], r.x[t][1][g]};
#pragma unroll
  for (int t = 0; t < S::WW; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      u32x2 v;
      if constexpr (sizeof(WT) == 2) {                                        // bfloat16 -> 32-bit: the bits, shifted (exact)
        const uint32_t lo = r.w[t][0][g >> 1], hi = r.w[t][0][2 + (g >> 1)];
        v = (g & 1) ? (u32x2){lo & 0xffff0000u, hi & 0xffff0000u} : (u32x2){lo << 16, hi << 16};
      } else {
        v = (u32x2){r.w[t][0][g], r.w[t][1][g]};
      }
      *reinterpret_cast<u32x2*>(stage + at_w[t][g]) = v;
    }
}
#endif

// What rotation and cache write in the epilogue need (rope_kvwrite_kernel's arguments).
struct F32RopeArgs {
  const int32_t* positions;
  const int32_t* row_seq;
  const int32_t* block_table;
  const float* cos_table;    // [positions, head_dim / 2]
  const float* sin_table;
  float* k_cache;
  float* v_cache;
  int heads, kv_heads, head_dim, page_size, page_shift, table_stride, write_cache;      // (page_shift: log2 of page_size, or -1)
};

// ROPE (two working waves): y is the stacked q|k|v product with q and k rotated, k and v also in their page slots: the statements of
// rope_kvwrite_kernel, which as a launch of its own reads and writes the 32-bit sums once more.  A workgroup's columns are 16 pairs of
// one head, first halves with one wave and second halves with the other, so that a lane's partner lies in the same lane of
// the other wave.  Replayed as graphs, us, product and kernel -> one: 8 rows of 96 heads of 64, K = 2048, 15.1 -> 13.2 (the product alone
// 12.0), 32-bit weights 19.4 -> 16.1; 8 rows of 48 heads of 128, K = 4096, 23.8 -> 22.4; 64 rows of 12 heads, K = 1024, 9.6 -> 8.2; 0.72 to 0.94 of
// the time at 14 such products.
template <typename WT, int WC, int D, bool ROPE>
__global__ __launch_bounds__(64 * (WC + 2)) void gemm_f32_strips_kernel(const float* __restrict__ x, const WT* __restrict__ w, float* __restrict__ y, int M,
                                                                       int N, int K, int ldx, int ldy, int accumulate, int row_tiles, F32RopeArgs ra) {
#if defined(__HIP_DEVICE_COMPILE__)
  using S = F32SShape<WT, WC, D>;
  extern __shared__ __attribute__((aligned(16))) unsigned char f32s_lds[];
  const int wave = wave_index(), lane = threadIdx.x & 63;
  static_assert(!ROPE || WC == 2, "a wave for the first halves of the pairs, one for the second");
  const int m0 = 16 * ((int)blockIdx.x % row_tiles), tile = (int)blockIdx.x / row_tiles;
  const int half = ROPE ? ra.head_dim >> 1 : S::COLS;                          // (a tile's second 16 columns are half a head behind its first)
  const int head = ROPE ? tile / (half >> 4) : 0, pair0 = ROPE ? 16 * (tile % (half >> 4)) : 0;
  const int n0 = ROPE ? head * ra.head_dim + pair0 : tile * S::COLS;
  const int steps = K / S::KB;
  if (wave >= WC) {
    // ---- a loading wave: runs of 8 k, lane l run l % 8 of row (column) l / 8 of its 8
    const int loader = wave - WC;
    const int x_rows = min(16, M - m0), w_rows = ROPE ? half + 16 : min(S::COLS, N - n0);   // (ROPE: whole tiles)
    const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(x + (size_t)m0 * ldx), 0, (int)((((size_t)x_rows - 1) * ldx + K) * sizeof(float)), 0x00020000);
    const __amdgpu_buffer_rsrc_t rs_w =
        __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)n0 * K), 0, (int)((size_t)w_rows * K * sizeof(WT)), 0x00020000);
    int voff_x[S::XW], voff_w[S::WW], at_x[S::XW][4], at_w[S::WW][4];
    const int run = lane % S::RUNS;
#pragma unroll
    for (int t = 0; t < S::XW; ++t) {
      const int row = (loader + t * S::LW) * (64 / S::RUNS) + lane / S::RUNS;
      voff_x[t] = min(row, x_rows - 1) * ldx * 4 + run * 32;                   // (rows past the operand are clamped to its last)
#pragma unroll
      for (int g = 0; g < 4; ++g) at_x[t][g] = (run >> 1) * S::XBLOCK + row * 64 + f32s_chunk(g, row, run >> 1) + 8 * (run & 1);
    }
#pragma unroll
    for (int t = 0; t < S::WW; ++t) {
      const int row = (loader + t * S::LW) * (64 / S::RUNS) + lane / S::RUNS;
      voff_w[t] = (ROPE ? (row < 16 ? row : row - 16 + half) : min(row, w_rows - 1)) * K * (int)sizeof(WT) + run * 8 * (int)sizeof(WT);
#pragma unroll
      for (int g = 0; g < 4; ++g) at_w[t][g] = S::XBYTES + (run >> 1) * S::WBLOCK + row * 64 + f32s_chunk(g, row, run >> 1) + 8 * (run & 1);
    }
    F32SRegs<S, WT> r[D];
#pragma unroll
    for (int d = 0; d < D; ++d) f32s_load<S, WT>(rs_x, rs_w, voff_x, voff_w, d, steps, r[d]);
    // stages 0 to steps + 1 (the last two: zeros, never used), a barrier behind each but the first
    for (int base = 0; base < steps + 2; base += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int stage = base + d;
        if (stage >= steps + 2) break;                                         // scalar
        f32s_store<S, WT>(f32s_lds + (d % 3) * S::STAGE, at_x, at_w, r[d]);
        f32s_load<S, WT>(rs_x, rs_w, voff_x, voff_w, stage + D, steps, r[d]);
        if (stage > 0) {
          __builtin_amdgcn_s_waitcnt(0xc07f);                                  // the writes are done (lgkmcnt 0)
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
        }
      }
    }
    return;
  }
  // ---- a working wave: blocks of 16 k in pairs, the next pair's operands read under this pair's eight instructions
  const int row = lane & 15, g = lane >> 4;
  int xa[2], wa[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    xa[i] = row * 64 + f32s_chunk(g, row, i);
    wa[i] = S::XBYTES + (wave * 16 + row) * 64 + f32s_chunk(g, row, i);
  }
  f32x4 acc[1][1] = {{{0.f, 0.f, 0.f, 0.f}}};
  f32x4 hx[2][2], hw[2][2];
  int pos[4] = {-1, -1, -1, -1}, page[4] = {0, 0, 0, 0};
  float cosine[4] = {}, sine[4] = {};
  int seq[4] = {0, 0, 0, 0};
  if constexpr (ROPE) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = min(m0 + 4 * g + i, M - 1);
      pos[i] = ra.positions[m];
      seq[i] = ra.row_seq[m];
    }
  }
  __builtin_amdgcn_s_barrier();                                                // stages 0 and 1 are there
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    hw[0][i] = *reinterpret_cast<const f32x4*>(f32s_lds + i * S::WBLOCK + wa[i]);
    hx[0][i] = *reinterpret_cast<const f32x4*>(f32s_lds + i * S::XBLOCK + xa[i]);
  }
  for (int base = 0; base < steps; base += 3) {
    if constexpr (ROPE) {
      // what hangs on the positions is asked for once those are there for certain, a turn later (in front of the first stage the wait
      // for them took 0.3 us a layer more)
      if (base == (steps > 3 ? 3 : 0)) {                                       // scalar
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int at = max(pos[i], 0);                                       // (a padding row: the product as it is, whatever is loaded)
          cosine[i] = ra.cos_table[(size_t)at * half + pair0 + row];
          sine[i] = ra.sin_table[(size_t)at * half + pair0 + row];
          page[i] = ra.block_table[(size_t)(pos[i] < 0 ? 0 : seq[i]) * ra.table_stride + (ra.page_shift >= 0 ? at >> ra.page_shift : at / ra.page_size)];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      if (base + u >= steps) break;                                            // scalar
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        __builtin_amdgcn_sched_barrier(0);
        if (p == 1) {
          // this stage has been read: behind the barrier its place is filled again, and the stage after the next is there
          __builtin_amdgcn_s_waitcnt(0xc07f);
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
        }
        const unsigned char* from = f32s_lds + (p == 1 ? (u + 1) % 3 : u) * S::STAGE;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int blk = 2 * (p ^ 1) + i;
          hw[p ^ 1][i] = *reinterpret_cast<const f32x4*>(from + blk * S::WBLOCK + wa[i]);
          hx[p ^ 1][i] = *reinterpret_cast<const f32x4*>(from + blk * S::XBLOCK + xa[i]);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)                                          // k ascending
            acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(hx[p][i][e], hw[p][i][e], acc[0][0], 0, 0, 0);
        f32_order<8, 4>();
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  if constexpr (ROPE) {
    // (the loading waves are done: their last stores lie before the barrier behind the last stage)
    const f32x4 own = acc[0][0];
    f32x4* sums = reinterpret_cast<f32x4*>(f32s_lds);
    sums[64 * wave + lane] = own;
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const f32x4 other = sums[64 * (wave ^ 1) + lane];
    const int n = n0 + half * wave + row, in_head = pair0 + half * wave + row;
    const bool turns = head < ra.heads + ra.kv_heads;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + 4 * g + i;
      if (m >= M) continue;
      float v = own[i];
      if (turns && pos[i] >= 0) v = wave == 0 ? own[i] * cosine[i] - other[i] * sine[i] : own[i] * cosine[i] + other[i] * sine[i];
      y[(size_t)m * ldy + n] = v;
      if (head >= ra.heads && pos[i] >= 0 && ra.write_cache) {
        float* cache = turns ? ra.k_cache : ra.v_cache;
        const int kv = head - ra.heads - (turns ? 0 : ra.kv_heads);
        const int slot = ra.page_shift >= 0 ? pos[i] & (ra.page_size - 1) : pos[i] % ra.page_size;
        cache[(((size_t)page[i] * ra.kv_heads + kv) * ra.page_size + slot) * ra.head_dim + in_head] = v;
      }
    }
  } else {
    f32_write<1, 1>(acc, y, ldy, m0, n0 + 16 * wave, M, N, accumulate);
  }
#endif
}

template <typename WT, int WC, int D, bool ROPE = false>
static void launch_f32_strips(const float* x, const WT* w, float* y, int M, int N, int K, int ldx, int ldy, int accumulate, hipStream_t s,
                              const F32RopeArgs& ra = F32RopeArgs{}) {
  using S = F32SShape<WT, WC, D>;
  const int row_tiles = (M + 15) / 16;
  hipLaunchKernelGGL((gemm_f32_strips_kernel<WT, WC, D, ROPE>), dim3(row_tiles * ((N + S::COLS - 1) / S::COLS)), dim3(64 * (WC + S::LW)), S::LDS, s, x, w, y, M, N,
                     K, ldx, ldy, accumulate, row_tiles, ra);
}
