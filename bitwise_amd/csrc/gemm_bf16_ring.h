// Part of gemm_bf16.hip (included there behind gemm_bf16_tiles.h; not a unit of its own): the tiles of prompt portions,
// fed through LDS rings.
//
// What bounds them, a step of 256 x 256 outputs: a compute unit's loads from the L2s take 0.8 us (64 KB at the 80 KB a microsecond
// that a kernel of nothing but such loads gets), its operand reads 0.4 (24 a wave, by the counter of LDS at work), the matrix
// instructions 1.0 (64 a wave), at the 2.0 GHz that the part runs at under this load; the step takes 1.41.  What is lost is where
// they wait for each other.  So
//   * the wait for a step and its barrier stand two turns before the end of the step before, and the step's first operands
//     are read under the last turns' matrix instructions: no wave starts a step by waiting for LDS;
//   * where only two steps of W fit beside three of x, a barrier in the middle of a step gives the half ring back early, so that
//     every load has a step and a half to arrive (192 x 256 tiles without it: 147 us a product that takes 120);
//   * the tile's shape goes by the product (ring_choice): as few bytes an output as its registers allow, but rounds of the
//     256 compute units that are not left part empty.
// Against one kernel each for 256 x 256, 128 x 256 and 128 x 128 tiles that waited at the step's edge and were chosen by counts
// of steps (one machine, both in turn, us): gate|up + SwiGLU of 2048 x 16384 x 2048 107 -> 99, of 2048 x 28672 x 4096 420 -> 365 (in
// 192 x 256 tiles, 1.32 PFLOP/s), of 777 rows 209 -> 186 (160 x 256); q|k|v with rotation of 2048 x 6144 x 2048 53 -> 46, of 1348 rows
// 51 -> 41, the plain product of K = 4096 118 -> 81 (256 x 192, one round); the residual adds of 2048 x 2048 x 8192 78 -> 73 (before with
// 67 MB of scratch, now without), of 777 x 4096 x 4096 48 -> 34, of K = 14336 120 in two launches -> 102.  The results are the same bits.
#pragma once

// A workgroup of eight waves computes BM x BN outputs (gated epilogues: BM x BN / 2, from BN / 2 gate and BN / 2 up rows of
// W) in steps of 64 along K; the waves lie WY x 8/WY over the tile, each with MI x NJ blocks of 16 x 16 outputs.  Tiles of
// x and W travel from memory straight into LDS (buffer loads with LDS as their destination: no registers, no LDS write
// instructions).  One load of a wave brings 8 rows of a step, 128 bytes each (whole cache lines), into 1 KB of LDS, lane l's
// 16 bytes to 16 * l.  Which 16 bytes of its row a lane fetches is permuted: slot c' of row r (r counted within its block
// of 16 rows) holds the row's chunk c' ^ (r >> 1), so that the 16 lanes that read one chunk of 16 different rows as a matrix
// operand hit 16 different groups of banks.
template <int EPI, int WY_, int MI_, int NJ_>
struct RingTile {
  static constexpr int WY = WY_, WX = 8 / WY_, MI = MI_, NJ = NJ_;
  static constexpr int BM = 16 * WY * MI, BN = 16 * WX * NJ;
  static constexpr bool GLU = epi_is_glu(EPI), ROPE = EPI == EPI_QKV_ROPE;
  static constexpr int COLS = GLU ? BN / 2 : BN;                   // output columns
  static constexpr int A_SLOT = BM * 128, B_SLOT = BN * 128;       // bytes of a step's rows
  static constexpr int LA = (BM + 63) / 64, LB = BN / 64;          // loads a wave and step
  static constexpr bool JUNK = BM % 64 != 0;                       // some of those have no rows: they go to 1 KB of their own
  // as many steps in LDS as fit; where three steps do not, three of x and two of W
  static constexpr bool FOUR = 4 * (A_SLOT + B_SLOT) <= BW_LDS_LIMIT, THREE = 3 * (A_SLOT + B_SLOT) + (JUNK ? 1024 : 0) <= BW_LDS_LIMIT;
  static constexpr int RA = FOUR ? 4 : 3, RB = FOUR ? 4 : (THREE ? 3 : 2);
  static constexpr int B_AT = RA * A_SLOT, JUNK_AT = B_AT + RB * B_SLOT;
  static constexpr int BYTES = JUNK_AT + (JUNK ? 1024 : 0);
  // two steps of W: a second barrier in the middle of a step, where every wave has its last operands of the step's W, lets the
  // step after next overwrite them at once
  static constexpr bool MID = RA != RB;
  static constexpr int DA = RA - 1, DB = MID ? RB : RB - 1;        // how many steps ahead the loads of a step's first and last turns are
  // loads of a wave that are younger than those of the next step, when a step has issued all of its own
  static constexpr int YOUNGER = (DA - 1) * LA + (DB - 1) * LB;
  static constexpr int U = 2 * MI;                                 // a step's turns: one block of x rows times NJ blocks of W rows
  // Three or four steps of both in LDS: the turn before which load n of a step is issued.  The first of them stand behind the
  // barrier, in the last two turns (-2, -1) of the step before, whose slots they overwrite.
  static constexpr int turn(int n) { return n * U / (LA + LB) - 2; }
  static constexpr int NA = U % 4 == 0 && MI < 6 ? 4 : (U % 3 == 0 ? 3 : (U % 4 == 0 ? 4 : 5));   // registers' ring of x blocks; divides U
  static constexpr int BPT = (NJ + MI - 2) / (MI - 1);             // W blocks of the second half read a turn
  static constexpr int B_FROM = MI - 1 - (NJ + BPT - 1) / BPT;     // and from which turn on
  static_assert(BN % 64 == 0 && BM % 32 == 0 && U % NA == 0 && BYTES <= BW_LDS_LIMIT && (NJ % 2 == 0 || !(GLU || ROPE)), "tile shapes");
};

template <int EPI>
__device__ __forceinline__ float glu_value(float g, float u, const QkvRopeArgs& rp) {
  if constexpr (EPI == EPI_CLAMPED_GLU_BF16) return clamped_swish_times<true>(g, u, rp.glu_limit, rp.glu_alpha);
  else if constexpr (EPI == EPI_GELU_GLU_BF16) return gelu_tanh_times(g, u);
  else return silu_times(g, u);
}

template <int EPI, int WY, int MI, int NJ, bool JOIN>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_bf16_ring_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ out, int M, int N, int K, int ldx,
    int ldo, int m_tiles, int n_tiles, int n_from, QkvRopeArgs rp, size_t seg_stride) {
  using T = RingTile<EPI, WY, MI, NJ>;
  constexpr bool GLU = T::GLU, ROPE = T::ROPE, ADD_FIRST = EPI == EPI_ADD_F32 && JOIN;
  constexpr int BM = T::BM, COLS = T::COLS, NH = NJ / 2, U = T::U, NA = T::NA;
  extern __shared__ __attribute__((aligned(16))) unsigned char ring[];
  // gridDim.y > 1: workgroup (tile, y) works on segment y of K alone and leaves its sums at out + y * seg_stride
  // elements (a residual add's segments, joined in order by add_segments_kernel afterwards)
  const int k_base = (int)blockIdx.y * GEMM_SEG, k_all = K;
  if (gridDim.y > 1) {
    out = (void*)((float*)out + (size_t)blockIdx.y * seg_stride);
    K = min(GEMM_SEG, K - k_base);
  }
  const int wave = wave_index(), lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const int wy = wave / T::WX, wx = wave % T::WX;
  // consecutive workgroups go to different dies: die d takes a run of tiles, so that an n tile's workgroups share a die
  const int nblocks = m_tiles * n_tiles, die = blockIdx.x & 7;
  const int bid = die * (nblocks >> 3) + min(die, nblocks & 7) + (int)(blockIdx.x >> 3);
  const int m0 = (bid % m_tiles) * BM;
  const int n0 = n_from + (bid / m_tiles) * COLS;                  // (n_from: the first of this launch's outputs)

  // this wave's loads of a step: groups of 8 rows LA * wave .. of x, LB * wave .. of W (gated: waves 0 to 3 the gate rows n0..,
  // waves 4 to 7 the up rows N + n0..).  Rows past M or N lie outside the descriptors and read as zeros.
  const int a_rows = min(BM, M - m0), b_rows = min(COLS, N - n0);
  const __amdgpu_buffer_rsrc_t rs_a = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(x + (size_t)m0 * ldx), 0, (int)((((size_t)a_rows - 1) * ldx + k_all) * 2), 0x00020000);
  const bool up = GLU && wave >= 4;
  const __amdgpu_buffer_rsrc_t rs_b = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(w + ((size_t)(up ? N : 0) + n0) * k_all), 0, (int)((size_t)b_rows * k_all * 2), 0x00020000);
  const int lrow = lane >> 3, lslot = lane & 7;
  // (arrays that lambdas take have plain sizes: the host pass drops a kernel whose lambdas capture arrays of dependent size)
  int voff_a[4], voff_b[4];
#pragma unroll
  for (int t = 0; t < T::LA; ++t) {
    const int row = 8 * (T::LA * wave + t) + lrow;
    voff_a[t] = T::JUNK && T::LA * wave + t >= BM / 8 ? 0x7ffffff0 : (row * ldx + 8 * (lslot ^ ((row & 15) >> 1))) * 2;
  }
#pragma unroll
  for (int t = 0; t < T::LB; ++t) {
    const int row = 8 * (T::LB * wave + t) + lrow;
    voff_b[t] = ((GLU && wave >= 4 ? row - COLS : row) * k_all + 8 * (lslot ^ ((row & 15) >> 1))) * 2;
  }
  typedef __attribute__((address_space(3))) void* lds_ptr;
  const int steps = K / 64;
  // (past K: outside the descriptors, no traffic, zeros into slots that the last step reads ahead from and whose values nobody uses)
  auto issue_a = [&](int step, int slot, int t) {
    const int q = T::LA * wave + t;
    const int at = T::JUNK && q >= BM / 8 ? T::JUNK_AT : slot * T::A_SLOT + q * 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_a, (lds_ptr)(ring + at), 16, step < steps ? voff_a[t] : 0x7ffffff0,
                                             k_base * 2 + step * 128, 0, 0);
  };
  auto issue_b = [&](int step, int slot, int t) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_b, (lds_ptr)(ring + T::B_AT + slot * T::B_SLOT + (T::LB * wave + t) * 1024), 16,
                                             step < steps ? voff_b[t] : 0x7ffffff0, k_base * 2 + step * 128, 0, 0);
  };

  f32x4 acc[MI][NJ], tot[JOIN ? MI : 1][JOIN ? NJ : 1];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if constexpr (JOIN) tot[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
  if constexpr (ADD_FIRST) {                                        // the chain of a residual add starts at the residual
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int m = m0 + 16 * (MI * wy + i) + 4 * g + q, n = n0 + 16 * (NJ * wx + j) + r;
          tot[i][j][q] = (m < M && n < N) ? ((const float*)out)[(size_t)m * ldo + n] : 0.0f;
        }
  }
  // Operands.  A block of 16 rows is 2 KB; lane (g, r) wants row r, chunk 4*kk + g: slot (4*kk + g) ^ (r >> 1) of that row.
  // x blocks MI*wy + i; W blocks NJ*wx + j.  Gated: gate blocks NH*wx + j (j < NH), then the up blocks of the same columns.
  // Rotary: pair blocks p = NH*wx + j (16 pairs (d, d + 32) of a head: its blocks p % 2 and p % 2 + 2), first halves, then second.
  const int row_off = (r >> 3) * 1024 + (r & 7) * 128;
  int slot_off[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) slot_off[kk] = row_off + (((4 * kk + g) ^ (r >> 1)) * 16);
  int b_blk[6];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int p = NH * wx + (j % NH);
    if constexpr (GLU) b_blk[j] = p + (j / NH) * (T::BN / 32);
    else if constexpr (ROPE) b_blk[j] = 4 * (p >> 1) + (p & 1) + 2 * (j / NH);
    else b_blk[j] = NJ * wx + j;
  }

  // Loads are issued in the order in which their steps are worked on; "all but the youngest" is the wait for a step.
#pragma unroll
  for (int st = -T::DB; st < 0; ++st) {
    if (st + T::DA >= 0) {
#pragma unroll
      for (int t = 0; t < T::LA; ++t) issue_a(st + T::DA, st + T::DA, t);
    }
#pragma unroll
    for (int t = 0; t < T::LB; ++t) issue_b(st + T::DB, st + T::DB, t);
  }
  u32x4 fa[5], fb[2][6];
  int sa = 0, sb = 0;                                             // slots of the step at hand
  auto next = [](int s, int n) { return s + 1 == n ? 0 : s + 1; };
  auto read_a = [&](int slot, int kk, int i, int to) {
    fa[to] = *reinterpret_cast<const u32x4*>(ring + slot * T::A_SLOT + (MI * wy + i) * 2048 + slot_off[kk]);
  };
  auto read_b = [&](int slot, int kk, int j) {
    fb[kk][j] = *reinterpret_cast<const u32x4*>(ring + T::B_AT + slot * T::B_SLOT + b_blk[j] * 2048 + slot_off[kk]);
  };
  // (the sums are zeroed here, while the first loads travel; left to itself the compiler does it behind the wait: 2048 x 8192
  // outputs of K = 64 stored in bfloat16 13.1 us, so 12.8)
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) asm volatile("" : "+v"(acc[i][j]));
  __builtin_amdgcn_s_waitcnt(vmcnt_only(T::YOUNGER));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if constexpr (!T::MID) {
#pragma unroll
    for (int n = 0; n < T::LA + T::LB; ++n)
      if (T::turn(n) < 0) {
        if (n < T::LA) issue_a(T::RA - 1, T::RA - 1, n);
        else issue_b(T::RB - 1, T::RB - 1, n - T::LA);
      }
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) read_b(0, 0, j);
  read_a(0, 0, 0, 0);
  read_a(0, 0, 1, 1);
  for (int step = 0; step < steps; ++step) {
    const int sa_next = next(sa, T::RA), sb_next = next(sb, T::RB);
    const int sa_fill = sa == 0 ? T::RA - 1 : sa - 1, sb_fill = sb == 0 ? T::RB - 1 : sb - 1;   // worked on a step ago
    __builtin_amdgcn_sched_barrier(0);
    // A step is 2 MI turns: one block of x against the wave's NJ blocks of W.  A turn reads the x block of the turn after next
    // (and, spread over the first half's turns, the W blocks of the second half), and one in so many issues a load for a
    // step further on.  The wait for the next step and the one barrier stand two turns before the step's end, so that
    // the next step's first operands are read under the last turns' matrix instructions.
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kk = u / MI;
      int reads = 1;
      if constexpr (T::MID) {
        if (u == MI + 1) {
          asm volatile("" ::: "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int n = 0; n < T::LA; ++n)
          if (n * MI / T::LA == u) issue_a(step + T::RA - 1, sa_fill, n);
#pragma unroll
        for (int n = 0; n < T::LB; ++n)
          if (MI + 1 + n * (MI > 3 ? MI - 3 : 1) / T::LB == u) issue_b(step + T::RB, sb, n);
      } else
#pragma unroll
      for (int n = 0; n < T::LA + T::LB; ++n)
        if (T::turn(n) == u) {
          if (n < T::LA) issue_a(step + T::RA - 1, sa_fill, n);
          else issue_b(step + T::RB - 1, sb_fill, n - T::LA);
        }
      if (u == U - 2) {
        // the next step's rows have landed, for every wave; and every wave has its last operands of this step, whose slots
        // the next loads overwrite
        __builtin_amdgcn_s_waitcnt(vmcnt_only(T::YOUNGER) & ~0x0f00);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      if constexpr (!T::MID) {
        // (this step's own slots, from here on)
#pragma unroll
        for (int n = 0; n < T::LA + T::LB; ++n)
          if (T::turn(n) + U == u) {
            if (n < T::LA) issue_a(step + T::RA, sa, n);
            else issue_b(step + T::RB, sb, n - T::LA);
          }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (u + 2 < U) read_a(sa, (u + 2) / MI, (u + 2) % MI, (u + 2) % NA);
      else read_a(sa_next, 0, u + 2 - U, (u + 2) % NA);
      if (kk == 0 && u >= T::B_FROM) {
#pragma unroll
        for (int t = 0; t < T::BPT; ++t) {
          const int j = (u - T::B_FROM) * T::BPT + t;
          if (j < NJ) {
            read_b(sb, 1, j);
            ++reads;
          }
        }
      }
      if (u >= U - 2) {
#pragma unroll
        for (int j = u == U - 2 ? 0 : NH; j < (u == U - 2 ? NH : NJ); ++j) read_b(sb_next, 0, j);
        reads += u == U - 2 ? NH : NJ - NH;
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        acc[u % MI][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(fa[u % NA]), as_bf16x8(fb[kk][j]), acc[u % MI][j], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < 5; ++t)
        if (t < reads) {
          if (t < NJ) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    sa = sa_next;
    sb = sb_next;
    if constexpr (JOIN) {
      const int kn = (step + 1) * 64;
      if (kn % GEMM_SEG == 0 && kn < K) {                // a segment ends before the last: joined left to right
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            tot[i][j] = !ADD_FIRST && kn == GEMM_SEG ? acc[i][j] : tot[i][j] + acc[i][j];
            acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
          }
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_only(0));                       // the padding loads too, before the waves end
  if constexpr (JOIN) {
    if (ADD_FIRST || K > GEMM_SEG) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = tot[i][j] + acc[i][j];
    }
  }

  if constexpr (ROPE) {
    // What the rows of the tile need from memory is fetched once for the workgroup, into the ring (free now), not
    // by every lane for each of its rows: position and page of each row (a thread a row), then the
    // rows' cosines and sines (16-byte loads; a row of 32 + 32 floats, 36 apart against bank conflicts).
    constexpr int CS = 36, HEADS = T::BN / 64;
    __syncthreads();                                                // every wave is done with the ring
    int* pos_lds = reinterpret_cast<int*>(ring);                    // [BM]
    int* page_lds = pos_lds + BM;                                   // [BM]
    float* cos_lds = reinterpret_cast<float*>(page_lds + BM);       // [BM][CS]
    float* sin_lds = cos_lds + BM * CS;                             // [BM][CS]
    const int first_head = n0 >> 6;
    const bool any_cache = first_head + HEADS > rp.heads;           // some of the tile's heads are k or v heads
    const bool any_rotary = first_head < rp.heads + rp.kv_heads;
    if (threadIdx.x < BM) {
      const int m = m0 + (int)threadIdx.x;
      const int mm = m < M ? m : M - 1;
      const int pos = rp.positions[mm];
      int page = 0;
      if (any_cache) page = rp.block_table[(size_t)rp.row_seq[mm] * rp.table_stride + ((pos > 0 ? pos : 0) >> rp.page_shift)];
      pos_lds[threadIdx.x] = m < M ? pos : -1;
      page_lds[threadIdx.x] = page;
    }
    __syncthreads();
    if (any_rotary && threadIdx.x < 2 * BM) {
      const int row = threadIdx.x >> 1, part = threadIdx.x & 1;     // 16 cosines and 16 sines of a row a thread
      const int pos = pos_lds[row];
      const size_t at = (size_t)(pos > 0 ? pos : 0) * 32 + 16 * part;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        *reinterpret_cast<f32x4*>(cos_lds + row * CS + 16 * part + 4 * t) = *reinterpret_cast<const f32x4*>(rp.cos_table + at + 4 * t);
        *reinterpret_cast<f32x4*>(sin_lds + row * CS + 16 * part + 4 * t) = *reinterpret_cast<const f32x4*>(rp.sin_table + at + 4 * t);
      }
    }
    __syncthreads();
    const int q_dim = rp.heads * 64;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int lrow0 = 16 * (MI * wy + i) + 4 * g;                 // the lane's four rows of the block, within the tile
      int pos4[4], page4[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        pos4[q] = pos_lds[lrow0 + q];
        page4[q] = page_lds[lrow0 + q];
      }
      // values lie transposed in their page ([d][slot]).  The lane's four rows are most often four consecutive
      // slots of one page starting at a multiple of four: then all four are stored at once.
      bool quad = pos4[0] >= 0 && (pos4[0] & 3) == 0;
#pragma unroll
      for (int t = 1; t < 4; ++t) quad = quad && pos4[t] == pos4[0] + t && page4[t] == page4[0];
      // (one or two pairs a wave belong to one head, and the stores to a row of it lie next to each other: by pairs instead, a
      // row's second half eight stores behind its first, 256 x 256 tiles took 3 us a round more)
      constexpr int OF_HEAD = NH <= 2 ? NH : 1;
#pragma unroll
      for (int j0 = 0; j0 < NH; j0 += OF_HEAD) {
        const int p0 = NH * wx + j0, head = first_head + (p0 >> 1);
        if (head < rp.heads + rp.kv_heads) {
          if (head >= rp.heads && !rp.write_cache) continue;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int pos = pos4[q];
            if (pos < 0) continue;
            const int m = m0 + lrow0 + q;
            bf16_t* dst = head < rp.heads
                              ? (bf16_t*)out + (size_t)m * q_dim + (size_t)head * 64
                              : rp.k_cache + (((size_t)page4[q] * rp.kv_heads + (head - rp.heads)) * rp.page_size + (pos & (rp.page_size - 1))) * 64;
#pragma unroll
            for (int j = j0; j < j0 + OF_HEAD; ++j) {
              const int d = 16 * ((p0 & 1) + j - j0) + r;           // pairs (d, d + 32) of the head
              const float c = cos_lds[(lrow0 + q) * CS + d], sn = sin_lds[(lrow0 + q) * CS + d];
              const float x1 = acc[i][j][q], x2 = acc[i][j + NH][q];
              dst[d] = f32_to_bf16(x1 * c - x2 * sn);
              dst[d + 32] = f32_to_bf16(x2 * c + x1 * sn);
            }
          }
        } else if (head < rp.heads + 2 * rp.kv_heads && rp.write_cache) {
          const int vh = head - rp.heads - rp.kv_heads;
#pragma unroll
          for (int j = j0; j < j0 + OF_HEAD; ++j) {
            const int d = 16 * ((p0 & 1) + j - j0) + r;
            if (quad) {
              bf16_t* dst = rp.v_cache + ((size_t)page4[0] * rp.kv_heads + vh) * 64 * rp.page_size + (pos4[0] & (rp.page_size - 1));
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                const f32x4& a = acc[i][j + h * NH];
                const u32x2 four = {pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3])};
                *reinterpret_cast<u32x2*>(dst + (size_t)(d + 32 * h) * rp.page_size) = four;
              }
            } else {
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                if (pos4[q] < 0) continue;
                bf16_t* dst = rp.v_cache + ((size_t)page4[q] * rp.kv_heads + vh) * 64 * rp.page_size + (pos4[q] & (rp.page_size - 1));
#pragma unroll
                for (int h = 0; h < 2; ++h) dst[(size_t)(d + 32 * h) * rp.page_size] = f32_to_bf16(acc[i][j + h * NH][q]);
              }
            }
          }
        }
      }
    }
  } else if constexpr (GLU) {
    // Whole rows of the tile leave as 16-byte stores: the waves put their outputs into the ring (free now) as the tile
    // lies in memory, [BM rows][COLS columns] with 16 bytes between rows, and the threads then store 16 bytes each.
    // (Two bytes a lane straight from the accumulators were 64 stores a wave, each of them four
    // pieces of 32 bytes.)  Outputs that are not 16-byte aligned take the element-wise way below; which way it is is asked once, not
    // for every value, between whose chains of exponential and reciprocal nothing else could run (2048 x 16384 x 64 in 256 x 256
    // tiles 21.6 us, so 17.9).
    constexpr int TROW = COLS * 2 + 16, CHUNKS = COLS / 8;
    const bool wide = (reinterpret_cast<uintptr_t>(out) & 15) == 0 && (ldo & 7) == 0 && (N & 7) == 0;
    if (wide) {
      __syncthreads();                                              // every wave is done with the ring
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int j = 0; j < NH; ++j)
            *reinterpret_cast<bf16_t*>(ring + (16 * (MI * wy + i) + 4 * g + q) * TROW + (16 * (NH * wx + j) + r) * 2) =
                f32_to_bf16(glu_value<EPI>(acc[i][j][q], acc[i][j + NH][q], rp));
      __syncthreads();
#pragma unroll
      for (int pass = 0; pass < (BM * CHUNKS + 511) / 512; ++pass) {
        const int c = 512 * pass + (int)threadIdx.x, row = c / CHUNKS, chunk = c % CHUNKS;
        const int m = m0 + row, n = n0 + 8 * chunk;
        if (row < BM && m < M && n < N)
          *reinterpret_cast<u32x4*>((bf16_t*)out + (size_t)m * ldo + n) = *reinterpret_cast<const u32x4*>(ring + row * TROW + 16 * chunk);
      }
    } else {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int m = m0 + 16 * (MI * wy + i) + 4 * g + q;
          if (m >= M) continue;
#pragma unroll
          for (int j = 0; j < NH; ++j) {
            const int n = n0 + 16 * (NH * wx + j) + r;
            if (n < N) ((bf16_t*)out)[(size_t)m * ldo + n] = f32_to_bf16(glu_value<EPI>(acc[i][j][q], acc[i][j + NH][q], rp));
          }
        }
    }
  } else {
    // (a residual add without joined sums meets the residual here: the loads of two block rows go out together, in front of
    // those rows' stores.  One by one between the stores 2048 x 8192 outputs of K = 64 took 37.7 us, so 28.9)
    constexpr bool ADD_LAST = EPI == EPI_ADD_F32 && !JOIN;
    constexpr int STEP = ADD_LAST ? 2 : 1;
    static_assert(MI % STEP == 0, "block rows in pairs");
#pragma unroll
    for (int i0 = 0; i0 < MI; i0 += STEP) {
      if constexpr (ADD_LAST) {
        f32x4 old[2][NJ];
#pragma unroll
        for (int i = 0; i < STEP; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
              const int m = m0 + 16 * (MI * wy + i0 + i) + 4 * g + q, n = n0 + 16 * (NJ * wx + j) + r;
              old[i][j][q] = (m < M && n < N) ? ((const float*)out)[(size_t)m * ldo + n] : 0.0f;
            }
#pragma unroll
        for (int i = 0; i < STEP; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) acc[i0 + i][j] = old[i][j] + acc[i0 + i][j];
      }
#pragma unroll
      for (int i = i0; i < i0 + STEP; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int m = m0 + 16 * (MI * wy + i) + 4 * g + q;
          if (m >= M) continue;
#pragma unroll
          for (int j = 0; j < NJ; ++j) {
            const int n = n0 + 16 * (NJ * wx + j) + r;
            if (n >= N) continue;
            if constexpr (EPI == EPI_ADD_F32) ((float*)out)[(size_t)m * ldo + n] = acc[i][j][q];
            else epilogue_store<EPI>(out, (size_t)m * ldo + n, acc[i][j][q], acc[i][j][q]);
          }
        }
    }
  }
}

// The shapes, and how long a round of the compute units takes with one (hundredths of a microsecond, all 256 at work):
// ``step`` for each 64 of K, ``ends`` for its first loads and its epilogue, ``brief`` the same for one or two steps, where nothing
// hides either and tiles of twice the size take more nearly twice as long, ``erf`` what the exact GELU adds, ``far`` what a step takes
// more from K = 4096 on (64 x 128: its rows are fewer than its rows of W, which come from memory and not from the L2s where K
// is long: 320 rows of 4096 x 4096 29 us, 25 in 128 x 64; of K = 14336 101 and 78).  Measured on products of 65 to 2,048 rows, 512 to 14336
// columns and K of 64 to 14336, every shape timed at each; over those with K of 512 or more a product takes 0.7 % more than in the
// shape that is best for it (mean; 7 % in one of 100).
// A tile of 256 x 256 has no registers left for the sums of earlier segments.
// (The two of 8,192 outputs are for products that would leave half of the chip idle in larger ones: gate|up of 117 x 16384 x 2048
// 23.4 us in 128 x 128 tiles, 18.6 in 128 x 64; 320 rows of 6144 x 2048 18.7 and 14.3 in 64 x 128.)
enum { RING_128, RING_128X256, RING_160X256, RING_192X256, RING_256X192, RING_256X256, RING_128X64, RING_64X128, RING_SHAPES };
struct RingCost {
  int rows, cols, step, ends, brief, erf, far;
  bool joins;
};
static const RingCost ring_costs[RING_SHAPES] = {{128, 128, 52, 650, 330, 240, 0, true},  {128, 256, 81, 750, 480, 500, 0, true},
                                                 {160, 256, 98, 820, 570, 600, 0, true},  {192, 256, 107, 865, 670, 740, 0, true},
                                                 {256, 192, 117, 940, 715, 740, 0, true}, {256, 256, 141, 900, 840, 980, 0, false},
                                                 {128, 64, 37, 500, 220, 110, 0, true},   {64, 128, 38, 500, 217, 110, 6, true}};

// The time of a product's tiles in that measure.  A last round that is part empty runs faster than a full one, the memory and
// the L2s being shared by fewer (0.6 of its time at the least; 160 x 256 tiles of 777 x 28672 x 4096, 2.19 rounds: 190 us
// against 67.5 a full round; 0.73 of one or two steps); not where one tile takes all rows: the weights' way through fewer compute units
// is what takes the time there (130 x 28672 x 4096: 112 tiles of 160 x 256 69 us, 224 of 128 x 256 60).
static long long ring_time(const RingCost& c, long long tiles, int K, bool one_row_tile, bool erf = false, int least_of_256 = 154) {
  const bool brief = K <= 128;
  if (brief) least_of_256 = 187;
  const long long last = tiles % 256;
  const long long rounds256 =
      tiles / 256 * 256 + (last ? (one_row_tile && !brief ? 256 : least_of_256 + last * (256 - least_of_256) / 256) : 0);
  return rounds256 * ((long long)(K / 64) * (c.step + (K >= 2 * GEMM_SEG ? c.far : 0)) + (brief ? c.brief : c.ends) + (erf ? c.erf : 0)) / 256;
}
static long long ring_tiles(const RingCost& c, int M, long long cols) { return (long long)((M + c.rows - 1) / c.rows) * ((cols + c.cols - 1) / c.cols); }

// The shape that takes the least time, all of K a workgroup.  ``cols``: rows of W; ``gated``: the outputs are half of those.
static int ring_choice(int M, long long cols, int K, bool gated, long long* time, bool erf = false) {
  int best = RING_128;
  long long least = -1;
  for (int i = 0; i < RING_SHAPES; ++i) {
    if (K > GEMM_SEG && !ring_costs[i].joins) continue;
    if (gated && i == RING_256X192) continue;
    const long long t = ring_time(ring_costs[i], ring_tiles(ring_costs[i], M, cols), K, M <= ring_costs[i].rows, erf);
    if (least < 0 || t < least) {
      least = t;
      best = i;
    }
  }
  if (time != nullptr) *time = least;
  return best;
}

// Columns of whole rounds in one shape, the others in the shape that is best for them: worth it where the whole product's last
// round is a small part of one.  A second launch and the first one's end cost RING_GAP; an estimated gain under 4.5 % is left.
// 140 products for which this holds (65 to 2,300 rows, K of 256 to 14336) took 7.9 % less than whole in the mean, the least 2 % more, within
// what runs differ: gate|up of 777 x 28672 x 4096 194 -> 174 us (510 tiles of 160 x 256, then 140 of 128 x 128), 1,288 rows of 20000 x 4096
// 220 -> 191.  Those with 3 to 4.5 % estimated took from 3 % more to 8 % less.
#define RING_GAP 250
struct RingParts {
  int shape, rest;
  long long first;                               // rows of W in ``shape``; 0: the product goes whole
};

static RingParts ring_parts(int M, long long cols, int K, bool gated, bool erf = false) {
  RingParts best{0, 0, 0};
  long long whole;
  ring_choice(M, cols, K, gated, &whole, erf);
  long long least = whole * 200 / 209;
  for (int i = 0; i < RING_SHAPES; ++i) {
    const RingCost& c = ring_costs[i];
    if ((K > GEMM_SEG && !c.joins) || (gated && i == RING_256X192)) continue;
    const long long mt = (M + c.rows - 1) / c.rows, rounds = ring_tiles(c, M, cols) / 256;
    for (long long r = rounds > 4 ? rounds - 3 : 1; r <= rounds; ++r) {
      const long long nt = r * 256 / mt, first = nt * c.cols;
      if (nt == 0 || first >= cols) continue;
      long long rest;
      const int shape = ring_choice(M, cols - first, K, gated, &rest, erf);
      const long long t = ring_time(c, nt * mt, K, M <= c.rows, erf) + RING_GAP + rest;
      if (t < least) {
        least = t;
        best = {i, shape, first};
      }
    }
  }
  return best;
}

extern "C" int bw_gemm_prompt_parts(int M, long long w_rows, int K, int gated, long long* first) {
  if (M <= 64 || w_rows <= 0 || K <= 0 || K % 64 || first == nullptr) return -2;
  *first = ring_parts(M, w_rows, K, gated != 0 && gated != 2, gated == 2).first;
  return 0;
}

extern "C" int bw_gemm_prompt_tile(int M, long long w_rows, int K, int gated, int* rows, int* columns) {
  if (M <= 64 || w_rows <= 0 || K <= 0 || K % 64 || rows == nullptr || columns == nullptr) return -2;
  const RingCost& c = ring_costs[ring_choice(M, w_rows, K, gated != 0 && gated != 2, nullptr, gated == 2)];
  *rows = c.rows;
  *columns = c.cols;
  return 0;
}

template <int EPI, int WY, int MI, int NJ, bool JOIN>
static int launch_ring_shape(const bf16_t* x, const bf16_t* w, void* out, int M, int N, int K, int ldx, int ldo, hipStream_t s,
                             const QkvRopeArgs& rp, int segments, size_t seg_stride, int n_from, int n_to) {
  using T = RingTile<EPI, WY, MI, NJ>;
  const int mt = (M + T::BM - 1) / T::BM, nt = (n_to - n_from + T::COLS - 1) / T::COLS;
  static bool allowed = false;                   // more than 64 KB of dynamic LDS has to be asked for once
  if (!allowed) {
    (void)hipFuncSetAttribute((const void*)gemm_bf16_ring_kernel<EPI, WY, MI, NJ, JOIN>, hipFuncAttributeMaxDynamicSharedMemorySize, T::BYTES);
    allowed = true;
  }
  BW_LAUNCH((gemm_bf16_ring_kernel<EPI, WY, MI, NJ, JOIN>), dim3(mt * nt, segments), dim3(512), T::BYTES, s, x, w, out, M, N, K, ldx,
            ldo, mt, nt, n_from, rp, seg_stride);
  return BW_LAUNCH_CHECK();
}

// ``segments`` > 1 (a 32-bit store): a workgroup per tile and segment of K, the sums of segment y at out + y * seg_stride.
// ``n_to`` > 0: of the outputs n_from .. n_to - 1 only (whole tiles, unless they end with the product's).
template <int EPI>
static int launch_ring(int shape, const bf16_t* x, const bf16_t* w, void* out, int M, int N, int K, int ldx, int ldo, hipStream_t s,
                       const QkvRopeArgs& rp = QkvRopeArgs{}, int segments = 1, size_t seg_stride = 0, int n_from = 0,
                       int n_to = 0) {
  constexpr bool JOIN = EPI != EPI_QKV_ROPE;     // (the rotary product has one segment)
  if (n_to == 0) n_to = N;
  switch (shape) {
    case RING_128: return launch_ring_shape<EPI, 2, 4, 2, JOIN>(x, w, out, M, N, K, ldx, ldo, s, rp, segments, seg_stride, n_from, n_to);
    case RING_128X64: return launch_ring_shape<EPI, 4, 2, 2, JOIN>(x, w, out, M, N, K, ldx, ldo, s, rp, segments, seg_stride, n_from, n_to);
    case RING_64X128: return launch_ring_shape<EPI, 2, 2, 2, JOIN>(x, w, out, M, N, K, ldx, ldo, s, rp, segments, seg_stride, n_from, n_to);
    case RING_128X256: return launch_ring_shape<EPI, 2, 4, 4, JOIN>(x, w, out, M, N, K, ldx, ldo, s, rp, segments, seg_stride, n_from, n_to);
    case RING_160X256: return launch_ring_shape<EPI, 2, 5, 4, JOIN>(x, w, out, M, N, K, ldx, ldo, s, rp, segments, seg_stride, n_from, n_to);
    case RING_192X256: return launch_ring_shape<EPI, 2, 6, 4, JOIN>(x, w, out, M, N, K, ldx, ldo, s, rp, segments, seg_stride, n_from, n_to);
    case RING_256X192:
      // (rotary pairs want whole pairs of blocks a wave: four by two waves of 64 x 96 outputs, where the others are two by four)
      if constexpr (EPI == EPI_QKV_ROPE) return launch_ring_shape<EPI, 4, 4, 6, JOIN>(x, w, out, M, N, K, ldx, ldo, s, rp, segments, seg_stride, n_from, n_to);
      else if constexpr (!epi_is_glu(EPI)) return launch_ring_shape<EPI, 2, 8, 3, JOIN>(x, w, out, M, N, K, ldx, ldo, s, rp, segments, seg_stride, n_from, n_to);
      break;
    case RING_256X256: return launch_ring_shape<EPI, 2, 8, 4, false>(x, w, out, M, N, K, ldx, ldo, s, rp, segments, seg_stride, n_from, n_to);
  }
  return -2;
}

// The tiles of a product, all of K a workgroup: of one shape, or, where that would leave a last round of few tiles, columns of whole
// rounds in one shape and the rest in tiles that fill the chip once more (a launch of its own: RING_GAP).
template <int EPI>
static int launch_ring_tiles(const bf16_t* x, const bf16_t* w, void* out, int M, int N, int K, int ldx, int ldo, hipStream_t s, const QkvRopeArgs& rp) {
  constexpr bool GLU = epi_is_glu(EPI);
  const long long cols = GLU ? 2LL * N : N;
  if constexpr (EPI != EPI_QKV_ROPE) {             // (whose tiles end with heads)
    const RingParts parts = ring_parts(M, cols, K, GLU, EPI == EPI_GELU_BF16);
    if (parts.first > 0) {
      const int n1 = (int)(GLU ? parts.first / 2 : parts.first);
      const int rc = launch_ring<EPI>(parts.shape, x, w, out, M, N, K, ldx, ldo, s, rp, 1, 0, 0, n1);
      return rc ? rc : launch_ring<EPI>(parts.rest, x, w, out, M, N, K, ldx, ldo, s, rp, 1, 0, n1, N);
    }
  }
  return launch_ring<EPI>(ring_choice(M, cols, K, GLU, nullptr, EPI == EPI_GELU_BF16), x, w, out, M, N, K, ldx, ldo, s, rp);
}
