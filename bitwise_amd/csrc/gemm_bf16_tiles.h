// Part of gemm_bf16.hip (included there, after its epilogues and launch macro; not a unit of its own):
// the 128 x 128 tiles of prompt portions that are staged through registers (K no multiple of 64), and their epilogue.
#pragma once

// ------------------------------------------------------------------------------ tile epilogue

// What a wave does with its NI x 4 accumulators (16 x 16 outputs each: rows row0 + 16 i + 4 g + q,
// columns 16 j + r of the wave's 64).  Plain epilogues: output columns col0 + 16 j + r.  SwiGLU:
// accumulators j = 0, 1 are gate columns col0 + 16 j + r, j = 2, 3 the up columns of the same outputs.
// Rotary q|k|v: the wave's 64 columns are head ``head``; accumulators j and j + 2 hold the rotary pairs
// (d, d + 32) in the same lane; q heads go to the q buffer, k heads rotated and v heads as they are to
// the row's page slot (v transposed).  ``residual_in``: the values already contain the residual.
template <int EPI, int NI>
__device__ __forceinline__ void tile_epilogue(const f32x4 (&acc)[NI][4], void* __restrict__ out, int M, int N, int ldo,
                                              int row0, int col0, int head, int r, int g, bool residual_in,
                                              const QkvRopeArgs& rp) {
  // Rotary: what the rows need from memory (position, then the page it selects) is asked for at once for all of
  // them, from addresses that are always valid, so that the waits for it are two and not two a row.
  constexpr int NR = EPI == EPI_QKV_ROPE ? NI : 1;
  int pos_all[NR][4], page_all[NR][4];
  if constexpr (EPI == EPI_QKV_ROPE) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = row0 + 16 * i + 4 * g + q;
        pos_all[i][q] = rp.positions[m < M ? m : M - 1];
      }
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = row0 + 16 * i + 4 * g + q;
        const int seq = rp.row_seq[m < M ? m : M - 1];
        const int pidx = (pos_all[i][q] > 0 ? pos_all[i][q] : 0) >> rp.page_shift;
        page_all[i][q] = head >= rp.heads ? rp.block_table[(size_t)seq * rp.table_stride + pidx] : 0;
      }
  }
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    // Rotary: the cosines and sines of the block's four rows are asked for together, from addresses that are
    // always valid (a padding row's position counts as 0), so that their latency is paid once a block, not once a row.
    float cs[4][2], sn[4][2];
    if constexpr (EPI == EPI_QKV_ROPE) {
      if (head < rp.heads + rp.kv_heads) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const size_t at = (size_t)(pos_all[i][q] > 0 ? pos_all[i][q] : 0) * 32 + 16 * j + r;
            cs[q][j] = rp.cos_table[at];
            sn[q][j] = rp.sin_table[at];
          }
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int m = row0 + 16 * i + 4 * g + q;
      if (m >= M) continue;
      if constexpr (EPI == EPI_QKV_ROPE) {
        const int pos = pos_all[i][q];
        if (head >= rp.heads + 2 * rp.kv_heads || pos < 0) continue;
        const int q_dim = rp.heads * 64;
        const size_t page = (size_t)page_all[i][q];
        const int slot = pos & (rp.page_size - 1);
        if (head < rp.heads + rp.kv_heads) {
          bf16_t* dst = head < rp.heads ? (bf16_t*)out + (size_t)m * q_dim + (size_t)head * 64
                                        : rp.k_cache + ((page * rp.kv_heads + (head - rp.heads)) * rp.page_size + slot) * 64;
          if (head < rp.heads || rp.write_cache) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const int d = 16 * j + r;
              const float c = cs[q][j], s = sn[q][j];
              const float x1 = acc[i][j][q], x2 = acc[i][j + 2][q];
              const float o1 = x1 * c - x2 * s;
              const float o2 = x2 * c + x1 * s;
              dst[d] = f32_to_bf16(o1);
              dst[d + 32] = f32_to_bf16(o2);
            }
          }
        } else if (rp.write_cache) {
          // values lie transposed in their page ([d][slot]).  The lane's four rows are most often four consecutive
          // slots of one page starting at a multiple of four: then the first row stores all four at once.
          bool quad = row0 + 16 * i + 4 * g + 3 < M && (pos_all[i][0] & 3) == 0;
#pragma unroll
          for (int t = 1; t < 4; ++t) quad = quad && pos_all[i][t] == pos_all[i][0] + t && page_all[i][t] == page_all[i][0];
          bf16_t* dst = rp.v_cache + (page * rp.kv_heads + (head - rp.heads - rp.kv_heads)) * 64 * rp.page_size + slot;
          if (quad) {
            if (q == 0) {
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                const u32x2 four = {pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3])};
                *reinterpret_cast<u32x2*>(dst + (size_t)(16 * j + r) * rp.page_size) = four;
              }
            }
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) dst[(size_t)(16 * j + r) * rp.page_size] = f32_to_bf16(acc[i][j][q]);
          }
        }
      } else if constexpr (epi_is_glu(EPI)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int n = col0 + 16 * j + r;
          if (n < N) epilogue_store<EPI>(out, (size_t)m * ldo + n, acc[i][j][q], acc[i][j + 2][q], rp.glu_limit, rp.glu_alpha);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int n = col0 + 16 * j + r;
          if (n >= N) continue;
          if (EPI == EPI_ADD_F32 && residual_in) ((float*)out)[(size_t)m * ldo + n] = acc[i][j][q];
          else epilogue_store<EPI>(out, (size_t)m * ldo + n, acc[i][j][q], acc[i][j][q]);
        }
      }
    }
  }
}

// ------------------------------------------------------------------------------ wide

#define WIDE_BM 128
#define WIDE_BN 128
#define WIDE_BK 64
#define WIDE_LDS_ROW 72   // bf16 elements per LDS row: 64 of data + 8 of padding (144 bytes)

template <int EPI, bool MULTI, bool FAST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_bf16_wide_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                             void* __restrict__ out, int M, int N, int K, int ldx,
                                                             int ldo, int m_tiles, int n_tiles, QkvRopeArgs rp) {
  // In SwiGLU mode a block covers 64 output columns: B rows 0-63 are gate rows, 64-127 up rows.
  constexpr int COLS = epi_is_glu(EPI) ? 64 : 128;
  __shared__ __attribute__((aligned(16))) bf16_t lds_a[2][WIDE_BM * WIDE_LDS_ROW];
  __shared__ __attribute__((aligned(16))) bf16_t lds_b[2][WIDE_BN * WIDE_LDS_ROW];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int r = lane & 15, g = lane >> 4;
  const int wy = wave >> 1, wx = wave & 1;
  // Blocks that run at the same time share an n tile (its weights are fetched once from HBM);
  // consecutive block ids go to different XCDs, so ids are regrouped by XCD first.
  int bid = blockIdx.x;
  const int nblocks = m_tiles * n_tiles;
  if (nblocks % 8 == 0) bid = (bid % 8) * (nblocks / 8) + bid / 8;
  const int m0 = (bid % m_tiles) * WIDE_BM;
  const int n0 = (bid / m_tiles) * COLS;

  // This thread's share of the global -> LDS copies: rows lr + 32j, 16-byte chunk lc.  The loads
  // go through buffer descriptors that cover exactly the block's rows of x and of W, so a row
  // past M or N reads as zeros by itself and one 32-bit offset per operand is all a thread keeps.
  const int lr = tid >> 3, lc = tid & 7;
  const int a_rows = min(WIDE_BM, M - m0);
  const __amdgpu_buffer_rsrc_t rs_a = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(x + (size_t)m0 * ldx), 0, (int)((((size_t)a_rows - 1) * ldx + K) * 2), 0x00020000);
  const int b_rows = min(COLS, N - n0);              // gate rows and up rows alike in SwiGLU mode
  const __amdgpu_buffer_rsrc_t rs_b0 =
      __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)n0 * K), 0, (int)((size_t)b_rows * K * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_b1 = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(w + ((size_t)N + n0) * K), 0, (int)((size_t)b_rows * K * 2), 0x00020000);
  const int voff_a = (lr * ldx + lc * 8) * 2, voff_b = (lr * K + lc * 8) * 2;
  // LDS rows of this wave's four B tiles
  int brow[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (epi_is_glu(EPI)) brow[j] = (j >> 1) * 64 + 32 * wx + 16 * (j & 1);
    else brow[j] = 64 * wx + 16 * j;
  }

  static_assert(!(MULTI && FAST), "the fast path is for one segment");
  constexpr bool TOT = MULTI;
  f32x4 acc[4][4], tot[TOT ? 4 : 1][TOT ? 4 : 1];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if constexpr (TOT) tot[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }

  // Tiles travel global -> registers -> LDS.  A tile is asked for two steps before it is used
  // and parked in one of two register sets meanwhile, so that a load has about two steps of
  // matrix work to arrive in; it is written to LDS (two buffers) one step before its use.
  // Loads are unconditional; a chunk past K (it would read the next row) is zeroed when it is
  // written to LDS.
  const u32x4 zero = {0u, 0u, 0u, 0u};
  u32x4 ra[2][4], rb[2][4];
  auto fetch = [&](int set, int k0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ra[set][j] = __builtin_amdgcn_raw_buffer_load_b128(rs_a, voff_a, (32 * j * ldx + k0) * 2, 0);
      if constexpr (epi_is_glu(EPI))
        rb[set][j] = __builtin_amdgcn_raw_buffer_load_b128(j < 2 ? rs_b0 : rs_b1, voff_b, (32 * (j & 1) * K + k0) * 2, 0);
      else
        rb[set][j] = __builtin_amdgcn_raw_buffer_load_b128(rs_b0, voff_b, (32 * j * K + k0) * 2, 0);
    }
  };
  auto stash = [&](int set, int buf, int k0) {
    // the loaded registers are only ever read here: writing zeros into them instead would make
    // the compiler wait for every load in flight first
    if (k0 + WIDE_BK > K) {                           // a last step that K does not fill
      const bool in = k0 + lc * 8 < K;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        *reinterpret_cast<u32x4*>(&lds_a[buf][(lr + 32 * j) * WIDE_LDS_ROW + lc * 8]) = in ? ra[set][j] : zero;
        *reinterpret_cast<u32x4*>(&lds_b[buf][(lr + 32 * j) * WIDE_LDS_ROW + lc * 8]) = in ? rb[set][j] : zero;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        *reinterpret_cast<u32x4*>(&lds_a[buf][(lr + 32 * j) * WIDE_LDS_ROW + lc * 8]) = ra[set][j];
        *reinterpret_cast<u32x4*>(&lds_b[buf][(lr + 32 * j) * WIDE_LDS_ROW + lc * 8]) = rb[set][j];
      }
    }
  };
  auto step = [&](int k0, int buf) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      u32x4 fa[4], fb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        fa[i] = *reinterpret_cast<const u32x4*>(&lds_a[buf][(64 * wy + 16 * i + r) * WIDE_LDS_ROW + kk * 32 + g * 8]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        fb[j] = *reinterpret_cast<const u32x4*>(&lds_b[buf][(brow[j] + r) * WIDE_LDS_ROW + kk * 32 + g * 8]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(fa[i]), as_bf16x8(fb[j]), acc[i][j], 0, 0, 0);
    }
    if constexpr (TOT) {
      const int kn = k0 + WIDE_BK;
      if (kn % GEMM_SEG == 0 || kn >= K) {          // a segment ends: join it to the total, left to right
        const bool first = k0 < GEMM_SEG;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if constexpr (EPI == EPI_ADD_F32) {
              if (first) {                          // the chain of additions starts at the residual
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  const int m = m0 + 64 * wy + 16 * i + 4 * g + q, n = n0 + 64 * wx + 16 * j + r;
                  tot[i][j][q] = (m < M && n < N) ? ((const float*)out)[(size_t)m * ldo + n] : 0.0f;
                }
              }
              tot[i][j] = tot[i][j] + acc[i][j];
            } else {
              tot[i][j] = first ? acc[i][j] : tot[i][j] + acc[i][j];
            }
            acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
          }
      }
    }
  };

  fetch(0, 0);
  fetch(1, WIDE_BK);
  stash(0, 0, 0);
  __syncthreads();
  if constexpr (FAST) {
    // K is a multiple of 128: every step is whole, and a step's body is one straight run of
    // instructions that the scheduler is told how to interleave, so that the LDS traffic and the
    // global loads hide behind the matrix instructions of the same wave:
    //   8 operand reads (first half of the step);
    //   8 x [2 matrix instructions, 1 operand read (second half), 1 global load (the tile after next)];
    //   8 x [2 matrix instructions, 1 LDS write (the next tile, loaded a step ago)].
    // (What then bounds the kernel is how many bytes of tile loads a compute unit can keep in
    // flight: about 45 KB, which at the latency of the L2 is a little more than the 64 KB a step
    // of two resident workgroups asks for.)
    auto fast_step = [&](int k0, int set_fetch, int buf) {
      const int set_stash = set_fetch ^ 1;
      fetch(set_fetch, k0 + 2 * WIDE_BK);             // past K: outside the descriptors, zeros, never used
      u32x4 fa[2][4], fb[2][4];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          fa[kk][i] = *reinterpret_cast<const u32x4*>(&lds_a[buf][(64 * wy + 16 * i + r) * WIDE_LDS_ROW + kk * 32 + g * 8]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          fb[kk][j] = *reinterpret_cast<const u32x4*>(&lds_b[buf][(brow[j] + r) * WIDE_LDS_ROW + kk * 32 + g * 8]);
      }
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(fa[kk][i]), as_bf16x8(fb[kk][j]), acc[i][j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        *reinterpret_cast<u32x4*>(&lds_a[buf ^ 1][(lr + 32 * j) * WIDE_LDS_ROW + lc * 8]) = ra[set_stash][j];
        *reinterpret_cast<u32x4*>(&lds_b[buf ^ 1][(lr + 32 * j) * WIDE_LDS_ROW + lc * 8]) = rb[set_stash][j];
      }
      __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
      }
      __syncthreads();
    };
    for (int k0 = 0; k0 < K; k0 += 2 * WIDE_BK) {
      fast_step(k0, 0, 0);
      fast_step(k0 + WIDE_BK, 1, 1);
    }
  } else
  // steps in pairs, so that register sets and buffers are named at compile time
  for (int k0 = 0; k0 < K; k0 += 2 * WIDE_BK) {
    fetch(0, k0 + 2 * WIDE_BK);
    step(k0, 0);
    stash(1, 1, k0 + WIDE_BK);
    __syncthreads();
    if (k0 + WIDE_BK >= K) break;
    fetch(1, k0 + 3 * WIDE_BK);
    step(k0 + WIDE_BK, 1);
    stash(0, 0, k0 + 2 * WIDE_BK);
    __syncthreads();
  }

  if constexpr (TOT) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = tot[TOT ? i : 0][TOT ? j : 0];
  }
  tile_epilogue<EPI, 4>(acc, out, M, N, ldo, m0 + 64 * wy, n0 + (epi_is_glu(EPI) ? 32 : 64) * wx, (n0 >> 6) + wx, r, g,
                        TOT, rp);
}
