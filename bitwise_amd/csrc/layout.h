// Index arithmetic of the kernels that normalise rows into LDS in front of a matrix product, as plain functions
// that compile for the host too: which shapes a launcher admits, how many bytes of LDS it asks for, where a lane
// stores and reads there, and which vector of a row a lane loads from memory.  The kernels call these functions
// and nothing else for those addresses, so a host program can walk every admitted shape, wave, lane and step and
// check each offset against the launch's own sizes (tests/layout_sweep.cpp does, with the compiler's address and
// undefined-behaviour checks switched on).  No HIP header is needed to include this file.
#pragma once

#include <stddef.h>

#if defined(__HIPCC__)
#define BW_HD __host__ __device__ __forceinline__
#else
#define BW_HD inline
#endif

enum { EPI_F32 = 0, EPI_BF16 = 1, EPI_ADD_F32 = 2, EPI_SWIGLU_BF16 = 3, EPI_QKV_ROPE = 4, EPI_CLAMPED_GLU_BF16 = 5, EPI_GELU_BF16 = 6, EPI_SIDE_BF16 = 7, EPI_GELU_GLU_BF16 = 8 };

// Epilogues that take the stacked weight [gate rows; up rows] and store act(gate) * up.
BW_HD constexpr bool epi_is_glu(int epi) { return epi == EPI_SWIGLU_BF16 || epi == EPI_CLAMPED_GLU_BF16 || epi == EPI_GELU_GLU_BF16; }

#define GEMM_SEG 2048                 // a segment of K: sums of different segments are joined left to right
#define BW_LDS_LIMIT (160 * 1024)     // bytes of LDS a workgroup of gfx950 may ask for

// ------------------------------------------------------------------------------ rows held in a wave's registers

// Lane ``lane`` owns the 16-byte vectors lane, lane + 64, ... of a row of ``nvec`` vectors; its j-th register
// holds vector 64 j + lane, or, past the row's end, the row's last vector again (loaded so that no load is
// conditional, never used).
BW_HD int norm_vec_index(int j, int lane, int nvec) {
  const int c = 64 * j + lane;
  return c < nvec ? c : nvec - 1;
}
BW_HD bool norm_vec_in_row(int j, int lane, int nvec) { return 64 * j + lane < nvec; }

// ------------------------------------------------------------------------------ gemm_bf16_mid_kernel

// The shape of gemm_bf16_mid_kernel's workgroup and ring for one set of template arguments (see the kernel).
template <int EPI, int NRB, bool NORM, bool NARROW = false, bool EIGHT = false>
struct MidShape {
  static constexpr bool GLU = EPI == EPI_SWIGLU_BF16;
  static constexpr bool HALVES = GLU || NARROW;                     // waves are (strip, half of the row blocks)
  static constexpr int NW = EIGHT ? 8 : 4;                          // waves
  static constexpr int COLS = HALVES ? 32 : 64;                     // output columns a workgroup
  static constexpr int B_ROWS = NARROW ? 32 : 64;                   // rows of W a step (SwiGLU: 32 gate, 32 up)
  static constexpr int SUB = EIGHT ? (B_ROWS == 64 ? (NORM || NRB == 4 ? 1 : 2) : (NORM ? 2 : 4)) : 1;   // steps of 64 along K a stage (NORM: weights only)
  static constexpr int STRIPS = COLS / 16, GROUPS = NW / STRIPS;    // wave = (strip of the columns, group of the row blocks)
  static constexpr int A_LOADS = NORM ? 0 : (SUB * 2 * NRB + NW - 1) / NW; // per wave and stage: 8 rows of x each
  static constexpr int B_LOADS = SUB * B_ROWS / 8 / NW;             // 8 rows of W each
  static constexpr int LPW = A_LOADS + B_LOADS;
  static constexpr int A_BYTES = NORM ? 0 : NRB * 2048, STEP_BYTES = A_BYTES + B_ROWS * 128, STAGE = SUB * STEP_BYTES;
  static constexpr int NI = NRB >= GROUPS ? NRB / GROUPS : 1;       // blocks of rows a wave works on (fewer blocks than groups: waves that only load)
  static constexpr int NJ = GLU ? 2 : 1;
  static constexpr bool ROPE_NARROW = NARROW && EPI == EPI_QKV_ROPE;  // a workgroup = 16 rotary pairs of a head
  // 17 rows or more: a ring of at most 72 KB, so that two workgroups share a compute unit and one's first loads
  // and epilogue lie under the other's steps (products with more workgroups than compute units: gate|up 17.2 ->
  // 16.0 us, the 8B shape's 53 -> 50 and its down projection 37 -> 35; the others unchanged); never fewer than 3
  static constexpr int FIT0 = (NORM || NRB < 2 ? 150 : 72) * 1024 / STAGE;
  static constexpr int FIT = FIT0 < 3 ? 3 : FIT0;
  static constexpr int STAGES = EIGHT ? (NORM ? 8 : (FIT > 6 ? 6 : FIT))
                                      : (ROPE_NARROW && NRB <= 2 ? 16 : 8);   // (half the weights a stage: twice the stages, where they fit)
  static constexpr int PENDING = LPW * (STAGES - 2);                // loads that may still be in flight at a step's start
  static constexpr int RING = STAGES * STAGE + 1024;                // and 1 KB where padding loads put their zeros
  static_assert(PENDING < 64, "the wait count has six bits");
  static_assert(STAGES >= 3, "a stage at hand, one landing, one asked for");
  static_assert(!NORM || NRB == 1, "rows are normalised in the kernel only up to 16 of them");
  static_assert(!NARROW || (!GLU && (EPI == EPI_QKV_ROPE || NRB >= 2)), "narrow tiles: plain epilogues of 17 rows or more, or the rotary one");
  static_assert(!EIGHT || NORM || (NRB >= 2 && (SUB * 2 * NRB) % NW == 0), "eight waves: 17 rows or more, or rows normalised in the kernel");
};

// A block of 16 rows of one step of 64 along K is 2 KB: rows 0-7 then rows 8-15, 128 bytes a row, the row's eight
// 16-byte chunks permuted by the row's number so that the operand reads of a wave hit distinct banks.  Lane
// (g = lane / 16, r = lane % 16) of a matrix instruction wants row r, chunk 4 kk + g for the half step kk.
BW_HD int mid_operand_offset(int r, int g, int kk) {
  return (r >> 3) * 1024 + (r & 7) * 128 + (((4 * kk + g) ^ (r >> 1)) * 16);
}

// The ring: stage ``step % STAGES``; a load is 8 rows of one step of 64 along K (1 KB).  Of x: block ``id % (2 NRB)``
// of step ``id / (2 NRB)`` of the stage for the wave's t-th load (ids past the stage's blocks are padding loads, whose
// zeros go behind the ring); of W likewise (SwiGLU with eight waves: the first four waves take the gate rows, the
// others the up rows, so that a wave's loads share a descriptor).  A step's bytes: the blocks of x, then those of W.
template <class S> BW_HD int mid_stage_offset(int step) { return (step % S::STAGES) * S::STAGE; }
template <class S> BW_HD int mid_padding_offset() { return S::STAGES * S::STAGE; }
template <class S, int NRB> BW_HD bool mid_a_load(int wave, int t, int& sub, int& block) {
  const int id = wave * S::A_LOADS + t;
  sub = id / (2 * NRB);
  block = id % (2 * NRB);
  return id < S::SUB * 2 * NRB;
}
template <class S> BW_HD int mid_a_dst(int sub, int block) { return sub * S::STEP_BYTES + block * 1024; }
template <class S> BW_HD void mid_b_load(int wave, int t, int& sub, int& blk) {
  constexpr int PER_STEP = S::B_ROWS / 8;
  if (S::NW == 8 && S::GLU) {                                        // waves 0-3: the gate rows, 4-7: the up rows
    const int id = (wave & 3) * S::B_LOADS + t;
    sub = id / (PER_STEP / 2);
    blk = id % (PER_STEP / 2) + (PER_STEP / 2) * (wave >> 2);
  } else {
    const int id = wave * S::B_LOADS + t;
    sub = id / PER_STEP;
    blk = id % PER_STEP;
  }
}
template <class S> BW_HD int mid_b_dst(int sub, int blk) { return sub * S::STEP_BYTES + S::A_BYTES + blk * 1024; }
// a wave's operand reads of W inside a step: its (gate) strip, the up strip 4 KB further
template <class S> BW_HD int mid_b_read_offset(int strip, int j, int r, int g, int kk) {
  return S::A_BYTES + strip * 2048 + j * 4096 + mid_operand_offset(r, g, kk);
}
// which block of 16 rows a wave starts at, and whether it has rows to work on at all (waves beyond the blocks of
// rows only load)
template <class S> BW_HD int mid_first_block(int wave) { return S::NI * (wave / S::STRIPS); }

// NORM variant: what the launcher admits.  Rows of one segment of K: up to 16 of them (LDS holds blocks of 16 rows,
// 2048 bytes a step).  Rows of up to two segments: up to 8, a row a wave, blocks of 8 rows, 1024 bytes a step.
// ``tiles``: workgroups of the launch (the kernel is for products with at least 64).
BW_HD bool mid_norm_admits(int M, int K, int tiles) {
  if (M < 1 || M > 16 || K < 64 || K % 64 || tiles < 64) return false;
  if (K > GEMM_SEG && (M > 8 || K > 2 * GEMM_SEG || K % 128)) return false;
  return true;
}
BW_HD int mid_norm_row_step(int K) { return K > GEMM_SEG ? 1024 : 2048; }

// Which rows a wave normalises: rows wave, wave + NW, ..., as many at a time as the rows need (a slot without a row
// would fetch a row for nothing); and how many 16-byte vectors of a row a lane holds: 8 (rows of one segment), or
// 16 (rows of two, which by the admission above are at most a row a wave of the eight-wave variant).
BW_HD int mid_norm_row_of(int wave, int i, int nw) { return wave + i * nw; }
BW_HD int mid_norm_rows_a_wave(int M, int nw) { return (M + nw - 1) / nw; }
BW_HD int mid_norm_vectors_a_lane(int K) { return K > GEMM_SEG ? 16 : 8; }

// Where vector c (elements 4c..4c+3 as four bfloat16, 8 bytes) of row m goes, relative to the rows' area: step
// c / 16, chunk (c % 16) / 2 of the step permuted as above, half c % 2 of the chunk.
BW_HD int mid_norm_store_offset(int c, int m, int row_step) {
  return (c >> 4) * row_step + (m >> 3) * 1024 + (m & 7) * 128 + ((((c & 15) >> 1) ^ ((m & 15) >> 1)) * 16) + (c & 1) * 8;
}

// Where lane (g, r) reads its 16 bytes of step ``k_step`` (of 64 along K) for the half step kk, relative to the rows' area.
BW_HD int mid_norm_read_offset(int k_step, int a_block, int row_step, int r, int g, int kk) {
  return k_step * row_step + a_block * 2048 + mid_operand_offset(r, g, kk);
}

// Bytes of LDS of a NORM launch: the ring, then the rows (8-row blocks: the reads of rows 8 to 15, which do not
// exist, end a block further).
BW_HD int mid_norm_lds_bytes(int ring, int K, int row_step) {
  return ring + (K / 64) * row_step + (row_step == 1024 ? 1024 : 0);
}

// ------------------------------------------------------------------------------ gemm_bf16_norm_strips_kernel

// A workgroup of eight waves takes ``strips`` (five to eight) strips of 16 rows of W, a wave each (SwiGLU: eight gate rows and the
// eight up rows of the same outputs).  LDS: [strips][stages][16 rows of W of a step, 128 bytes each, chunks permuted as above], then the
// rows as in the NORM variant.
#define NORM_STRIP_STAGE 2048
BW_HD constexpr int norm_strips_cols(bool glu) { return glu ? 8 : 16; }                                  // outputs a strip
BW_HD constexpr int norm_strips_stages(int strips) { return strips == 5 ? 9 : strips == 6 ? 7 : strips == 7 ? 6 : 5; }   // (as many as LDS holds beside the rows' 65 KB)
BW_HD constexpr int norm_strips_ring(int strips, int stages) { return strips * stages * NORM_STRIP_STAGE; }
BW_HD constexpr int norm_strips_ring_of(int wave, int stages) { return wave * stages * NORM_STRIP_STAGE; }
BW_HD constexpr int norm_strips_next(int at, int stages) { return at == (stages - 1) * NORM_STRIP_STAGE ? 0 : at + NORM_STRIP_STAGE; }
BW_HD constexpr int norm_strips_before(int at, int stages) { return at == 0 ? (stages - 1) * NORM_STRIP_STAGE : at - NORM_STRIP_STAGE; }

// A wave's strip: its first output, and the rows of W behind its two descriptors (strip rows 0 to 7 and 8 to 15; ``working`` false: the wave
// has no strip and only normalises).  A descriptor of no rows gives zeros wherever a lane points in it.
struct NormStrip {
  bool working;
  int n0, have;                        // first output, and how many of the strip's outputs there are
  size_t row[2];                       // first row of W of each half
  int rows[2];
};
BW_HD NormStrip norm_strips_of_wave(bool glu, int block, int strips, int wave, int N) {
  NormStrip s;
  const int cols = norm_strips_cols(glu), first = (block * strips + wave) * cols;
  s.working = wave < strips && first < N;
  s.n0 = s.working ? first : 0;
  s.have = cols < N - s.n0 ? cols : N - s.n0;
  s.rows[0] = s.have < 8 ? s.have : 8;
  s.rows[1] = glu ? s.have : (s.have > 8 ? s.have - 8 : 0);
  s.row[0] = (size_t)s.n0;
  s.row[1] = (size_t)(glu ? N + s.n0 : (s.rows[1] ? s.n0 + 8 : s.n0));
  return s;
}
// Where a lane points in the descriptor of half ``half``, in bytes (a step further: 128 more), and where its 16 bytes land in the stage.
BW_HD int norm_strips_load_offset(int half, int lane, int K) {
  const int row = lane >> 3, slot = lane & 7;
  return (row * K + 8 * (slot ^ ((8 * half + row) >> 1))) * 2;
}
BW_HD constexpr int norm_strips_half(int half) { return half * 1024; }

// How many strips a workgroup takes, or 0: the NORM variant of the kernel for up to 64 rows.  Counted in what a strip of a full round
// of the compute units takes (2.9 us for K = 2048, at 5.4 TB/s): a round its strips and 0.8 for its beginning, a part-empty last
// round no less than 0.44 of its strips (what one compute unit pulls).  5 rows, us, that variant -> strips as many as the count takes (the best of 5 to 8):
//   SwiGLU   11008 x 4096 46.4 -> 38.4 (7)   14336 x 4096 50.1 -> 47.7 (7)   18432 x 4096 68.6 -> 63.4 with 6 (62.6 with 5)
//            9728 x 2560 28.7 -> 22.6 with 7 (22.1 with 6)   12000 x 2048 25.5 -> 24.6 with 6 (23.8 with 8)   16384 x 2048 32.0 -> 31.4 (8)
//   stores   128256 x 4096 202 -> 194 (7)   20000 x 1024 14.6 -> 11.2 with 5 (10.9 with 7)
// Where both make whole rounds the variant is as fast or faster (8192 x 2048 17.7, 17.9 with 8; stores of K = 2048: 49152 columns 44.4
// and 46.1 with 7, 32000 29.7 and 30.7 with 8), so it stays unless the count says 4 % less, 10 % for stores of one segment, 6 % for those of
// two (47936 x 2176 stays at 42.8, 42.2 with 6).  385 products drawn over all of that: 0.62 to 1.03 of the variant's time (two above 1.01), 0.88 in the mean.
inline int norm_strips_admits(int M, int N, int K, int epilogue) {
  const bool glu = epilogue == EPI_SWIGLU_BF16;
  if ((!glu && epilogue != EPI_F32) || !mid_norm_admits(M, K, (N + (glu ? 31 : 63)) / (glu ? 32 : 64))) return 0;
  const auto cost = [&](int strips) {                                  // in 1/10000
    const int cols = strips * norm_strips_cols(glu);
    const long long wgs = (N + cols - 1) / cols, left = wgs % 256;
    const long long rounds = wgs / 256 * 10000 + (left ? (left * 10000 / 256 > 4400 ? left * 10000 / 256 : 4400) : 0);
    return strips * rounds + (wgs + 255) / 256 * 8000;
  };
  const long long variant = cost(4);
  long long least = variant * (glu ? 96 : K <= GEMM_SEG ? 90 : 94) / 100;
  int best = 0;
  for (int strips = 5; strips <= 8; ++strips) {
    // eight: a ring of five stages; seven in more than one round: where the count is even with six those are faster (21000 x 2944 46.8 and
    // 50.1, variant 47.3; stores of 42000 x 2944 49.0 and 52.3, 51.3)
    const bool rounds = (N + strips * norm_strips_cols(glu) - 1) / (strips * norm_strips_cols(glu)) > 256;
    const long long c = strips == 8 ? cost(strips) * 103 / 100 : strips == 7 && rounds ? cost(strips) * 1005 / 1000 : cost(strips);
    if (c < least) {
      least = c;
      best = strips;
    }
  }
  return best;
}

// ------------------------------------------------------------------------------ decode_gemm_kernel (fused_decode.hip)

#define DEC_SEG 2048
#define DEC_MAX_LDS (BW_LDS_LIMIT - 1024)

// LDS: [M rows of K + 8 bfloat16 (16 bytes of padding: operand reads hit distinct banks)] rounded up to 16 bytes,
// then a ring of ``stages`` stages of ``stage_bytes`` for each wave.
BW_HD int decode_lds_row(int K) { return K + 8; }                                  // bfloat16 elements
BW_HD size_t decode_rows_bytes(int M, int K) { return ((size_t)M * decode_lds_row(K) * 2 + 15) & ~(size_t)15; }
BW_HD size_t decode_ring_offset(int M, int K, int wave, int stages, int stage_bytes) {
  return decode_rows_bytes(M, K) + (size_t)wave * stages * stage_bytes;
}
BW_HD size_t decode_lds_bytes(int M, int K, int waves, int stages, int stage_bytes) {
  return decode_rows_bytes(M, K) + (size_t)waves * stages * stage_bytes;
}
// Can the rows live in LDS beside 64 KB of rings, and does a row fit a wave's registers?
BW_HD bool decode_gemm_admits(int M, int N, int K, int lda) {
  if (M <= 0 || M > 16 || N <= 0 || K <= 0 || (K % 64)) return false;
  if (K > DEC_SEG || (lda % 4) || lda < K) return false;
  if ((size_t)M * decode_lds_row(K) * 2 + 64 * 1024 > DEC_MAX_LDS) return false;
  return true;
}
// bfloat16 element where vector c of row m is stored, and where lane (g, r) reads its 8 elements of a step's half kk
// (rows past M read row 0; their products are thrown away).
BW_HD size_t decode_norm_store_elem(int m, int c, int K) { return (size_t)m * decode_lds_row(K) + 4 * c; }
BW_HD size_t decode_operand_elem(int r, int M, int g, int step, int kk, int K) {
  return (size_t)(r < M ? r : 0) * decode_lds_row(K) + 8 * g + 64 * step + 32 * kk;
}
// Byte offset inside a stage of a wave's ring (16 rows of W, 128 bytes each, chunks permuted as above).
BW_HD int decode_ring_operand_offset(int r, int g, int kk) { return mid_operand_offset(r, g, kk); }
