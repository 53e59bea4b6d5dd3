// bfloat16 matrix product on the matrix cores: y[m][n] = sum_k x[m][k] * W[n][k],
// x bfloat16 [M][K], W bfloat16 row-major [N][K], 32-bit accumulation.
//
// Arithmetic, the same for every M (one row or thousands): K is cut into segments of 2048
// (a property of the weight, never of the batch).  Within a segment each 16x16 block of
// outputs is one accumulator that runs v_mfma_f32_16x16x32_bf16 over k ascending in steps
// of 32 from zero; within an instruction lane group g holds k = kk+8g..kk+8g+7.  Segment
// results are added in 32-bit left to right: y = ((p0 + p1) + p2) + ..., and where the product
// is added into a residual the chain starts there: y = ((res + p0) + p1) + ...  An output's bits
// therefore depend only on its own row of x and row of W (and its own residual).
//
// Several kernels run this arithmetic; which one is a matter of the shape alone (rows, columns, K), never of the
// values, and they agree bit for bit (the tests compare them).  What bounds them all is how many bytes of loads
// a compute unit keeps in flight and fetches through its L1, so each shape gets the kernel that fetches least:
//   * up to 64 rows (decode steps, short prompt portions):
//       - many columns: the "mid" kernel, a workgroup per 64 columns (32 of SwiGLU, or 32 where there are few
//         columns and more than 16 rows), the rows of x shared by its four strips; optionally RMSNorm of up to 16
//         rows fused in front (the rows normalised into LDS by the workgroup) and rotation + cache write behind
//         (a head a workgroup, or with fewer than 256 heads 16 rotary pairs of one);
//         a residual add of 17 to 64 rows over several segments gives every segment workgroups of its own, which
//         meet in device scratch and are added in segment order by the last to arrive;
//       - up to 16 rows and few columns, or several segments: the "stream" kernel, a wave per strip and segment;
//       - both stream weights and x through rings in LDS filled by buffer loads with LDS as their destination,
//         8 rows of 128 bytes an instruction (whole cache lines; half lines cost nearly as much as whole ones),
//         no registers in between, so the rings are deep; the 16-byte chunks of a row are permuted so that operand
//         reads hit distinct banks; a wave waits for "all but the loads of the stages after this one", which
//         works because loads complete in the order they are issued and nothing else is loaded meanwhile;
//       - anything else (K no multiple of 64, SwiGLU with few columns): the "skinny" kernel, a wave per strip
//         and segment streaming through a ring of registers;
//   * more rows (prompt portions): tiles of 8,192 to 65,536 outputs (64 x 128 to 256 x 256), eight waves, steps of 64 along K fed through
//     rings in LDS by the same kind of loads (gemm_bf16_ring.h); the shape is the one whose rounds of the compute units
//     take the least time.  Several segments are joined in registers, or, for a residual add with scratch and few tiles, a
//     workgroup per tile and segment leaves its sums for a second kernel that joins them in order.  The "wide" kernel (128 x
//     128 tiles staged through registers by four waves) takes K that is no multiple of 64.
//
// Epilogues: store 32-bit, store bfloat16, add into a 32-bit residual (each output owned
// by one lane: no atomics), SwiGLU of two products (gate rows n, up rows N+n of a
// stacked weight) stored as bfloat16: h = g * (1/(1+exp(-g))) * u in 32-bit, the exact GELU stored as bfloat16, or rotary encoding of the
// stacked q|k|v product and the write of k and v to their page slots (heads of 64; up to 64 rows: head sizes
// in multiples of 64).
#include <algorithm>
#include <mutex>

#include "common.h"
#include "api.h"
#include "layout.h"        // the epilogues' numbers, GEMM_SEG, MidShape and the LDS layout of the rows normalised in the kernel

// What the rotary epilogue of the stacked q|k|v product needs: the statements of
// rope_kvwrite_kernel on the 32-bit products while they are still in registers.
struct QkvRopeArgs {
  const int32_t* positions;    // [rows]; negative = padding row
  const int32_t* row_seq;      // [rows] -> row of the block table
  const int32_t* block_table;
  const float* cos_table;      // [max_pos, 32]
  const float* sin_table;
  bf16_t* k_cache;
  bf16_t* v_cache;
  int heads, kv_heads, page_size, table_stride, write_cache;
  int page_shift;              // page_size is a power of two: positions are split by shift and mask, not by division
  int head_dim = 64;           // (the kernels for up to 64 rows take multiples of 64; the tiled ones 64)
  float glu_limit = 0.0f, glu_alpha = 1.0f;   // EPI_CLAMPED_GLU_BF16 only: the clamp and the sigmoid's slope
};

// ------------------------------------------------------------------------------ phases of one launch
//
// A decode step is a row of small kernels, each of which has to wait for the one before it, and the end of one
// kernel and the start of the next cost as much as many of them take to stream their weights.  The kernels for up
// to 16 rows can therefore also run as phases of ONE launch: the workgroups of phase 0 come first in block order, then
// those of phase 1, and so on.  Workgroups are handed to the compute units in block order, so when a workgroup runs
// every workgroup of the phases before it is running or done; it asks for its weights at once (they depend on
// nothing), then waits until the phase before it has counted all of its workgroups in (a flag that the last of them
// sets; the wait is bounded: a wave that gives up sets a bit of an error word and goes on, nothing hangs), and only
// then reads what that phase wrote.  What one phase writes and a later one reads travels with stores and loads
// of device scope: the dies' L2s are not coherent with each other, a plain load could hit a stale line.  The
// arithmetic of a phase is the statements of its kernel: the same bits.
struct ChainCtx {
  int bx, by, bz, gx, gy, gz;      // the workgroup's place in its phase's grid, and that grid
  int waves;                       // waves of a workgroup of this phase
  const int* wait_flag;            // null: this phase waits for nothing
  int* err;                        // a word that gets bit err_bit when a wait gives up
  int err_bit, spin_limit;
};

__device__ __forceinline__ ChainCtx launch_ctx() {
  return ChainCtx{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, (int)gridDim.x, (int)gridDim.y, (int)gridDim.z,
                  (int)(blockDim.x >> 6), nullptr, nullptr, 0, 0};
}

// The workgroup waits for the phase before its own (every wave of the workgroup calls this).
template <bool CH>
__device__ __forceinline__ void chain_wait(const ChainCtx& cc) {
  if constexpr (CH) {
    if (cc.wait_flag == nullptr) return;
    if (threadIdx.x == 0) {
      int spins = 0;
      while (__hip_atomic_load(cc.wait_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
        if (++spins > cc.spin_limit) {
          atomicOr(cc.err, 1 << cc.err_bit);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    __syncthreads();
    asm volatile("" ::: "memory");
  }
}

// Loads and stores of what another phase of the same launch wrote or will read (DEV), else plain ones.
template <bool DEV>
__device__ __forceinline__ float ld_f32(const float* p) {
  if constexpr (DEV) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else return *p;
}
template <bool DEV>
__device__ __forceinline__ void st_f32(float* p, float v) {
  if constexpr (DEV) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}
template <bool DEV>
__device__ __forceinline__ void st_bf16(bf16_t* p, bf16_t v) {
  if constexpr (DEV) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}

template <int EPI, bool DEV = false>
__device__ __forceinline__ void epilogue_store(void* __restrict__ out, size_t o, float v, float u, float limit = 0.0f,
                                               float alpha = 1.0f) {
  if constexpr (EPI == EPI_F32) st_f32<DEV>((float*)out + o, v);
  else if constexpr (EPI == EPI_BF16) st_bf16<DEV>((bf16_t*)out + o, f32_to_bf16(v));
  else if constexpr (EPI == EPI_GELU_BF16) st_bf16<DEV>((bf16_t*)out + o, f32_to_bf16(gelu_erf(v)));
  else if constexpr (EPI == EPI_ADD_F32) st_f32<DEV>((float*)out + o, ld_f32<DEV>((const float*)out + o) + v);
  else if constexpr (EPI == EPI_SWIGLU_BF16) st_bf16<DEV>((bf16_t*)out + o, f32_to_bf16(silu_times(v, u)));
  else if constexpr (EPI == EPI_CLAMPED_GLU_BF16) st_bf16<DEV>((bf16_t*)out + o, f32_to_bf16(clamped_swish_times<true>(v, u, limit, alpha)));
  else if constexpr (EPI == EPI_GELU_GLU_BF16) st_bf16<DEV>((bf16_t*)out + o, f32_to_bf16(gelu_tanh_times(v, u)));
}

// EPI_SIDE_BF16 (up to 16 rows): an output is the GELU (tanh form) of its sum times the element of its row's token in a table, rounded
// to bfloat16: the statements of side_gate_kernel on the sums while they are still in registers.
struct SideGateArgs {
  const int32_t* tokens = nullptr;
  const int32_t* feedback = nullptr;
  const bf16_t* table = nullptr;       // [vocab] rows of ldt elements, column n of the product at element n
  int ldt = 0, vocab = 0;
};
template <int EPI>
__device__ __forceinline__ int side_token(const SideGateArgs& sg, int m) {
  if constexpr (EPI == EPI_SIDE_BF16) {
    int tok = sg.tokens[m];
    if (tok == BW_TOKEN_FROM_FEEDBACK && sg.feedback != nullptr) tok = sg.feedback[m];
    return tok;
  } else {
    return 0;
  }
}
__device__ __forceinline__ void side_store(const SideGateArgs& sg, int tok, int n, bf16_t* out, float z) {
  float v = 0.0f;
  if (tok >= 0 && tok < sg.vocab) v = gelu_tanh(z) * bf16_to_f32(sg.table[(size_t)tok * sg.ldt + n]);
  *out = f32_to_bf16(v);
}

// (host) The phases asked for while a chain is open wait in a list and leave as one launch (further down).
struct MidCall;
struct RowsCall;
static bool chain_is_open();
static int chain_flush(hipStream_t s);
static int chain_record_mid(int kind, const MidCall& c, int wgs, int lds_bytes, hipStream_t s);
static int chain_record_rows(int kind, const RowsCall& c, int wgs, int waves, int lds_bytes, hipStream_t s);

// Every other launch of this file: what waits in an open chain goes first.
#define BW_LAUNCH(kernel, grid, block, lds, stream, ...)                \
  do {                                                                  \
    if (chain_is_open()) (void)chain_flush(stream);                     \
    hipLaunchKernelGGL(kernel, grid, block, lds, stream, __VA_ARGS__);  \
  } while (0)

#include "gemm_bf16_skinny.h"
#include "gemm_bf16_tiles.h"
#include "gemm_bf16_ring.h"
#include "gemm_bf16_rows.h"
#include "gemm_bf16_phases.h"

// ------------------------------------------------------------------------------ launch

// How a residual add of 17 to 64 rows runs in the kernel above: 64 or 32 columns a workgroup (as many workgroups
// as there are compute units, if the product has them), a workgroup per tile and segment of K if there are several
// (they meet in device scratch the caller brings).  tiles 0: it does not run there.
// out = (((out + p[0]) + p[1]) + ...) + p[S-1], element by element: the segments of a residual add that
// the tiles left in scratch ([S][M][N]), joined in segment order (ADD false: a store, the chain starts at p[0]).
template <bool ADD>
__global__ __launch_bounds__(256) void add_segments_kernel(float* __restrict__ out, const float* __restrict__ parts, int S,
                                                           int M, int N, int ldo) {
  const size_t quads = (size_t)M * (N >> 2);
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= quads) return;
  const int m = (int)(i / (N >> 2)), n = 4 * (int)(i % (N >> 2));
  float* o = out + (size_t)m * ldo + n;
  f32x4 y = *reinterpret_cast<const f32x4*>(ADD ? o : parts + (size_t)m * N + n);
  for (int sg = ADD ? 0 : 1; sg < S; ++sg) y = y + *reinterpret_cast<const f32x4*>(parts + ((size_t)sg * M + m) * N + n);
  *reinterpret_cast<f32x4*>(o) = y;
}

static void add_rows_shape(int M, int N, int K, int& tiles, bool& narrow) {
  const int S = (K + GEMM_SEG - 1) / GEMM_SEG;
  tiles = 0;
  narrow = false;
  if (M <= 16 || M > 64 || K % 64) return;
  narrow = ((N + 63) / 64) * S < 256;
  tiles = narrow ? (N + 31) / 32 : (N + 63) / 64;
  if (tiles * S < 32) tiles = 0;
}

// How a residual add (or 32-bit store) of more than 64 rows is laid out.
//   blocks at once  the kernel for up to 64 rows with all blocks of 64 rows in one launch (its
//               grid's third dimension), while the workgroups fit the chip at once (512; a store of one segment: as
//               store_in_blocks has it): the output projection of 2048 columns takes 8.4 us at 128 rows and 13.3 at 512,
//               where 128 x 128 tiles took 16.4 and 21.6.  The q|k|v product with rotation and cache write goes the
//               same way (launch_qkv_rope_mid).
//   row blocks  the kernel for up to 64 rows once per block of 64 rows, with its workgroup per 32 or 64 columns and
//               segment of K (its scratch if K has several segments): up to 128 rows and three segments, where a
//               launch more costs less than the join below (K = 2048: 16 and 19 us at 65 and 128 rows, for 24).
//   whole       a workgroup per tile with all of K, the segments joined in registers: needs no scratch.
//   split       a workgroup per tile and segment, the segments' sums whole in scratch and joined in order
//               afterwards: where few tiles of all of K would leave most of the chip idle (128 rows of 2048 columns are 16
//               of 128 x 128, each 128 steps long for K = 8192: 76 us; 25 split).
// All give the same bits.  Which shapes are asked to bring scratch for a split is a count of rounds and steps
// (add_takes_scratch: what callers of bw_gemm_add_scratch size by, so it stays as it is while the kernels change); whether one that
// brings it is split or goes whole, and in which tiles, the estimated times decide (split_shape, which bw_gemm_split_tile
// and bw_gemm_split_rows tell callers that do not want to hold scratch for nothing).
// tiles64: what the 64-row kernel's scratch is sized by.
enum AddRoute { ADD_WHOLE, ADD_ROW_BLOCKS, ADD_SPLIT };

// "Blocks at once" for a residual add of more than 64 rows: how many blocks of 64 rows, tiles of 64 or (narrow) 32
// columns; tiles 0: it does not run that way (more than 512 workgroups, or too few to matter).  Several segments of K
// meet in scratch: 4096 floats a workgroup, a counter a (block, tile).
#define ADD_BLOCKS_MAX_WGS 512
static void add_blocks_shape(int M, int N, int K, int& tiles, bool& narrow, int& zb) {
  const int S = (K + GEMM_SEG - 1) / GEMM_SEG;
  tiles = 0;
  narrow = false;
  zb = (M + 63) / 64;
  if (M <= 64 || K % 64 || N <= 0) return;
  const int wide = (N + 63) / 64;
  narrow = wide * zb * S < 192;
  const int t = narrow ? (N + 31) / 32 : wide;
  if (t * zb * S >= 32 && t * zb * S <= ADD_BLOCKS_MAX_WGS) tiles = t;
}

// A store of more than 64 rows and one workgroup for all of K: the 64-row kernel with all blocks of 64 rows in one launch, or
// tiles?  While every workgroup has a compute unit to itself (256) the blocks take 0.75 to 0.9 of the tiles' time at any K; two of
// them on a compute unit take turns, and from 257 to 512 workgroups the blocks win only where K is short (0.96 to 1.03 of the tiles'
// time at K = 512, 1.04 to 1.17 at K = 2048; the exact GELU's many instructions run beside the other's products: 0.85 to 0.96 up to K = 1024),
// up to 384 of them at K = 2048 for the GELU (0.95 to 0.99) and for three blocks (192 rows of 8192 columns 15.4 us and 17.0), and up to 320
// for K of several segments (0.92 to 1.02; 1.04 to 1.4 beyond).
static bool store_in_blocks(int M, int N, int K, bool erf) {
  const long long wgs = (long long)((N + 63) / 64) * ((M + 63) / 64);
  if (K <= (erf ? 1024 : 512)) return wgs <= 512;
  if (K <= GEMM_SEG) return wgs <= (erf || M <= 192 ? 384 : 256);
  return wgs <= 320;
}

// Steps of a round times rounds, a step of 256 x 256 tiles counted as two of 128 x 128 and one of 128 x 256 as 8/5 (with
// all of K) or 7/4; the join as the steps it takes time for.  Scratch where a split of some shape saves a tenth.
static bool add_takes_scratch(int M, int N, int K, int ldo) {
  const int S = (K + GEMM_SEG - 1) / GEMM_SEG;
  if (S < 2 || N % 4 || ldo % 4) return false;
  auto tiles = [&](int rows, int cols) { return (long long)((M + rows - 1) / rows) * ((N + cols - 1) / cols); };
  auto rounds = [](long long wgs) { return (wgs + 255) / 256; };
  const long long seg = GEMM_SEG / 64, join = (long long)S * M * N / 500000 + 8;
  const long long whole = rounds(tiles(128, 128)) * (K / 64), whole256 = rounds(tiles(128, 256)) * (K / 64) * 8 / 5;
  const long long by128 = rounds(tiles(128, 128) * S) * seg + join, by256 = rounds(tiles(128, 256) * S) * seg * 7 / 4 + join;
  const long long by_big = M >= 512 ? rounds(tiles(256, 256) * S) * 2 * seg + join : whole;
  const long long split = std::min(std::min(by128, by_big), by256);
  return !(whole256 < whole && whole256 <= split) && 10 * split < 9 * whole;
}

static AddRoute add_route(int M, int N, int K, int ldo, int& tiles64) {
  const int S = (K + GEMM_SEG - 1) / GEMM_SEG;
  tiles64 = 0;
  if (M <= 64 || K % 64) return ADD_WHOLE;
  bool narrow;
  add_rows_shape(64, N, K, tiles64, narrow);
  if (tiles64 && M <= 128 && S <= 3) return ADD_ROW_BLOCKS;
  tiles64 = 0;
  return add_takes_scratch(M, N, K, ldo) ? ADD_SPLIT : ADD_WHOLE;
}

// The join is a launch (3 us) and moves 8 bytes an element and segment and 8 more an element, the stores of the sums among them
// (2048 x 2048, four segments: 28 us in all), at about 9 TB/s, much of it in caches.
static long long add_join_time(int M, int N, int S) { return (8LL * S + 8) * M * N / 90000 + 300; }

// The tiles of a split.  Up to 192 rows always one of 128 x 128 or 128 x 256, counted in rounds and steps as where scratch is asked
// for: the weights' way from memory takes the time there, not the matrix cores, and the times below do not see it (33 products of 129
// to 192 rows, 4096 to 8192 columns and K of 4096 to 14336, every shape timed, split and whole: by the count four take more than 5 %
// longer than the best, up to 27 %; by the times ten, up to 18 %).  More rows: the shape that takes less time than all of K a
// workgroup in one launch (not in the two that ring_parts might make of it); -1: none does (204 products of up to 2,048 rows: 0.8 %
// from the best in the mean).
static int add_split_shape(int M, int N, int K) {
  const int S = (K + GEMM_SEG - 1) / GEMM_SEG;
  if (M <= 192) {
    const long long wgs128 = ring_tiles(ring_costs[RING_128], M, N) * S, wgs256 = ring_tiles(ring_costs[RING_128X256], M, N) * S;
    return (wgs256 + 255) / 256 * 7 < (wgs128 + 255) / 256 * 4 ? RING_128X256 : RING_128;
  }
  long long least;
  int shape = -1;
  ring_choice(M, N, K, false, &least);
  const long long join = add_join_time(M, N, S);
  for (int i = 0; i < RING_SHAPES; ++i) {
    const long long t = ring_time(ring_costs[i], ring_tiles(ring_costs[i], M, N) * S, GEMM_SEG, false) + join;
    if (t < least) {
      least = t;
      shape = i;
    }
  }
  return shape;
}

// The tiles in which a residual add (store: a 32-bit store) of more than 64 rows leaves its segments' sums in scratch of S M N
// floats; -1: it does not, whatever scratch it is given for that.
static int split_shape(int M, int N, int K, int ldo, bool store) {
  int tiles, zb;
  bool narrow;
  add_blocks_shape(M, N, K, tiles, narrow, zb);
  if (tiles || add_route(M, N, K, ldo, tiles) != ADD_SPLIT) return -1;
  // (a store splits only what leaves compute units idle)
  if (store && ((M + 127) / 128) * ((N + 127) / 128) >= 256) return -1;
  return add_split_shape(M, N, K);
}

template <int EPI>
static int launch_gemm_bf16(const bf16_t* x, const bf16_t* w, void* out, int M, int N, int K, int ldx, int ldo,
                            hipStream_t s, const QkvRopeArgs& rp = QkvRopeArgs{}, const MidSplitArgs& sp = MidSplitArgs{},
                            size_t scratch_floats = 0, int num_counters = 0) {
  const int S = (K + GEMM_SEG - 1) / GEMM_SEG;
  constexpr int NB = epi_is_glu(EPI) ? 2 : 1;
  // a 32-bit store may give the segments of K workgroups of their own, too, where the caller brings the scratch
  const bool split_ok = sp.scratch != nullptr && sp.counters != nullptr;
  if (M <= 64) {
    // (the rotary epilogue belongs to the wide kernel; the clamped and the GELU unit of few rows are a kernel behind the 32-bit product)
    if constexpr (EPI == EPI_QKV_ROPE || EPI == EPI_CLAMPED_GLU_BF16 || EPI == EPI_GELU_GLU_BF16) return -2;
    else {
      // one segment and enough columns: the rows of x are shared through LDS
      constexpr int MID_COLS = epi_is_glu(EPI) ? 32 : 64;
      const int wgs = (N + MID_COLS - 1) / MID_COLS;
      // (the descriptors of W cover a tile's rows each, so only the rows of x have to fit 31 bits of offset)
      const bool fits = (size_t)M * ldx * 2 < ((size_t)1 << 31);
      // (a residual add of several segments starts its chain at the residual: the kernels further down do that)
      // (and so does a 32-bit store of up to 16 rows, whose segments those kernels give waves of their own, or with scratch
      // of up to 64 and four segments: 4,096 columns of K = 21,504 at 8 rows took 65 us as 64 workgroups with all of K
      // each, 29 as strips; at 64 rows of K = 8,192 21 us and 17.5, of K = 21,504, where the join weighs more, 33 and 39)
      const bool whole_k = S == 1 || (EPI != EPI_ADD_F32 && !(EPI == EPI_F32 && (M <= 16 ? S <= 40 : split_ok && S <= 4)) &&
                                     !(EPI == EPI_GELU_BF16 && M <= 16 && S <= 40));
      // (up to 16 rows stored as they are: a wave per strip is faster where the workgroups of 64 columns leave half the compute
      // units idle or go into a second round: 5,120 columns of K = 2,048 at 8 rows 12.2 us and 7.8, 17,472 columns 23.4
      // and 19.3)
      const bool strips_win = (EPI == EPI_F32 || EPI == EPI_GELU_BF16) && M <= 16 && S <= 40 && (wgs < 112 || wgs > 256);
      if (whole_k && K % 64 == 0 && wgs >= 64 && fits && !strips_win) {
        if (M <= 16) return launch_mid<EPI, 1, false>(x, w, out, M, N, K, ldx, ldo, wgs, s);
        if (M <= 32) return launch_mid<EPI, 2, false>(x, w, out, M, N, K, ldx, ldo, wgs, s);
        // 33 to 64 rows and so few columns that twice the workgroups still fit the chip at once: two blocks of 32 rows,
        // 32 columns a workgroup, which then pulls half the rows of x and half the weights (4096 columns of K = 2048
        // at 64 rows: 9.5 us against 14.1; 2048 columns, further down: 8.4 against 10.7)
        if constexpr (EPI == EPI_ADD_F32 || EPI == EPI_F32 || EPI == EPI_BF16 || EPI == EPI_GELU_BF16) {
          if (2 * ((N + 31) / 32) <= 256)
            return launch_mid<EPI, 2, false, true>(x, w, out, M, N, K, ldx, ldo, (N + 31) / 32, s, MidNormArgs{}, QkvRopeArgs{}, 1,
                                                   MidSplitArgs{}, 2);
        }
        return launch_mid<EPI, 4, false>(x, w, out, M, N, K, ldx, ldo, wgs, s);
      }
      // a residual add of more than 16 rows and fewer columns (the other kernel for it fetches W once per block of
      // 16 rows): narrower tiles, and several segments if the caller brought scratch for them to meet in
      if constexpr (EPI == EPI_ADD_F32 || EPI == EPI_F32) {
        int tiles;
        bool narrow;
        add_rows_shape(M, N, K, tiles, narrow);
        if (tiles && fits && (S == 1 || split_ok)) {
          if (S > 1 && (scratch_floats < (size_t)tiles * S * 4096 || num_counters < tiles)) return -6;
          const MidNormArgs na{};
          const QkvRopeArgs no{};
          if (narrow) {
            if (M <= 32) return launch_mid<EPI, 2, false, true>(x, w, out, M, N, K, ldx, ldo, tiles, s, na, no, S, sp);
            // one segment and so few tiles that twice as many still fit the chip at once: two blocks of 32 rows, each
            // workgroup then pulls half the rows of x beside its weights
            if (S == 1 && 2 * tiles <= 256)
              return launch_mid<EPI, 2, false, true>(x, w, out, M, N, K, ldx, ldo, tiles, s, na, no, S, sp, 2);
            return launch_mid<EPI, 4, false, true>(x, w, out, M, N, K, ldx, ldo, tiles, s, na, no, S, sp);
          }
          if (M <= 32) return launch_mid<EPI, 2, false>(x, w, out, M, N, K, ldx, ldo, tiles, s, na, no, S, sp);
          return launch_mid<EPI, 4, false>(x, w, out, M, N, K, ldx, ldo, tiles, s, na, no, S, sp);
        }
      }
    }
    if constexpr (!epi_is_glu(EPI) && EPI != EPI_QKV_ROPE) {
      // up to 16 rows: a wave per strip and segment, streaming through its own ring in LDS
      if (M <= 16 && K % 64 == 0 && S <= 40 && (size_t)M * ldx * 2 < ((size_t)1 << 31)) {
        // one segment and few columns: everything asked for at once
        if ((N + 15) / 16 < 256 && K <= 64 * BURST_STEPS) return launch_burst<EPI>(x, w, out, M, N, K, ldx, ldo, s);
        // (two segments and 256 strips, the 8B shape's output projection: half strips, 512 workgroups of two waves of which
        // two share a compute unit, were slower: 10.7 us against 9.6)
        if ((N + 15) / 16 < 256) return launch_stream<EPI, 8>(x, w, out, M, N, K, ldx, ldo, S, s);
        return launch_stream<EPI, 16>(x, w, out, M, N, K, ldx, ldo, S, s);
      }
    }
    const int row_blocks = (M + 15) / 16, strips = (N + 15) / 16;
    // Few columns and more than 16 rows: a workgroup per block of 16 rows (the strips of W are then
    // fetched once per block of rows, from cache after the first, by four times the waves).  Many
    // columns: one wave takes all rows of its strip.
    const bool split_rows = row_blocks > 1 && strips < 256;
    const int wm = split_rows ? 1 : row_blocks;
    const int waves = S < 4 ? S : 4;      // one wave per SIMD: the operand ring may use up to 512 registers
    // few columns: half strips, so that there are at least as many workgroups as compute units
    const bool half = strips < 256 && row_blocks == 1;
    dim3 grid(half ? (N + 7) / 8 : strips, split_rows ? row_blocks : 1), block(64 * waves);
    const size_t lds = S > 1 ? (size_t)S * NB * wm * 4 * 64 * sizeof(float) : 0;
    if (lds > 64 * 1024) return -2;
    if ((size_t)M * ldx * 2 >= ((size_t)1 << 31) || (size_t)16 * K * 2 >= ((size_t)1 << 31)) return -2;   // offsets within x, within a strip of W
#define BW_SKINNY(WMV, DV, CWV)                                                                                    \
  if (K % 32)                                                                                                      \
    BW_LAUNCH((gemm_bf16_skinny_kernel<WMV, EPI, DV, true, CWV>), grid, block, lds, s, x, w, out, M, N, K, ldx, ldo, S); \
  else                                                                                                             \
    BW_LAUNCH((gemm_bf16_skinny_kernel<WMV, EPI, DV, false, CWV>), grid, block, lds, s, x, w, out, M, N, K, ldx, ldo, S);
    switch (wm) {
      case 1:
        if (half) { BW_SKINNY(1, 16, 8) }
        else { BW_SKINNY(1, 16, 16) }
        break;
      case 2: BW_SKINNY(2, (NB == 2 ? 8 : 16), 16) break;
      case 3: BW_SKINNY(3, 8, 16) break;
      default: BW_SKINNY(4, 8, 16) break;
    }
#undef BW_SKINNY
  } else {
    if constexpr (EPI == EPI_ADD_F32 || EPI == EPI_F32) {
      // Few enough workgroups to be on the chip at once (the output projection of a short prompt is 16 tiles of 128 x 128
      // for 128 rows and 2048 columns, whatever is idle): the kernel for up to 64 rows, a workgroup per block of 64 rows,
      // 64 or 32 columns and segment of K, all blocks in one launch.
      if ((size_t)M * ldx * 2 < ((size_t)1 << 31)) {
        // (one segment, and blocks of 32 rows by 32 columns still fit the chip at once: as for 33 to 64 rows above)
        if (S == 1 && K % 64 == 0 && ((N + 31) / 32) * ((M + 31) / 32) <= 256 && ((N + 31) / 32) * ((M + 31) / 32) >= 32)
          return launch_mid<EPI, 2, false, true>(x, w, out, M, N, K, ldx, ldo, (N + 31) / 32, s, MidNormArgs{}, QkvRopeArgs{}, 1,
                                                 MidSplitArgs{}, (M + 31) / 32);
        int tiles, zb;
        bool narrow;
        add_blocks_shape(M, N, K, tiles, narrow, zb);
        // (a store of one segment whose workgroups would share compute units: by time, further down)
        if (EPI == EPI_F32 && S == 1 && !narrow && !store_in_blocks(M, N, K, false)) tiles = 0;
        const bool scratch_ok = S == 1 || (split_ok &&
                                           scratch_floats >= (size_t)tiles * zb * S * 4096 && num_counters >= tiles * zb);
        if (tiles && scratch_ok) {
          const MidNormArgs na{};
          const QkvRopeArgs no{};
          if (narrow) return launch_mid<EPI, 4, false, true>(x, w, out, M, N, K, ldx, ldo, tiles, s, na, no, S, sp, zb);
          return launch_mid<EPI, 4, false>(x, w, out, M, N, K, ldx, ldo, tiles, s, na, no, S, sp, zb);
        }
      }
      int tiles;
      AddRoute route = add_route(M, N, K, ldo, tiles);
      // (a store splits only what leaves compute units idle)
      if (EPI == EPI_F32 && ((M + 127) / 128) * ((N + 127) / 128) >= 256) route = ADD_WHOLE;
      if (EPI == EPI_ADD_F32 && route == ADD_ROW_BLOCKS && (size_t)M * ldx * 2 < ((size_t)1 << 31) &&
          (S == 1 || (sp.scratch != nullptr && sp.counters != nullptr && scratch_floats >= (size_t)tiles * S * 4096 &&
                      num_counters >= tiles))) {
        for (int m0 = 0; m0 < M; m0 += 64) {
          const int rc = launch_gemm_bf16<EPI>(x + (size_t)m0 * ldx, w, (float*)out + (size_t)m0 * ldo, M - m0 < 64 ? M - m0 : 64, N, K,
                                               ldx, ldo, s, rp, sp, scratch_floats, num_counters);
          if (rc) return rc;
        }
        return 0;
      }
      if (route == ADD_SPLIT && sp.scratch != nullptr && ((uintptr_t)out & 15) == 0) {
        if (scratch_floats < (size_t)S * M * N) return -6;
        const int shape = add_split_shape(M, N, K);
        if (shape >= 0) {
          const int rc = launch_ring<EPI_F32>(shape, x, w, (void*)sp.scratch, M, N, K, ldx, N, s, QkvRopeArgs{}, S, (size_t)M * N);
          if (rc) return rc;
          const size_t quads = (size_t)M * (N >> 2);
          BW_LAUNCH(add_segments_kernel<EPI == EPI_ADD_F32>, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s, (float*)out, sp.scratch, S,
                             M, N, ldo);
          return BW_LAUNCH_CHECK();
        }
      }
    }
    if constexpr (EPI == EPI_F32 || EPI == EPI_BF16 || EPI == EPI_GELU_BF16) {
      const int wgs = (N + 63) / 64, zb = (M + 63) / 64;
      if (K % 64 == 0 && wgs >= 64 && store_in_blocks(M, N, K, EPI == EPI_GELU_BF16) && (size_t)M * ldx * 2 < ((size_t)1 << 31))
        return launch_mid<EPI, 4, false>(x, w, out, M, N, K, ldx, ldo, wgs, s, MidNormArgs{}, QkvRopeArgs{}, 1, MidSplitArgs{}, zb);
    }
    // K in whole steps of 64: tiles through LDS rings, of the shape that takes the least time
    if (K % 64 == 0)
      return launch_ring_tiles<EPI>(x, w, out, M, N, K, ldx, ldo, s, rp);
    constexpr int COLS = epi_is_glu(EPI) ? 64 : 128;
    const int m_tiles = (M + WIDE_BM - 1) / WIDE_BM, n_tiles = (N + COLS - 1) / COLS;
    dim3 grid(m_tiles * n_tiles), block(256);
    if (S > 1)
      BW_LAUNCH((gemm_bf16_wide_kernel<EPI, true, false>), grid, block, 0, s, x, w, out, M, N, K, ldx, ldo, m_tiles, n_tiles, rp);
    else if (K % (2 * WIDE_BK) == 0)
      BW_LAUNCH((gemm_bf16_wide_kernel<EPI, false, true>), grid, block, 0, s, x, w, out, M, N, K, ldx, ldo, m_tiles, n_tiles, rp);
    else
      BW_LAUNCH((gemm_bf16_wide_kernel<EPI, false, false>), grid, block, 0, s, x, w, out, M, N, K, ldx, ldo, m_tiles, n_tiles, rp);
  }
  return BW_LAUNCH_CHECK();
}

// Whether a gated GELU of more than 64 rows takes less time in the epilogue of its stacked product (bw_gemm_gelu_glu_bf16) than as a
// kernel behind the 32-bit store.  The epilogue saves the sums' way through memory (writing 2 N of them a row, reading them, a
// launch: 2,048 rows of 2 x 8192 columns and K = 2048 122 + 38 us -> 111), but its product goes in tiles with all of K a workgroup, where
// the store of few rows or few columns gives blocks of 64 rows or segments of K workgroups of their own (128 rows of 2 x 512 columns and K =
// 14336: 20 us and 70).  Both times are estimated, in hundredths of a microsecond: a workgroup of the 64-row kernel 300 and 25 a
// step of 64 (15 with 32 columns), half as much again where two share a compute unit, 200 more where segments meet; tiles as in
// ring_time, a part-empty round counted as 0.73 of a full one at the least; the activation 250 and its bytes at 3.5 TB/s.  K of several
// segments in tiles of few rows is slower than that (the weights' way), so there the epilogue has to win by a quarter.  Over
// 1,704 products (65 to 2,048 rows, 2 x 512 to 2 x 14336 columns, K of 64 to 14336) both ways timed: no choice more than 5 % slower than the
// kernel behind the store, 0.3 % from the better one in the mean.
extern "C" int bw_gemm_gelu_glu_wins(int M, int N, int K) {
  if (M <= 64 || N <= 0 || K <= 0 || N > (1 << 29)) return 0;
  if (K % 64) return 1;                                     // (the same kernel either way)
  const int S = (K + GEMM_SEG - 1) / GEMM_SEG, cols = 2 * N, per = std::min(K, GEMM_SEG) / 64;
  const long long squares = (long long)((cols + 31) / 32) * ((M + 31) / 32);
  long long store;
  int tiles, zb;
  bool narrow;
  add_blocks_shape(M, cols, K, tiles, narrow, zb);
  if (S == 1 && squares >= 32 && squares <= 256) {
    store = 300 + 15 * per;
  } else if (tiles && (S > 1 || narrow || store_in_blocks(M, cols, K, false))) {
    store = 300 + (narrow ? 15 : 25) * per;
    if ((long long)tiles * zb * S > 256) store = store * 29 / 20;
    if (S > 1) store += 200;
  } else {
    const int shape = split_shape(M, cols, K, cols, true);
    if (shape < 0) return 1;
    store = ring_time(ring_costs[shape], ring_tiles(ring_costs[shape], M, cols) * S, GEMM_SEG, false) + add_join_time(M, cols, S);
  }
  long long epilogue = -1;
  for (int i = 0; i < RING_SHAPES; ++i) {
    if (i == RING_256X192 || (K > GEMM_SEG && !ring_costs[i].joins)) continue;
    const long long t = ring_time(ring_costs[i], ring_tiles(ring_costs[i], M, cols), K, M <= ring_costs[i].rows, false, 187);
    if (epilogue < 0 || t < epilogue) epilogue = t;
  }
  if (S > 1) epilogue = epilogue * 5 / 4;
  return epilogue <= store + 250 + 5LL * M * cols / 70000;
}

// bw_gemm_add_scratch asks for the S M N floats of a split by a count that its callers rely on; whether one takes place goes by time.
// The tiles (rows, columns) in which a residual add (store: a 32-bit store) of M > 64 rows leaves its segments' sums there; 0, 0: it
// goes whole, with the scratch as without.
extern "C" int bw_gemm_split_tile(int M, int N, int K, int store, int* rows, int* columns) {
  if (M <= 0 || N <= 0 || K <= 0 || rows == nullptr || columns == nullptr) return -2;
  const int shape = M > 64 ? split_shape(M, N, K, 4, store != 0) : -1;
  *rows = shape < 0 ? 0 : ring_costs[shape].rows;
  *columns = shape < 0 ? 0 : ring_costs[shape].cols;
  return 0;
}

// The most rows, up to max_rows, with which it does; 0: it never does.
extern "C" int bw_gemm_split_rows(int max_rows, int N, int K, int store) {
  if (N <= 0 || K <= 0) return 0;
  for (int M = max_rows; M > 64; --M)
    if (split_shape(M, N, K, 4, store != 0) >= 0) return M;
  return 0;
}

// What a residual add wants beside its operands to give every segment of K workgroups of its own: floats of
// scratch and counters (int32, zero before the first launch; every launch leaves them zero).  Both 0: it would not.
extern "C" int bw_gemm_add_scratch(int M, int N, int K, long long* scratch_floats, int* counters) {
  int tiles = 0;
  bool narrow = false;
  const int S = K > 0 ? (K + GEMM_SEG - 1) / GEMM_SEG : 0;
  if (M > 64 && N > 0 && S > 1) {                           // a few blocks of 64 rows at once: a cell a workgroup
    int zb;
    add_blocks_shape(M, N, K, tiles, narrow, zb);
    if (tiles) {
      *scratch_floats = (long long)ADD_BLOCKS_MAX_WGS * 4096;   // (the same for every shape: one buffer serves all)
      *counters = ADD_BLOCKS_MAX_WGS;
      return 0;
    }
  }
  const AddRoute route = M > 64 && N > 0 ? add_route(M, N, K, 4, tiles) : ADD_WHOLE;
  if (route == ADD_SPLIT) {      // a prompt portion: the segments' sums, whole
    *scratch_floats = (long long)S * M * N;
    *counters = 1;                                          // (none is used)
    return 0;
  }
  if (M > 0 && M <= 64 && N > 0 && S > 1) add_rows_shape(M, N, K, tiles, narrow);
  else if (S == 1) tiles = 0;                               // (blocks of 64 rows of one segment share nothing)
  *scratch_floats = (long long)tiles * S * 4096;
  *counters = tiles;
  return 0;
}

// out += x W^T with the scratch that bw_gemm_add_scratch asks for: the bits of bw_gemm_bf16's residual add.
extern "C" int bw_gemm_add_bf16(const void* x, const void* w, void* out, int M, int N, int K, int ldx, int ldo,
                                float* scratch, long long scratch_floats, int32_t* counters, int num_counters,
                                void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || (K % 8) || (ldx % 8) || ldx < K || ldo < N) return -2;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) return -3;
  return launch_gemm_bf16<EPI_ADD_F32>((const bf16_t*)x, (const bf16_t*)w, out, M, N, K, ldx, ldo, (hipStream_t)stream,
                                       QkvRopeArgs{}, MidSplitArgs{scratch, counters}, (size_t)scratch_floats, num_counters);
}

// out[m][n] = bf16(gelu_tanh(x W^T [m][n]) * table[token of m][n]) for up to 16 rows and fewer than 4,096 columns, K in steps of 64:
// the bits of bw_gemm_bf16's 32-bit store followed by bw_side_gate.  -7: not this shape.
extern "C" int bw_gemm_side_bf16(const void* x, const void* w, void* out, int M, int N, int K, int ldx, int ldo, const int32_t* tokens,
                                 const int32_t* feedback, const void* table, int ldt, int vocab, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || ldx < K || (ldx % 8) || ldo < N || ldt < N || vocab <= 0 || tokens == nullptr || table == nullptr) return -2;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) return -3;
  const int S = (K + GEMM_SEG - 1) / GEMM_SEG;
  if (M > 16 || K % 64 || S > 40 || (N + 15) / 16 >= 256 || (size_t)M * ldx * 2 >= ((size_t)1 << 31)) return -7;
  const SideGateArgs sg{tokens, feedback, (const bf16_t*)table, ldt, vocab};
  hipStream_t s = (hipStream_t)stream;
  if (K <= 64 * BURST_STEPS) return launch_burst<EPI_SIDE_BF16>((const bf16_t*)x, (const bf16_t*)w, out, M, N, K, ldx, ldo, s, sg);
  return launch_stream<EPI_SIDE_BF16, 8>((const bf16_t*)x, (const bf16_t*)w, out, M, N, K, ldx, ldo, S, s, sg);
}

// out = x W^T (32-bit store) with that scratch: the bits of bw_gemm_bf16's store.
extern "C" int bw_gemm_store_bf16(const void* x, const void* w, void* out, int M, int N, int K, int ldx, int ldo,
                                  float* scratch, long long scratch_floats, int32_t* counters, int num_counters, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || (K % 8) || (ldx % 8) || ldx < K || ldo < N) return -2;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) return -3;
  return launch_gemm_bf16<EPI_F32>((const bf16_t*)x, (const bf16_t*)w, out, M, N, K, ldx, ldo, (hipStream_t)stream,
                                   QkvRopeArgs{}, MidSplitArgs{scratch, counters}, (size_t)scratch_floats, num_counters);
}

extern "C" int bw_gemm_bf16(const void* x, const void* w, void* out, int M, int N, int K, int ldx, int ldo,
                            int epilogue, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || (K % 8) || (ldx % 8) || ldx < K || ldo < N) return -2;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) return -3;
  hipStream_t s = (hipStream_t)stream;
  const bf16_t* xp = (const bf16_t*)x;
  const bf16_t* wp = (const bf16_t*)w;
  switch (epilogue) {
    case EPI_F32: return launch_gemm_bf16<EPI_F32>(xp, wp, out, M, N, K, ldx, ldo, s);
    case EPI_BF16: return launch_gemm_bf16<EPI_BF16>(xp, wp, out, M, N, K, ldx, ldo, s);
    case EPI_ADD_F32: return launch_gemm_bf16<EPI_ADD_F32>(xp, wp, out, M, N, K, ldx, ldo, s);
    case EPI_GELU_BF16: return launch_gemm_bf16<EPI_GELU_BF16>(xp, wp, out, M, N, K, ldx, ldo, s);
    case EPI_SWIGLU_BF16: return launch_gemm_bf16<EPI_SWIGLU_BF16>(xp, wp, out, M, N, K, ldx, ldo, s);
  }
  return -2;
}

// The stacked gate|up product of more than 64 rows with the clamped gated unit in its epilogue:
// out[m, n] = bf16(g' sigmoid(alpha g') (u' + 1)), g' = min(x.W[n], limit), u' = clamp(x.W[N + n], -limit, limit); w is
// [2N, K].  The bits of gemm_bf16 (32-bit store) + glu.
extern "C" int bw_gemm_clamped_glu_bf16(const void* x, const void* w, void* out, int M, int N, int K, int ldx, int ldo,
                                        float limit, float alpha, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M <= 64 || !(limit > 0.0f)) return -2;
  if (K <= 0 || (K % 8) || (ldx % 8) || ldx < K || ldo < N) return -2;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) return -3;
  QkvRopeArgs rp{};
  rp.glu_limit = limit;
  rp.glu_alpha = alpha;
  return launch_gemm_bf16<EPI_CLAMPED_GLU_BF16>((const bf16_t*)x, (const bf16_t*)w, out, M, N, K, ldx, ldo,
                                                (hipStream_t)stream, rp);
}

// The same with the GELU (tanh form) of the gate: out[m, n] = bf16(gelu(x.W[n]) (x.W[N + n])).  The bits of gemm_bf16
// (32-bit store) + glu, which at 2,048 rows of 2 x 8192 columns and K = 2048 write and read 134 MB of sums: 122 + 38 us -> 111
// (bw_gemm_gelu_glu_wins: where it is the faster way).
extern "C" int bw_gemm_gelu_glu_bf16(const void* x, const void* w, void* out, int M, int N, int K, int ldx, int ldo, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M <= 64) return -2;
  if (K <= 0 || (K % 8) || (ldx % 8) || ldx < K || ldo < N) return -2;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) return -3;
  return launch_gemm_bf16<EPI_GELU_GLU_BF16>((const bf16_t*)x, (const bf16_t*)w, out, M, N, K, ldx, ldo, (hipStream_t)stream);
}

// The stacked q|k|v product with rotation and cache write in its epilogue (heads of 64 elements, K of one
// segment; more than 64 rows, or up to 64 with at least 64 heads and K in steps of 64): q rotated to q_out [M, heads*64],
// k rotated and v to their page slots.  The bits of gemm_bf16 (32-bit store) + rope_kvwrite.
extern "C" int bw_gemm_qkv_rope_bf16(const void* x, int ldx, const void* w_qkv, void* q_out, const int32_t* positions,
                                     const int32_t* row_seq, const int32_t* block_table, int table_stride,
                                     const float* cos_table, const float* sin_table, void* k_cache, void* v_cache,
                                     int M, int heads, int kv_heads, int head_dim, int K, int page_size,
                                     int write_cache, void* stream) {
  if (M <= 0) return 0;
  if (head_dim % 64) return -4;
  if (K <= 0 || (K % 8) || (ldx % 8) || ldx < K || page_size <= 0) return -2;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w_qkv)) & 15) return -3;
  if (page_size <= 0 || (page_size & (page_size - 1))) return -5;
  QkvRopeArgs rp{positions, row_seq, block_table, cos_table, sin_table, (bf16_t*)k_cache, (bf16_t*)v_cache,
                 heads, kv_heads, page_size, table_stride, write_cache, __builtin_ctz((unsigned)page_size), head_dim};
  // up to 64 rows, or a few blocks of 64 rows at once: a workgroup per 32 or 16 rotary pairs of a head
  const int mid = launch_qkv_rope_mid((const bf16_t*)x, ldx, (const bf16_t*)w_qkv, q_out, M, K, rp, (hipStream_t)stream);
  if (mid != -7) return mid;
  if (M <= 64) return -2;
  if (head_dim != 64) return -4;                                   // the tiled kernels' epilogue: heads of 64 ...
  if (K > GEMM_SEG) return -2;                                     // ... and one segment of K
  const int N = (heads + 2 * kv_heads) * 64;
  return launch_gemm_bf16<EPI_QKV_ROPE>((const bf16_t*)x, (const bf16_t*)w_qkv, q_out, M, N, K, ldx, heads * 64,
                                        (hipStream_t)stream, rp);
}

// ------------------------------------------------------------------------------ a residual add that allocates nothing

// out += x W^T like bw_gemm_add_bf16, for callers that can neither allocate device memory nor bring a
// workspace (code under graph capture, tight serving loops, harnesses that forbid hipMalloc): the
// segments' sums and the tiles' counters live in one array in the library's own device image.  Every GPU
// that loads the library holds a copy of the array at an address of its own until the process ends; the
// name of the array is no device address in host code, so the address is asked for once per device and
// kept.  Calls on one GPU share the array: calls that overlap there (two streams, two threads) race.
#define BW_STATIC_SCRATCH_FLOATS (2 * 1024 * 1024)          // 8 MB of sums
#define BW_STATIC_SCRATCH_COUNTERS 1024                      // 4 KB of counters behind them
#define BW_STATIC_MAX_DEVICES 64
static __device__ __align__(256) float scratch[BW_STATIC_SCRATCH_FLOATS + BW_STATIC_SCRATCH_COUNTERS];

__global__ __launch_bounds__(256) void zero_words_kernel(int32_t* __restrict__ p, int n) {
  const int i = (int)(blockIdx.x * 256 + threadIdx.x);
  if (i < n) p[i] = 0;
}

static float* static_scratch_of_device[BW_STATIC_MAX_DEVICES];
static std::mutex static_scratch_mutex;

// The current device's copy of the array (asked for at the first call on that device).
static int static_scratch_address(float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= BW_STATIC_MAX_DEVICES) return -2;
  std::lock_guard<std::mutex> hold(static_scratch_mutex);
  if (static_scratch_of_device[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (p == nullptr) return -2;
    static_scratch_of_device[dev] = (float*)p;
  }
  *out = static_scratch_of_device[dev];
  return 0;
}

extern "C" int bw_gemm_add_bf16_static_max(long long* scratch_floats, int* counters) {
  *scratch_floats = BW_STATIC_SCRATCH_FLOATS;
  *counters = BW_STATIC_SCRATCH_COUNTERS;
  return 0;
}

extern "C" int bw_gemm_add_bf16_static(const void* x, const void* w, void* out, int M, int N, int K, int ldx, int ldo,
                                       void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || (K % 8) || (ldx % 8) || ldx < K || ldo < N) return -2;
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) return -3;
  long long need_floats = 0;
  int need_counters = 0;
  bw_gemm_add_scratch(M, N, K, &need_floats, &need_counters);
  if (need_floats > BW_STATIC_SCRATCH_FLOATS || need_counters > BW_STATIC_SCRATCH_COUNTERS) return -7;
  if (need_floats == 0)      // this shape's kernel joins its segments in registers: nothing to share
    return launch_gemm_bf16<EPI_ADD_F32>((const bf16_t*)x, (const bf16_t*)w, out, M, N, K, ldx, ldo, (hipStream_t)stream);
  float* base = nullptr;
  const int rc = static_scratch_address(&base);
  if (rc != 0) return rc;
  int32_t* count = reinterpret_cast<int32_t*>(base + BW_STATIC_SCRATCH_FLOATS);
  // The counters must be zero when the kernel starts.  Every launch leaves them so, but the array outlives a
  // launch that was aborted half way; a small kernel clears them (a memset node in a captured graph is no
  // safe thing on this hardware's runtime).  The sums need no clearing: every cell is written before it is read.
  BW_LAUNCH(zero_words_kernel, dim3((need_counters + 255) / 256), dim3(256), 0, (hipStream_t)stream, count,
                     need_counters);
  return launch_gemm_bf16<EPI_ADD_F32>((const bf16_t*)x, (const bf16_t*)w, out, M, N, K, ldx, ldo, (hipStream_t)stream,
                                       QkvRopeArgs{}, MidSplitArgs{base, count}, (size_t)need_floats, need_counters);
}
