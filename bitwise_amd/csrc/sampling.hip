// Token choice and logits fingerprints on the device, one workgroup per logits row.
//
// Greedy: the first maximum wins (the reference scans with a strict '>', src/engine.cpp:40-45).
// Temperature: w[i] = bw_expf((l[i] - max) / T) in 32-bit, sums in double, the token is the first
// i whose running sum exceeds u * total, else the last i with positive weight
// (src/engine.cpp:50-73).  The reference adds the weights one after the other; here each of
// the 256 threads adds its own contiguous stretch of the vocabulary in order and the
// stretches are joined in thread order, which moves the running sum by a few units of
// 2^-53 and depends on nothing but the row itself.  u comes from the host's counter-based
// generator keyed by (seed, position, stream).
#include "common.h"
#include "api.h"

#define SMP_THREADS 256

__global__ __launch_bounds__(SMP_THREADS) void sample_kernel(const float* __restrict__ logits, int vocab, int ld,
                                                             const float* __restrict__ temperature,
                                                             const double* __restrict__ uniform,
                                                             int32_t* __restrict__ out) {
  __shared__ float s_val[SMP_THREADS];
  __shared__ int s_idx[SMP_THREADS];
  __shared__ double s_sum[SMP_THREADS];
  __shared__ int s_pick[SMP_THREADS];
  __shared__ int s_lastpos[SMP_THREADS];
  __shared__ double s_total;
  const int row = blockIdx.x, tid = threadIdx.x;
  const float* l = logits + (size_t)row * ld;
  const int chunk = (vocab + SMP_THREADS - 1) / SMP_THREADS;
  const int begin = tid * chunk < vocab ? tid * chunk : vocab;
  const int end = begin + chunk < vocab ? begin + chunk : vocab;

  // maximum and its first index: every thread scans an interleaved share of the row in ascending
  // order (16-byte loads where the row allows), the shares are joined below with ties going to
  // the smaller index, so the first maximum of the whole row wins whatever the split
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  if ((vocab & 3) == 0 && (ld & 3) == 0 && (reinterpret_cast<uintptr_t>(logits) & 15) == 0) {
    const f32x4* lv = reinterpret_cast<const f32x4*>(l);
    const int nv = vocab >> 2;
    auto scan = [&](const f32x4& x, int v) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (x[e] > best || best_i == 0x7fffffff) {  // the share's first element, or strictly greater
          best = x[e];
          best_i = 4 * v + e;
        }
    };
    int v = tid;
    for (; v + 3 * SMP_THREADS < nv; v += 4 * SMP_THREADS) {   // four loads in flight, scanned in ascending order
      const f32x4 x0 = lv[v], x1 = lv[v + SMP_THREADS], x2 = lv[v + 2 * SMP_THREADS], x3 = lv[v + 3 * SMP_THREADS];
      scan(x0, v);
      scan(x1, v + SMP_THREADS);
      scan(x2, v + 2 * SMP_THREADS);
      scan(x3, v + 3 * SMP_THREADS);
    }
    for (; v < nv; v += SMP_THREADS) scan(lv[v], v);
  } else {
    for (int i = tid; i < vocab; i += SMP_THREADS)
      if (l[i] > best || best_i == 0x7fffffff) {
        best = l[i];
        best_i = i;
      }
  }
  s_val[tid] = best;
  s_idx[tid] = best_i;
  __syncthreads();
  for (int off = SMP_THREADS / 2; off >= 1; off >>= 1) {
    if (tid < off) {
      const float ov = s_val[tid + off];
      const int oi = s_idx[tid + off];
      if (oi != 0x7fffffff && (s_idx[tid] == 0x7fffffff || ov > s_val[tid] || (ov == s_val[tid] && oi < s_idx[tid]))) {
        s_val[tid] = ov;
        s_idx[tid] = oi;
      }
    }
    __syncthreads();
  }
  const float mx = s_val[0];
  const float T = temperature[row];
  if (T <= 0.0f) {
    if (tid == 0) out[row] = s_idx[0];
    return;
  }

  double part = 0.0;
  int lastpos = -1;
  for (int i = begin; i < end; ++i) {
    const float w = bw_expf((l[i] - mx) / T);
    if (w > 0.0f) {
      part += (double)w;
      lastpos = i;
    }
  }
  s_sum[tid] = part;
  s_lastpos[tid] = lastpos;
  s_pick[tid] = -1;
  __syncthreads();
  if (tid == 0) {  // exclusive prefix in thread order; s_sum[t] becomes the sum before stretch t
    double run = 0.0;
    int last = 0;
    for (int t = 0; t < SMP_THREADS; ++t) {
      const double p = s_sum[t];
      s_sum[t] = run;
      run += p;
      if (s_lastpos[t] >= 0) last = s_lastpos[t];
    }
    s_lastpos[0] = last;
    s_total = run;
  }
  __syncthreads();
  const double total = s_total;
  const double target = uniform[row] * total;
  double cum = s_sum[tid];
  if (cum <= target) {
    for (int i = begin; i < end; ++i) {
      const float w = bw_expf((l[i] - mx) / T);
      if (w <= 0.0f) continue;
      cum += (double)w;
      if (cum > target) {
        s_pick[tid] = i;
        break;
      }
    }
  }
  __syncthreads();
  if (tid == 0) {
    int pick = s_lastpos[0];
    for (int t = 0; t < SMP_THREADS; ++t)
      if (s_pick[t] >= 0) {
        pick = s_pick[t];
        break;
      }
    out[row] = pick;
  }
}

extern "C" int bw_sample(const float* logits, int vocab, int ld, int rows, const float* temperature,
                         const double* uniform, int32_t* out, void* stream) {
  if (rows <= 0) return 0;
  if (vocab <= 0 || ld < vocab) return -2;
  hipLaunchKernelGGL(sample_kernel, dim3(rows), dim3(SMP_THREADS), 0, (hipStream_t)stream, logits, vocab, ld,
                     temperature, uniform, out);
  return BW_LAUNCH_CHECK();
}

// Fingerprint chain of the reference (src/engine.cpp:18-29): h = (h ^ word) * 1099511628211
// over the row's 8-byte words, single trailing bytes likewise, then the splitmix64 finaliser.
//
// One wave a row, link by link: the chain as it is written.  The row's
// address is the same for every lane, so the words arrive through the scalar unit, sixteen of them a load and the
// next sixteen asked for before these are used, and the chain runs in scalar registers, a link every 13 ns (eight scalar
// instructions): 318 us for 49,152 logits, whatever the number of rows.  For short rows, and for very many.
#define FP_BLOCK 16        // words of 8 bytes a block
__device__ __forceinline__ uint64_t fp_link(uint64_t h, uint32_t lo, uint32_t hi) {
  return (h ^ ((uint64_t)lo | ((uint64_t)hi << 32))) * 1099511628211ull;
}

// an odd row's last element byte by byte, and the finaliser
__device__ __forceinline__ uint64_t fp_finish(uint64_t h, const uint32_t* __restrict__ p, int vocab) {
  if (vocab & 1) {
    const uint32_t t = p[vocab - 1];
    for (int k = 0; k < 4; ++k) h = (h ^ ((t >> (8 * k)) & 0xffu)) * 1099511628211ull;
  }
  h = (h ^ (h >> 30)) * 0xBF58476D1CE4E5B9ull;
  h = (h ^ (h >> 27)) * 0x94D049BB133111EBull;
  return h ^ (h >> 31);
}

struct FpBlock {
  uint32_t d[2 * FP_BLOCK];
};

__device__ __forceinline__ void fp_load(FpBlock& blk, const uint32_t* __restrict__ p) {
#pragma unroll
  for (int j = 0; j < 2 * FP_BLOCK; ++j) blk.d[j] = p[j];
}

__device__ __forceinline__ uint64_t fp_chain(uint64_t h, const FpBlock& blk) {
#pragma unroll
  for (int j = 0; j < FP_BLOCK; ++j) h = fp_link(h, blk.d[2 * j], blk.d[2 * j + 1]);
  return h;
}

__global__ __launch_bounds__(64) void fingerprint_kernel(const float* __restrict__ logits, int vocab, int ld, int rows,
                                                         const uint64_t* __restrict__ h_in, uint64_t* __restrict__ h_out) {
  const int row = blockIdx.x;                                         // the same for every lane: scalar from here on
  if (row >= rows) return;
  const uint32_t* __restrict__ p = reinterpret_cast<const uint32_t*>(logits + (size_t)row * ld);
  uint64_t h = h_in[row];
  const int words = vocab >> 1;
  const int blocks = words / FP_BLOCK;
  // two blocks in turn: while one is chained the other is on its way (scalar loads come back in any order, so a
  // wait is for all of them; each block is asked for a whole chain of sixteen links before it is needed)
  FpBlock even, odd;
  if (blocks > 0) fp_load(even, p);
  int b = 0;
  for (; b + 2 <= blocks; b += 2) {
    __builtin_amdgcn_s_waitcnt(0xc07f);                                // lgkmcnt(0): the block to be chained now is there ...
    __builtin_amdgcn_sched_barrier(0);
    fp_load(odd, p + (size_t)(b + 1) * 2 * FP_BLOCK);                  // ... before the next one is asked for
    __builtin_amdgcn_sched_barrier(0);
    h = fp_chain(h, even);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_sched_barrier(0);
    fp_load(even, p + (size_t)(b + 2 < blocks ? b + 2 : b) * 2 * FP_BLOCK);      // (past the end: a block once more, unused)
    __builtin_amdgcn_sched_barrier(0);
    h = fp_chain(h, odd);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (b < blocks) h = fp_chain(h, even);                               // an odd number of blocks: the last one
  for (int i = blocks * FP_BLOCK; i < words; ++i) h = fp_link(h, p[2 * i], p[2 * i + 1]);
  if (threadIdx.x == 0) h_out[row] = fp_finish(h, p, vocab);
}

// Bit by bit, all links at once.  The chain is serial in its links but not in its bits: bit j of a link's product
// is bit j of x = h ^ word plus carries and shifted copies that depend on lower bits of x alone, so that
//   h_j(n + 1) = h_j(n) ^ word_j(n) ^ K_j(n),      K_j made of bits below j of the same link,
// and once the bits below j are known at every link, bit j of all of them is an exclusive or over the links before: a scan.  A
// row is therefore 64 scans, one behind the other, instead of one step a word.
//
// A workgroup holds 32 links a thread as 64 slices of a bit each: link i * T + t is bit i of thread t's slices (T threads;
// consecutive threads read consecutive words, and a 32 x 32 transposition in registers makes the slices).  The factor is
// 2^40 + 3 (1 + 16 + 128): y = 3 x, z = y + 16 y, u = z + 128 y, v = u + 2^40 x, sums of two numbers each, a bit of all 32 links
// in two instructions (exclusive or and majority of three).  A bit's scan runs over the lanes of a wave for all 32 values
// of i at once, over the waves through LDS, and over i in scalar registers.  A row longer than a workgroup holds takes
// several passes; slots past a pass's links hold zero words, and the first of them reads the pass's result.
//
// What bounds it: the 64 rounds, each some thirty instructions a wave and one meeting of the workgroup.  49,152 logits: 318 us as a
// chain, 42 so (eight rows 43, 256 rows 46); 128,256: 831 and 85; 32,000: 208 and 31.
__device__ __forceinline__ uint32_t fp_xor3(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return (uint32_t)__builtin_amdgcn_bitop3_b32((int)a, (int)b, (int)c, 0x96);
#else
  return a ^ b ^ c;
#endif
}

__device__ __forceinline__ uint32_t fp_major(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return (uint32_t)__builtin_amdgcn_bitop3_b32((int)a, (int)b, (int)c, 0xe8);
#else
  return (a & b) | (a & c) | (b & c);
#endif
}

template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t fp_scan_step(uint32_t v) {
  return v ^ (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, true);
}

// bit i of a[j] and bit j of a[i] change places
__device__ __forceinline__ void fp_transpose(uint32_t (&a)[32]) {
#pragma unroll
  for (int s = 16; s; s >>= 1) {
    const uint32_t low = s == 16 ? 0x0000ffffu : s == 8 ? 0x00ff00ffu : s == 4 ? 0x0f0f0f0fu : s == 2 ? 0x33333333u : 0x55555555u;
#pragma unroll
    for (int k = 0; k < 32; ++k)
      if (!(k & s)) {
        const uint32_t x = a[k], y = a[k + s];
        a[k] = (x & low) | ((y << s) & ~low);
        a[k + s] = ((x >> s) & low) | (y & ~low);
      }
  }
}

template <int WAVES>
__global__ __launch_bounds__(64 * WAVES, 4) void fingerprint_slices_kernel(const float* __restrict__ logits, int vocab, int ld,
                                                                        const uint64_t* __restrict__ h_in, uint64_t* __restrict__ h_out) {
  constexpr int T = 64 * WAVES;
  static_assert(WAVES == 4 || WAVES == 8 || WAVES == 16, "the waves' totals are scanned in a row of 16 lanes");
  __shared__ uint32_t totals[2][16];
  __shared__ uint32_t state[2];
  const int row = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t* __restrict__ p = reinterpret_cast<const uint32_t*>(logits + (size_t)row * ld);
  const int words = vocab >> 1;
  uint64_t h = h_in[row];
  if (t < 16) totals[0][t] = totals[1][t] = 0;                       // (lanes past the waves read zeros)
  __syncthreads();
  for (int at = 0; at < words; at += 32 * T - 1) {
    const int n = words - at < 32 * T - 1 ? words - at : 32 * T - 1;   // the pass's links
    uint32_t x[64], y[64];
    {
      uint32_t lo[32], hi[32];
#pragma unroll
      for (int i = 0; i < 32; ++i) {
        const int link = i * T + t;
        lo[i] = link < n ? p[2 * (size_t)(at + link)] : 0u;
        hi[i] = link < n ? p[2 * (size_t)(at + link) + 1] : 0u;
      }
      fp_transpose(lo);
      fp_transpose(hi);
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        x[j] = lo[j];
        x[32 + j] = hi[j];
      }
    }
    uint32_t cy = 0, cz = 0, cu = 0, cv = 0;
#pragma unroll
    for (int j = 0; j < 64; ++j) {
      const uint32_t x1 = j >= 1 ? x[j - 1] : 0u, y4 = j >= 4 ? y[j - 4] : 0u, y7 = j >= 7 ? y[j - 7] : 0u, x40 = j >= 40 ? x[j - 40] : 0u;
      const uint32_t d = fp_xor3(fp_xor3(fp_xor3(x[j] ^ x40, y4, y7), x1, cy), cz, cu ^ cv);
      uint32_t v = fp_scan_step<0x111, 0xf>(d);                       // row_shr 1, 2, 4, 8: sixteen lanes
      v = fp_scan_step<0x112, 0xf>(v);
      v = fp_scan_step<0x114, 0xf>(v);
      v = fp_scan_step<0x118, 0xf>(v);
      v = fp_scan_step<0x142, 0xa>(v);                                // row_bcast 15 and 31: the whole wave
      v = fp_scan_step<0x143, 0xc>(v);
      if (lane == 63) totals[j & 1][wave] = v;
      __syncthreads();                                                // (a buffer is written again two meetings on)
      uint32_t w = totals[j & 1][lane & 15];
      w = fp_scan_step<0x111, 0xf>(w);
      w = fp_scan_step<0x112, 0xf>(w);
      if (WAVES > 4) w = fp_scan_step<0x114, 0xf>(w);
      if (WAVES > 8) w = fp_scan_step<0x118, 0xf>(w);
      const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)w, WAVES - 1);
      const uint32_t before = wave ? (uint32_t)__builtin_amdgcn_readlane((int)w, wave - 1) : 0u;
      uint32_t base = all << 1;                                       // exclusive or of the totals of smaller i
      base ^= base << 1;
      base ^= base << 2;
      base ^= base << 4;
      base ^= base << 8;
      base ^= base << 16;
      base ^= before ^ (0u - (uint32_t)((h >> j) & 1));
      // v ^ d: the lanes before; ^ base: h_j at the own links; ^ the word's bit: x_j
      const uint32_t xj = fp_xor3(v, x[j] ^ d, base);
      x[j] = xj;
      const uint32_t yj = fp_xor3(xj, x1, cy), zj = fp_xor3(yj, y4, cz), uj = fp_xor3(zj, y7, cu);
      y[j] = yj;
      cy = fp_major(xj, x1, cy);
      cz = fp_major(yj, y4, cz);
      cu = fp_major(zj, y7, cu);
      cv = fp_major(uj, x40, cv);
    }
    // the slot behind the last link: its word is zero, so x is h there
    const int slot = n / T;
    if (t == n - slot * T) {
      uint32_t lo = 0, hi = 0;
#pragma unroll
      for (int j = 0; j < 32; ++j) {
        lo |= ((x[j] >> slot) & 1u) << j;
        hi |= ((x[32 + j] >> slot) & 1u) << j;
      }
      state[0] = lo;
      state[1] = hi;
    }
    __syncthreads();
    h = (uint64_t)__builtin_amdgcn_readfirstlane((int)state[0]) & 0xffffffffull;
    h |= (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)state[1]) << 32;
  }
  if (t == 0) h_out[row] = fp_finish(h, p, vocab);
}

// Which kernel, by nanoseconds: the waves of a workgroup of slices, or 0 for the chain.  A link of the chain takes 13, 15 with 787 rows and
// 16 with 1,024, whose waves share compute units; 1,100 rows take 1.8 times as long, 2,048 2 to 3.7 times.  A pass of 4, 8 or 16 waves
// over their 8,191, 16,383 or 32,767 words takes 26, 30 or 42 us on a compute unit of its own, 34 with two of four waves on one, 47 with
// four; beyond that sixteen waves' worth of rows share one at about 42.
// 4,096 logits are 26 us so and 28 as a chain, 3,072 are 26 and 21; 787 rows of 5,645 47 and 42, 1,024 rows of 7,000 47 and 59, of 8,192 47 and
// 67, 4,096 of them 237 as a chain.
static int fingerprint_waves(int rows, int words) {
  const long long link = rows <= 512 ? 13000 : rows <= 1024 ? 13000 + 6ll * (rows - 512) : 13000ll * (2048 + rows) / 2048;   // ps
  const int pass_ns[3] = {26000, 30000, 42000};
  int waves = 0;
  long long best = words * link / 1000;
  for (int k = 0; k < 3; ++k) {
    const int w = 4 << k, slots = 2048 * w - 1, a_round = 256 * 16 / w;
    const long long passes = (words + slots - 1) / slots;
    long long ns = rows <= 256 ? pass_ns[k] : (rows + a_round - 1) / a_round * (long long)pass_ns[2];
    if (k == 0 && rows > 256 && rows <= 1024) ns = rows <= 512 ? 34000 : 47000;
    if (passes * ns < best) {
      best = passes * ns;
      waves = w;
    }
  }
  return waves;
}

extern "C" int bw_fingerprint_waves(int rows, int vocab) { return rows > 0 && vocab > 0 ? fingerprint_waves(rows, vocab >> 1) : 0; }

extern "C" int bw_fingerprint(const float* logits, int vocab, int ld, int rows, const void* h_in, void* h_out,
                              void* stream) {
  if (rows <= 0) return 0;
  const uint64_t* from = (const uint64_t*)h_in;
  uint64_t* to = (uint64_t*)h_out;
  const int waves = fingerprint_waves(rows, vocab >> 1);
  const hipStream_t s = (hipStream_t)stream;
  if (waves == 16) hipLaunchKernelGGL((fingerprint_slices_kernel<16>), dim3(rows), dim3(1024), 0, s, logits, vocab, ld, from, to);
  else if (waves == 8) hipLaunchKernelGGL((fingerprint_slices_kernel<8>), dim3(rows), dim3(512), 0, s, logits, vocab, ld, from, to);
  else if (waves == 4) hipLaunchKernelGGL((fingerprint_slices_kernel<4>), dim3(rows), dim3(256), 0, s, logits, vocab, ld, from, to);
  else hipLaunchKernelGGL(fingerprint_kernel, dim3(rows), dim3(64), 0, s, logits, vocab, ld, rows, from, to);
  return BW_LAUNCH_CHECK();
}
