// Matrix memories walked in stages: a portion of one or a few requests over the whole chip (included by sequence_mix.hip).
//
// The walk (linear_recurrence_kernel, PHASE 0) gives a column of the memory as many lanes as its sum has parts, each with a chain of
// eight channels: 16 heads of 64 x 128 are 256 waves on 64 of 256 compute units, and what bounds it is that a wave issues an
// instruction every 2.3 to 2.8 ns, 44 of them a token.  A part cannot be cut into more chains without other bits.
// But one chain can be handed on: here a part is F lanes of 8 / F channels, lane ``stage`` of it works on token i - stage in step i,
// and each starts its chain from what the lane before it reached in the step before.  The same chains, the same joins of the parts
// (a tree over neighbouring lanes), F times as many lanes with a fraction of the instructions each.
// One request, us, walk -> stages:                                  64 tokens     128          512          2,048
//   16 heads of 64 x 128, decays given                              12.4 -> 11.3  20.1 -> 14.5  67 -> 36    257 -> 129
//   8 heads of 128 x 256, scalar gates (their launch included)      21.6 -> 22.1  37 -> 31      131 -> 70   509 -> 253
// Of 129 us (63 ns a token) the steps alone take 77 (11 vector instructions, 2 LDS reads), the rest is staging, barriers and the
// sums' way out.  Two requests of 1,024 tokens at once 133 -> 95 and 259 -> 164; where requests fill the chip the walk, which needs
// fewer instructions a column, is the better one (three of 683: 93 and 98; the caller's rule).
// Tried: 8-byte operands as they lie in memory (an 8-byte read costs LDS what a 16-byte one does: 163 us); the compiler's order of the
// steps (the same instructions, 167); a branch around the sums' store (180); chunks of 32 tokens in three buffers (164).
// A token outside the portion (the first and last steps of the later and earlier stages) is one that leaves the memory as it is, to the
// bit: decay 1, k = -0 and v = 1, so that S' = fma(1, S, -0).
#pragma once

template <int MODE, int DPAD>
struct StagesShape {
  static constexpr bool CHANNELS = MODE == RECUR_DECAY_GIVEN;                 // a decay a channel; otherwise a factor a token
  static constexpr int PARTS = recur_split(DPAD), F = 32 / PARTS, DH = DPAD / PARTS / F;   // lanes a column: 32
  static constexpr int RC = 16, RING = 4 * RC, PRE = F - 1;                   // tokens staged together; rows of the rings
  static constexpr int WCOLS = 2 * RW, VW = CHANNELS ? 1 : 2;                 // columns a workgroup; numbers a token and column (v, or the token's factor and v as it enters)
  static constexpr int KQ_ROW = 2 * DPAD, A_ROW = DPAD, LINE = RING + 4;      // floats
  static constexpr int KQ = RING * KQ_ROW, A = CHANNELS ? RING * A_ROW : 0, V = VW * WCOLS * F * LINE, OUT = WCOLS * LINE;
  static constexpr int LDS = (KQ + A + V + OUT) * 4;
  static constexpr int VECS = DPAD / 4, NL = RC * VECS / (64 * RW);           // 16-byte loads of q, of k (and of decays) a thread and chunk
  static_assert(DH * F * PARTS == DPAD && DH >= 2 && DH <= 4 && PARTS <= 16, "a part is F lanes of two or four channels");
  static_assert(LDS <= BW_LDS_LIMIT && NL * 64 * RW == RC * VECS, "four chunks have to fit, whole loads");
};

// What a lane needs of four tokens.
template <int DH, bool CH, int VW>
struct StagesOps {
  float k[4][DH], q[4][DH], a[CH ? 4 : 1][CH ? DH : 1], v[VW][4];
};

// What a thread brings of a chunk: its vectors of q, k and decays, one v and its token's gates.
template <int NL, bool CH>
struct StagesLoads {
  f32x4 q[NL], k[NL], a[CH ? NL : 1];
  float v, f, i;
};

typedef const __attribute__((address_space(3))) float* lds_floats;
typedef const __attribute__((address_space(3))) f32x4* lds_vectors;

template <int CTRL>
__device__ __forceinline__ float stages_dpp(float v) {
  return __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}

// RECUR_DECAY_GIVEN, or RECUR_SCALAR_GATES with ``gate`` as scalar_gates_kernel leaves it.
// Operands lie in rings of four chunks in LDS, in the row of the step at which their stage wants them (token + stage) and side by
// side as a lane reads them, 16 bytes at a time (an 8-byte read costs LDS as much): two channels of k and of q; two channels of
// two tokens' decays; four tokens of v, a line for every column and stage.  Chunk c is worked on while chunk c + 2 is written and
// chunks c + 3 to c + 6 are on their way from memory, a barrier a chunk; the sums of chunk c leave two chunks later.
template <int MODE, int DPAD>
__global__ __launch_bounds__(64 * RW) void recurrence_stages_kernel(RecurArgs a) {
  using S = StagesShape<MODE, DPAD>;
  constexpr bool CHANNELS = S::CHANNELS;
  constexpr int F = S::F, DH = S::DH, RC = S::RC, RING = S::RING, PRE = S::PRE, WCOLS = S::WCOLS, VW = S::VW, LINE = S::LINE;
  extern __shared__ __attribute__((aligned(16))) float stages_lds[];
  float* kqs = stages_lds;                                                    // F = 4: [row][lane][k0 k1 q0 q1]; F = 2: [row][k or q][lane][4]
  float* as = kqs + S::KQ;                                                    // F = 4: [row / 2][lane][row % 2][2]; F = 2: [row][lane][4]
  float* vs = as + S::A;                                                      // [VW][column][stage][row]
  float* outs = vs + S::V;                                                    // [column][row]
  const int tid = threadIdx.x, lane = tid & 63, wv = wave_index();
  // (all of a head's workgroups on one die, where the heads divide: its q, k and decays come from memory once)
  int h = blockIdx.y, block = blockIdx.x;
  if (a.heads % 8 == 0) {
    const int lin = (int)(blockIdx.y * gridDim.x + blockIdx.x), i = lin >> 3;
    h = (lin & 7) + 8 * (i / (int)gridDim.x);
    block = i % (int)gridDim.x;
  }
  const int first = a.seq_rows[2 * blockIdx.z], count = a.seq_rows[2 * blockIdx.z + 1], slot = a.slots[blockIdx.z];
  if (count <= 0 || slot < 0) return;
  if (a.positions[first] < 0) return;
  const int vdim = a.vdim, j_wg = block * WCOLS, hk = h / a.heads_per_key;
  const int in_col = lane & 31, stage = in_col % F, part = in_col / F;
  const int col = 2 * wv + (lane >> 5);
  const int chan = (stage * DH >> 2) * 4 * S::PARTS + 4 * part + (stage * DH & 3);   // this lane's channels, as the walk deals them to a part
  float* Sp = a.state + (size_t)slot * a.state_ld + ((size_t)h * vdim + j_wg + col) * DPAD + chan;
  float Sx[2][DH];                                                            // the memory at the tokens of even and of odd steps
#pragma unroll
  for (int d = 0; d < DH; ++d) Sx[1][d] = Sp[d];
  unsigned hand = stage == 0 ? 0u : 0xffffffffu;                              // the first stage starts its chains from zero
  asm("" : "+v"(hand));                                                       // (a mask: one instruction with the move between the lanes)

  // What a thread moves: a vector of q, k and decays (or two) of its token of a chunk; of waves 0 and 1 a v, of waves 2 and 3 a sum.
  // Every address is a scalar that moves with the chunk and an offset that does not (but for the last chunk's tokens past the portion).
  using Loads = StagesLoads<S::NL, CHANNELS>;
  static_assert(RC * WCOLS == 2 * 64, "a v a thread of two waves, a sum a thread of the others");
  const int vt = (tid & 127) / WCOLS, vc = tid % WCOLS;
  const bool brings = wv < 2;                                                 // (scalar)
  unsigned proj_at[S::NL], gate_at[S::NL], v_at;
  auto offsets = [&](int tokens) {                                            // with the chunk's first ``tokens`` tokens in the portion
#pragma unroll
    for (int u = 0; u < S::NL; ++u) {
      const int e = tid + 64 * RW * u, t = min(e / S::VECS, tokens - 1), d = 4 * (e % S::VECS);
      proj_at[u] = (unsigned)(t * a.ldp + d) * 4u;
      gate_at[u] = (unsigned)(t * a.ldg + d) * 4u;
    }
    v_at = (unsigned)(min(vt, tokens - 1) * a.ldp + vc) * 4u;
  };
  offsets(min(RC, count));
  auto at = [](const float* base, unsigned bytes) { return reinterpret_cast<const char*>(base) + bytes; };
  auto fetch = [&](Loads& l, int c) {
    const int t0 = min(c * RC, count - 1);                                    // (past the portion: not used)
    if (c * RC + RC > count) offsets(max(count - c * RC, 1));                 // (scalar; nothing comes behind)
    const float* row = a.proj + (size_t)(first + t0) * a.ldp;
    const float* qp = row + a.q_off + hk * DPAD;
    const float* kp = row + a.k_off + hk * DPAD;
    const float* gate = CHANNELS ? a.gate + (size_t)(first + t0) * a.ldg + a.gate_off + h * DPAD : nullptr;
#pragma unroll
    for (int u = 0; u < S::NL; ++u) {
      l.q[u] = *reinterpret_cast<const f32x4*>(at(qp, proj_at[u]));
      l.k[u] = *reinterpret_cast<const f32x4*>(at(kp, proj_at[u]));
      if constexpr (CHANNELS) l.a[u] = *reinterpret_cast<const f32x4*>(at(gate, gate_at[u]));
    }
    if (brings) {
      l.v = *reinterpret_cast<const float*>(at(row + a.v_off + h * vdim + j_wg, v_at));
      if constexpr (!CHANNELS) {
        const float* g = a.gate + (size_t)(first + min(c * RC + vt, count - 1)) * a.ldg;
        l.f = g[a.gate_off + h];
        l.i = g[a.gate2_off + h];
      }
    }
  };
  auto stash = [&](const Loads& l, int c) {
    const bool whole = c * RC + RC <= count;                                  // (scalar)
    const int row0 = (c * RC) & (RING - 1);
#pragma unroll
    for (int u = 0; u < S::NL; ++u) {
      const int e = tid + 64 * RW * u, t = e / S::VECS, i = e % S::VECS;
      f32x4 q4 = l.q[u], k4 = l.k[u], a4;
      if constexpr (CHANNELS) a4 = l.a[u];
#pragma unroll
      for (int x = 0; x < 4; ++x) q4[x] *= a.qscale;
      if (a.kscale != 1.0f) {                                                 // (scalar)
#pragma unroll
        for (int x = 0; x < 4; ++x) k4[x] *= a.kscale;
      }
      if (!whole && c * RC + t >= count) {
        q4 = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        k4 = (f32x4){-0.0f, -0.0f, -0.0f, -0.0f};
        if constexpr (CHANNELS) a4 = (f32x4){1.0f, 1.0f, 1.0f, 1.0f};
      }
      const int half = i / S::PARTS, p = i % S::PARTS;
      if constexpr (F == 4) {
#pragma unroll
        for (int w = 0; w < 2; ++w) {                                         // four channels are two stages'
          const int s = 2 * half + w, row = (row0 + t + s) & (RING - 1), to = p * 4 + s;
          *reinterpret_cast<f32x4*>(kqs + (row * 32 + to) * 4) = (f32x4){k4[2 * w], k4[2 * w + 1], q4[2 * w], q4[2 * w + 1]};
          if constexpr (CHANNELS) *reinterpret_cast<u32x2*>(as + (((row >> 1) * 32 + to) * 2 + (row & 1)) * 2) = (u32x2){__float_as_uint(a4[2 * w]), __float_as_uint(a4[2 * w + 1])};
        }
      } else {
        const int row = (row0 + t + half) & (RING - 1), to = p * 2 + half;
        *reinterpret_cast<f32x4*>(kqs + (row * 64 + to) * 4) = k4;
        *reinterpret_cast<f32x4*>(kqs + (row * 64 + 32 + to) * 4) = q4;
        if constexpr (CHANNELS) *reinterpret_cast<f32x4*>(as + (row * 32 + to) * 4) = a4;
      }
    }
    if (brings) {
      float w[VW];
      if constexpr (CHANNELS) {
        w[0] = l.v;
      } else {
        w[0] = l.f;
        w[1] = l.i * l.v;
      }
      if (!whole && c * RC + vt >= count)
#pragma unroll
        for (int x = 0; x < VW; ++x) w[x] = 1.0f;
#pragma unroll
      for (int s = 0; s < F; ++s)
#pragma unroll
        for (int x = 0; x < VW; ++x) vs[((x * WCOLS + vc) * F + s) * LINE + ((row0 + vt + s) & (RING - 1))] = w[x];
    }
  };
  // the tokens before the first one, which the later stages start with
  if (tid < 32) {
    const int s = tid % F;
    for (int r = 0; r < s; ++r) {
      if constexpr (F == 4) {
        *reinterpret_cast<f32x4*>(kqs + (r * 32 + tid) * 4) = (f32x4){-0.0f, -0.0f, 0.0f, 0.0f};
        if constexpr (CHANNELS)
          for (int x = 0; x < 2; ++x) as[(((r >> 1) * 32 + tid) * 2 + (r & 1)) * 2 + x] = 1.0f;
      } else {
        *reinterpret_cast<f32x4*>(kqs + (r * 64 + tid) * 4) = (f32x4){-0.0f, -0.0f, -0.0f, -0.0f};
        *reinterpret_cast<f32x4*>(kqs + (r * 64 + 32 + tid) * 4) = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (CHANNELS) *reinterpret_cast<f32x4*>(as + (r * 32 + tid) * 4) = (f32x4){1.0f, 1.0f, 1.0f, 1.0f};
      }
    }
  } else if (tid >= 64 && tid < 64 + VW * WCOLS * F) {
    const int s = (tid - 64) % F;
    for (int r = 0; r < s; ++r) vs[(tid - 64) * LINE + r] = 1.0f;
  }

  // A wave is alone on its SIMD, and an instruction that needs the result of the one before it costs twice its time.  So the
  // operations of a step are written in the order in which they issue, those of four tokens between one another (the product k v of
  // the token after the next, the memory at the next one, the chain of this one, the joins of the one before), each three
  // places and more behind what it needs.
  using Ops = StagesOps<DH, CHANNELS, VW>;
#define BW_NEXT __builtin_amdgcn_sched_barrier(0)
  float kv[2][DH], reached = 0.0f, joined = 0.0f;
  f32x4 left = {0.f, 0.f, 0.f, 0.f};
  auto product = [&](const Ops& o, int n, int d, float& r) { r = o.k[n][d] * o.v[VW - 1][n]; };
  auto memory = [&](const Ops& o, int n, int d, float before, float in, float& r) {
    if constexpr (CHANNELS) r = fmaf(o.a[n][d], before, in);
    else r = fmaf(o.v[0][n], before, in);
  };
  auto hand_on = [&]() { return __uint_as_float(__float_as_uint(stages_dpp<F == 4 ? 0x90 : 0xa0>(reached)) & hand); };   // (quads of lanes: from stage - 1 of the part)
  // token N of the group ``o``, the group behind it ``p`` (loaded under tokens 0 and 1: ``load0``, ``load1``)
  auto advance = [&](const Ops& o, Ops& p, auto index, auto load0, auto load1) {
    constexpr int N = decltype(index)::value, CUR = N & 1, NXT = CUR ^ 1;
    const Ops& o1 = N + 1 < 4 ? o : p;
    const Ops& o2 = N + 2 < 4 ? o : p;
    float c = hand_on();
    BW_NEXT;
    if constexpr (F == 2) joined += stages_dpp<0x112>(joined);                // row_shr:2: the parts' sums, neighbours first
    else joined += stages_dpp<0x114>(joined);                                 // row_shr:4
    BW_NEXT;
    memory(o1, (N + 1) & 3, 0, Sx[CUR][0], kv[NXT][0], Sx[NXT][0]);
    BW_NEXT;
    if constexpr (N == 0) {
      load0();
      BW_NEXT;
    }
    if constexpr (N == 1) {
      load1();
      BW_NEXT;
    }
    c = fmaf(Sx[CUR][0], o.q[N][0], c);
    BW_NEXT;
    memory(o1, (N + 1) & 3, 1, Sx[CUR][1], kv[NXT][1], Sx[NXT][1]);
    BW_NEXT;
    if constexpr (F == 2) joined += stages_dpp<0x114>(joined);
    else joined += stages_dpp<0x118>(joined);                                 // row_shr:8
    BW_NEXT;
    if constexpr (DH == 2) {
      product(o2, (N + 2) & 3, 0, kv[CUR][0]);
      BW_NEXT;
      c = fmaf(Sx[CUR][1], o.q[N][1], c);
      BW_NEXT;
      product(o2, (N + 2) & 3, 1, kv[CUR][1]);
      BW_NEXT;
    } else {
      memory(o1, (N + 1) & 3, 2, Sx[CUR][2], kv[NXT][2], Sx[NXT][2]);
      BW_NEXT;
      c = fmaf(Sx[CUR][1], o.q[N][1], c);
      BW_NEXT;
      memory(o1, (N + 1) & 3, 3, Sx[CUR][3], kv[NXT][3], Sx[NXT][3]);
      BW_NEXT;
      product(o2, (N + 2) & 3, 0, kv[CUR][0]);
      BW_NEXT;
      if constexpr (F == 2) joined += stages_dpp<0x118>(joined);
      BW_NEXT;
      c = fmaf(Sx[CUR][2], o.q[N][2], c);
      BW_NEXT;
      product(o2, (N + 2) & 3, 1, kv[CUR][1]);
      BW_NEXT;
      product(o2, (N + 2) & 3, 2, kv[CUR][2]);
      BW_NEXT;
      c = fmaf(Sx[CUR][3], o.q[N][3], c);
      BW_NEXT;
    }
    joined += stages_dpp<0x142>(joined);                                      // row_bcast:15: the last stage's last part holds the whole sum
    left[(N + 3) & 3] = joined;                                               // (of the token before)
    BW_NEXT;
    if constexpr (DH == 4) {
      product(o2, (N + 2) & 3, 3, kv[CUR][3]);
      BW_NEXT;
    }
    reached = joined = c;
  };
  const unsigned out0 = (unsigned)(uintptr_t)(lds_floats)(outs + col * LINE);
  // the two lanes that hold sums store four steps' (a branch costs as much as five instructions)
  auto store = [&](int row) {
    asm volatile("s_mov_b64 exec, %2\n\tds_write_b128 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(out0 + (unsigned)(row & (RING - 1)) * 4), "v"(left),
                 "s"(0x8000000080000000ull)
                 : "memory");
  };
  // four tokens' operands, of rows row .. row + 3 of the rings: from the block of eight rows that the pointers are at
  const lds_vectors kq0 = (lds_vectors)(kqs + in_col * 4), a0 = (lds_vectors)(as + in_col * 4);
  const lds_vectors v0 = (lds_vectors)(vs + (col * F + stage) * LINE);
  lds_vectors kqp = kq0, ap = a0, vp = v0;
  auto at_block = [&](int row) {                                              // (scalar)
    kqp = kq0 + row * (S::KQ_ROW / 4);
    ap = a0 + row * (S::A_ROW / 4);
    vp = v0 + row / 4;
    asm("" : "+v"(kqp), "+v"(ap), "+v"(vp));                                  // (a register each: offsets within the instructions)
  };
  auto load_kq = [&](Ops& o, int n0, int from, int to) {
#pragma unroll
    for (int n = from; n < to; ++n) {
      const f32x4 x = kqp[(n0 + n) * (S::KQ_ROW / 4)];
      if constexpr (F == 4) {
        o.k[n][0] = x[0];
        o.k[n][1] = x[1];
        o.q[n][0] = x[2];
        o.q[n][1] = x[3];
      } else {
        const f32x4 y = kqp[(n0 + n) * (S::KQ_ROW / 4) + 32];
#pragma unroll
        for (int d = 0; d < DH; ++d) {
          o.k[n][d] = x[d];
          o.q[n][d] = y[d];
        }
      }
    }
  };
  auto load_v = [&](Ops& o, int n0) {
#pragma unroll
    for (int x = 0; x < VW; ++x) {
      const f32x4 v = vp[x * (WCOLS * F * LINE / 4) + n0 / 4];
#pragma unroll
      for (int n = 0; n < 4; ++n) o.v[x][n] = v[n];
    }
  };
  auto load_a = [&](Ops& o, int n0) {
    if constexpr (CHANNELS) {
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        if constexpr (F == 4) {
          if (n % 2 == 0) {
            const f32x4 x = ap[(n0 + n) / 2 * 32];
            o.a[n][0] = x[0];
            o.a[n][1] = x[1];
            o.a[n + 1][0] = x[2];
            o.a[n + 1][1] = x[3];
          }
        } else {
          const f32x4 x = ap[(n0 + n) * 32];
#pragma unroll
          for (int d = 0; d < DH; ++d) o.a[n][d] = x[d];
        }
      }
    }
  };
  const int chunks = (count + PRE + RC - 1) / RC;
  Loads ahead[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) fetch(ahead[c], c);
  stash(ahead[0], 0);
  fetch(ahead[0], 4);
  stash(ahead[1], 1);
  fetch(ahead[1], 5);
  __syncthreads();
  Ops even, odd;
  load_kq(even, 0, 0, 4);
  load_v(even, 0);
  load_a(even, 0);
#pragma unroll
  for (int d = 0; d < DH; ++d) {
    product(even, 0, d, kv[0][d]);
    product(even, 1, d, kv[1][d]);
    memory(even, 0, d, Sx[1][d], kv[0][d], Sx[0][d]);
  }
  BW_NEXT;
  // sums leave by waves 2 and 3; what they are divided by is fetched a chunk ahead
  float den = 1.0f;
  const unsigned out_at = (unsigned)(vt * a.ldo + vc) * 4u;
  auto divisor = [&](int c) {
    if constexpr (CHANNELS) return 1.0f;
    else return brings ? 1.0f : a.gate[(size_t)(first + max(min(c * RC + vt - PRE, count - 1), 0)) * a.ldg + 2 * a.heads + h];
  };
  auto sum_of = [&](int c) { return outs[vc * LINE + ((c * RC + vt) & (RING - 1))]; };
  auto leave = [&](int c, float sum) {
    if (brings) return;                                                       // (scalar)
    const int t0 = c * RC - PRE;
    if (t0 + vt < 0 || t0 + vt >= count) return;
    float* to = a.out + ((long long)first + t0) * a.ldo + h * vdim + j_wg;
    *reinterpret_cast<float*>(reinterpret_cast<char*>(to) + out_at) = CHANNELS ? sum : sum / den;
  };
  auto chunk = [&](int c, Loads& l) {
    const float sum = sum_of(max(c - 2, 0));
#pragma unroll
    for (int half = 0; half < RC / 8; ++half) {
      const int row = c * RC + 8 * half;
      advance(even, odd, std::integral_constant<int, 0>{}, [&] { load_kq(odd, 4, 0, 2); load_v(odd, 4); }, [&] {});
      store(row - 4);
      advance(even, odd, std::integral_constant<int, 1>{}, [&] {}, [&] { load_a(odd, 4); load_kq(odd, 4, 2, 4); });
      at_block((row + 8) & (RING - 1));
      advance(even, odd, std::integral_constant<int, 2>{}, [&] {}, [&] {});
      advance(even, odd, std::integral_constant<int, 3>{}, [&] {}, [&] {});
      advance(odd, even, std::integral_constant<int, 0>{}, [&] { load_kq(even, 0, 0, 2); load_v(even, 0); }, [&] {});
      store(row);
      advance(odd, even, std::integral_constant<int, 1>{}, [&] {}, [&] { load_a(even, 0); load_kq(even, 0, 2, 4); });
      advance(odd, even, std::integral_constant<int, 2>{}, [&] {}, [&] {});
      advance(odd, even, std::integral_constant<int, 3>{}, [&] {}, [&] {});
      if (half == 0) {
        if (c + 2 < chunks) stash(l, c + 2);
        if (c >= 2) leave(c - 2, sum);
        den = divisor(max(c - 1, 0));
        if (c + 6 < chunks) fetch(l, c + 6);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);                                        // (the stores above are not the compiler's to count)
    __syncthreads();
  };
  // (left in the middle, not skipped through: a way back to the top that is never taken would have every wait for a set of loads
  // be a wait for the set just asked for)
  for (int c = 0;;) {
    chunk(c, ahead[2]);
    if (++c == chunks) break;
    chunk(c, ahead[3]);
    if (++c == chunks) break;
    chunk(c, ahead[0]);
    if (++c == chunks) break;
    chunk(c, ahead[1]);
    if (++c == chunks) break;
  }
  // the last token's joins, and what has not left yet
  if constexpr (F == 2) joined += stages_dpp<0x112>(joined);
  joined += stages_dpp<0x114>(joined);
  joined += stages_dpp<0x118>(joined);
  joined += stages_dpp<0x142>(joined);
  left[3] = joined;
  store(chunks * RC - 4);
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __syncthreads();
  for (int c = max(chunks - 2, 0); c < chunks; ++c) {
    den = divisor(c);
    leave(c, sum_of(c));
  }
#undef BW_NEXT
#pragma unroll
  for (int d = 0; d < DH; ++d) Sp[d] = Sx[1][d];
}

// The scalar gates of a portion, a workgroup a head and request: for every token the factor of the memory, that of the token's own
// k v^T, and what the read-out is divided by ([rows, 3 heads]), and the normaliser and the maximum in the slot (every copy of
// them).  The statements of the walk's preparation of a chunk.  The gates themselves by all threads; then four kinds of waves a chunk
// of 32 tokens behind one another, a barrier a chunk: the running maximum, which is the one chain; the factors (a token a lane); the
// normaliser (a channel a lane); its product with q, summed over the lanes.
// What bounds it: the instructions of a compute unit's four SIMDs, of which the keeping waves and the summing ones share two.  Sums of
// eight tokens go through the lanes together (wave_sums_of_eight): 2,048 tokens of 8 heads of 128 77 -> 72 us.  Then the keys' way: loads a token were more than a
// wave may count, so no more than two chunks were on their way; four tokens a load, straight into LDS, five chunks ahead: 72 -> 61.
#define SG_CHUNK 32
#define SG_TOKENS 2048   // whose gates lie in LDS together
#define SG_SUMS 4        // waves that sum
#define SG_SLOTS 6       // chunks of keys in LDS

// wave_sum of eight values: the same additions, but where a step of a butterfly leaves both halves with the same sums, here each half
// goes on with another value's (20 instructions for what eight butterflies take some 90).  A lane has the sum of value number
// sum_of_eight_at(lane).
__device__ __forceinline__ int sum_of_eight_at(int lane) { return 4 * ((lane >> 3) & 1) + 2 * ((lane >> 4) & 1) + (lane >> 5); }
__device__ __forceinline__ float wave_sums_of_eight(const float (&v)[8], int lane) {
  typedef __attribute__((ext_vector_type(2))) unsigned u2;
  float x[4], y[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {                                                // values 2 i in the lower half of the wave, 2 i + 1 in the upper
    const u2 h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[2 * i]), __float_as_uint(v[2 * i + 1]), false, false);
    x[i] = __uint_as_float(h[0]) + __uint_as_float(h[1]);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {                                                // rows of 16 lanes: values 4 i, 4 i + 2, 4 i + 1, 4 i + 3
    const u2 h = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[2 * i]), __float_as_uint(x[2 * i + 1]), false, false);
    y[i] = __uint_as_float(h[0]) + __uint_as_float(h[1]);
  }
  const bool upper = (lane & 8) != 0;                                          // halves of a row: y[0] and y[1]
  float z = (upper ? y[1] : y[0]) + lane_xor<8>(upper ? y[0] : y[1]);
  z += lane_xor<4>(z);
  z += lane_xor<2>(z);
  z += lane_xor<1>(z);
  return z;
}

template <int NN>
__global__ __launch_bounds__(64 * (2 + NN + SG_SUMS)) void scalar_gates_kernel(RecurArgs a, float* __restrict__ gates, int copies) {
#if defined(__HIP_DEVICE_COMPILE__)                                            // (buffer descriptors are a type of the device pass)
  constexpr int T = SG_CHUNK, DIM = 64 * NN, THREADS = 64 * (2 + NN + SG_SUMS), MINE = T / SG_SUMS;
  __shared__ __attribute__((aligned(16))) float gi[SG_TOKENS], gf[SG_TOKENS], mx[2][T], before[2], ems[4][T], fib[2][T][2];
  extern __shared__ __attribute__((aligned(16))) float sg_n[];                // [2][T][DIM], then the keeping waves' keys
  const int lane = threadIdx.x & 63, wave = wave_index(), h = blockIdx.x;
  const int first = a.seq_rows[2 * blockIdx.y], count = a.seq_rows[2 * blockIdx.y + 1], slot = a.slots[blockIdx.y];
  if (count <= 0 || slot < 0) return;
  if (a.positions[first] < 0) return;
  const int hk = h / a.heads_per_key, ldo = 3 * a.heads;
  const size_t copy = (size_t)a.heads * DIM + a.heads;
  float* nv = a.state + (size_t)slot * a.state_ld + (size_t)a.heads * DIM * a.vdim + (size_t)h * DIM;
  float* mv = a.state + (size_t)slot * a.state_ld + (size_t)a.heads * DIM * a.vdim + (size_t)a.heads * DIM + h;
  const int ch = 64 * (wave - 2) + lane, w = wave - 2 - NN;
  const bool keeps = wave >= 2 && wave < 2 + NN;
  float m = *mv, n = keeps ? nv[ch] : 0.0f;
  __syncthreads();                                                             // (the state is read before anybody writes it)
  const float cap = a.param, bi = a.bias[h], bf = a.bias2[h];
  for (int base = 0; base < count; base += SG_TOKENS) {
    const int tokens = min(SG_TOKENS, count - base), chunks = (tokens + T - 1) / T;
    float* g0 = gates + (size_t)(first + base) * ldo + h;
    for (int t = threadIdx.x; t < tokens; t += THREADS) {
      const float* g = a.gate + (size_t)(first + base + t) * a.ldg;
      gi[t] = cap * tanhf((g[a.gate_off + h] + bi) / cap);
      gf[t] = log_sigmoid(cap * tanhf((g[a.gate2_off + h] + bf) / cap));
    }
    __syncthreads();
    auto rows_of = [&](int c) { return min(T, tokens - c * T); };
    // a wave's part of a step: chunk s behind the chunks that the waves before it are at
    auto steps = [&](int behind, auto work) {
      for (int s = 0; s < chunks + 3; ++s) {
        const int c = s - behind;
        if (c >= 0 && c < chunks) work(c);
        __syncthreads();
      }
    };
    if (wave == 0) {
      steps(0, [&](int c) {
        const int tc = rows_of(c);
        const float* f0 = gf + c * T;
        const float* i0 = gi + c * T;
        if (lane == 0) before[c & 1] = m;
        if (tc == T) {
          f32x4 f[T / 4], i[T / 4];
#pragma unroll
          for (int e = 0; e < T / 4; ++e) {
            f[e] = *reinterpret_cast<const f32x4*>(f0 + 4 * e);
            i[e] = *reinterpret_cast<const f32x4*>(i0 + 4 * e);
          }
#pragma unroll
          for (int e = 0; e < T / 4; ++e) {
            f32x4 m4;
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              m = fmaxf(f[e][x] + m, i[e][x]);
              m4[x] = m;
            }
            *reinterpret_cast<f32x4*>(&mx[c & 1][4 * e]) = m4;
          }
        } else {
          for (int t = 0; t < tc; ++t) {
            m = fmaxf(f0[t] + m, i0[t]);
            mx[c & 1][t] = m;
          }
        }
      });
    } else if (wave == 1) {
      steps(1, [&](int c) {
        const int t = lane & (T - 1);
        const bool in = lane < rows_of(c);
        const float was = t == 0 ? before[c & 1] : mx[c & 1][max(t - 1, 0)];
        const float mn = mx[c & 1][t], x = gf[c * T + t] + was;
        const float fa = bw_expf(x - mn), ib = bw_expf(gi[c * T + t] - mn), em = bw_expf(-mn);
        if (in) {
          fib[c & 1][t][0] = fa;
          fib[c & 1][t][1] = ib;
          ems[c & 3][t] = em;
          float* g = g0 + (size_t)(c * T + t) * ldo;
          g[0] = fa;
          g[a.heads] = ib;
        }
      });
    } else {
      // queries: four chunks in registers, three of them on their way
      const bool sums = wave >= 2 + NN;
      const float* from = a.proj + (size_t)(first + base) * a.ldp + (sums ? a.q_off : a.k_off) + hk * DIM;   // (scalar)
      const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc((void*)from, 0, (int)((((size_t)tokens - 1) * a.ldp + DIM) * 4), 0x00020000);
      const int row_bytes = a.ldp * 4;
      if (!sums) {
        // A wave's keys: [SG_SLOTS chunks][T][64 channels] of LDS that nobody else touches, filled straight from memory (four tokens
        // a load), SG_SLOTS - 1 chunks ahead.  Rows past the portion's end lie outside the descriptor (zeros, never used).
        float* keys = sg_n + 2 * T * DIM + (wave - 2) * SG_SLOTS * T * 64;
        const unsigned at = (unsigned)(lane >> 4) * row_bytes + 256 * (wave - 2) + 16 * (lane & 15);
        auto fetch = [&](int c, int slot) {
          typedef __attribute__((address_space(3))) void* lds_ptr;
#pragma unroll
          for (int t = 0; t < T / 4; ++t)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (lds_ptr)(keys + (slot * T + 4 * t) * 64), 16, (int)(at + (unsigned)(c * T + 4 * t) * row_bytes), 0, 0, 0);
        };
        auto run = [&](int c, int slot) {
          const int tc = rows_of(c);
          const float* kc = keys + slot * T * 64 + lane;
          float* out = sg_n + (c & 1) * T * DIM + ch;
          if (tc == T) {
            float k[T];
#pragma unroll
            for (int t = 0; t < T; ++t) k[t] = kc[t * 64];
#pragma unroll
            for (int t = 0; t < T; t += 2) {
              const f32x4 two = *reinterpret_cast<const f32x4*>(&fib[c & 1][t][0]);
              n = fmaf(two[0], n, two[1] * (k[t] * a.kscale));
              out[t * DIM] = n;
              n = fmaf(two[2], n, two[3] * (k[t + 1] * a.kscale));
              out[(t + 1) * DIM] = n;
            }
          } else {
            for (int t = 0; t < tc; ++t) {
              n = fmaf(fib[c & 1][t][0], n, fib[c & 1][t][1] * (kc[t * 64] * a.kscale));
              out[t * DIM] = n;
            }
          }
        };
        for (int c = 0; c < SG_SLOTS - 1; ++c) fetch(c, c);
        for (int i = 0; i < 2; ++i) __syncthreads();
        int slot = 0;
        for (int c = 0; c < chunks; ++c) {
          fetch(c + SG_SLOTS - 1, slot == 0 ? SG_SLOTS - 1 : slot - 1);        // (where the chunk before lay)
          __builtin_amdgcn_s_waitcnt(vmcnt_only((SG_SLOTS - 1) * (T / 4)));    // this chunk's have landed: loads land in order
          asm volatile("" ::: "memory");
          run(c, slot);
          slot = slot == SG_SLOTS - 1 ? 0 : slot + 1;
          __syncthreads();
        }
        __builtin_amdgcn_s_waitcnt(vmcnt_only(0));                             // (those past the end, too, before the places are used again)
        for (int i = 2; i < 3; ++i) __syncthreads();
      } else {
        float q0[MINE][NN], q1[MINE][NN], q2[MINE][NN], q3[MINE][NN];
        auto fetch = [&](float (&q)[MINE][NN], int c) {
#pragma unroll
          for (int t = 0; t < MINE; ++t)
#pragma unroll
            for (int i = 0; i < NN; ++i)
              q[t][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rows, lane * 4 + 256 * i, min(c * T + w * MINE + t, tokens - 1) * row_bytes, 0));
        };
        auto run = [&](const float (&q)[MINE][NN], int c) {
          const float* in = sg_n + (c & 1) * T * DIM + w * MINE * DIM + lane;
          static_assert(MINE == 8, "a wave's tokens of a chunk are summed together");
          float sum[MINE];
#pragma unroll
          for (int t = 0; t < MINE; ++t) {
            sum[t] = 0.0f;
#pragma unroll
            for (int i = 0; i < NN; ++i) sum[t] = fmaf(in[t * DIM + 64 * i], q[t][i] * a.qscale, sum[t]);
          }
          const float mine = wave_sums_of_eight(sum, lane);
          const int t = w * MINE + sum_of_eight_at(lane);
          if ((lane & 7) == 0 && t < rows_of(c)) g0[(size_t)(c * T + t) * ldo + 2 * a.heads] = fmaxf(fabsf(mine), ems[c & 3][t]) + 1e-6f;
        };
        fetch(q0, 0);
        fetch(q1, 1);
        fetch(q2, 2);
        for (int i = 0; i < 3; ++i) __syncthreads();
        for (int c = 0;;) {                                                     // (left in the middle, as the walk in stages is)
          fetch(q3, c + 3); run(q0, c); __syncthreads(); if (++c == chunks) break;
          fetch(q0, c + 3); run(q1, c); __syncthreads(); if (++c == chunks) break;
          fetch(q1, c + 3); run(q2, c); __syncthreads(); if (++c == chunks) break;
          fetch(q2, c + 3); run(q3, c); __syncthreads(); if (++c == chunks) break;
        }
        for (int i = 3; i < 3; ++i) __syncthreads();
      }
    }
  }
  for (int k = 0; k < copies; ++k) {
    if (wave == 0 && lane == 0) mv[k * copy] = m;
    if (keeps) nv[k * copy + ch] = n;
  }
#endif
}

// Whether the kernel takes the layout: whole heads of 64 or 128 channels, whole vectors.
static bool stages_fit(const RecurArgs& a, int mode) {
  return (a.dim == 64 || a.dim == 128) && a.vdim % (2 * RW) == 0 && ((a.q_off | a.k_off | a.ldp) & 3) == 0 && (reinterpret_cast<uintptr_t>(a.proj) & 15) == 0 &&
         a.ldp < (1 << 18) && a.ldg < (1 << 18) && a.ldo < (1 << 18) &&
         (mode != RECUR_DECAY_GIVEN || (((a.ldg | a.gate_off) & 3) == 0 && (reinterpret_cast<uintptr_t>(a.gate) & 15) == 0));
}

template <int MODE, int DPAD>
static int launch_stages(const RecurArgs& a, int nseq, hipStream_t s) {
  using S = StagesShape<MODE, DPAD>;
  static bool allowed = false;                       // more than 64 KB of dynamic LDS has to be asked for once
  if (S::LDS > 48 * 1024 && !allowed) {
    (void)hipFuncSetAttribute((const void*)recurrence_stages_kernel<MODE, DPAD>, hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS);
    allowed = true;
  }
  hipLaunchKernelGGL((recurrence_stages_kernel<MODE, DPAD>), dim3(a.vdim / S::WCOLS, a.heads, nseq), dim3(64 * RW), S::LDS, s, a);
  return BW_LAUNCH_CHECK();
}

template <int NN>
static int launch_scalar_gates(const RecurArgs& a, float* gates, int nseq, hipStream_t s) {
  constexpr int lds = (2 + SG_SLOTS) * SG_CHUNK * 64 * NN * 4;
  static bool allowed = false;
  if (lds > 48 * 1024 && !allowed) {
    (void)hipFuncSetAttribute((const void*)scalar_gates_kernel<NN>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    allowed = true;
  }
  hipLaunchKernelGGL((scalar_gates_kernel<NN>), dim3(a.heads, nseq), dim3(64 * (2 + NN + SG_SUMS)), lds, s, a, gates, recur_blocks(a.dim, a.vdim));
  return BW_LAUNCH_CHECK();
}

static int launch_in_stages(int mode, const RecurArgs& a, float* gates, int nseq, hipStream_t s) {
  if (mode == RECUR_DECAY_GIVEN) return a.dim == 64 ? launch_stages<RECUR_DECAY_GIVEN, 64>(a, nseq, s) : launch_stages<RECUR_DECAY_GIVEN, 128>(a, nseq, s);
  const int rc = a.dim == 64 ? launch_scalar_gates<1>(a, gates, nseq, s) : launch_scalar_gates<2>(a, gates, nseq, s);
  if (rc != 0) return rc;
  RecurArgs b = a;
  b.gate = gates;
  b.ldg = 3 * a.heads;
  b.gate_off = 0;
  b.gate2_off = a.heads;
  return a.dim == 64 ? launch_stages<RECUR_SCALAR_GATES, 64>(b, nseq, s) : launch_stages<RECUR_SCALAR_GATES, 128>(b, nseq, s);
}
