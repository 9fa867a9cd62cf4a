// Recurrent matrix-memory mixers for ragged batches.
//
//   S_t = a_t S_(t-1) + b_t k_t v_t^T,    o_t = S_t^T q_t
//
// per head, with a 32-bit state S [D][E] per (slot, head) that lives across
// steps.  Four gatings share the kernels:
//
//   decay  a_t = decay_h, b_t = 1; q, k and v pass through silu.
//   gated  log gates i, f from a projection, soft-capped:
//            i = cap tanh(x_i / cap), f = logsigmoid(cap tanh(x_f / cap)),
//          a running maximum m keeps S and the normaliser n in range:
//            m_t = max(f + m_(t-1), i), a_t = exp(f + m_(t-1) - m_t),
//            b_t = exp(i - m_t), n_t = a_t n_(t-1) + b_t k_t,
//            o_t = S_t^T q_t / (max(|n_t . q_t|, exp(-m_t)) + 1e-6);
//          q is scaled by qscale.  S, n and m are zero at position 0.
//   timed  a time step from a projection (state-space duality):
//            b_t = softplus(x + bias), a_t = exp(-exp(A_log) b_t),
//          heads share q and k in groups, o_t + skip v_t is multiplied by
//          silu(z).
//   turned a_t = decay_h, b_t = kscale; q and k are rotated at their position,
//          in halves: elements i and i + rot / 2 turn together.
//
//   sv_memory_steps   token after token; single-token decoding, the 32-bit
//                     mode and sizes the chunk kernels do not take
//   sv_memory_chunks  256-token chunks on MFMA for bf16 prompt portions
//
// Every group of 32 state columns keeps its own copy of n and m, so the
// workgroups of a head never wait for each other.
//
// A segment whose context is empty starts from zero instead of reading its
// slot, so a slot needs no clearing when it changes hands.

#include "serving.h"

#define GATED_EPS 1e-6f

enum Gating { DECAY = 0, GATED = 1, TIMED = 2, TURNED = 3 };

struct MemoryArgs {
  const void *q, *k, *v;    // first row of the step's projections
  long qst, kst, vst;       // row strides (elements)
  const float* gates;       // [T][2 H] raw i then f (gated); [T][H] (timed)
  const void *ib, *fb;      // [H] biases, T: of i and f (gated); of the time
                            //   step, and A_log (timed)
  const float* decay;       // [H] (decay, turned)
  const float* log2_decay;  // [H] (decay, turned)
  float* S;                 // [slots][H][D][E]
  float* n;                 // [slots][H][ceil(E / 32)][D] (gated)
  float* m;                 // [slots][H][ceil(E / 32)] (gated)
  const int* seg;           // [n_seg][4]: slot, first row, rows, context
  void* out;                // [T][H * E]
  int H, D, E;
  float gate_cap, qscale;
  // timed only
  int G;                    // heads of q and k
  const void* skip;         // [H], T
  const void* z;            // [T][H * E] rows
  long zst;
  // q, k and v of single tokens before their causal convolution (steps only)
  const void *cw, *cb;      // [taps][C], [C]; cw null: they have passed it
  void* ring;               // [slots][taps][C]: position p in place p % taps
  int taps, C, kch, qch;    // channels of v, k, q start at 0, kch, qch
  // turned only
  const double* freq;       // [rot / 2] radians a position
  int rot;
  float amp, kscale;        // cos and sin are multiplied by amp
};

__device__ __forceinline__ float softplus_f(float x) {
  return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x)));
}

__device__ __forceinline__ void log_gates(const MemoryArgs& a, float gi, float gf,
                                          float ib, float fb, float& i, float& f) {
  i = a.gate_cap * tanhf((gi + ib) / a.gate_cap);
  f = log_sigmoid_f(a.gate_cap * tanhf((gf + fb) / a.gate_cap));
}
__device__ __forceinline__ void log_gates(const MemoryArgs& a, long row,
                                          int h, float ib, float fb,
                                          float& i, float& f) {
  const float* g = a.gates + row * 2 * a.H;
  log_gates(a, g[h], g[a.H + h], ib, fb, i, f);
}

// ---------------------------------------------------------------------------
// token after token: a workgroup owns 32 columns of one head's state
// ---------------------------------------------------------------------------
// TAPS: 0 no convolution, 1 any number of taps, else this number
// once: states that no cache keeps.  Bound by reading and writing them.  One step's are
// in no cache at the next where there are more of them than the 256 MB behind the L2s,
// and are then read and written faster past it; fewer may be there still (us, kept and
// past: 32 heads of 128 x 128, 128 tokens (268 MB) 106, 87; 64: 54, 45; 32 (67 MB)
// 23, 25; 128 heads of 128 x 64, 32 tokens (134 MB) 55, 46.5).
template <typename T, int NI, int GATE, bool VEC, int TAPS>
__global__ void __launch_bounds__(256)
memory_steps_kernel(MemoryArgs a, bool once) {
  const int D = a.D, E = a.E;
  const int nt = (E + 31) / 32;
  const int vt = blockIdx.x % nt;
  const int h = blockIdx.x / nt % a.H;
  const int* sg = a.seg + 4 * (blockIdx.x / nt / a.H);
  const long slot = sg[0];
  const int row0 = sg[1], nrow = sg[2], ctx = sg[3];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int vq = tid & 7, dg = tid >> 3;
  const int e0 = vt * 32 + 4 * vq;

  __shared__ float sq[2][NI * 32], sk[2][NI * 32], sv[2][32];
  __shared__ float red[2][4][32], redn[2][4];

  float* Sp = a.S + (slot * a.H + h) * D * E;
  float S[NI][4];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) S[i][j] = 0.f;
  auto each_word = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int d = dg + 32 * i;
      if (d < D && e0 < E) f((f32x4*)(Sp + (long)d * E + e0), S[i]);
    }
  };
  if (ctx > 0) {
    if (VEC && once) {
      each_word([](f32x4* p, float* s) {
        const f32x4 w = __builtin_nontemporal_load(p);
#pragma unroll
        for (int j = 0; j < 4; ++j) s[j] = w[j];
      });
    } else if (VEC) {
      each_word([](f32x4* p, float* s) { load4((const float*)p, s); });
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int d = dg + 32 * i;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (d < D && e0 + j < E) S[i][j] = Sp[(long)d * E + e0 + j];
      }
    }
  }
  // n: dim d belongs to thread d (and d + 256)
  constexpr int NN = (NI * 32 + 255) / 256;
  float n[NN], m = 0.f, ib = 0.f, fb = 0.f;
  if (GATE == GATED) {
#pragma unroll
    for (int i = 0; i < NN; ++i) {
      const int d = tid + 256 * i;
      n[i] = ctx > 0 && d < D ? a.n[((slot * a.H + h) * nt + vt) * D + d] : 0.f;
    }
    if (ctx > 0) m = a.m[(slot * a.H + h) * nt + vt];
  }
  constexpr bool fixed = GATE == DECAY || GATE == TURNED;
  if (!fixed) {
    ib = to_f(((const T*)a.ib)[h]);
    fb = to_f(((const T*)a.fb)[h]);
  }
  const float decay = fixed ? a.decay[h] : 0.f;
  const int hk = GATE == TIMED ? h / (a.H / a.G) : h;   // head of q and k
  constexpr bool conv = TAPS > 0;
  // The convolution of a single token: channel c's filter and earlier inputs,
  // and its result; `keep` writes the token's own input into the ring.
  constexpr int NT = TAPS > 1 ? TAPS : 1;
  const int last = (TAPS > 1 ? TAPS : a.taps) - 1;
  const int here = conv ? ctx % (last + 1) : 0;
  auto place = [&](int k) {              // of the input last - k tokens ago
    const int i = here - last + k;
    return (long)(i < 0 ? i + last + 1 : i) * a.C;
  };
  auto convolve = [&](float x, int c, bool keep) {
    T* ring = (T*)a.ring + slot * (last + 1) * a.C + c;
    const T* w = (const T*)a.cw + c;
    float y = to_f(((const T*)a.cb)[c]);
    if (TAPS > 1) {
      float f[NT], in[NT];
#pragma unroll
      for (int k = 0; k < NT; ++k) {
        f[k] = to_f(w[(long)k * a.C]);
        in[k] = k < NT - 1 ? to_f(ring[place(k)]) : x;
      }
#pragma unroll
      for (int k = 0; k < NT; ++k)
        y += k >= last - ctx ? f[k] * in[k] : 0.f;
    } else {
      for (int k = max(0, last - ctx); k < last; ++k)
        y += to_f(w[(long)k * a.C]) * to_f(ring[place(k)]);
      y += to_f(w[(long)last * a.C]) * x;
    }
    if (keep) from_f(ring[(long)here * a.C], x);
    return silu_f(y);
  };

  for (int t = 0; t < nrow; ++t) {
    const long row = row0 + t;
    const int b = t & 1;
    for (int d = tid; d < NI * 32; d += 256) {
      float x = 0.f, y = 0.f;
      if (d < D) {
        x = to_f(((const T*)a.q)[row * a.qst + (long)hk * D + d]);
        y = to_f(((const T*)a.k)[row * a.kst + (long)hk * D + d]);
        if (GATE == GATED) x *= a.qscale;
        if (GATE == TURNED && d < a.rot) {
          const int half = a.rot / 2;
          const bool low = d < half;
          const int i = low ? d : d - half;
          const long o = (long)hk * D + (low ? d + half : i);
          float c, s;
          turn(a.freq[i], ctx + t, &c, &s);
          c *= a.amp;
          s *= low ? -a.amp : a.amp;
          x = x * c + to_f(((const T*)a.q)[row * a.qst + o]) * s;
          y = y * c + to_f(((const T*)a.k)[row * a.kst + o]) * s;
        }
        if (GATE == TURNED) y *= a.kscale;
        if (GATE == DECAY) { x = silu_f(x); y = silu_f(y); }
        if (conv) {
          const bool keep = vt == 0 && h % (a.H / a.G) == 0;
          x = convolve(x, a.qch + hk * D + d, keep);
          y = convolve(y, a.kch + hk * D + d, keep);
        }
      }
      sq[b][d] = x;
      sk[b][d] = y;
    }
    if (tid < 32) {
      const int e = vt * 32 + tid;
      float x = e < E ? to_f(((const T*)a.v)[row * a.vst + (long)h * E + e])
                      : 0.f;
      if (GATE == DECAY) x = silu_f(x);
      if (conv && e < E) x = convolve(x, h * E + e, true);
      sv[b][tid] = x;
    }
    float fs = decay, is = 1.f;
    if (GATE == TIMED) {
      is = softplus_f(a.gates[row * a.H + h] + ib);
      fs = expf(-expf(fb) * is);
    }
    if (GATE == GATED) {
      float gi, gf;
      log_gates(a, row, h, ib, fb, gi, gf);
      const float mn = fmaxf(gf + m, gi);
      fs = expf(gf + m - mn);
      is = expf(gi - mn);
      m = mn;
    }
    __syncthreads();
    float v[4], o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = sv[b][4 * vq + j] * is;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const float kd = sk[b][dg + 32 * i], qd = sq[b][dg + 32 * i];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        S[i][j] = fs * S[i][j] + kd * v[j];
        o[j] += qd * S[i][j];
      }
    }
#pragma unroll
    for (int off = 8; off < 64; off <<= 1)
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] += __shfl_xor(o[j], off, 64);
    if (lane < 8)
#pragma unroll
      for (int j = 0; j < 4; ++j) red[b][wid][4 * vq + j] = o[j];
    if (GATE == GATED) {
      float nq = 0.f;
#pragma unroll
      for (int i = 0; i < NN; ++i) {
        const int d = tid + 256 * i;
        if (d < NI * 32) {
          n[i] = fs * n[i] + is * sk[b][d];
          nq += n[i] * sq[b][d];
        }
      }
      nq = wave_reduce(nq, SumOp());
      if (lane == 0) redn[b][wid] = nq;
    }
    __syncthreads();
    if (tid < 32 && vt * 32 + tid < E) {
      float r = red[b][0][tid] + red[b][1][tid] + red[b][2][tid] +
                red[b][3][tid];
      if (GATE == GATED) {
        const float nq = redn[b][0] + redn[b][1] + redn[b][2] + redn[b][3];
        r /= fmaxf(fabsf(nq), expf(-m)) + GATED_EPS;
      }
      if (GATE == TIMED) {
        const long at = (long)h * E + vt * 32 + tid;
        r += to_f(((const T*)a.skip)[h]) * sv[b][tid];
        r *= silu_f(to_f(((const T*)a.z)[row * a.zst + at]));
      }
      from_f(((T*)a.out)[row * a.H * E + (long)h * E + vt * 32 + tid], r);
    }
  }

  if (VEC && once) {
    each_word([](f32x4* p, float* s) {
      __builtin_nontemporal_store(f32x4{s[0], s[1], s[2], s[3]}, p);
    });
  } else if (VEC) {
    each_word([](f32x4* p, float* s) { store4((float*)p, s); });
  } else {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int d = dg + 32 * i;
      if (d >= D) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (e0 + j < E) Sp[(long)d * E + e0 + j] = S[i][j];
    }
  }
  if (GATE == GATED) {
#pragma unroll
    for (int i = 0; i < NN; ++i) {
      const int d = tid + 256 * i;
      if (d < D) a.n[((slot * a.H + h) * nt + vt) * D + d] = n[i];
    }
    if (tid == 0) a.m[(slot * a.H + h) * nt + vt] = m;
  }
}

template <typename T, int GATE, int TAPS>
static int launch_steps(const MemoryArgs& a, int n_seg, hipStream_t stream) {
  const long grid = (long)n_seg * a.H * ((a.E + 31) / 32);
  const bool vec = a.E % 4 == 0;
  const bool once = (long)n_seg * a.H * a.D * a.E * 4 > 100L << 20;
#define MS(N, V) \
  memory_steps_kernel<T, N, GATE, V, TAPS><<<grid, 256, 0, stream>>>(a, once)
#define MSV(N) do { if (vec) MS(N, true); else MS(N, false); } while (0)
  if (a.D <= 64) MSV(2);
  else if (a.D <= 128) MSV(4);
  else if (a.D <= 256) MSV(8);
  else if (a.D <= 512) MSV(16);
  else return 1;
#undef MSV
#undef MS
  return (int)hipGetLastError();
}

extern "C" int sv_memory_steps(const MemoryArgs* a, int n_seg, int gating,
                               int f32, hipStream_t stream) {
  if (n_seg <= 0) return 0;
#define MST(T, K) launch_steps<T, TIMED, K>(*a, n_seg, stream)
#define MS(T)                                                            \
  (gating == GATED   ? launch_steps<T, GATED, 0>(*a, n_seg, stream)      \
   : gating == DECAY ? launch_steps<T, DECAY, 0>(*a, n_seg, stream)      \
   : gating == TURNED ? launch_steps<T, TURNED, 0>(*a, n_seg, stream)    \
   : !a->cw ? MST(T, 0) : a->taps == 4 ? MST(T, 4) : MST(T, 1))
  if (gating == TURNED && (a->rot % 2 || a->rot > a->D)) return 1;
  return f32 ? MS(float) : MS(short);
#undef MS
#undef MST
}


// ---------------------------------------------------------------------------
// Chunks on MFMA (bf16 projections, 32-bit everything else)
//
// A portion is cut into chunks of 256 tokens, and every chunk is computed in
// parallel; only a scan over the chunks' states is sequential.  With local
// inclusive sums b_t of the log forgets, c_t = max(f_t + c_(t-1), i_t) from
// c = -inf, and m, S, n before the chunk:
//
//   gates    b_t, i_t, c_t of every token
//   states   U = sum_s e^(b_L - b_s + i_s - c_L) k_s v_s^T   (and N with k_s)
//   scan     m' = max(b_L + m, c_L)
//            S' = e^(b_L + m - m') S + e^(c_L - m') U        (n' likewise)
//   outputs  m_t = max(b_t + m, c_t)
//            o_t ~ e^(b_t + m - m_t) S^T q_t
//                  + sum_(s<=t) e^(b_t - b_s + i_s - m_t) (q_t . k_s) v_s
//
// every exponent is <= 0.  b is kept per 64 tokens (with the four totals of
// a chunk), so near tokens never cancel large sums.  The fixed decays have
// e^(b_t - b_s + i_s - m_t) = decay^(t-s) and no m; the timed gating has
// e^(b_t - b_s) times the time step of s, and no m.
//
// 32-bit operands meet bf16 ones exactly: an f32 value is split into three
// bf16 planes (8 + 8 + 8 bits) and each plane is multiplied on its own.
// Rotated queries and keys are split into two planes (a rest below 2^-17);
// where two split values meet, products below 2^-24 are left out.
// Scores are produced transposed (lane = query), so they feed the next
// product as its B operand from registers: the accumulator's row order is
// the contraction order, and V^T is read from LDS in that same order.
// ---------------------------------------------------------------------------
#define MC_L 256

struct ChunkArgs {
  MemoryArgs a;
  const int* chunks;        // [n_chunks][4]: segment, first row, rows, ctx > 0
                            //   or not the first chunk of its segment
  const int* first;         // [n_seg + 1] first chunk of a segment
  int n_chunks, n_seg, T;
  float *b, *i, *c;         // [H][T] (gated; timed: i is the step, no c)
  float *tot, *cend;        // [n_chunks][H][4], [n_chunks][H] (gated; timed:
                            //   no cend)
  float* U;                 // [n_chunks][H][E][D]; or null (no VT): a state is
                            //   carried from chunk to chunk
  float* N;                 // [n_chunks][H][D] (gated): N, then n before
  short* P;                 // [n_chunks][H][3][E][D] state before the chunk; if
                            //   there is no U [n_chunks][H][E / 32][3][D / 16]
                            //   [64][8]: keys 16 c + 8 hi + 0..7 of column col;
                            //   or null: nothing is left between chunks (not
                            //   turned, D 128, E a multiple of 64, no VT and U)
  float* mst;               // [n_chunks][H] m before the chunk (gated)
  short* VT;                // [n_chunks][H][E][256] V^T, activated; or null
                            //   (timed, D 64 or 128, or not turned and no P; E a
                            //   multiple of 64)
  short* KA;                // [T][H][D] activated K (decay); two planes of
                            //   rotated K (turned)
  short* QA;                // two planes of rotated Q (turned)
  float norm_eps;           // turned, with z: every head over its root mean
                            //   square, times silu(z)
};

__host__ __device__ constexpr bool fixed_decay(int gate) {
  return gate == DECAY || gate == TURNED;
}
// planes of queries and keys
__host__ __device__ constexpr int qk_planes(int gate) {
  return gate == TURNED ? 2 : 1;
}

// split a pair of floats into three planes of packed bf16
__device__ __forceinline__ void split3(float x, float y, uint* w) {
#pragma unroll
  for (int z = 0; z < 3; ++z) {
    w[z] = pack_bf16x2(x, y);
    x -= __uint_as_float(w[z] << 16);
    y -= __uint_as_float(w[z] & 0xffff0000u);
  }
}
// The same, cut off instead of rounded, since three of 8 bits hold all 24 either way.
// Masks take fewer cycles than shifts and packed conversions: one pass over 2731 and
// 1365 tokens 104.4 -> 103.1 us (two runs differ by 0.1), 1293 decayed ones 65.9 -> 65.0; but chunks' states and
// outputs of decayed memories took 2.5 % longer with it, of others 0.5 % less.
__device__ __forceinline__ void cut3(float x, float y, uint* w) {
#pragma unroll
  for (int z = 0; z < 3; ++z) {
    w[z] = __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302);
    x -= __uint_as_float(__float_as_uint(x) & 0xffff0000u);
    y -= __uint_as_float(__float_as_uint(y) & 0xffff0000u);
  }
}

__device__ __forceinline__ void unpack8(uint4v u, float* v) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[2 * j] = __uint_as_float(u[j] << 16);
    v[2 * j + 1] = __uint_as_float(u[j] & 0xffff0000u);
  }
}
template <bool ON>
__device__ __forceinline__ uint4v silu8(uint4v u) {
  if (ON) {
    float v[8];
    unpack8(u, v);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      u[j] = pack_bf16x2(silu_f(v[2 * j]), silu_f(v[2 * j + 1]));
  }
  return u;
}

// ---- gates: one block per (chunk, head), one thread per token -------------
template <int GATE>
__global__ void __launch_bounds__(MC_L)
memory_gates_kernel(ChunkArgs x) {
  const MemoryArgs& a = x.a;
  const int h = blockIdx.x % a.H, ch = blockIdx.x / a.H;
  const int row0 = x.chunks[4 * ch + 1], nrow = x.chunks[4 * ch + 2];
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  float i = -INFINITY, f = 0.f;
  const float ib = bits2f(((const short*)a.ib)[h]);
  const float fb = bits2f(((const short*)a.fb)[h]);
  if (t < nrow) {
    if (GATE == TIMED) {
      i = softplus_f(a.gates[(long)(row0 + t) * a.H + h] + ib);
      f = -expf(fb) * i;
    } else {
      log_gates(a, row0 + t, h, ib, fb, i, f);
    }
  }
  float F = f, I = i;                    // scan of (F, I) by (+, max)
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float F0 = __shfl_up(F, off, 64), I0 = __shfl_up(I, off, 64);
    if (lane >= off) {
      I = fmaxf(I0 + F, I);
      F += F0;
    }
  }
  __shared__ float sF[4], sI[4];
  if (lane == 63) {
    sF[wid] = F;
    sI[wid] = I;
  }
  __syncthreads();
  float c = -INFINITY;
  for (int w = 0; w < wid; ++w) c = fmaxf(c + sF[w], sI[w]);
  c = fmaxf(c + F, I);
  if (t < nrow) {
    const long o = (long)h * x.T + row0 + t;
    x.b[o] = F;
    x.i[o] = i;
    if (GATE == GATED) x.c[o] = c;
  }
  const long ci = (long)ch * a.H + h;
  if (lane == 63) x.tot[ci * 4 + wid] = F;
  if (GATE == GATED && t == MC_L - 1) x.cend[ci] = c;
}

// ---- rotation: one workgroup per token, q and k of all heads into planes ---
template <bool VEC>
__global__ void __launch_bounds__(256) memory_turn_kernel(ChunkArgs x) {
  extern __shared__ float cs[];          // cos [rot / 2], sin [rot / 2]
  const MemoryArgs& a = x.a;
  const int ch = blockIdx.x / MC_L, t = blockIdx.x % MC_L;
  if (t >= x.chunks[4 * ch + 2]) return;
  const long row = x.chunks[4 * ch + 1] + t;
  const int* sg = a.seg + 4L * x.chunks[4 * ch];
  const int p = sg[3] + (int)row - sg[1];
  const int half = a.rot / 2, D = a.D;
  for (int i = threadIdx.x; i < half; i += 256) {
    float c, s;
    turn(a.freq[i], p, &c, &s);
    cs[i] = c * a.amp;
    cs[half + i] = s * a.amp;
  }
  __syncthreads();
  const long HD = (long)a.H * D, plane = (long)x.T * HD;
  constexpr int V = VEC ? 8 : 1;
  const int items = (D - half) / V;      // of a head: pairs, then the rest
  auto get = [&](const short* s, float* v) {
    if (VEC) unpack8(*(const uint4v*)s, v); else v[0] = bits2f(s[0]);
  };
  auto put = [&](short* d, const float* v) {
    if (VEC) {
      uint4v w0, w1;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float u = v[2 * j % V], w = v[(2 * j + 1) % V];
        w0[j] = pack_bf16x2(u, w);
        w1[j] = pack_bf16x2(u - __uint_as_float(w0[j] << 16),
                            w - __uint_as_float(w0[j] & 0xffff0000u));
      }
      *(uint4v*)d = w0;
      *(uint4v*)(d + plane) = w1;
    } else {
      d[0] = f2bits(v[0]);
      d[plane] = f2bits(v[0] - bits2f(d[0]));
    }
  };
  for (int it = threadIdx.x; it < 2 * a.H * items; it += 256) {
    const int h = it / items % a.H, i = it % items * V;
    const bool key = it >= a.H * items;
    const short* src = (key ? (const short*)a.k + row * a.kst
                            : (const short*)a.q + row * a.qst) + (long)h * D;
    short* dst = (key ? x.KA : x.QA) + row * HD + (long)h * D;
    float u[V], w[V];
    get(src + half + i, w);
    if (i < half) {
      get(src + i, u);
#pragma unroll
      for (int j = 0; j < V; ++j) {
        const float c = cs[i + j], s = cs[half + i + j], y = u[j];
        u[j] = y * c - w[j] * s;
        w[j] = w[j] * c + y * s;
      }
      put(dst + i, u);
    }
    put(dst + half + i, w);
  }
}

// ---- states: U of a chunk, 64 columns per workgroup ------------------------
template <int DP, int GATE>
__global__ void __launch_bounds__(256)
memory_states_kernel(ChunkArgs x) {
  constexpr int KZ = qk_planes(GATE);
  constexpr int CPR = DP / 8, PAIRS = 32 * CPR / 256;
  constexpr int MT = DP / 32, NT = DP / 64;   // m tiles; tiles of a wave
  const MemoryArgs& a = x.a;
  const int D = a.D, E = a.E;
  const int nt = (E + 63) / 64;
  const int et = blockIdx.x % nt, h = blockIdx.x / nt % a.H;
  const int ch = blockIdx.x / nt / a.H;
  const int row0 = x.chunks[4 * ch + 1], nrow = x.chunks[4 * ch + 2];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int e0 = et * 64;
  const long ci = (long)ch * a.H + h;
  __shared__ __attribute__((aligned(16))) short kt[KZ][DP * 64];
  __shared__ __attribute__((aligned(16))) short vw[3][64 * 64];
  __shared__ __attribute__((aligned(16))) short vu[64 * 64];  // V^T as it is
  __shared__ float s_w[MC_L];
  {
    float w = 0.f;
    if (tid < nrow) {
      if (!fixed_decay(GATE)) {
        const long o = (long)h * x.T + row0 + tid;
        float d = x.tot[ci * 4 + wid] - x.b[o];
        for (int j = wid + 1; j < 4; ++j) d += x.tot[ci * 4 + j];
        w = GATE == TIMED ? expf(d) * x.i[o]
                          : expf(d + (x.i[o] - x.cend[ci]));
      } else {
        w = __builtin_amdgcn_exp2f((nrow - 1 - tid) * a.log2_decay[h]);
        if (GATE == TURNED) w *= a.kscale;
      }
    }
    s_w[tid] = w;
  }
  const int hk = GATE == TIMED ? h / (a.H / a.G) : h;
  const short* kp = (GATE == TURNED ? x.KA : (const short*)a.k) + (long)hk * D;
  const long kst = GATE == TURNED ? (long)a.H * D : a.kst;
  const short* vp = (const short*)a.v + (long)h * E + e0;
  const uint4v zero = {0, 0, 0, 0};
  uint4v kreg[KZ][2 * PAIRS], vreg[2];
  const int v_r = tid >> 3 << 1, v_c = (tid & 7) * 8;
  const TileWrite vtw(v_c, v_r);
  const TileRead tr(col, 0);
  auto issue = [&](int c0) {
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
      const int it = p * 256 + tid;
      const int r = it / CPR * 2, c = it % CPR * 8;
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int z = 0; z < KZ; ++z)
          kreg[z][2 * p + y] = c0 + r + y < nrow && c < D
              ? *(const uint4v*)(kp + ((long)z * x.T + row0 + c0 + r + y) * kst + c)
              : zero;
    }
#pragma unroll
    for (int y = 0; y < 2; ++y)
      vreg[y] = c0 + v_r + y < nrow && e0 + v_c < E
          ? *(const uint4v*)(vp + (long)(row0 + c0 + v_r + y) * a.vst + v_c)
          : zero;
  };
  f32x16 acc[NT] = {};
  float nacc = 0.f;
  const bool with_n = GATE == GATED && et == 0;
  issue(0);
  for (int c0 = 0; c0 < nrow; c0 += 64) {
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
      const int it = p * 256 + tid;
      const int r = it / CPR * 2, c = it % CPR * 8;
      union { uint4v u; unsigned short s[8]; } y0, y1;
      const TileWrite tw(c, r);
#pragma unroll
      for (int z = 1; z < KZ; ++z) {
        y0.u = kreg[z][2 * p];
        y1.u = kreg[z][2 * p + 1];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          *(uint*)(&kt[z][tw.at(j)]) = (uint)y0.s[j] | ((uint)y1.s[j] << 16);
      }
      y0.u = silu8<GATE == DECAY>(kreg[0][2 * p]);
      y1.u = silu8<GATE == DECAY>(kreg[0][2 * p + 1]);
      if (GATE == DECAY && et == 0 && c < D) {
        short* ka = x.KA + ((long)(row0 + c0 + r) * a.H + h) * D + c;
        if (c0 + r < nrow) *(uint4v*)ka = y0.u;
        if (c0 + r + 1 < nrow) *(uint4v*)(ka + (long)a.H * D) = y1.u;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
        *(uint*)(&kt[0][tw.at(j)]) = (uint)y0.s[j] | ((uint)y1.s[j] << 16);
    }
    {
      float f0[8], f1[8];
      unpack8(silu8<GATE == DECAY>(vreg[0]), f0);
      unpack8(silu8<GATE == DECAY>(vreg[1]), f1);
      const float w0 = s_w[c0 + v_r], w1 = s_w[c0 + v_r + 1];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        uint w[3];
        split3(f0[j] * w0, f1[j] * w1, w);
        const int o = vtw.at(j);
        *(uint*)(vu + o) = pack_bf16x2(f0[j], f1[j]);
#pragma unroll
        for (int z = 0; z < 3; ++z) *(uint*)(&vw[z][o]) = w[z];
      }
    }
    __syncthreads();
    if (c0 + 64 < nrow) issue(c0 + 64);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int e = (i * 256 + tid) >> 3, sl = tid & 7;
      if (x.VT && e0 + e < E)
        *(uint4v*)(x.VT + (ci * E + e0 + e) * MC_L + c0 + 8 * sl) =
            *(const uint4v*)(vu + tslot(e, 8 * sl));
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
      for (int y = 0; y < NT; ++y) {
        const int tile = wid + 4 * y;
        const int m = tile % MT, n = tile / MT;
        frag_u kf[KZ];
#pragma unroll
        for (int z = 0; z < KZ; ++z)
          kf[z].u4 = *(const uint4v*)(&kt[z][tr.at(m, 2 * kk + hi)]);
#pragma unroll
        for (int z = 0; z < 3; ++z) {
          frag_u vf;
          vf.u4 = *(const uint4v*)(&vw[z][tr.at(n, 2 * kk + hi)]);
#pragma unroll
          for (int w = 0; w < KZ && w + z < 3; ++w)
            acc[y] = mfma_bf16(kf[w].bf, vf.bf, acc[y]);
        }
      }
    }
    if (with_n && tid < DP) {
#pragma unroll
      for (int s = 0; s < 64; s += 8) {
        float kv[8];
        unpack8(*(const uint4v*)(&kt[0][tslot(tid, s)]), kv);
#pragma unroll
        for (int j = 0; j < 8; ++j) nacc += s_w[c0 + s + j] * kv[j];
      }
    }
  }
  float* U = x.U + ci * E * D;
#pragma unroll
  for (int y = 0; y < NT; ++y) {
    const int tile = wid + 4 * y;
    const int m = tile % MT, e = e0 + 32 * (tile / MT) + col;
    if (e >= E) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = 32 * m + 8 * r + 4 * hi;
      if (d < D)
        *(f32x4*)(U + (long)e * D + d) =
            f32x4{acc[y][4 * r], acc[y][4 * r + 1], acc[y][4 * r + 2],
                  acc[y][4 * r + 3]};
    }
  }
  if (with_n && tid < D) x.N[ci * D + tid] = nacc;
}

// ---- scan over the chunks of a segment: tiles of 64 keys x 16 columns ------
template <int GATE>
__global__ void __launch_bounds__(256)
memory_scan_kernel(ChunkArgs x) {
  const MemoryArgs& a = x.a;
  const int D = a.D, E = a.E;
  const int nd = (D + 63) / 64, ne = (E + 15) / 16;
  const int dt = blockIdx.x % nd, et = blockIdx.x / nd % ne;
  const int h = blockIdx.x / nd / ne % a.H;
  const int sg = blockIdx.x / nd / ne / a.H;
  const long slot = a.seg[4 * sg];
  const int ctx = a.seg[4 * sg + 3];
  const int tid = threadIdx.x;
  const int d = dt * 64 + (tid & 15) * 4, e = et * 16 + (tid >> 4);
  const bool live = d < D && e < E;
  const int nt = (E + 31) / 32;
  float* Sp = a.S + (slot * a.H + h) * D * E;
  __shared__ float tr[64][17];
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  float m = 0.f;
  if (ctx > 0) {
    for (int i = tid; i < 64 * 16; i += 256) {
      const int dd = dt * 64 + i / 16, ee = et * 16 + i % 16;
      tr[i / 16][i % 16] = dd < D && ee < E ? Sp[(long)dd * E + ee] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) S[j] = tr[(tid & 15) * 4 + j][tid >> 4];
    __syncthreads();
    if (GATE == GATED) m = a.m[(slot * a.H + h) * nt];
  }
  // the first column tile also carries n
  const bool with_n = GATE == GATED && et == 0 && tid < 64 && dt * 64 + tid < D;
  float n = 0.f;
  const long nat = (slot * a.H + h) * nt * D + dt * 64 + tid;
  if (with_n && ctx > 0) n = a.n[nat];
  // the state factors of up to 64 chunks at a time, then the chunks with the
  // next four U in flight
  constexpr int PF = 4;
  __shared__ float s_b[64], s_c[64];
  const int c0 = x.first[sg], c1 = x.first[sg + 1];
  const float l2d = fixed_decay(GATE) ? a.log2_decay[h] : 0.f;
  const long at = (long)e * D + d, step = (long)a.H * E * D;
  const float* Up = x.U + ((long)c0 * a.H + h) * E * D + at;
  f32x4 Un[PF] = {};
#pragma unroll
  for (int j = 0; j < PF; ++j)
    if (live && c0 + j < c1) Un[j] = *(const f32x4*)(Up + j * step);
  for (int cb = c0; cb < c1; cb += 64) {
    __syncthreads();
    if (tid < 64 && cb + tid < c1) {
      const long ci = (long)(cb + tid) * a.H + h;
      if (!fixed_decay(GATE)) {
        const float* tt = x.tot + ci * 4;
        const float b = tt[0] + tt[1] + tt[2] + tt[3];
        s_b[tid] = GATE == TIMED ? expf(b) : b;
        if (GATE == GATED) s_c[tid] = x.cend[ci];
      } else {
        s_b[tid] = __builtin_amdgcn_exp2f(x.chunks[4 * (cb + tid) + 2] * l2d);
      }
    }
    __syncthreads();
    const int ce = min(c1, cb + 64);
    for (int ch0 = cb; ch0 < ce; ch0 += PF) {
#pragma unroll
      for (int j = 0; j < PF; ++j) {
        const int ch = ch0 + j;
        if (ch >= ce) break;
        const long ci = (long)ch * a.H + h;
        const f32x4 U = Un[j];
        if (live && ch + PF < c1)
          Un[j] = *(const f32x4*)(Up + (long)(ch - c0 + PF) * step);
        if (live && (ch > c0 || ctx > 0)) {
          uint w0[3], w1[3];
          split3(S[0], S[1], w0);
          split3(S[2], S[3], w1);
#pragma unroll
          for (int z = 0; z < 3; ++z)
            *(uint2*)(x.P + (ci * 3 + z) * E * D + at) = uint2{w0[z], w1[z]};
        }
        float fs, us = 1.f;
        if (GATE == GATED) {
          const float bm = s_b[ch - cb] + m;
          const float mn = fmaxf(bm, s_c[ch - cb]);
          fs = expf(bm - mn);
          us = expf(s_c[ch - cb] - mn);
          if (dt == 0 && et == 0 && tid == 0) x.mst[ci] = m;
          if (with_n) {
            const long o = ci * D + dt * 64 + tid;
            const float N = x.N[o];
            x.N[o] = n;
            n = fs * n + us * N;
          }
          m = mn;
        } else {
          fs = s_b[ch - cb];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) S[i] = fs * S[i] + us * U[i];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) tr[(tid & 15) * 4 + j][tid >> 4] = S[j];
  __syncthreads();
  for (int i = tid; i < 64 * 16; i += 256) {
    const int dd = dt * 64 + i / 16, ee = et * 16 + i % 16;
    if (dd < D && ee < E) Sp[(long)dd * E + ee] = tr[i / 16][i % 16];
  }
  if (with_n)
    for (int j = 0; j < nt; ++j) a.n[nat + (long)j * D] = n;
}

// ---- outputs: 128 queries x VT columns per workgroup -----------------------
template <int DP, int VT, int GATE>
__global__ void __launch_bounds__(
    256, DP <= 128 || (VT <= 64 && GATE != TURNED) ? 2 : 1)
memory_outputs_kernel(ChunkArgs x) {
  constexpr int KZ = qk_planes(GATE);
  constexpr int NC = DP / 16, NB = VT / 32;
  constexpr int KP = DP * 2;             // K row pitch (bytes)
  constexpr int CPR = DP / 8, PAIRS = 32 * CPR / 256;
  constexpr int VN = VT / 32;            // 16-byte pieces of V^T a thread
  constexpr int KV_B = KZ * 64 * KP + VT * 64 * 2;
  constexpr int ST_B = 3 * 32 * KP;
  const MemoryArgs& a = x.a;
  const int D = a.D, E = a.E;
  const int nt = (E + VT - 1) / VT;
  const int et = blockIdx.x % nt, half = blockIdx.x / nt % 2;
  const int h = blockIdx.x / nt / 2 % a.H, ch = blockIdx.x / nt / 2 / a.H;
  const int row0 = x.chunks[4 * ch + 1], nrow = x.chunks[4 * ch + 2];
  const bool carried = x.chunks[4 * ch + 3];
  if (GATE == GATED && et == 0 && half == 0) {
    // m after the portion: nothing reads the slot's m any more
    const int sg = x.chunks[4 * ch];
    if (ch == x.first[sg + 1] - 1) {
      const long ci = (long)ch * a.H + h;
      const float* tt = x.tot + ci * 4;
      const float m = fmaxf(tt[0] + tt[1] + tt[2] + tt[3] + x.mst[ci],
                            x.cend[ci]);
      const int mt = (E + 31) / 32;
      for (int j = threadIdx.x; j < mt; j += 256)
        a.m[((long)a.seg[4 * sg] * a.H + h) * mt + j] = m;
    }
  }
  if (half * 128 >= nrow) return;        // the whole workgroup
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int e0 = et * VT;
  const long ci = (long)ch * a.H + h;
  const int t = half * 128 + wid * 32 + col;   // place in the chunk
  const int jt = half * 2 + (wid >> 1);        // its 64-token group
  __shared__ __attribute__((aligned(16))) char
      buf[KV_B > ST_B ? KV_B : ST_B];
  char* kb = buf;
  short* vb = (short*)(buf + KZ * 64 * KP);
  __shared__ float s_col[64], s_step[GATE == TIMED ? 64 : 1];
  __shared__ float s_n[GATE == GATED ? DP : 1];
  auto kswz = [](int row, int byte) {
    return CPR >= 16 ? swz16(row, byte) : swz(row, byte);
  };

  const int hk = GATE == TIMED ? h / (a.H / a.G) : h;
  frag_u qf[KZ][NC];
#pragma unroll
  for (int z = 0; z < KZ; ++z) {
    const long r = row0 + min(t, nrow - 1);
    const short* src =
        GATE == TURNED ? x.QA + (((long)z * x.T + r) * a.H + h) * D
                       : (const short*)a.q + r * a.qst + (long)hk * D;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d = c * 16 + hi * 8;
      qf[z][c].u4 = d < D ? silu8<GATE == DECAY>(*(const uint4v*)(src + d))
                          : uint4v{0, 0, 0, 0};
    }
  }
  // row terms of the weights
  float row = 0.f, inter, em = 0.f, l2d = 0.f;
  const float qs = GATE == GATED ? a.qscale : 1.f;
  float tot[4];
  if (!fixed_decay(GATE)) {
    const long o = (long)h * x.T + row0 + min(t, nrow - 1);
    float before = GATE == GATED ? x.mst[ci] : 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      tot[j] = x.tot[ci * 4 + j];
      if (j < jt) before += tot[j];
    }
    const float bt = x.b[o];
    const float mt = GATE == GATED ? fmaxf(bt + before, x.c[o]) : 0.f;
    inter = __expf(bt + before - mt) * qs;
    row = bt - mt;
    if (GATE == GATED) em = expf(-mt);
  } else {
    l2d = a.log2_decay[h];
    inter = __builtin_amdgcn_exp2f((t + 1) * l2d);
  }

  f32x16 ot[NB] = {};
  float den = 0.f;
  if (carried) {
    // the carried state: its planes pass through LDS 32 columns at a time
    if (GATE == GATED) {
      for (int d = tid; d < DP; d += 256)
        s_n[d] = d < D ? x.N[ci * D + d] : 0.f;
    }
    const short* P = x.P + ci * 3 * E * D;
    constexpr int NP = 3 * 32 * CPR / 256;
    uint4v preg[NP];
    auto fetch = [&](int nb) {
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int it = i * 256 + tid;
        const int c = it % CPR * 8, r = it / CPR;     // r: plane * 32 + row
        const int e = e0 + 32 * nb + (r & 31);
        preg[i] = e < E && c < D
            ? *(const uint4v*)(P + ((long)(r >> 5) * E + e) * D + c)
            : uint4v{0, 0, 0, 0};
      }
    };
    fetch(0);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if (e0 + 32 * nb >= E) continue;   // uniform
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int it = i * 256 + tid;
        const int c = it % CPR * 8, r = it / CPR;
        *(uint4v*)(buf + r * KP + kswz(r & 31, c * 2)) = preg[i];
      }
      __syncthreads();
      if (nb + 1 < NB) fetch(nb + 1);
#pragma unroll
      for (int z = 0; z < 3; ++z)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          frag_u sf;
          sf.u4 = *(const uint4v*)(buf + (z * 32 + col) * KP +
                                   kswz(col, (c * 16 + hi * 8) * 2));
#pragma unroll
          for (int w = 0; w < KZ && w + z < 3; ++w)
            ot[nb] = mfma_bf16(sf.bf, qf[w][c].bf, ot[nb]);
        }
      ot[nb] *= inter;
    }
    if (GATE == GATED) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        float qv[8];
        unpack8(qf[0][c].u4, qv);
#pragma unroll
        for (int j = 0; j < 8; ++j) den += qv[j] * s_n[c * 16 + hi * 8 + j];
      }
      den *= inter;
    }
  }

  // ---- keys of the chunk, 64 at a time, from the newest back ---------------
  const short* kp =
      (fixed_decay(GATE) ? x.KA : (const short*)a.k) + (long)hk * D;
  const long kst = fixed_decay(GATE) ? (long)a.H * D : a.kst;
  const short* vp = x.VT + (ci * E + e0) * MC_L;
  const uint4v zero = {0, 0, 0, 0};
  uint4v kreg[KZ][2 * PAIRS], vreg[VN];
  float colr = 0.f, stepr = 0.f;
  auto issue = [&](int J) {
    const int c0 = 64 * J;
#pragma unroll
    for (int p = 0; p < 2 * PAIRS; ++p) {
      const int it = p * 256 + tid;
      const int r = it / CPR, c = it % CPR * 8;
#pragma unroll
      for (int z = 0; z < KZ; ++z)
        kreg[z][p] = c0 + r < nrow && c < D
            ? *(const uint4v*)(kp + ((long)z * x.T + row0 + c0 + r) * kst + c)
            : zero;
    }
#pragma unroll
    for (int p = 0; p < VN; ++p) {
      const int e = (p * 256 + tid) >> 3;
      vreg[p] = e0 + e < E
          ? *(const uint4v*)(vp + (long)e * MC_L + c0 + 8 * (tid & 7)) : zero;
    }
    if (!fixed_decay(GATE) && tid < 64) {
      colr = -INFINITY;
      stepr = 0.f;
      if (c0 + tid < nrow) {
        const long o = (long)h * x.T + row0 + c0 + tid;
        stepr = x.i[o];
        colr = GATE == TIMED ? -x.b[o] : stepr - x.b[o];
      }
    }
  };
  const TileRead vr(col, 4 * hi);
  const int J1 = min(half * 2 + 1, (nrow - 1) / 64);
  issue(J1);
  for (int J = J1; J >= 0; --J) {
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 2 * PAIRS; ++p) {
      const int it = p * 256 + tid;
      const int r = it / CPR, c = it % CPR * 8;
#pragma unroll
      for (int z = 0; z < KZ; ++z)
        *(uint4v*)(kb + (z * 64 + r) * KP + kswz(r, c * 2)) = kreg[z][p];
    }
#pragma unroll
    for (int p = 0; p < VN; ++p)
      *(uint4v*)(vb + tslot((p * 256 + tid) >> 3, 8 * (tid & 7))) = vreg[p];
    if (!fixed_decay(GATE) && tid < 64) s_col[tid] = colr;
    if (GATE == TIMED && tid < 64) s_step[tid] = stepr;
    __syncthreads();
    if (J > 0) issue(J - 1);
    if (J > jt || half * 128 + wid * 32 >= nrow) continue;  // wave-uniform

    // row part of the exponent for keys of group J
    float base = row;
    if (!fixed_decay(GATE) && J < jt) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j >= J && j < jt) base += tot[j];
    }
    // 32 keys at a time keeps the registers for two workgroups per CU
#pragma unroll 1
    for (int k2 = 0; k2 < 2; ++k2) {
      const int kr = col + 32 * k2;
      f32x16 acc = {};
#pragma unroll
      for (int c = 0; c < NC; ++c) {
#pragma unroll
        for (int z = 0; z < KZ; ++z) {
          frag_u kf;
          kf.u4 = *(const uint4v*)(kb + (z * 64 + kr) * KP +
                                   kswz(kr, (c * 16 + hi * 8) * 2));
#pragma unroll
          for (int w = 0; w < KZ && w + z < 2; ++w)
            acc = mfma_bf16(kf.bf, qf[w][c].bf, acc);
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int s = 32 * k2 + acc_row(r, hi);
        float w;
        if (GATE == TIMED) w = __expf(base + s_col[s]) * s_step[s];
        else if (GATE == GATED) w = __expf(base + s_col[s]) * qs;
        else w = __builtin_amdgcn_exp2f((float)(t - 64 * J - s) * l2d);
        if (GATE == TURNED) w *= a.kscale;
        if (J == jt && 64 * J + s > t) w = 0.f;
        acc[r] *= w;
        if (GATE == GATED) den += acc[r];
      }
#pragma unroll
      for (int cc = 0; cc < 2; ++cc) {
        frag_u pf[3];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          uint w[3];
          split3(acc[8 * cc + 2 * u], acc[8 * cc + 2 * u + 1], w);
#pragma unroll
          for (int z = 0; z < 3; ++z) pf[z].u[u] = w[z];
        }
        const int slot = 4 * k2 + 2 * cc;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          frag_u vf;
          *(uint2*)&vf.u[0] = *(const uint2*)(vb + vr.at(nb, slot));
          *(uint2*)&vf.u[2] = *(const uint2*)(vb + vr.at(nb, slot + 1));
#pragma unroll
          for (int z = 0; z < 3; ++z)
            ot[nb] = mfma_bf16(vf.bf, pf[z].bf, ot[nb]);
        }
      }
    }
  }

  float inv = 1.f;
  if (GATE == GATED) {
    den += __shfl_xor(den, 32, 64);
    inv = 1.f / (fmaxf(fabsf(den), em) + GATED_EPS);
  }
  if (GATE == TURNED && a.z) {           // the head's norm; e0 is 0
    float sq = 0.f;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) sq += ot[nb][r] * ot[nb][r];
    sq += __shfl_xor(sq, 32, 64);
    inv = 1.f / sqrtf(sq / E + x.norm_eps);
  }
  if (t >= nrow) return;
  const float skip = GATE == TIMED ? bits2f(((const short*)a.skip)[h]) : 0.f;
  short* dst = (short*)a.out + ((long)(row0 + t) * a.H + h) * E + e0;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      const int e = 32 * nb + 8 * rg + 4 * hi;
      if (e0 + e >= E) continue;
      float o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = ot[nb][4 * rg + j] * inv;
      if (GATE == TURNED && a.z) {
        float z[4];
        load4((const short*)a.z + (long)(row0 + t) * a.zst + (long)h * E + e, z);
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] *= silu_f(z[j]);
      }
      if (GATE == TIMED) {
        float v[4], z[4];
        const long at = (long)h * E + e0 + e;
        load4((const short*)a.v + (long)(row0 + t) * a.vst + at, v);
        load4((const short*)a.z + (long)(row0 + t) * a.zst + at, z);
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = (o[j] + skip * v[j]) * silu_f(z[j]);
      }
      *(uint2*)(dst + e) = uint2{pack_bf16x2(o[0], o[1]),
                                 pack_bf16x2(o[2], o[3])};
    }
}

// ---- timed states of D = 64 by a multiple of 64, chunk after chunk ----------
// One workgroup carries DP keys x ET columns of a head's state through its
// segment: the state stays in the accumulators, is scaled by what a chunk
// forgets, and the chunk's weighted keys and values are added to it, 64 tokens a
// piece.  Before a chunk its three planes go out as the outputs' fragments, 16
// bytes a lane.  Keys come straight into LDS, two pieces ahead, and are turned by
// transposing reads; values come through registers, two ahead as well, where
// they are weighted and split.  One barrier a piece, which waits by count.
//
// The states of all chunks at once and a scan over them move 32 bits out and back and
// take two launches; the planes and the values are what is left.
__global__ void __launch_bounds__(256, 2) memory_carry_kernel(ChunkArgs x) {
  constexpr int DP = 64, MT = DP / 32, ET = 128 / MT;   // tiles of keys; columns
  constexpr int NC = DP / 16, SL = DP / 8, VS = ET / 8;
  constexpr int LK = DP / 32, LV = ET / 32;    // words of a thread and piece
  constexpr int PLANE = 64 * ET * 2, VA = 6;   // pieces that values are ahead
  // apart by name, so that a read of one need not wait for the words on their
  // way into another
  __shared__ __attribute__((aligned(16))) char k0[64 * DP * 2], k1[64 * DP * 2],
      k2[64 * DP * 2];
  __shared__ __attribute__((aligned(16))) char v0[3 * PLANE], v1[3 * PLANE];
  __shared__ float s_w[2][MC_L];
  const MemoryArgs& a = x.a;
  const int E = a.E;
  // an XCD has the same heads of all segments: heads that share keys, and long
  // segments beside short ones
  const int units = a.H * (E / ET), per = (units + 7) / 8;
  const int unit = blockIdx.x % 8 * per + blockIdx.x / 8 % per;
  const int sg = blockIdx.x / 8 / per;
  if (unit >= units) return;
  const int h = unit / (E / ET), e0 = unit % (E / ET) * ET;
  const int row0 = a.seg[4 * sg + 1], rows = a.seg[4 * sg + 2];
  const int ctx = a.seg[4 * sg + 3];
  const int ch0 = x.first[sg], ch1 = x.first[sg + 1];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int m = wid % MT, n = wid / MT;

  auto turn = [](int r) { return value_turn<SL>(r); };
  const short* kp = (const short*)a.k + row0 * a.kst + h / (a.H / a.G) * DP;
  const short* vp = (const short*)a.v + row0 * a.vst + (long)h * E + e0;
  // Pieces past the last are that one again, so that the words on their way keep
  // their number.  As buffer loads: behind other loads into LDS the compiler
  // waits for all of them where it needs a value.
  const int last = max(0, rows - 1) / 64;
  const int kst = (int)a.kst * 2, vst = (int)a.vst * 2;
  auto issue_k = [&](int i, char* buf) __attribute__((always_inline)) {
    i = min(i, last);
    const auto src = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(kp + 64L * i * a.kst), 0, 0x7fffffff, 0x00027000);
#pragma unroll
    for (int p = 0; p < LK; ++p) {
      const int r = (p * 256 + tid) / SL, s = tid % SL ^ turn(r);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          src, (lds_ptr)(buf + (p * 256 + wid * 64) * 16), 16,
          min(r, rows - 1 - 64 * i) * kst + s * 16, 0, 0, 0);
    }
  };
  auto load_v = [&](int i, uint4v* v) __attribute__((always_inline)) {
    i = min(i, last);
    const char* src = (const char*)(vp + 64L * i * a.vst);
#pragma unroll
    for (int p = 0; p < LV; ++p) {
      const int r = (p * 256 + tid) / VS;
      v[p] = *(const uint4v*)(src + (uint)(min(r, rows - 1 - 64 * i) * vst +
                                           tid % VS * 16));
    }
  };
  // the weight of this thread's token of a chunk, at its end; what the chunk
  // leaves of the state before it
  float wb, wi, keep = 0.f;
  f32x4 wt;
  auto load_w = [&](int ch) __attribute__((always_inline)) {
    const long o = (long)h * x.T + row0 + min((ch - ch0) * MC_L + tid, rows - 1);
    wb = x.b[o];
    wi = x.i[o];
    wt = *(const f32x4*)(x.tot + ((long)ch * a.H + h) * 4);
  };
  auto weight = [&](int ch, float& keep) __attribute__((always_inline)) {
    float d = wt[3] * (wid < 3);
    d += wt[2] * (wid < 2);
    d += wt[1] * (wid < 1);
    d += wt[wid] - wb;
    keep = expf(wt[0] + wt[1] + wt[2] + wt[3]);
    return (ch - ch0) * MC_L + tid < rows ? expf(d) * wi : 0.f;
  };
  // the compiler knows nothing of the order that the wait below counts on
  auto in_order = []() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
  };

  f32x16 acc = {};
  float* Sp = a.S + ((long)a.seg[4 * sg] * a.H + h) * DP * E + e0 + 32 * n + col;
  if (ctx > 0)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      acc[r] = Sp[(long)(32 * m + acc_row(r, hi)) * E];

  // this lane's part of the addresses of transposing reads (bytes)
  const int tr_key = 4 * hi + ((lane & 15) >> 2);
  const int tr_col = ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
  const int kx = tr_key * DP * 2 + tr_col + value_turn<SL>(tr_key) * 16;
  const int vx = tr_key * ET * 2 + tr_col + value_turn<8>(tr_key) * 16;
  // the weighted values of a piece, split
  auto convert = [&](int i, const float* w, char* vb, const uint4v* v)
      __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < LV; ++p) {
      const int r = (p * 256 + tid) / VS;
      const int s = tid % VS ^ value_turn<8>(r);
      float f[8];
      uint4v u[3];
      unpack8(64 * i + r < rows ? v[p] : uint4v{0, 0, 0, 0}, f);
      const float wr = w[r];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint t[3];
        split3(f[2 * j] * wr, f[2 * j + 1] * wr, t);
#pragma unroll
        for (int z = 0; z < 3; ++z) u[z][j] = t[z];
      }
#pragma unroll
      for (int z = 0; z < 3; ++z)
        *(uint4v*)(vb + z * PLANE + r * ET * 2 + s * 16) = u[z];
    }
  };
  // piece i; w: of the piece behind it, whose values are made ready
  auto piece = [&](int i, bool fresh, const float* w, char* kb, char* kn, char* vb, char* vn,
                   uint4v* v) __attribute__((always_inline)) {
    // The keys of this piece are here: behind them only those of the next were
    // asked for, twice values, and the planes of the chunk's state if it is the
    // first or second of a chunk (of the first chunk, these keys are here).
    if (64 * i + 64 > rows) {
      __builtin_amdgcn_s_waitcnt(0xf70);           // vmcnt(0)
      in_order();
#pragma unroll
      for (int p = 0; p < LK; ++p)
        if (64 * i + (p * 256 + tid) / SL >= rows)
          *(uint4v*)(kb + (p * 256 + tid) * 16) = uint4v{0, 0, 0, 0};
    }
    in_order();
    static_assert(LK + 2 * LV + 6 < 16, "");
    if (fresh) __builtin_amdgcn_s_waitcnt(0x70 | (LK + 2 * LV + 6));
    else __builtin_amdgcn_s_waitcnt(0x70 | (LK + 2 * LV));   // and lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    in_order();
    issue_k(i + 2, kn);
    in_order();
    __builtin_amdgcn_sched_barrier(0);
    union { tr4 t[2]; bf16x8 bf; } kf[4], vf[4][3];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        kf[c].t[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr4)(
            kb + (kx ^ (64 * m)) + (16 * c + 8 * u) * DP * 2));
#pragma unroll
        for (int z = 0; z < 3; ++z)
          vf[c][z].t[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr4)(
              vb + z * PLANE + (vx ^ (64 * n)) + (16 * c + 8 * u) * ET * 2));
      }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int z = 0; z < 3; ++z) acc = mfma_bf16(kf[c].bf, vf[c][z].bf, acc);
    convert(i + 1, w, vn, v);
    __builtin_amdgcn_sched_group_barrier(0x100, 16, 0);
#pragma unroll
    for (int y = 0; y < 12; ++y) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x2, 7 * LV, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    in_order();
    load_v(i + 1 + VA, v);
    in_order();
  };
  // the planes as fragments of the outputs' products: lane (col, hi) has keys 16 c
  // + 8 hi ... of column col
  auto leave = [&](int ch) __attribute__((always_inline)) {
    short* P = x.P + ((((long)ch * a.H + h) * (E / 32) + e0 / 32 + n) * 3 * NC +
                      2 * m) * 512 + lane * 8;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      uint w[4][3];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        split3(acc[8 * c + 2 * u], acc[8 * c + 2 * u + 1], w[u]);
#pragma unroll
      for (int z = 0; z < 3; ++z) {
        const auto r0 = __builtin_amdgcn_permlane32_swap(w[0][z], w[2][z], false,
                                                         false);
        const auto r1 = __builtin_amdgcn_permlane32_swap(w[1][z], w[3][z], false,
                                                         false);
        *(uint4v*)(P + (z * NC + c) * 512) = uint4v{r0[0], r1[0], r0[1], r1[1]};
      }
    }
  };

  if (rows > 0) {
    uint4v v[VA][LV];
#pragma unroll
    for (int i = 0; i < VA; ++i) load_v(i, v[i]);
    load_w(ch0);
    in_order();
    issue_k(0, k0);
    in_order();
    issue_k(1, k1);
    s_w[0][tid] = weight(ch0, keep);
    __syncthreads();
    convert(0, s_w[0], v0, v[0]);
    in_order();
    load_v(VA, v[0]);
    char *const kr[3] = {k0, k1, k2}, *const vr[2] = {v0, v1};
    const int pieces = last + 1;
    if (ctx > 0) leave(ch0);
    for (int cb = ch0; cb < ch1; cb += 3) {
#pragma unroll
      for (int y = 0; y < 3; ++y) {
        const int ch = cb + y;
        if (ch >= ch1) break;
        acc *= keep;
        const int i = 4 * (ch - ch0), now = (ch - ch0) & 1;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          if (i + p >= pieces) break;
          if (p == 2) s_w[now ^ 1][tid] = weight(min(ch + 1, ch1 - 1), keep);
          piece(i + p, p < 2, p < 3 ? s_w[now] + 64 * p + 64 : s_w[now ^ 1],
                kr[(4 * y + p) % 3], kr[(4 * y + p + 2) % 3], vr[p % 2],
                vr[(p + 1) % 2], v[(4 * y + p + 1) % VA]);
          if (p == 0) load_w(min(ch + 1, ch1 - 1));
        }
        if (ch + 1 < ch1) leave(ch + 1);
      }
    }
    __builtin_amdgcn_s_waitcnt(0xf70);             // vmcnt(0): LDS is given back
  }
#pragma unroll
  for (int r = 0; r < 16; ++r)
    Sp[(long)(32 * m + acc_row(r, hi)) * E] = acc[r];
}

// ---- timed outputs of D = 64 or 128, 64 columns per workgroup ---------------
// The same 128 queries, but all tiles come straight into LDS (DMA), up to three
// ahead of the one that is multiplied, in a ring of four: the carried state's
// planes, as fragments, then keys and values, 32 tokens a tile, the oldest first;
// values are turned by transposing reads.  One barrier a tile, which waits by
// count.  Bound by latency: three workgroups share a CU, vector work fills 40 % of
// the time, products 25 %.  2 x 2048 tokens, 128 heads of 128 x 64: tiles of 64
// tokens, one ahead, with all words waited for at every barrier 129 us, now 117
// (200 MB: 40).  Keys of 64 fitted four times on a CU before and fit three times:
// calls of all kinds take 0.97 to 0.99 of the time then, at worst 1.04 (3052 tokens
// and 1188 more, 80 heads of 64 x 64: 107 and 111 us); smaller tiles for four spill
// 19 registers, 1.06.
// The weights of an earlier group's keys are products: what is left at the end
// of their group, and from there to the query.  The skip is part of a token's
// weight on itself.
template <int DP>
__global__ void __launch_bounds__(256, 3) memory_timed_kernel(ChunkArgs x) {
  constexpr int NC = DP / 16, SL = DP / 8, KP = DP * 2;
  constexpr int TILE = 12288, KEYS = 32 * KP;
  constexpr int NS = DP / 32;            // tiles of the state: 8 NC / NS fragments
  constexpr int LS = 3, LK = DP / 64, LT = LK + 1;   // words of a thread and tile
  constexpr int OP = 68;                 // pitch of a wave's results
  static_assert(32 * OP * 4 <= TILE && KEYS + 32 * 128 <= TILE &&
                2 * 3 * NC * 1024 == NS * TILE, "");
  // apart by name, so that a read of one need not wait for the words on their
  // way into another
  __shared__ __attribute__((aligned(16))) char b0[TILE], b1[TILE], b2[TILE], b3[TILE];
  __shared__ float s_col[MC_L], s_step[MC_L], s_far[MC_L];
  const MemoryArgs& a = x.a;
  const int E = a.E, nt = E / 64;
  // the halves and the heads that share keys follow each other on one XCD
  int id = blockIdx.x;
  {
    const int total = gridDim.x, per = total / 8, rest = total % 8, xcd = id % 8;
    id = xcd * per + min(xcd, rest) + id / 8;
  }
  const int half = id & 1, et = id / 2 % nt;
  const int h = id / 2 / nt % a.H, ch = id / 2 / nt / a.H;
  const int row0 = x.chunks[4 * ch + 1], nrow = x.chunks[4 * ch + 2];
  const bool carried = x.chunks[4 * ch + 3];
  if (half * 128 >= nrow) return;        // the whole workgroup
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int e0 = et * 64;
  const long ci = (long)ch * a.H + h;
  const int t = half * 128 + wid * 32 + col;   // place in the chunk
  const int tt = half * 4 + wid, jt = tt >> 1; // its 32 and 64 tokens
  const int hk = h / (a.H / a.G);

  frag_u qf[NC];
  const short* q = (const short*)a.q + (row0 + min(t, nrow - 1)) * a.qst + hk * DP;
#pragma unroll
  for (int c = 0; c < NC; ++c) qf[c].u4 = *(const uint4v*)(q + c * 16 + hi * 8);
  const long ho = (long)h * x.T + row0;
  const float bt = x.b[ho + min(t, nrow - 1)];
  const float b_tok = x.b[ho + min(tid, nrow - 1)];
  const float i_tok = x.i[ho + min(tid, nrow - 1)];
  const f32x4 tot = *(const f32x4*)(x.tot + ci * 4);
  const float skip = bits2f(((const short*)a.skip)[h]);
  // the loads below are counted, these are not
  auto in_order = []() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
  };
  in_order();

  // Thread tid fills 16-byte places tid, tid + 256, ... of a tile.  Buffer loads:
  // behind other loads into LDS the compiler waits for all of them where it needs
  // a value.  Tiles 4 - NS to 3: the state, then keys and values.
  auto turn = [](int r) { return SL == 16 ? row_turn(r) : key_turn<SL>(r); };
  const auto state_src = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(x.P + ci * 3 * E * DP + (x.U ? e0 : 3 * e0) * DP), 0, 0x7fffffff,
      0x00027000);
  const auto key_src = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const short*)a.k + (long)row0 * a.kst + hk * DP), 0, 0x7fffffff,
      0x00027000);
  const auto value_src = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const short*)a.v + (long)row0 * a.vst + (long)h * E + e0), 0,
      0x7fffffff, 0x00027000);
  const int kst = (int)a.kst * 2, vst = (int)a.vst * 2;
  auto issue = [&](int i, char* buf) __attribute__((always_inline)) {
    in_order();
    if (i < 4) {
#pragma unroll
      for (int p = 0; p < LS; ++p) {
        // fragments, or from rows of planes
        const int f = 12 * (i - (4 - NS)) + 4 * p + wid;
        const int row = f % (3 * NC) / NC * E + f / (3 * NC) * 32 + col;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            state_src, (lds_ptr)(buf + (p * 256 + wid * 64) * 16), 16,
            x.U ? row * DP * 2 + f % NC * 32 + hi * 16 : f * 1024 + lane * 16, 0,
            0, 0);
      }
    } else {
      const int s0 = (i - 4) * 32;
#pragma unroll
      for (int p = 0; p < LK; ++p) {
        const int r = (p * 256 + tid) / SL, s = tid % SL ^ turn(r);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            key_src, (lds_ptr)(buf + (p * 256 + wid * 64) * 16), 16,
            min(s0 + r, nrow - 1) * kst + s * 16, 0, 0, 0);
      }
      const int r = tid >> 3, s = (tid & 7) ^ value_turn<8>(r);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          value_src, (lds_ptr)(buf + KEYS + wid * 1024), 16,
          min(s0 + r, nrow - 1) * vst + s * 16, 0, 0, 0);
    }
    in_order();
  };
  // A tile is here, in all waves, and the one before is read; `behind` words of this
  // thread were asked for after it.  Full halves have 4 or 8 tiles of keys; others
  // too, with their last row for those that they do not have.
  auto arrive = [&](int behind) __attribute__((always_inline)) {
    in_order();
    // a constant, but the builtin wants a literal
    if (behind == 6) __builtin_amdgcn_s_waitcnt(0x76);
    else if (behind == 5) __builtin_amdgcn_s_waitcnt(0x75);
    else if (behind == 7) __builtin_amdgcn_s_waitcnt(0x77);
    else __builtin_amdgcn_s_waitcnt(0x74);   // 4 is right for all: no less
    __builtin_amdgcn_s_barrier();
    in_order();
  };
  char *const ring[4] = {b0, b1, b2, b3};
  float inter;
  auto weights = [&]() __attribute__((always_inline)) {
    float before = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < jt) before += tot[j];
    const float c = tid < nrow ? -b_tok : -INFINITY;
    const float s = tid < nrow ? i_tok : 0.f;
    s_col[tid] = c;
    s_step[tid] = s;
    s_far[tid] = __expf(tot[0] * (wid == 0) + tot[1] * (wid == 1) +
                        tot[2] * (wid == 2) + tot[3] * (wid == 3) + c) * s;
    inter = __expf(bt + before);
  };

  // this lane's part of the addresses: slot 2 c + hi of row col; a transposing
  // read, where 16 lanes turn 4 keys by 16 columns
  const int kx = SL == 16 ? row_lane(col, hi)
                          : col * KP + (hi ^ key_turn<SL>(col)) * 16;
  const int tr_key = 4 * hi + ((lane & 15) >> 2);
  const int vx = (tr_key * 64 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4 +
                  value_turn<8>(tr_key) * 8) * 2;
  f32x16 ot[2] = {};
  // part y of the state: fragments c of plane z of 32 columns nb, c fastest
  auto state = [&](int y, const char* buf) __attribute__((always_inline)) {
#pragma unroll
    for (int f = 0; f < 12; ++f) {
      const int at = 12 * y + f, nb = at / (3 * NC), c = at % NC;
      frag_u sf;
      sf.u4 = *(const uint4v*)(buf + f * 1024 + lane * 16);
      ot[nb] = mfma_bf16(sf.bf, qf[c].bf, ot[nb]);
    }
  };
  const bool rows = half * 128 + wid * 32 < nrow;
  auto keys = [&](int i, const char* buf) __attribute__((always_inline)) {
    if (i > tt || !rows) return;         // later keys; wave-uniform
    const int J = i >> 1, s0 = i * 32;
    f32x16 acc = {};
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      frag_u kf;
      kf.u4 = *(const uint4v*)(buf + (kx ^ (32 * c)));
      acc = mfma_bf16(kf.bf, qf[c].bf, acc);
    }
    if (J < jt) {
      float from = bt;                   // from the end of the group
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j > J && j < jt) from += tot[j];
      from = __expf(from);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[r] *= s_far[s0 + acc_row(r, hi)] * from;
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int s = s0 + acc_row(r, hi);
        const float w = __expf(bt + s_col[s]) * s_step[s];
        acc[r] *= s > t ? 0.f : w;
        acc[r] += s == t ? skip : 0.f;
      }
    }
#pragma unroll
    for (int cc = 0; cc < 2; ++cc) {
      frag_u pf[3];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        uint w[3];
        split3(acc[8 * cc + 2 * u], acc[8 * cc + 2 * u + 1], w);
#pragma unroll
        for (int z = 0; z < 3; ++z) pf[z].u[u] = w[z];
      }
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        union { tr4 t[2]; bf16x8 bf; } vf;
#pragma unroll
        for (int u = 0; u < 2; ++u)
          vf.t[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_tr4)(buf + KEYS + (vx ^ (nb * 64)) + (16 * cc + 8 * u) * 128));
#pragma unroll
        for (int z = 0; z < 3; ++z) ot[nb] = mfma_bf16(vf.bf, pf[z].bf, ot[nb]);
      }
    }
  };
  // (weights in both branches, where the compiler knows what was asked for)
  if (carried) {
#pragma unroll
    for (int i = 4 - NS; i < 7 - NS; ++i) issue(i, ring[i % 4]);
    weights();
#pragma unroll
    for (int i = 4 - NS; i < 4; ++i) {
      arrive((i + 1 < 4 ? LS : LT) + (i + 2 < 4 ? LS : LT));
      issue(i + 3, ring[(i + 3) % 4]);
      state(i - (4 - NS), ring[i % 4]);
    }
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) ot[nb] *= inter;
  } else {
#pragma unroll
    for (int i = 4; i < 7; ++i) issue(i, ring[i % 4]);
    weights();
  }
  // through LDS, so that every row is read and written as a whole (8 bytes a
  // lane, each of another row: 163 us in place of 121)
  const int r0 = half * 128 + wid * 32 + (lane >> 3), c0 = (lane & 7) * 8;
  const long at = (long)h * E + e0 + c0;
  uint4v zz[4];
  if (half)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      arrive(LT + LT);
      issue(i + 7, ring[(i + 3) % 4]);
      keys(i, ring[i]);
    }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    arrive(i < 2 ? LT + LT : i == 2 ? LT + 4 : 4);
    if (i == 0) issue(half * 4 + 7, b3);
    if (i == 1)
#pragma unroll
      for (int y = 0; y < 4; ++y)
        zz[y] = *(const uint4v*)((const short*)a.z +
                                 (row0 + min(r0 + 8 * y, nrow - 1)) * a.zst + at);
    keys(half * 4 + i, ring[i]);
  }

  float* o = (float*)(wid == 0 ? b0 : wid == 1 ? b1 : wid == 2 ? b2 : b3);
  __syncthreads();
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg)
      *(f32x4*)(o + col * OP + 32 * nb + 8 * rg + 4 * hi) =
          f32x4{ot[nb][4 * rg], ot[nb][4 * rg + 1], ot[nb][4 * rg + 2],
                ot[nb][4 * rg + 3]};
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (r0 + 8 * i >= nrow) break;
    const float* src = o + ((lane >> 3) + 8 * i) * OP + c0;
    float y[8], z[8];
    load4(src, y);
    load4(src + 4, y + 4);
    unpack8(zz[i], z);
    uint4v w;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = pack_bf16x2(y[2 * j] * silu_f(z[2 * j]),
                         y[2 * j + 1] * silu_f(z[2 * j + 1]));
    *(uint4v*)((short*)a.out + (long)(row0 + r0 + 8 * i) * a.H * E + at) = w;
  }
}

// ---- memories of D = 128, states and outputs in one pass (not turned) -----------
// One workgroup takes 64 columns of a head through its segment, 64 tokens a piece:
// nothing but queries, keys, values, gates and results moves.  Three waves of a SIMD
// do different things, since one alone issues a vector instruction every eight
// cycles.  Four hold the state in accumulators, 16 columns each; for every piece they
// multiply its planes by the queries (the accumulators' row order is the contraction
// order), scale it and add the weighted keys and values.  Four weight the scores
// within the piece, 16 tokens each, and add their products a piece later; the one with
// the fewest scores also makes the next piece's gates.  Four ask for the next piece's
// tiles, which come straight into LDS, and write the results of two pieces ago.  One
// barrier a piece.  Bound by what a SIMD issues: up to 136 products of 16 cycles and
// 720 vector instructions of 2.4 to 5, which products hardly hide, are 4200 of a
// piece's 4770 cycles; the tiles alone take half of them, a piece's latency each time.
// 128 heads of 128 x 64 in us, carried states and outputs in chunks of 256 as above |
// one pass:
//   2 x 2048 tokens 181 | 105      4 x 500 104 | 62     1 x 4096 177 | 158
//   64 heads: 1500 tokens 60 | 56, 3 x 500 52 | 38, 50 35 | 19 (its one launch)
// With two waves a SIMD, states and everything else, 2 x 2048 took 130; with four of
// 128 registers 133, and with two of them for the halves of the state 120; the gates
// beside the results' waves 116.
constexpr int PASS_D = 128;
template <int N> struct Count { static constexpr int value = N; };

// DECAY: queries, keys and values pass through registers and silu on their way into
// LDS, the weights are the same for every piece, and the results are written as they
// are.  32 heads of 128 x 128 in us, activated copies, states of all chunks at once, a
// scan and outputs | one pass:
//   50 tokens 17.7 | 7.1    500 43.6 | 28.4    4 x 500 40.6 | 18.1    3 x 2000 72 | 56
// GATED: the waves that hold the state carry 32 keys of the normaliser each, the same
// in 16 columns, and leave its planes for the scores' waves, which multiply them by the
// queries.  Exponents are summed from the piece's end and with the running maxima taken
// from each other first, which halves the state's error.  16 heads of 128 x 256:
//   50 tokens 21.9 | 7.5    500 49.8 | 25.9    4 x 500 48.0 | 17.4    3 x 2000 75 | 50
template <int GATE>
__global__ void __launch_bounds__(768) memory_pass_kernel(ChunkArgs x) {
  constexpr int DP = PASS_D, L = 64, ET = 64;
  constexpr int TILE = L * DP * 2, VT = L * ET * 2, PART = ET * L * 4;
  // apart by name, so that a read of one need not wait for the words on their
  // way into another
  __shared__ __attribute__((aligned(16))) char q0[TILE], q1[TILE], k0[TILE], k1[TILE],
      v0[VT], v1[VT];
  // the results: four columns of a token in a word, the tokens of 16 words turned by
  // the columns
  __shared__ __attribute__((aligned(16))) char s_part[3 * PART];
  // log forgets and steps; what is left of a token at the end of its 16, and of the
  // piece; what a piece leaves of the state.  GATED: the parts of a weight's exponent
  // that are the query's and the key's, and what is left of the state at a token
  __shared__ __attribute__((aligned(16))) float s_b[2 * L], s_i[2 * L], s_far[2 * L],
      s_w[2 * L];
  __shared__ float s_keep[2];
  // GATED: e^-m, and in three planes the weights and the normaliser before the piece
  __shared__ float s_em[GATE == GATED ? 2 * L : 1];
  __shared__ __attribute__((aligned(16))) short s_wp[GATE == GATED ? 2 * 3 * L : 8],
      s_np[GATE == GATED ? 2 * 3 * DP : 8];
  const MemoryArgs& a = x.a;
  const int E = a.E;
  // heads that share keys are on one XCD
  const int units = a.H * (E / ET), per = (units + 7) / 8;
  const int unit = blockIdx.x % 8 * per + blockIdx.x / 8 % per;
  const int sg = blockIdx.x / 8 / per;
  if (unit >= units) return;             // the whole workgroup
  const int h = unit / (E / ET), e0 = unit % (E / ET) * ET;
  const int row0 = a.seg[4 * sg + 1], rows = a.seg[4 * sg + 2];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, quad = lane >> 4;
  const int pieces = (rows + L - 1) / L;
  auto meet = []() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);              // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // transposing reads: 16 lanes turn 4 tokens by 16 columns; tokens 32 c + 16 u + 4
  // quad ... of columns 16 n ... are at (kx ^ 32 n) + (32 c + 16 u) rows
  const int turn_row = 4 * quad + (col >> 2), turn_slot = col >> 1 & 1;
  const int kx0 = turn_row * 256 + (row_turn(turn_row) ^ turn_slot) * 16 + (col & 1) * 8;
  const int vx = turn_row * 128 + (value_turn<8>(turn_row) ^ turn_slot) * 16 +
                 (col & 1) * 8;
  union Turned { tr4 t[2]; bf16x8 bf; uint u[4]; };
  auto turned = [&](const char* at, int pitch) __attribute__((always_inline)) {
    Turned f;
#pragma unroll
    for (int u = 0; u < 2; ++u)
      f.t[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr4)(at + 16 * u * pitch));
    return f;
  };
  // four columns e4 of token t
  auto part_at = [](int e4, int t) __attribute__((always_inline)) {
    return (e4 * 64 + (t ^ (e4 >> 1))) * 16;
  };

  if (wid < 4) {
    const long head = (long)a.seg[4 * sg] * a.H + h;
    float* Sp = a.S + head * DP * E + (long)(4 * quad) * E + e0 + 16 * wid + col;
    // GATED: each wave carries two of the normaliser's blocks, and begins with them
    const int d0 = GATE == GATED ? 2 * wid : 0;
    f32x4 S[8] = {};                     // keys 16 (d ^ d0) + 4 quad ... of column col
    if (a.seg[4 * sg + 3] > 0)
#pragma unroll
      for (int d = 0; d < 8; ++d)
#pragma unroll
        for (int j = 0; j < 4; ++j) S[d][j] = Sp[(long)(16 * (d ^ d0) + j) * E];
    f32x4 N[2] = {};                     // the same of the normaliser, in all columns
    float* Np = GATE == GATED
                    ? a.n + (head * (E / 32) + e0 / 32) * DP + 16 * d0 + 4 * quad
                    : nullptr;
    if (GATE == GATED && a.seg[4 * sg + 3] > 0)
#pragma unroll
      for (int d = 0; d < 2; ++d) N[d] = *(const f32x4*)(Np + 16 * d);
    auto put_n = [&](int now) __attribute__((always_inline)) {
      if (GATE != GATED) return;
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        uint t0[3], t1[3];
        cut3(N[d][0], N[d][1], t0);
        cut3(N[d][2], N[d][3], t1);
        if (col == 0)
#pragma unroll
          for (int z = 0; z < 3; ++z)
            *(uint2*)(s_np + (now * 3 + z) * DP + 16 * (d + d0) + 4 * quad) =
                uint2{t0[z], t1[z]};
      }
    };
    put_n(0);
    // 8 bytes of row col, slot s: at ^ 16 s
    const int qx = (col * 256 + (row_turn(col) ^ (quad >> 1)) * 16 + (quad & 1) * 8) ^
                   32 * d0;
    const int kx = kx0 ^ 32 * d0;
    const int wx = vx ^ (32 * wid), ox = part_at(4 * wid + quad, col);
    // Words are read from LDS a part ahead of the products that need them, and
    // converted beside the products before.
    auto piece = [&](int i, const char* qb, const char* kb, const char* vb, char* part)
        __attribute__((always_inline)) {
      const int now = i & 1;
      f32x4 o[4] = {}, w[2][2];
      frag_u pf[2][3], vf[2][3];
      Turned qf[2][4], kf[2][8], v[2];
      auto read_q = [&](int p) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int u = 0; u < 2; ++u)
            qf[p & 1][n].t[u] =
                *(const tr4*)(qb + n * 4096 + (qx ^ (64 * p + 32 * u)));
      };
      auto read_k = [&](int c, int d0) __attribute__((always_inline)) {
#pragma unroll
        for (int d = d0; d < d0 + 4; ++d)
          kf[c][d] = turned(kb + (kx ^ (32 * d)) + c * 32 * 256, 256);
      };
      auto split_s = [&](int p) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          uint t[3];
          cut3(S[2 * p + u / 2][u % 2 * 2], S[2 * p + u / 2][u % 2 * 2 + 1], t);
#pragma unroll
          for (int z = 0; z < 3; ++z) pf[p & 1][z].u[u] = t[z];
        }
      };
      auto split_v = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          uint t[3];
          cut3(__uint_as_float(v[c].u[u] << 16) * w[c][u / 2][u % 2 * 2],
               __uint_as_float(v[c].u[u] & 0xffff0000u) * w[c][u / 2][u % 2 * 2 + 1],
               t);
#pragma unroll
          for (int z = 0; z < 3; ++z) vf[c][z].u[u] = t[z];
        }
      };
      auto outputs = [&](int p) __attribute__((always_inline)) {
#pragma unroll
        for (int z = 0; z < 3; ++z)
#pragma unroll
          for (int n = 0; n < 4; ++n)
            o[n] = mfma16(pf[p & 1][z].bf, qf[p & 1][n].bf, o[n]);
      };
      auto updates = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int z = 0; z < 3; ++z)
#pragma unroll
          for (int d = 0; d < 8; ++d) S[d] = mfma16(kf[c][d].bf, vf[c][z].bf, S[d]);
      };
      // reads first, then `each` other instructions behind every product
      auto order = [](auto reads, auto products, auto each)
          __attribute__((always_inline)) {
        __builtin_amdgcn_sched_group_barrier(0x100, decltype(reads)::value, 0);
#pragma unroll
        for (int y = 0; y < decltype(products)::value; ++y) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, decltype(each)::value, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      __builtin_amdgcn_sched_barrier(0);
      read_q(0);
      const float keep = s_keep[now];
      read_q(1);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        v[c] = turned(vb + wx + c * 32 * 128, 128);
#pragma unroll
        for (int u = 0; u < 2; ++u)
          w[c][u] = *(const f32x4*)(s_w + now * L + 32 * c + 16 * u + 4 * quad);
      }
      __builtin_amdgcn_sched_barrier(0);
      split_s(0);
      __builtin_amdgcn_sched_barrier(0);
      outputs(0);
      split_s(1);
      order(Count<0>{}, Count<12>{}, Count<4>{});
      read_q(2);
      outputs(1);
      split_s(2);
      order(Count<0>{}, Count<12>{}, Count<4>{});
      read_q(3);
      outputs(2);
      split_s(3);
      order(Count<8>{}, Count<12>{}, Count<4>{});
      read_k(0, 0);
      read_k(0, 4);
      outputs(3);
      split_v(0);
#pragma unroll
      for (int d = 0; d < 8; ++d) S[d] *= keep;
      order(Count<16>{}, Count<12>{}, Count<8>{});
#pragma unroll
      for (int n = 0; n < 4; ++n) *(f32x4*)(part + ox + 256 * n) = o[n];
      read_k(1, 0);
      read_k(1, 4);
      updates(0);
      split_v(1);
      order(Count<16>{}, Count<24>{}, Count<3>{});
      updates(1);
      if (GATE == GATED) {
        frag_u wp[2][3];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int z = 0; z < 3; ++z)
#pragma unroll
            for (int u = 0; u < 2; ++u)
              *(uint2*)&wp[c][z].u[2 * u] = *(const uint2*)(
                  s_wp + (now * 3 + z) * L + 32 * c + 16 * u + 4 * quad);
#pragma unroll
        for (int d = 0; d < 2; ++d) N[d] *= keep;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
          for (int z = 0; z < 3; ++z)
#pragma unroll
            for (int d = 0; d < 2; ++d)
              N[d] = mfma16(kf[c][d].bf, wp[c][z].bf, N[d]);
        put_n(1 - now);
      }
    };
    meet();
    char *part = s_part, *next = s_part + PART, *after = s_part + 2 * PART;
    for (int i = 0; i < pieces; ++i) {
      piece(i, i & 1 ? q1 : q0, i & 1 ? k1 : k0, i & 1 ? v1 : v0, part);
      meet();
      char* p = part;
      part = next, next = after, after = p;
    }
#pragma unroll
    for (int d = 0; d < 8; ++d)
#pragma unroll
      for (int j = 0; j < 4; ++j) Sp[(long)(16 * (d ^ d0) + j) * E] = S[d][j];
    if (GATE == GATED && col < 2)        // a copy for every 32 columns
#pragma unroll
      for (int d = 0; d < 2; ++d) *(f32x4*)(Np + col * DP + 16 * d) = N[d];
    meet();
    return;
  }

  if (wid < 8) {
    const float skip = GATE == TIMED ? bits2f(((const short*)a.skip)[h]) : 0.f;
    const float ib = GATE == DECAY ? 0.f : bits2f(((const short*)a.ib)[h]);
    const float fb = GATE == DECAY ? 0.f : bits2f(((const short*)a.fb)[h]);
    const float rate = GATE == TIMED ? -expf(fb) : 0.f;
    const float l2d = GATE == DECAY ? a.log2_decay[h] : 0.f;
    float* mp = nullptr;
    float m = 0.f;                       // before the next piece (GATED)
    if (GATE == GATED) {
      mp = a.m + (((long)a.seg[4 * sg] * a.H + h) * E + e0) / 32;
      if (a.seg[4 * sg + 3] > 0) m = mp[0];
    }
    struct Raw { float i, f; };
    auto load_gate = [&](int i) __attribute__((always_inline)) {
      const long r = row0 + min(L * i + lane, rows - 1);
      if (GATE == TIMED) return Raw{a.gates[r * a.H + h], 0.f};
      if (GATE == GATED)
        return Raw{a.gates[2 * r * a.H + h], a.gates[(2 * r + 1) * a.H + h]};
      return Raw{0.f, 0.f};
    };
    auto gates = [&](int i, Raw g) __attribute__((always_inline)) {
      const int at = (i & 1) * L + lane;
      if (GATE == GATED) {
        float in = -INFINITY, F = 0.f;
        if (L * i + lane < rows) log_gates(a, g.i, g.f, ib, fb, in, F);
        float I = in;                    // scan of (F, I) by (+, max)
        float R = __shfl_down(F, 1, 64); // what comes after, without F's rounding
        if (lane == 63) R = 0.f;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const float F0 = __shfl_up(F, off, 64), I0 = __shfl_up(I, off, 64);
          const float R0 = __shfl_down(R, off, 64);
          if (lane >= off) {
            I = fmaxf(I0 + F, I);
            F += F0;
          }
          if (lane + off < 64) R += R0;
        }
        const float mt = fmaxf(F + m, I);
        const float end = __shfl(F, 63, 64), mn = __shfl(mt, 63, 64);
        const float w = expf(R + (in - mn));   // large ones first, exactly
        s_b[at] = F - mt;
        s_i[at] = in - F;
        s_far[at] = __expf(F + (m - mt)) * a.qscale;
        s_em[at] = expf(-mt);
        s_w[at] = w;
        uint t[3];
        cut3(w, 0.f, t);
#pragma unroll
        for (int z = 0; z < 3; ++z) s_wp[((i & 1) * 3 + z) * L + lane] = (short)t[z];
        if (lane == 0) s_keep[i & 1] = expf(end + (m - mn));
        m = mn;
        return;
      }
      if (GATE == DECAY) {               // only what the state needs
        const int n = min(rows - L * i, L);
        s_w[at] =
            lane < n ? __builtin_amdgcn_exp2f((n - 1 - lane) * l2d) : 0.f;
        if (lane == 0) s_keep[i & 1] = __builtin_amdgcn_exp2f(n * l2d);
        return;
      }
      const float step = L * i + lane < rows ? softplus_f(g.i + ib) : 0.f;
      float F = rate * step;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const float before = __shfl_up(F, off, 64);
        if (lane >= off) F += before;
      }
      const float end = __shfl(F, 63, 64), near = __shfl(F, lane | 15, 64);
      s_b[at] = F;
      s_i[at] = step;
      s_far[at] = expf(near - F) * step;
      s_w[at] = expf(end - F) * step;
      if (lane == 0) s_keep[i & 1] = expf(end);
    };
    const int rx = col * 256 + (row_turn(col) ^ quad) * 16;
    // tokens 16 n ... of a piece
    auto run = [&](auto number) __attribute__((always_inline)) {
      constexpr int n = decltype(number)::value, NP = n / 2 + 1;
      f32x4 pv[4];                       // columns 16 et + 4 quad ... of token t
      const int t = 16 * n + col;
      float inter = GATE == DECAY ? __builtin_amdgcn_exp2f((t + 1) * l2d) : 0.f;
      float inv = 1.f;                   // GATED: 1 / the normaliser
      // (of keys 4 quad + j of block J, seen from token t)
      f32x4 weight[GATE == DECAY ? n + 1 : 1];
      if (GATE == DECAY)
#pragma unroll
        for (int J = 0; J <= n; ++J)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int away = max(t - 16 * J - 4 * quad - j, 0);
            weight[GATE == DECAY ? J : 0][j] = __builtin_amdgcn_exp2f(away * l2d);
          }
      int at[4];
#pragma unroll
      for (int et = 0; et < 4; ++et) at[et] = part_at(4 * et + quad, t);
      auto add = [&](char* part) __attribute__((always_inline)) {
        f32x4 o[4];
#pragma unroll
        for (int et = 0; et < 4; ++et) o[et] = *(f32x4*)(part + at[et]);
#pragma unroll
        for (int et = 0; et < 4; ++et)
          *(f32x4*)(part + at[et]) = GATE == GATED ? (inter * o[et] + pv[et]) * inv
                                                   : inter * o[et] + pv[et];
      };
      auto piece = [&](int i, const char* qb, const char* kb, const char* vb)
          __attribute__((always_inline)) {
        frag_u qf[4], kf[4][n + 1];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          qf[c].u4 = *(const uint4v*)(qb + n * 4096 + (rx ^ (64 * c)));
#pragma unroll
          for (int J = 0; J <= n; ++J)
            kf[c][J].u4 = *(const uint4v*)(kb + J * 4096 + (rx ^ (64 * c)));
        }
        f32x4 acc[2 * NP] = {};
        if (GATE == DECAY) {
#pragma unroll
          for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int J = 0; J <= n; ++J) acc[J] = mfma16(kf[c][J].bf, qf[c].bf, acc[J]);
#pragma unroll
          for (int J = 0; J <= n; ++J) acc[J] *= weight[GATE == DECAY ? J : 0];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (4 * quad + j > col) acc[n][j] = 0.f;
        } else if (GATE == GATED) {
          f32x4 nq = {};                 // the same in all rows
#pragma unroll
          for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int z = 0; z < 3; ++z) {
              frag_u nf;
              nf.u4 = *(const uint4v*)(s_np + ((i & 1) * 3 + z) * DP + 32 * c + 8 * quad);
              nq = mfma16(nf.bf, qf[c].bf, nq);
            }
#pragma unroll
          for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int J = 0; J <= n; ++J) acc[J] = mfma16(kf[c][J].bf, qf[c].bf, acc[J]);
          const float bt = s_b[(i & 1) * L + t];
          inter = s_far[(i & 1) * L + t];
          float den = 0.f;
#pragma unroll
          for (int J = 0; J <= n; ++J) {
            const f32x4 key = *(const f32x4*)(s_i + (i & 1) * L + 16 * J + 4 * quad);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              acc[J][j] *= __expf(bt + key[j]) * a.qscale;
              if (J == n && 4 * quad + j > col) acc[J][j] = 0.f;
              den += acc[J][j];
            }
          }
          den += __shfl_xor(den, 16, 64);
          den += __shfl_xor(den, 32, 64);
          den += inter * nq[0];
          inv = 1.f / (fmaxf(fabsf(den), s_em[(i & 1) * L + t]) + GATED_EPS);
        } else {
          const float* b = s_b + (i & 1) * L;
          const float bt = b[t];
          const f32x4 bs = *(const f32x4*)(b + 16 * n + 4 * quad);
          const f32x4 step = *(const f32x4*)(s_i + (i & 1) * L + 16 * n + 4 * quad);
          f32x4 far[n + 1];
          float from[n + 1];
#pragma unroll
          for (int J = 0; J < n; ++J) {
            far[J] = *(const f32x4*)(s_far + (i & 1) * L + 16 * J + 4 * quad);
            from[J] = b[16 * J + 15];
          }
#pragma unroll
          for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int J = 0; J <= n; ++J) acc[J] = mfma16(kf[c][J].bf, qf[c].bf, acc[J]);
          inter = __expf(bt);
#pragma unroll
          for (int J = 0; J < n; ++J) acc[J] *= far[J] * __expf(bt - from[J]);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float w = acc[n][j] * (__expf(bt - bs[j]) * step[j]);
            const int s = 4 * quad + j;
            acc[n][j] = (s > col ? 0.f : w) + (s == col ? skip : 0.f);
          }
        }
#pragma unroll
        for (int et = 0; et < 4; ++et) pv[et] = f32x4{};
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          Turned v[4];
#pragma unroll
          for (int et = 0; et < 4; ++et)
            v[et] = turned(vb + (vx ^ (32 * et)) + p * 32 * 128, 128);
          frag_u pf[3];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            uint w[3];
            cut3(acc[2 * p + u / 2][u % 2 * 2], acc[2 * p + u / 2][u % 2 * 2 + 1], w);
#pragma unroll
            for (int z = 0; z < 3; ++z) pf[z].u[u] = w[z];
          }
#pragma unroll
          for (int z = 0; z < 3; ++z)
#pragma unroll
            for (int et = 0; et < 4; ++et)
              pv[et] = mfma16(v[et].bf, pf[z].bf, pv[et]);
        }
      };
      Raw g{0.f, 0.f};
      if (n == 0 && pieces) {
        gates(0, load_gate(0));
        g = load_gate(1);
      }
      meet();
      char *part = s_part + 2 * PART, *next = s_part, *after = s_part + PART;
      for (int i = 0; i < pieces; ++i) {
        if (n == 0) {
          gates(i + 1, g);
          g = load_gate(i + 2);
        }
        if (i) add(part);                // of the piece before
        piece(i, i & 1 ? q1 : q0, i & 1 ? k1 : k0, i & 1 ? v1 : v0);
        meet();
        char* p = part;
        part = next, next = after, after = p;
      }
      if (pieces) add(part);
      if (GATE == GATED && n == 0 && lane < 2) mp[lane] = m;
      meet();
    };
    if (wid == 4) run(Count<0>{});
    else if (wid == 5) run(Count<1>{});
    else if (wid == 6) run(Count<2>{});
    else run(Count<3>{});
    return;
  }

  const int ft = tid - 512, n = wid - 8;
  const int hk = h / (a.H / a.G);
  const short* qp = (const short*)a.q + row0 * a.qst + hk * DP;
  const short* kp = (const short*)a.k + row0 * a.kst + hk * DP;
  const short* vp = (const short*)a.v + row0 * a.vst + (long)h * E + e0;
  const int qst = (int)a.qst * 2, kst = (int)a.kst * 2, vst = (int)a.vst * 2;
  const int rt = ft / 16, rv = ft / 8, turn_t = (ft % 16 ^ row_turn(rt)) * 16;
  const int qo = rt * qst + turn_t, ko = rt * kst + turn_t;
  const int vo = rv * vst + (ft % 8 ^ value_turn<8>(rv)) * 16;
  // rows past the last come as zeros
  auto issue = [&](int i, char* qb, char* kb, char* vb) __attribute__((always_inline)) {
    const int end = min(rows - L * i, L) - 1;
    const auto qs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(qp + (long)L * i * a.qst), 0, end * qst + DP * 2, 0x00027000);
    const auto ks = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(kp + (long)L * i * a.kst), 0, end * kst + DP * 2, 0x00027000);
    const auto vs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(vp + (long)L * i * a.vst), 0, end * vst + ET * 2, 0x00027000);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int at = (p * 256 + n * 64) * 16;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(qs, (lds_ptr)(qb + at), 16,
                                               qo + p * 16 * qst, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ks, (lds_ptr)(kb + at), 16,
                                               ko + p * 16 * kst, 0, 0, 0);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          vs, (lds_ptr)(vb + (p * 256 + n * 64) * 16), 16, vo + p * 32 * vst, 0, 0, 0);
  };
  // the same through registers, asked for two pieces ahead
  uint4v words[GATE == DECAY ? 10 : 1];
  auto fetch = [&](int i) __attribute__((always_inline)) {
    const int end = min(rows - L * i, L) - 1;
    const auto qs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(qp + (long)L * i * a.qst), 0, end * qst + DP * 2, 0x00027000);
    const auto ks = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(kp + (long)L * i * a.kst), 0, end * kst + DP * 2, 0x00027000);
    const auto vs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(vp + (long)L * i * a.vst), 0, end * vst + ET * 2, 0x00027000);
    auto load = [](__amdgpu_buffer_rsrc_t src, int off) __attribute__((always_inline)) {
      return __builtin_bit_cast(uint4v,
                                __builtin_amdgcn_raw_buffer_load_b128(src, off, 0, 0));
    };
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      words[GATE == DECAY ? p : 0] = load(qs, qo + p * 16 * qst);
      words[GATE == DECAY ? 4 + p : 0] = load(ks, ko + p * 16 * kst);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
      words[GATE == DECAY ? 8 + p : 0] = load(vs, vo + p * 32 * vst);
  };
  auto put = [&](char* qb, char* kb, char* vb) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < 10; ++p) {
      char* to = p < 4 ? qb : p < 8 ? kb : vb;
      *(uint4v*)(to + ((p < 8 ? p % 4 : p - 8) * 256 + ft) * 16) =
          silu8<true>(words[GATE == DECAY ? p : 0]);
    }
  };
  // two rows of 64 columns, 16 bytes a lane
  const int r0 = 16 * n + (lane >> 3) * 2, c8 = lane & 7;
  const long at = (long)h * E + e0 + c8 * 8;
  uint4v z[2], znext[2];
  auto load_z = [&](int i) __attribute__((always_inline)) {
    if (GATE != TIMED) return;
#pragma unroll
    for (int y = 0; y < 2; ++y)
      znext[y] = *(const uint4v*)((const short*)a.z + at +
                                  (long)(row0 + min(L * i + r0 + y, rows - 1)) * a.zst);
  };
  uint4v w[2];
  auto results = [&](const char* part) __attribute__((always_inline)) {
    float v[2][8];
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        load4((const float*)(part + part_at(2 * c8 + u, r0 + y)), v[y] + 4 * u);
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      if (GATE == TIMED) {
        float g[8];
        unpack8(z[y], g);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[y][j] *= silu_f(g[j]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) w[y][j] = pack_bf16x2(v[y][2 * j], v[y][2 * j + 1]);
    }
  };
  auto store = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int y = 0; y < 2; ++y)
      if (L * i + r0 + y < rows)
        *(uint4v*)((short*)a.out + (long)(row0 + L * i + r0 + y) * a.H * E + at) = w[y];
  };
  // what was asked for is here
  auto arrive = []() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xf70);               // vmcnt(0)
    asm volatile("" ::: "memory");
  };
  if (pieces) {
    if (GATE == DECAY) {
      fetch(0);
      put(q0, k0, v0);
      if (pieces > 1) fetch(1);
    } else {
      issue(0, q0, k0, v0);
      arrive();
    }
  }
  meet();
  const char *part = s_part + PART, *next = s_part + 2 * PART, *after = s_part;
  for (int i = 0; i < pieces; ++i) {
    if (GATE == DECAY) {
      if (i + 1 < pieces) put(i & 1 ? q0 : q1, i & 1 ? k0 : k1, i & 1 ? v0 : v1);
      if (i + 2 < pieces) fetch(i + 2);
    } else if (i + 1 < pieces) {
      issue(i + 1, i & 1 ? q0 : q1, i & 1 ? k0 : k1, i & 1 ? v0 : v1);
    }
    if (i) load_z(i - 1);                // for the next turn
    if (i > 1) results(part);            // of two pieces ago
    if (GATE != DECAY) arrive();
    if (i > 1) store(i - 2);
    z[0] = znext[0], z[1] = znext[1];
    meet();
    const char* p = part;
    part = next, next = after, after = p;
  }
  if (pieces) load_z(pieces - 1);
  if (pieces > 1) {
    results(part);
    store(pieces - 2);
  }
  z[0] = znext[0], z[1] = znext[1];
  meet();
  if (pieces) {
    results(next);
    store(pieces - 1);
  }
}

// wider column tiles read the keys less often, as long as the accumulators
// leave registers for two workgroups per CU
template <int DP, int GATE>
static void launch_chunks(const ChunkArgs& x, hipStream_t stream) {
  const MemoryArgs& a = x.a;
  const long ch = (long)x.n_chunks * a.H;
  if constexpr (GATE != TURNED && DP == PASS_D)
    if (!x.P) {
      const int units = a.H * (a.E / 64);
      memory_pass_kernel<GATE>
          <<<(long)x.n_seg * 8 * ((units + 7) / 8), 768, 0, stream>>>(x);
      return;
    }
  if (!fixed_decay(GATE)) memory_gates_kernel<GATE><<<ch, MC_L, 0, stream>>>(x);
  if (GATE == TURNED) {
    const size_t lds = a.rot * sizeof(float);
    const long rows = (long)x.n_chunks * MC_L;
    if (a.rot % 16 == 0) memory_turn_kernel<true><<<rows, 256, lds, stream>>>(x);
    else memory_turn_kernel<false><<<rows, 256, lds, stream>>>(x);
  }
  if constexpr (GATE == TIMED && DP <= 128)
    if (!x.VT) {
      if (x.U) {
        memory_states_kernel<DP, GATE><<<ch * (a.E / 64), 256, 0, stream>>>(x);
        memory_scan_kernel<GATE><<<(long)x.n_seg * a.H * (DP / 64) * (a.E / 16),
                                   256, 0, stream>>>(x);
      } else if constexpr (DP == 64) {
        const int units = a.H * (a.E / 64);
        memory_carry_kernel<<<(long)x.n_seg * 8 * ((units + 7) / 8), 256, 0,
                              stream>>>(x);
      }
      memory_timed_kernel<DP><<<ch * 2 * (a.E / 64), 256, 0, stream>>>(x);
      return;
    }
  memory_states_kernel<DP, GATE>
      <<<ch * ((a.E + 63) / 64), 256, 0, stream>>>(x);
  memory_scan_kernel<GATE><<<(long)x.n_seg * a.H * ((a.D + 63) / 64) *
                                 ((a.E + 15) / 16), 256, 0, stream>>>(x);
  if (a.E <= 64 || DP > 128)
    memory_outputs_kernel<DP, 64, GATE>
        <<<ch * 2 * ((a.E + 63) / 64), 256, 0, stream>>>(x);
  else
    memory_outputs_kernel<DP, (DP > 128 ? 64 : 128), GATE>
        <<<ch * 2 * ((a.E + 127) / 128), 256, 0, stream>>>(x);
}

// bf16; D and E multiples of 8 with D <= 256; 16-byte aligned rows
extern "C" int sv_memory_chunks(const ChunkArgs* x, int gating,
                                hipStream_t stream) {
  if (x->n_seg <= 0) return 0;
  if (gating == TURNED &&
      (x->a.rot % 2 || x->a.rot > x->a.D ||
       (x->a.z && (x->a.E > 128 || (x->a.E > 64 && x->a.D > 128)))))
    return 1;
  if (!x->VT && ((gating != TIMED && (gating == TURNED || x->P)) || x->a.E % 64 ||
                 (x->a.D != 64 && x->a.D != 128)))
    return 1;
  if (!x->U && x->VT) return 1;
  // states are carried for 64 keys; one pass, for 128, leaves none behind
  if (!x->VT && !x->U && x->a.D != (x->P ? 64 : PASS_D)) return 1;
  if (!x->P && (x->VT || x->U || x->a.qst >= 1 << 22)) return 1;
  // offsets of a chunk's rows are of 32 bits
  if (!x->VT && (x->a.kst >= 1 << 22 || x->a.vst >= 1 << 22)) return 1;
#define MC(P)                                                     \
  do {                                                            \
    if (gating == GATED) launch_chunks<P, GATED>(*x, stream);     \
    else if (gating == TIMED) launch_chunks<P, TIMED>(*x, stream); \
    else if (gating == TURNED) launch_chunks<P, TURNED>(*x, stream); \
    else launch_chunks<P, DECAY>(*x, stream);                     \
  } while (0)
  if (x->a.D <= 64) MC(64);
  else if (x->a.D <= 128) MC(128);
  else if (x->a.D <= 256) MC(256);
  else return 1;
#undef MC
  return (int)hipGetLastError();
}
