// Attention over a paged KV cache for ragged batches.
//
// Cache layout: K [page][kv head][64][D], V [page][kv head][64][E]; a
// request's block table maps position / 64 to a page.  Visibility of key j
// for the query at position i:  j <= i and (i - j < window or j < keep).
// window <= 0 means plain causal.  Sizes D and E need not be equal.
//
// Scores and the softmax may be modified (ScoreArgs): a factor a head, a soft
// cap, a bias that falls with the distance, a sink in the denominator; the
// output may pass through one gate a head.
//
//   sv_kv_append   writes the K/V rows of a step into their pages
//   sv_qkv_append  the same with rotation and norm of queries and keys and with
//                  values mixed with another layer's
//   sv_attn_rows   one query row per workgroup group: single-token decoding
//                  (the row's own K/V is appended here) and the 32-bit mode
//   sv_attn_tiles  MFMA flash kernel over 128-row tiles for prompt portions

#include "serving.h"

#define NEG_BIG (-1e30f)
// The running maximum may lag behind by this much (in log 2): O is rescaled only
// when a row outgrows it.  The weights are 32-bit either way.
#define TILES_LAG 8.f

// ---------------------------------------------------------------------------
// append
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256)
kv_append_kernel(const T* __restrict__ k, const T* __restrict__ v, long kst,
                 long vst, T* __restrict__ kc, T* __restrict__ vc,
                 const int* __restrict__ pos, const int* __restrict__ seq,
                 const int* __restrict__ bt, int MB, int G, int D, int E) {
  const int t = blockIdx.x;
  const int p = pos[t];
  const long page = bt[(long)seq[t] * MB + p / SV_PAGE];
  const int in_page = p % SV_PAGE;
  for (int i = threadIdx.x; i < G * D; i += 256)
    kc[((page * G + i / D) * SV_PAGE + in_page) * D + i % D] = k[t * kst + i];
  for (int i = threadIdx.x; i < G * E; i += 256)
    vc[((page * G + i / E) * SV_PAGE + in_page) * E + i % E] = v[t * vst + i];
}

// 8 elements a thread when every row is a multiple of 8 elements
template <typename T>
__global__ void __launch_bounds__(256)
kv_append_vec_kernel(const T* __restrict__ k, const T* __restrict__ v,
                     long kst, long vst, T* __restrict__ kc,
                     T* __restrict__ vc, const int* __restrict__ pos,
                     const int* __restrict__ seq, const int* __restrict__ bt,
                     int MB, int G, int D, int E) {
  const int t = blockIdx.x;
  const int p = pos[t];
  const long page = bt[(long)seq[t] * MB + p / SV_PAGE];
  const int in_page = p % SV_PAGE;
  constexpr int NW = 8 * sizeof(T) / 16;
  for (int i = threadIdx.x * 8; i < G * D; i += 256 * 8) {
    const uint4v* s = (const uint4v*)(k + t * kst + i);
    uint4v* d = (uint4v*)(kc + ((page * G + i / D) * SV_PAGE + in_page) * D +
                          i % D);
#pragma unroll
    for (int j = 0; j < NW; ++j) d[j] = s[j];
  }
  for (int i = threadIdx.x * 8; i < G * E; i += 256 * 8) {
    const uint4v* s = (const uint4v*)(v + t * vst + i);
    uint4v* d = (uint4v*)(vc + ((page * G + i / E) * SV_PAGE + in_page) * E +
                          i % E);
#pragma unroll
    for (int j = 0; j < NW; ++j) d[j] = s[j];
  }
}

extern "C" int sv_kv_append(const void* k, const void* v, long kst, long vst,
                            void* kc, void* vc, const int* pos,
                            const int* seq, const int* bt, int MB, int T,
                            int G, int D, int E, int vec, int f32,
                            hipStream_t stream) {
  if (T <= 0) return 0;
#define KA(K, TT)                                                            \
  K<TT><<<T, 256, 0, stream>>>((const TT*)k, (const TT*)v, kst, vst,         \
                               (TT*)kc, (TT*)vc, pos, seq, bt, MB, G, D, E)
  if (f32) { if (vec) KA(kv_append_vec_kernel, float); else KA(kv_append_kernel, float); }
  else     { if (vec) KA(kv_append_vec_kernel, short); else KA(kv_append_kernel, short); }
#undef KA
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// append with what comes before the attention.  LPH lanes own a head of a row
// (8 elements each).  Queries are changed in place, keys and values go into
// their pages only.
// ---------------------------------------------------------------------------
struct QkvArgs {
  void* q;
  const void *k, *v;
  long qst, kst, vst;
  const double* freq;       // [rot / 2] radians a position: elements 2i and
                            //   2i + 1 turn; or null
  const void *qw, *kw;      // [D] weights of the norm, or null
  const void* first;        // values to mix in, or null
  long fst;
  const void* mix;          // their share (one number)
  void *kc, *vc;
  const int *pos, *seq, *bt;
  int MB, T, H, G, D, E, rot;
  int norm;                 // queries and keys over their root mean square
  int temp_every;           // > 0: queries times 1 + coef ln(floor((p + 1) /
  float temp_coef, eps;     //   every) + 1)
};

template <typename T, int LPH, bool VEC>
__global__ void __launch_bounds__(256) qkv_append_kernel(QkvArgs a) {
  constexpr int PER = 256 / LPH;         // heads of a workgroup
  const int heads = a.H + 2 * a.G;
  const long item = (long)blockIdx.x * PER + threadIdx.x / LPH;
  const long row = min(item / heads, (long)a.T - 1);
  const bool live = item < (long)a.T * heads;
  const int hh = item % heads, d0 = threadIdx.x % LPH * 8;
  const int p = a.pos[row];
  const long page = a.bt[(long)a.seq[row] * a.MB + p / SV_PAGE];
  const bool is_q = hh < a.H, is_v = hh >= a.H + a.G;
  const int g = is_q ? 0 : is_v ? hh - a.H - a.G : hh - a.H;
  const int size = is_v ? a.E : a.D;
  const int n = min(8, size - d0);       // elements of this lane; <= 0: none
  const T* src = is_q   ? (const T*)a.q + row * a.qst + (long)hh * a.D
                 : is_v ? (const T*)a.v + row * a.vst + (long)g * a.E
                        : (const T*)a.k + row * a.kst + (long)g * a.D;
  float x[8];
  load8<VEC>(src + d0, n, x);
  if (is_v && a.first) {
    const float m = to_f(((const T*)a.mix)[0]);
    float f[8];
    load8<VEC>((const T*)a.first + row * a.fst + (long)g * a.E + d0, n, f);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = (1.f - m) * x[j] + m * f[j];
  }
  if (!is_v && a.freq) {
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
      if (d0 + j >= a.rot) continue;
      float c, s;
      turn(a.freq[(d0 + j) / 2], p, &c, &s);
      const float u = x[j], w = x[j + 1];
      x[j] = u * c - w * s;
      x[j + 1] = w * c + u * s;
    }
  }
  if (a.norm) {                          // all lanes: values join the shuffles
    float sq = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) sq += x[j] * x[j];
#pragma unroll
    for (int off = LPH / 2; off > 0; off >>= 1) sq += __shfl_xor(sq, off, 64);
    if (!is_v) {
      const float rstd = 1.f / sqrtf(sq / a.D + a.eps);
      const T* w = (const T*)(is_q ? a.qw : a.kw);
      float u[8];
      if (w) load8<VEC>(w + d0, n, u);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] *= w ? rstd * u[j] : rstd;
    }
  }
  if (is_q && a.temp_every > 0) {
    const float t = 1.f + a.temp_coef * logf((float)((p + 1) / a.temp_every + 1));
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] *= t;
  }
  if (!live || n <= 0) return;
  const long at = (page * a.G + g) * SV_PAGE + p % SV_PAGE;
  T* dst = is_q   ? (T*)a.q + row * a.qst + (long)hh * a.D
           : is_v ? (T*)a.vc + at * a.E : (T*)a.kc + at * a.D;
  if (VEC) {
    store4(dst + d0, x);
    store4(dst + d0 + 4, x + 4);
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < n) from_f(dst[d0 + j], x[j]);
  }
}

// D and E at most 512; vec: D, E, strides and bases in 8 elements
extern "C" int sv_qkv_append(const QkvArgs* a, int vec, int f32,
                             hipStream_t stream) {
  if (a->T <= 0) return 0;
  if (a->rot % 2 || a->rot > a->D) return 1;
  const int big = a->D > a->E ? a->D : a->E;
  const long items = (long)a->T * (a->H + 2 * a->G);
#define QA(T, L, V)                                              \
  qkv_append_kernel<T, L, V>                                     \
      <<<(items + 256 / L - 1) / (256 / L), 256, 0, stream>>>(*a)
#define QAV(L)                                                   \
  do {                                                           \
    if (f32) { if (vec) QA(float, L, true); else QA(float, L, false); } \
    else     { if (vec) QA(short, L, true); else QA(short, L, false); } \
  } while (0)
  if (big <= 64) QAV(8);
  else if (big <= 128) QAV(16);
  else if (big <= 256) QAV(32);
  else if (big <= 512) QAV(64);
  else return 1;
#undef QAV
#undef QA
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// scores: s = q.k scale temp_h; s <- cap tanh(s / cap); s <- s - slope_h
// (i - j); the denominator also holds exp(sink_h); the output of head h is
// multiplied by sigmoid(gate[row][h]).  What is null or zero is left out.
// ---------------------------------------------------------------------------
struct ScoreArgs {
  const void *temp, *sink;  // [H], T
  const float* slope;       // [H]
  const void* gate;         // [rows][H], T
  long gst;
  float cap;
};

// ---------------------------------------------------------------------------
// rows
// ---------------------------------------------------------------------------
struct RowsArgs {
  const void *q, *k, *v;       // row 0 of the step's projections
  long qst, kst, vst;          // row strides (elements)
  void *kc, *vc;               // cache
  long kcs, vcs;               // elements from one cached row to the next
  const int *pos, *seq, *bt;   // per row: position, sequence; block table
  float* part;                 // [rows][H][splits][E + 2] or null (1 split)
  void* out;                   // [rows][H * E]
  int MB, rows, H, G, D, E, splits, append, window, keep;
  float scale;
  ScoreArgs mod;
  const float *cos, *sin;      // [positions][D / 2]: q and k are still to be
                               //   turned (form 2, plain scores); or null
};

// tanh, in the 32-bit mode to the last digits, else to 1e-7
__device__ __forceinline__ float tanh_t(float x, float) { return tanhf(x); }
__device__ __forceinline__ float tanh_t(float x, short) {
  return 1.f - 2.f * __builtin_amdgcn_rcpf(
                         1.f + __builtin_amdgcn_exp2f(2.f * SV_LOG2E * x));
}

// LPR lanes own one key row (DPL dims each); RC query heads share the row.
template <bool VEC, int DPL, typename T>
__device__ __forceinline__ void load_dims(const T* p, int n, float* v) {
#pragma unroll
  for (int j = 0; j < DPL; j += 8) load8<VEC>(p + j, n - j, v + j);
}

// MOD: scores and softmax as ScoreArgs say; without it they are plain.
template <bool MOD, typename T, int LPR, int RC, bool VEC, int DPL = 8>
__global__ void __launch_bounds__(256, RC <= 4 && DPL == 8 ? 4 : 1)
attn_rows_kernel(RowsArgs a) {
  constexpr int NR = 64 / LPR;     // key rows of one wave step
  constexpr int DV = LPR * DPL;
  const int rep = a.H / a.G;
  const int nrc = (rep + RC - 1) / RC;
  const int split = blockIdx.x % a.splits;
  const int unit = blockIdx.x / a.splits;
  const int rc = unit % nrc;
  const int g = unit / nrc % a.G;
  const int row = unit / nrc / a.G;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hl = lane % LPR, sub = lane / LPR;
  const int d0 = DPL * hl;
  // dims of this lane; <= 0: none
  const int nd = min(DPL, a.D - d0), ne = min(DPL, a.E - d0);
  const int D = a.D, E = a.E;

  const int i_pos = a.pos[row];
  const int* bt = a.bt + (long)a.seq[row] * a.MB;

  float qv[RC][DPL];
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    const int h = g * rep + min(rc * RC + r, rep - 1);
    load_dims<VEC, DPL>((const T*)a.q + row * a.qst + (long)h * D + d0, nd, qv[r]);
  }
  // scores in units of log 2; of the cap, if there is one
  const float cap = MOD ? a.mod.cap : 0.f;
  const float s2 = cap > 0.f ? a.scale / cap : a.scale * SV_LOG2E;
  float slope[RC];
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    float t = s2;
    if (MOD) {
      const int h = g * rep + min(rc * RC + r, rep - 1);
      if (a.mod.temp) t *= to_f(((const T*)a.mod.temp)[h]);
      // the same for all lanes: not in a vector register
      slope[r] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(
          a.mod.slope ? a.mod.slope[h] * SV_LOG2E : 0.f)));
    }
#pragma unroll
    for (int j = 0; j < DPL; ++j) qv[r][j] *= t;
  }

  const T* kn = (const T*)a.k + row * a.kst + (long)g * D;
  const T* vn = (const T*)a.v + row * a.vst + (long)g * E;
  if (a.append && split == 0 && rc == 0) {
    const long page = bt[i_pos / SV_PAGE];
    const long base = (page * a.G + g) * SV_PAGE + i_pos % SV_PAGE;
    for (int i = threadIdx.x; i < D; i += 256)
      ((T*)a.kc)[base * a.kcs + i] = kn[i];
    for (int i = threadIdx.x; i < E; i += 256)
      ((T*)a.vc)[base * a.vcs + i] = vn[i];
  }

  // visible keys as one list: the kept first ones, then the window.  With
  // append, the row's own key is handled from registers at the end.
  const int lo = a.window > 0 ? max(0, i_pos - a.window + 1) : 0;
  const int nfirst = min(a.keep, lo);
  const int total = nfirst + (i_pos - lo) + (a.append ? 0 : 1);
  const int per = (total + a.splits - 1) / a.splits;
  const int k0 = split * per, k1 = min(total, k0 + per);

  float m[RC], l[RC], o[RC][DPL];
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    m[r] = NEG_BIG;
    l[r] = 0.f;
#pragma unroll
    for (int j = 0; j < DPL; ++j) o[r][j] = 0.f;
  }

  auto fetch = [&](int idx, float* kf, float* vf) {
    const int j = idx < nfirst ? idx : lo + idx - nfirst;
    const long base =
        ((long)bt[j / SV_PAGE] * a.G + g) * SV_PAGE + j % SV_PAGE;
    load_dims<VEC, DPL>((const T*)a.kc + base * a.kcs + d0, nd, kf);
    load_dims<VEC, DPL>((const T*)a.vc + base * a.vcs + d0, ne, vf);
  };
  auto absorb = [&](const float* kf, const float* vf, bool live, int away) {
    float s[RC];
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      s[r] = 0.f;
#pragma unroll
      for (int j = 0; j < DPL; ++j) s[r] += qv[r][j] * kf[j];
    }
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1)
#pragma unroll
      for (int r = 0; r < RC; ++r) s[r] += __shfl_xor(s[r], off, 64);
    if (MOD) {
      if (cap > 0.f)
#pragma unroll
        for (int r = 0; r < RC; ++r) s[r] = cap * SV_LOG2E * tanh_t(s[r], T());
#pragma unroll
      for (int r = 0; r < RC; ++r) s[r] -= slope[r] * away;
    }
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      const float mn = live ? fmaxf(m[r], s[r]) : m[r];
      const float al = __builtin_amdgcn_exp2f(m[r] - mn);
      const float p = live ? __builtin_amdgcn_exp2f(s[r] - mn) : 0.f;
      m[r] = mn;
      l[r] = l[r] * al + p;
#pragma unroll
      for (int j = 0; j < DPL; ++j) o[r][j] = o[r][j] * al + p * vf[j];
    }
  };

  float kf[DPL], vf[DPL];
  int idx = k0 + wid * NR + sub;
#pragma unroll
  for (int j = 0; j < DPL; ++j) kf[j] = vf[j] = 0.f;
  if (idx < k1) fetch(idx, kf, vf);
  for (int b = k0 + wid * NR; b < k1; b += 4 * NR, idx += 4 * NR) {
    float kx[DPL], vx[DPL];
#pragma unroll
    for (int j = 0; j < DPL; ++j) kx[j] = vx[j] = 0.f;
    if (idx + 4 * NR < k1) fetch(idx + 4 * NR, kx, vx);
    absorb(kf, vf, idx < k1,
           MOD ? i_pos - (idx < nfirst ? idx : lo + idx - nfirst) : 0);
#pragma unroll
    for (int j = 0; j < DPL; ++j) {
      kf[j] = kx[j];
      vf[j] = vx[j];
    }
  }
  if (a.append && split == 0 && wid == 0) {
    load_dims<VEC, DPL>(kn + d0, nd, kf);
    load_dims<VEC, DPL>(vn + d0, ne, vf);
    absorb(kf, vf, sub == 0, 0);
  }

  // fold the NR row groups of the wave, then the 4 waves
#pragma unroll
  for (int off = 32; off >= LPR; off >>= 1)
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      const float m2 = __shfl_xor(m[r], off, 64);
      const float l2 = __shfl_xor(l[r], off, 64);
      const float mn = fmaxf(m[r], m2);
      const float c1 = __builtin_amdgcn_exp2f(m[r] - mn);
      const float c2 = __builtin_amdgcn_exp2f(m2 - mn);
      m[r] = mn;
      l[r] = l[r] * c1 + l2 * c2;
#pragma unroll
      for (int j = 0; j < DPL; ++j)
        o[r][j] = o[r][j] * c1 + __shfl_xor(o[r][j], off, 64) * c2;
    }
  __shared__ float so[4][RC][DV];
  __shared__ float sml[4][RC][2];
  if (sub == 0) {
#pragma unroll
    for (int r = 0; r < RC; ++r) {
#pragma unroll
      for (int j = 0; j < DPL; ++j) so[wid][r][d0 + j] = o[r][j];
      if (hl == 0) {
        sml[wid][r][0] = m[r];
        sml[wid][r][1] = l[r];
      }
    }
  }
  __syncthreads();
  for (int it = threadIdx.x; it < RC * DV; it += 256) {
    const int r = it / DV, e = it % DV;
    if (rc * RC + r >= rep || e >= E) continue;
    float mm = NEG_BIG;
#pragma unroll
    for (int w = 0; w < 4; ++w) mm = fmaxf(mm, sml[w][r][0]);
    float ll = 0.f, oo = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float c = __builtin_amdgcn_exp2f(sml[w][r][0] - mm);
      ll += sml[w][r][1] * c;
      oo += so[w][r][e] * c;
    }
    const int h = g * rep + rc * RC + r;
    if (MOD && a.mod.sink && split == 0) {   // once for all splits
      const float sink = to_f(((const T*)a.mod.sink)[h]) * SV_LOG2E;
      const float mn = fmaxf(mm, sink);
      const float c = __builtin_amdgcn_exp2f(mm - mn);
      ll = ll * c + __builtin_amdgcn_exp2f(sink - mn);
      oo *= c;
      mm = mn;
    }
    if (MOD && a.mod.gate)
      oo *= sigmoid_f(to_f(((const T*)a.mod.gate)[row * a.mod.gst + h]));
    if (a.splits == 1) {
      from_f(((T*)a.out)[((long)row * a.H + h) * E + e], oo / ll);
    } else {
      float* p = a.part +
                 (((long)row * a.H + h) * a.splits + split) * (E + 2);
      p[e] = oo;
      if (e == 0) {
        p[E] = mm;
        p[E + 1] = ll;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The same on MFMA, for bf16 heads of 64 or 128.  One workgroup = 4 waves, one
// query row, up to 16 heads that share their keys, a range of the keys in tiles
// of 32 (half a page); every wave takes every fourth tile with buffers of its
// own, so that waves never wait for each other.  Keys go straight into
// registers as fragments (a lane's 16 bytes of a row), values into LDS, from
// where transposing reads turn them.  S^T has its keys in the accumulator's
// rows, which is the order in which the values come; the weights stay 32-bit, in
// three planes that add up to them.
//
// Bound by memory: 8 waves a CU have 16 KB each on their way.  Values are read past the
// caches, as is right for what is read once a step (32 rows of up to 4096 keys, 309 MB:
// 61.1 -> 56.4 us; 64 rows of 1000, 16 heads: 33 -> 27.5); keys too are 2 % faster there
// but 13 % slower here, where their lines come in halves.  The kernel above
// spends its time on vector work (a key costs 140 cycles of a wave; here 30), but
// has more workgroups on a CU and less to start with: of many short rows whose
// heads have keys of their own it is the faster one (rows_kernel in
// ops/serving.py).
// ---------------------------------------------------------------------------
// the larger of the four lanes 16 apart
__device__ __forceinline__ float max_quarters(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x),
                                                  __float_as_uint(x), false,
                                                  false);
  return max_halves(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}

// ROT: the row's queries and key are turned here, an element with that half a head
// on, which the same lane holds.  As a kernel of its own, which every layer waits
// for, that took 4.6 us (4 layers, 16 steps: one request 7840 -> 7740 us).
// ONCE: up to 16 heads a group, nobody else reads a tile, and no cache keeps its values
// (32 heads of one group, 200 rows of 448, kept 20.1, past 21.0 us; of 180 12.3, 12.9).
template <bool MOD, int DE, bool ROT, bool ONCE>
__global__ void __launch_bounds__(256, 2) attn_rows_mfma_kernel(RowsArgs a) {
  constexpr int NC = DE / 32;            // chunks of a key
  constexpr int NB = DE / 16;            // 16-row blocks of O^T
  constexpr int CV = DE / 8;             // 16-byte slots of a value row
  constexpr int VB = 32 * DE * 2;        // bytes of a value tile
  // a tile a wave each; apart by name, so that a read of one need not wait for
  // the words on their way into the other
  __shared__ __attribute__((aligned(16))) char v0[4 * VB], v1[4 * VB];
  __shared__ float sml[4][16][2];

  const int rep = a.H / a.G, nrc = (rep + 15) / 16;
  const int split = blockIdx.x % a.splits;
  const int unit = blockIdx.x / a.splits;
  const int rc = unit % nrc, g = unit / nrc % a.G, row = unit / nrc / a.G;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15, grp = lane >> 4;
  const int h = g * rep + min(rc * 16 + c16, rep - 1);

  const int i_pos = a.pos[row];
  const int* bt = a.bt + (long)a.seq[row] * a.MB;
  const short* kn = (const short*)a.k + row * a.kst + (long)g * DE;
  const short* vn = (const short*)a.v + row * a.vst + (long)g * DE;
  if (a.append && split == 0 && rc == 0) {
    const long page = bt[i_pos / SV_PAGE];
    const long base = (page * a.G + g) * SV_PAGE + i_pos % SV_PAGE;
    for (int i = tid; i < DE; i += 256) {
      if (!ROT) ((short*)a.kc)[base * a.kcs + i] = kn[i];
      ((short*)a.vc)[base * a.vcs + i] = vn[i];
    }
  }

  frag_u qf[NC], own[ROT ? NC : 1];      // own: the row's key
  {
    const short* src = (const short*)a.q + row * a.qst + (long)h * DE + grp * 8;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      qf[c].u4 = *(const uint4v*)(src + c * 32);
      if (ROT) own[c].u4 = *(const uint4v*)(kn + c * 32 + grp * 8);
    }
  }
  float co[ROT ? NC / 2 : 1][8], si[ROT ? NC / 2 : 1][8];
  if constexpr (ROT)
#pragma unroll
    for (int c = 0; c < NC / 2; ++c)
#pragma unroll
      for (int j = 0; j < 8; j += 4) {
        const long at = (long)i_pos * (DE / 2) + c * 32 + grp * 8 + j;
        load4(a.cos + at, co[c] + j);
        load4(a.sin + at, si[c] + j);
      }
  // scores in units of log 2; of the cap, if there is one
  const float cap = MOD ? a.mod.cap : 0.f;
  float s2 = cap > 0.f ? a.scale / cap : a.scale * SV_LOG2E;
  if (MOD && a.mod.temp) s2 *= bits2f(((const short*)a.mod.temp)[h]);
  const float slope = MOD && a.mod.slope ? a.mod.slope[h] * SV_LOG2E : 0.f;

  // visible tiles as one list: those of the kept first keys, then the window's
  const int lo = a.window > 0 ? max(0, i_pos - a.window + 1) : 0;
  const int t_hi = i_pos / 32;
  const int nk = a.window > 0 ? min((a.keep + 31) / 32, t_hi + 1) : 0;
  const int t_lo = max(nk, lo / 32);
  const int total = nk + max(0, t_hi - t_lo + 1);
  const int per = (total + a.splits - 1) / a.splits;
  const int n1 = min(total, (split + 1) * per);
  auto tile_of = [&](int n) { return n < nk ? n : t_lo + n - nk; };

  // The page of a tile, asked for a turn before: a vector load, which the compiler
  // would wait for as soon as it has it.
  auto page_of = [&](int n) { return bt[tile_of(min(n, n1 - 1)) / 2]; };
  auto settle = [](int page) {
    asm volatile("" : "+v"(page));
    return __builtin_amdgcn_readfirstlane(page);
  };
  // Ask for a tile.  Keys past the newest read its row again, and the row's own
  // key and value come from the projection, also where they are not written
  // yet.
  auto issue = [&](int n, int page, frag_u (*kf)[NC], char* vd)
      __attribute__((always_inline)) {
    const int t = tile_of(n);
    const int newest = i_pos - t * 32;   // row of the tile
    const long base = ((long)settle(page) * a.G + g) * SV_PAGE + (t & 1) * 32;
    const short* kb = (const short*)a.kc + base * a.kcs;
    const short* vb = (const short*)a.vc + base * a.vcs;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = i * 16 + c16;
      const short* src = a.append && r >= newest
                             ? kn : kb + (long)min(r, newest) * a.kcs;
#pragma unroll
      for (int c = 0; c < NC; ++c)
        kf[i][c].u4 = *(const uint4v*)(src + c * 32 + grp * 8);
    }
#pragma unroll
    for (int p = 0; p < CV / 2; ++p) {
      const int it = p * 64 + lane, r = it / CV;
      // pairs of slots are rotated, so that 8 rows of a pair use every bank
      const int c = (it % CV ^ ((CV == 16 ? r : r >> 1) % (CV / 2)) * 2) * 8;
      const short* src = a.append && r >= newest
                             ? vn : vb + (long)min(r, newest) * a.vcs;
      __builtin_amdgcn_global_load_lds(
          (global_ptr)(src + c), (lds_ptr)(vd + wid * VB + p * 1024), 16, 0,
          ONCE ? 2 : 0);
    }
  };
  // a transposing read: 16 lanes turn 4 keys by 16 columns
  const int tr_row = 4 * grp + (c16 >> 2);
  const int tr_turn = (CV == 16 ? tr_row : tr_row >> 1) % (CV / 2);
  const int vx = wid * VB + tr_row * DE * 2 + tr_turn * 32 + (c16 & 3) * 8;

  f32x4 o[NB] = {};                      // O^T: rows d, col head
  float m = NEG_BIG, l = 0.f;            // l: of this lane's keys

  auto attend = [&](int n, frag_u (*kf)[NC], char* vbuf) __attribute__((always_inline)) {
    const int t = tile_of(n);
    if constexpr (ROT)
      if (t == t_hi)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (i * 16 + c16 >= i_pos - t * 32)
#pragma unroll
            for (int c = 0; c < NC; ++c) kf[i][c] = own[c];
    f32x4 s[2] = {};
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 2; ++i) s[i] = mfma16(kf[i][c].bf, qf[c].bf, s[i]);
    const int i0 = i_pos - t * 32 - 4 * grp;   // of this lane's key 0
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      s[i] *= s2;
      if (MOD) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (cap > 0.f) s[i][r] = cap * SV_LOG2E * tanh_t(s[i][r], short());
          s[i][r] -= slope * (float)(i0 - 16 * i - r);
        }
      }
    }
    if (t == t_hi || (a.window > 0 && t * 32 <= i_pos - a.window)) {
      asm volatile("");
      const int first = a.window > 0 ? i0 - a.window : -1 - 4 * grp;
      const int kept = a.window > 0 ? a.keep - t * 32 - 4 * grp : 0;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * i + r;
          s[i][r] = j > i0 || (j <= first && j >= kept) ? -INFINITY : s[i][r];
        }
    }
    float mt = -INFINITY;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) mt = fmaxf(mt, s[i][r]);
    mt = max_quarters(mt);
    if (__ballot(mt > m + TILES_LAG)) {
      const float mn = fmaxf(m, mt);
      const float al = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= al;
#pragma unroll
      for (int b = 0; b < NB; ++b) o[b] *= al;
    }
    frag_u pf[3];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float x = __builtin_amdgcn_exp2f(s[u >> 1][2 * (u & 1)] - m);
      float y = __builtin_amdgcn_exp2f(s[u >> 1][2 * (u & 1) + 1] - m);
      l += x + y;
#pragma unroll
      for (int z = 0; z < 3; ++z) {
        const uint w = pack_bf16x2(x, y);
        pf[z].u[u] = w;
        x -= __uint_as_float(w << 16);
        y -= __uint_as_float(w & 0xffff0000u);
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      union { tr4 t[2]; bf16x8 bf; } vf;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        vf.t[i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_tr4)(vbuf + (vx ^ (b * 32)) + i * 16 * DE * 2));
#pragma unroll
      for (int z = 0; z < 3; ++z) o[b] = mfma16(vf.bf, pf[z].bf, o[b]);
    }
  };
  // All words that this wave has asked for are there, and its reads are done.  The
  // compiler has to know: behind a wait in asm it waits for the next tile's words
  // before it multiplies this one's keys.
  auto arrived = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x70);              // vmcnt(0) lgkmcnt(0)
    asm volatile("" ::: "memory");
  };

  frag_u ka[2][NC], kb[2][NC];
  int n = split * per + wid;
  int page = 0;
  if (n < n1) {
    const int first = page_of(n);
    if (n + 4 < n1) page = page_of(n + 4);
    issue(n, first, ka, v0);
  }
  if constexpr (ROT) {                   // while the first tile is on its way
#pragma unroll
    for (int c = 0; c < NC / 2; ++c) {
#pragma unroll
      for (int z = 0; z < 2; ++z) {
        frag_u& lo = z ? own[c] : qf[c];
        frag_u& up = z ? own[c + NC / 2] : qf[c + NC / 2];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          float x[2], y[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const float p = __uint_as_float(e ? lo.u[u] & 0xffff0000u : lo.u[u] << 16);
            const float q = __uint_as_float(e ? up.u[u] & 0xffff0000u : up.u[u] << 16);
            x[e] = p * co[c][2 * u + e] - q * si[c][2 * u + e];
            y[e] = q * co[c][2 * u + e] + p * si[c][2 * u + e];
          }
          lo.u[u] = pack_bf16x2(x[0], x[1]);
          up.u[u] = pack_bf16x2(y[0], y[1]);
        }
      }
    }
    if (split == 0 && rc == 0 && wid == 0 && c16 == 0) {
      const long page = bt[i_pos / SV_PAGE];
      short* to = (short*)a.kc +
                  ((page * a.G + g) * SV_PAGE + i_pos % SV_PAGE) * a.kcs + grp * 8;
#pragma unroll
      for (int c = 0; c < NC; ++c) *(uint4v*)(to + c * 32) = own[c].u4;
    }
  }
  for (; n < n1; n += 8) {
    arrived();
    if (n + 4 < n1) {
      issue(n + 4, page, kb, v1);
      page = page_of(n + 8);
    }
    attend(n, ka, v0);
    if (n + 4 >= n1) break;
    arrived();
    if (n + 8 < n1) {
      issue(n + 8, page, ka, v0);
      page = page_of(n + 12);
    }
    attend(n + 4, kb, v1);
  }

  // the four waves
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (grp == 0) {
    sml[wid][c16][0] = m;
    sml[wid][c16][1] = l;
  }
  __syncthreads();                       // the tiles have been read
  float* so = (float*)(wid < 2 ? v0 : v1) + (wid & 1) * 16 * DE;  // [head][DE]
#pragma unroll
  for (int b = 0; b < NB; ++b)
    *(f32x4*)(so + c16 * DE + ((b * 16 + 4 * grp) ^ (c16 & 7) * 4)) = o[b];
  __syncthreads();
  for (int it = tid; it < min(16, rep - rc * 16) * DE; it += 256) {
    const int r = it / DE, e = it % DE;
    float mm = NEG_BIG;
#pragma unroll
    for (int w = 0; w < 4; ++w) mm = fmaxf(mm, sml[w][r][0]);
    float ll = 0.f, oo = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float c = __builtin_amdgcn_exp2f(sml[w][r][0] - mm);
      ll += sml[w][r][1] * c;
      oo += ((const float*)(w < 2 ? v0 : v1))[((w & 1) * 16 + r) * DE +
                                              (e ^ (r & 7) * 4)] * c;
    }
    const int hh = g * rep + rc * 16 + r;
    if (MOD && a.mod.sink && split == 0) {   // once for all splits
      const float sink = bits2f(((const short*)a.mod.sink)[hh]) * SV_LOG2E;
      const float mn = fmaxf(mm, sink);
      const float c = __builtin_amdgcn_exp2f(mm - mn);
      ll = ll * c + __builtin_amdgcn_exp2f(sink - mn);
      oo *= c;
      mm = mn;
    }
    if (MOD && a.mod.gate)
      oo *= sigmoid_f(bits2f(
          ((const short*)a.mod.gate)[row * a.mod.gst + hh]));
    const long rh = (long)row * a.H + hh;
    if (a.splits == 1) {
      ((short*)a.out)[rh * DE + e] = f2bits(oo / ll);
    } else {
      float* p = a.part + (rh * a.splits + split) * (DE + 2);
      p[e] = oo;
      if (e == 0) {
        p[DE] = mm;
        p[DE + 1] = ll;
      }
    }
  }
}

// One workgroup = one query row and head, 64 V columns; its four waves take
// every fourth split.  At most 64 splits.
template <typename T, int V>
__global__ void __launch_bounds__(256)
attn_rows_merge_kernel(const float* __restrict__ part, T* __restrict__ out,
                       int splits, int E) {
  __shared__ float coef[64], sum[4][64][V];
  const long rh = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float* p = part + rh * splits * (E + 2);
  if (wid == 0) {
    float m = NEG_BIG, l = 0.f;
    if (lane < splits) {
      m = p[(long)lane * (E + 2) + E];
      l = p[(long)lane * (E + 2) + E + 1];
    }
    float mm = m;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mm = fmaxf(mm, __shfl_xor(mm, off, 64));
    const float w = __builtin_amdgcn_exp2f(m - mm);
    l *= w;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off, 64);
    coef[lane] = w / l;
  }
  __syncthreads();
  const int e = (blockIdx.y * 64 + lane) * V;
  float acc[V] = {};
  if (e < E) {
    const float* src = p + e;
#pragma unroll 8
    for (int s = wid; s < splits; s += 4) {
      const float c = coef[s];
#pragma unroll
      for (int j = 0; j < V; ++j) acc[j] += c * src[(long)s * (E + 2) + j];
    }
  }
#pragma unroll
  for (int j = 0; j < V; ++j) sum[wid][lane][j] = acc[j];
  __syncthreads();
  if (wid > 0 || e >= E) return;
#pragma unroll
  for (int j = 0; j < V; ++j)
    from_f(out[rh * E + e + j], sum[0][lane][j] + sum[1][lane][j] +
                                    sum[2][lane][j] + sum[3][lane][j]);
}

extern "C" int sv_attn_merge(const float* part, void* out, long rows,
                             int splits, int E, int f32, hipStream_t stream) {
  if (splits > 64) return 1;
  const int v = E % 2 ? 1 : 2;
  const dim3 grid(rows, (E + 64 * v - 1) / (64 * v));
#define AM(T, V) attn_rows_merge_kernel<T, V><<<grid, 256, 0, stream>>>( \
      part, (T*)out, splits, E)
  if (f32) { if (v == 2) AM(float, 2); else AM(float, 1); }
  else     { if (v == 2) AM(short, 2); else AM(short, 1); }
#undef AM
  return (int)hipGetLastError();
}

// vec: 1 D, E, strides and bases in 8 elements; 2 on MFMA (bf16, D = E = 64 or
// 128)
template <bool MOD, typename T>
static int launch_rows(const RowsArgs& a, int vec, hipStream_t stream) {
  const int rep = a.H / a.G;
  const int big = a.D > a.E ? a.D : a.E;
  const int rcn = big > 512 ? (rep > 1 ? 2 : 1)
                            : rep >= 8 ? 8 : rep > 2 ? 4 : rep;
  const int nrc = vec == 2 ? (rep + 15) / 16 : (rep + rcn - 1) / rcn;
  const long grid = (long)a.rows * a.G * nrc * a.splits;
  if (a.cos && vec != 2) return 1;
  if (vec == 2) {
    if (sizeof(T) != 2 || a.D != a.E || (a.D != 64 && a.D != 128)) return 1;
#define ARMO(D, R, O) \
  attn_rows_mfma_kernel<MOD, D, R, O><<<grid, 256, 0, stream>>>(a)
#define ARM(D, R) \
  do { if (nrc == 1) ARMO(D, R, true); else ARMO(D, R, false); } while (0)
    if (a.cos) {
      if constexpr (MOD) return 1;
      else if (!a.append) return 1;
      else if (a.D == 64) ARM(64, true);
      else ARM(128, true);
    } else if (a.D == 64) ARM(64, false);
    else ARM(128, false);
#undef ARM
#undef ARMO
    if (a.splits > 1)
      return sv_attn_merge(a.part, a.out, (long)a.rows * a.H, a.splits, a.E, 0,
                           stream);
    return (int)hipGetLastError();
  }
#define AR(L, ...) \
  attn_rows_kernel<MOD, T, L, __VA_ARGS__><<<grid, 256, 0, stream>>>(a)
#define ARV(L, R) do { if (vec) AR(L, R, true); else AR(L, R, false); } while (0)
#define ARR(L)                                                         \
  do {                                                                 \
    if (rcn == 8) ARV(L, 8); else if (rcn == 4) ARV(L, 4);             \
    else if (rcn == 2) ARV(L, 2); else ARV(L, 1);                      \
  } while (0)
  if (big <= 64) ARR(8);
  else if (big <= 128) ARR(16);
  else if (big <= 256) ARR(32);
  else if (big <= 512) ARR(64);
  else if (big <= 1024) {
    if (rcn == 2) { if (vec) AR(64, 2, true, 16); else AR(64, 2, false, 16); }
    else { if (vec) AR(64, 1, true, 16); else AR(64, 1, false, 16); }
  } else return 1;
#undef ARR
#undef ARV
#undef AR
  if (a.splits > 1)
    return sv_attn_merge(a.part, a.out, (long)a.rows * a.H, a.splits, a.E,
                         sizeof(T) == 4, stream);
  return (int)hipGetLastError();
}

extern "C" int sv_attn_rows(const RowsArgs* a, int vec, int f32,
                            hipStream_t stream) {
  if (a->rows <= 0) return 0;
  const ScoreArgs& m = a->mod;
  const bool mod = m.temp || m.sink || m.slope || m.gate || m.cap > 0.f;
  if (f32)
    return mod ? launch_rows<true, float>(*a, vec, stream)
               : launch_rows<false, float>(*a, vec, stream);
  return mod ? launch_rows<true, short>(*a, vec, stream)
             : launch_rows<false, short>(*a, vec, stream);
}

// ---------------------------------------------------------------------------
// tiles: bf16 MFMA flash attention for prompt portions
//
// One workgroup = 4 waves x 32 query rows of one head; a key tile is one
// cache page.  S^T = K Q^T keeps every softmax statistic lane-local (a lane
// owns one query row).  The weights stay 32-bit: P is split exactly into
// NP bf16 planes (3 planes carry the full 24-bit significand) and V enters
// once per plane.  P never leaves registers: the accumulator's row order
// {4 hi + 0..3, 8 + 4 hi + 0..3} of a 16-key chunk is used as the
// contraction order of P V, and V^T is read from LDS in the same order
// (transposing loads).
//
// Bound by the matrix cores and by the vector work of the splits beside them:
// four products a tile where plain attention has two, which run at about 1.1
// PFLOP/s (a large matrix product: 1.3 to 1.5).  6000 tokens of three portions
// behind up to 4096, 32/8 heads: 621 -> 585 us with the next tile's scores
// beside this tile's exponentials, page numbers read two tiles ahead, keys
// rotated over all banks, and a maximum that lags; 568 with the order of the
// planes below, 556 with keys read ahead of their products, page numbers that
// nobody waits for and no branch a word on its way into LDS (latent attention of 2
// x 2048 tokens 355 -> 345, of 3 x 230 with 16 heads 196 -> 168).  An explicit order
// of products and vector work took 630, scores in one block with the weights of the
// tile before them spill 300 registers, splits by v_dot2c_f32_bf16 616.
// ---------------------------------------------------------------------------
//
// A key may end in columns that all heads share (kr): the rotated part of
// latent attention, whose other columns are expanded into a workspace first.
// The output may pass through sigmoid(gate).
struct TilesArgs {
  const short* q;
  long qst;                 // row stride of q
  const short *kc, *vc, *kr;
  long kpage, khead, krow;  // elements between pages, heads, rows
  long vpage, vhead, vrow;
  long rrow;                // between rows of kr (pages follow each other)
  const short* gate;        // [T][H * E] or null
  long gst;
  const int* tiles;         // [n_tiles][4]: seq, first row, rows, position
  const int* bt;
  short* out;               // [T][H * E]
  int MB, H, G, D, E, DS;   // DS: columns of a key before the shared ones
  int window, keep;
  float scale;
  ScoreArgs mod;            // its gate is one number a head
};

// MOD: 0 plain scores, 1 with a distance bias, 2 with a soft cap (and the bias,
// if there is one); a sink and the gates are handled in all.
template <int DK, int DE, int NP, bool SHARED, int MOD>
__global__ void __launch_bounds__(256, DE <= 128 ? 2 : 1)
attn_tiles_kernel(TilesArgs a) {
  constexpr int NC = DK / 16;        // 16-wide chunks of the key size
  constexpr int NB = DE / 32;        // 32-row blocks of O^T
  constexpr int KP = DK * 2;         // K row pitch (bytes)
  constexpr int CK = DK / 8, CV = DE / 8;  // 16-byte slots of a row
  // two key tiles, rows as in the cache; apart by name, so that a read of one
  // need not wait for the words on their way into the other
  __shared__ __attribute__((aligned(16))) char k0[64 * KP], k1[64 * KP];
  __shared__ __attribute__((aligned(16))) char v0[128 * DE], v1[128 * DE];

  // later tiles of a portion see more keys: they start first
  const int* tl = a.tiles + 4 * (gridDim.y - 1 - blockIdx.y);
  const int seq = tl[0], row0 = tl[1], nrow = tl[2], p0 = tl[3];
  const int h = near_head(blockIdx.x, a.H), g = h / (a.H / a.G);
  const int* bt = a.bt + (long)seq * a.MB;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int my = wid * 32 + col;              // query row in the tile
  const int my_pos = p0 + my;
  const int D = a.D, E = a.E;

  // A factor below zero turns the sign of the queries, so that the largest
  // product is the largest score; one of zero is as good as a tiny one, which
  // leaves a masked score at minus infinity.
  const float factor = a.scale * SV_LOG2E *
      (a.mod.temp ? bits2f(((const short*)a.mod.temp)[h]) : 1.f);
  const uint flip = MOD == 0 && factor < 0.f ? 0x80008000u : 0u;
  const float s2 = MOD == 0 ? fmaxf(fabsf(factor), 1e-37f) : factor;
  const float slope = MOD && a.mod.slope ? a.mod.slope[h] * SV_LOG2E : 0.f;
  // tanh(x) = 1 - 2 / (1 + e^2x), with x in units of log 2 / cap
  const float cap2 = MOD == 2 ? a.mod.cap * SV_LOG2E : 0.f;
  const float in_cap = MOD == 2 ? 2.f / a.mod.cap : 0.f;

  frag_u qf[NC];
  {
    const short* src =
        a.q + (long)(row0 + min(my, nrow - 1)) * a.qst + (long)h * D;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int d = c * 16 + hi * 8;
      qf[c].u4 = d < D ? *(const uint4v*)(src + d) : uint4v{0, 0, 0, 0};
      qf[c].u4 ^= flip;
    }
  }

  f32x16 ot[NB] = {};
  float m_run = NEG_BIG;
  float l_run = 0.f;                 // over this half wave's keys

  const int q_hi = p0 + nrow - 1;
  const int t_hi = q_hi / SV_PAGE;
  const int lo = a.window > 0 ? max(0, p0 - a.window + 1) : 0;
  const int nk = a.window > 0
                     ? min((a.keep + SV_PAGE - 1) / SV_PAGE, t_hi + 1) : 0;
  const int t_lo = max(nk, lo / SV_PAGE);
  const int ntiles = nk + max(0, t_hi - t_lo + 1);
  const int w_lo = p0 + wid * 32, w_hi = min(w_lo + 31, q_hi);

  // 32-bit within a page
  const int krow = (int)a.krow, vrow = (int)a.vrow, rrow = (int)a.rrow;
  auto tile_of = [&](int n) { return n < nk ? n : t_lo + n - nk; };
  // A page number is a vector load, which the compiler waits for, with all words on
  // their way into LDS, as soon as it has it: `settle` keeps that behind a barrier
  // that waits for them anyway.
  auto page_of = [&](int n) { return bt[tile_of(min(n, ntiles - 1))]; };
  auto settle = [](int page) {
    asm volatile("" : "+v"(page));
    return __builtin_amdgcn_readfirstlane(page);
  };
  // Ask for the rows of a page: a wave's 64 slots of 16 bytes follow each
  // other in LDS, so the rotation of a row's slots is done on the source.
  // Rows that fill the tile need no branch a word.
  auto issue_k = [&](long page, char* kd) {
    const short* kb = a.kc + page * a.kpage + g * a.khead;
    const short* rb = SHARED ? a.kr + page * SV_PAGE * rrow - a.DS : nullptr;
    auto word = [&](int p, bool all) __attribute__((always_inline)) {
      const int it = p * 256 + tid, r = it / CK;
      const int c = (it % CK ^ key_turn<CK>(r)) * 8;
      if (!all && c >= D) return;
      __builtin_amdgcn_global_load_lds(
          (global_ptr)(SHARED && c >= a.DS ? rb + (r * rrow + c)
                                           : kb + (r * krow + c)),
          (lds_ptr)(kd + (p * 256 + wid * 64) * 16), 16, 0, 0);
    };
    if (D == DK) {
#pragma unroll
      for (int p = 0; p < CK / 4; ++p) word(p, true);
    } else {
#pragma unroll
      for (int p = 0; p < CK / 4; ++p) word(p, false);
    }
  };
  auto issue_v = [&](long page, char* vd) {
    const short* vb = a.vc + page * a.vpage + g * a.vhead;
    auto word = [&](int p, bool all) __attribute__((always_inline)) {
      const int it = p * 256 + tid, r = it / CV;
      const int c = (it % CV ^ value_turn<CV>(r)) * 8;
      if (!all && c >= E) return;
      __builtin_amdgcn_global_load_lds(
          (global_ptr)(vb + (r * vrow + c)),
          (lds_ptr)(vd + (p * 256 + wid * 64) * 16), 16, 0, 0);
    };
    if (E == DE) {
#pragma unroll
      for (int p = 0; p < CV / 4; ++p) word(p, true);
    } else {
#pragma unroll
      for (int p = 0; p < CV / 4; ++p) word(p, false);
    }
  };
  // this lane's part of the addresses in a tile (bytes): slot 2 c + hi of key
  // row col; a transposing read, where 16 lanes turn 4 keys by 16 columns
  int kx[KeySlots<CK>::steps];
#pragma unroll
  for (int c = 0; c < KeySlots<CK>::steps; ++c)
    kx[c] = col * KP + ((2 * c + hi) ^ key_turn<CK>(col)) * 16;
  const int tr_key = 4 * hi + ((lane & 15) >> 2);
  const int vx = (tr_key * DE + ((lane >> 4) & 1) * 16 + (lane & 3) * 4 +
                  value_turn<CV>(tr_key) * 8) * 2;

  // S^T = K Q^T, the keys of two products AHEAD of them
  auto scores = [&](f32x16* s, const char* kbuf) __attribute__((always_inline)) {
    constexpr int AHEAD = 2;
    frag_u kf[AHEAD + 1][2];
    auto read = [&](int c) __attribute__((always_inline)) {
      constexpr int M = KeySlots<CK>::steps;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        kf[c % (AHEAD + 1)][kb].u4 = *(const uint4v*)(
            kbuf + kx[c % M] + (c / M) * M * 32 + kb * 32 * KP);
    };
    s[0] = s[1] = f32x16{};
#pragma unroll
    for (int c = 0; c < AHEAD; ++c) read(c);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (c + AHEAD < NC) read(c + AHEAD);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
        s[kb] = mfma_bf16(kf[c % (AHEAD + 1)][kb].bf, qf[c].bf, s[kb]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // scores of tile n as they enter the softmax, and the running maximum
  auto level = [&](int n, f32x16* s) __attribute__((always_inline)) {
    const int kv0 = tile_of(n) * SV_PAGE;
    const int i0 = my_pos - kv0 - 4 * hi;      // of this lane's key 0
    if (MOD) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) s[kb] *= s2;
      if (MOD == 2)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            s[kb][r] = cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(
                1.f + __builtin_amdgcn_exp2f(s[kb][r] * in_cap));
      if (MOD == 1 || slope != 0.f)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            s[kb][r] -= slope * (float)(i0 - 32 * kb - acc_row(r, 0));
    }
    if (kv0 + SV_PAGE - 1 > w_lo ||
        (a.window > 0 && w_hi - kv0 >= a.window && kv0 + SV_PAGE > a.keep)) {
      asm volatile("");          // a branch: not selects on every tile
      // key j is seen if j <= i0 and (j > first or j < kept)
      const int first = a.window > 0 ? i0 - a.window : -1 - 4 * hi;
      const int kept = a.window > 0 ? a.keep - kv0 - 4 * hi : 0;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = 32 * kb + acc_row(r, 0);
          const bool gone = j > i0 || (j <= first && j >= kept);
          s[kb][r] = gone ? -INFINITY : s[kb][r];
        }
    }
    float mt = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, s[kb][r]);
    mt = max_halves(mt);
    if (MOD == 0) mt *= s2;
    if (__ballot(mt > m_run + TILES_LAG)) {
      const float m_new = fmaxf(m_run, mt);
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) ot[nb] *= alpha;
    }
  };
  auto weigh = [&](f32x16* s) __attribute__((always_inline)) {
    float ps = 0.f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[kb][r] = __builtin_amdgcn_exp2f(MOD == 0 ? s[kb][r] * s2 - m_run
                                                   : s[kb][r] - m_run);
        ps += s[kb][r];
      }
    l_run += ps;
  };
  // O^T += V^T P, 16 keys after 16; the next ones' planes are made beside the
  // products
  auto gather = [&](const f32x16* s, char* vbuf) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      frag_u pf[NP];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float x = s[c >> 1][8 * (c & 1) + 2 * u];
        float y = s[c >> 1][8 * (c & 1) + 2 * u + 1];
#pragma unroll
        for (int z = 0; z < NP; ++z) {
          const uint w = pack_bf16x2(x, y);
          pf[z].u[u] = w;
          x -= __uint_as_float(w << 16);
          y -= __uint_as_float(w & 0xffff0000u);
        }
      }
      // a plane of all columns after the other: a product that adds to the one
      // before it waits for it (6000 prompt tokens: 590 -> 582 us, latent 395 ->
      // 381)
      union { tr4 t[2]; bf16x8 bf; } vf[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int u = 0; u < 2; ++u)
          vf[nb].t[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_tr4)(vbuf + (vx ^ (nb * 64)) + (16 * c + 8 * u) * DE * 2));
#pragma unroll
      for (int z = 0; z < NP; ++z)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          ot[nb] = mfma_bf16(vf[nb].bf, pf[z].bf, ot[nb]);
    }
  };
  auto active = [&](int n) {
    const int kv0 = tile_of(n) * SV_PAGE;
    return n < ntiles && wid * 32 < nrow && kv0 <= w_hi &&
        (a.window <= 0 || kv0 < a.keep || kv0 + SV_PAGE - 1 > w_lo - a.window);
  };
  // Tile n's weights and values, while the next tile's scores are made: the
  // products of one run beside the exponentials of the other.
  auto step = [&](int n, f32x16* s, f32x16* next, const char* kbuf, char* vbuf)
      __attribute__((always_inline)) {
    const bool now = active(n);
    if (now) level(n, s);
    if (now || active(n + 1)) scores(next, kbuf);
    if (now) {
      weigh(s);
      gather(s, vbuf);
    }
  };

  if (D < DK) {                // columns that no tile writes
    for (int i = tid; i < 64 * CK; i += 256) {
      *(uint4v*)(k0 + i * 16) = uint4v{0, 0, 0, 0};
      *(uint4v*)(k1 + i * 16) = uint4v{0, 0, 0, 0};
    }
    __syncthreads();
  }
  f32x16 sa[2], sb[2];
  int pa = page_of(0), pb = page_of(1), pc = page_of(2);
  issue_k(pa, k0);
  issue_v(pa, v0);
  if (ntiles > 1) issue_k(pb, k1);
  __syncthreads();             // also waits for the words on their way
  if (active(0)) scores(sa, k0);
  __syncthreads();
  for (int n = 0; n < ntiles; n += 2) {
    // keys of n + 1 and values of n are there; pb, pc: pages of n + 1, n + 2
    const int vd = page_of(n + 3);
    if (n + 2 < ntiles) issue_k(pc, k0);
    if (n + 1 < ntiles) issue_v(pb, v1);
    step(n, sa, sb, k1, v0);
    __syncthreads();
    if (n + 1 >= ntiles) break;
    pb = settle(vd);
    const int ve = page_of(n + 4);
    if (n + 3 < ntiles) issue_k(pb, k1);
    if (n + 2 < ntiles) issue_v(pc, v0);
    step(n + 1, sb, sa, k0, v1);
    __syncthreads();
    pc = settle(ve);
  }

  l_run += __shfl_xor(l_run, 32, 64);
  if (my >= nrow) return;
  float inv = 1.f / l_run;
  if (a.mod.sink) {
    const float sink = bits2f(((const short*)a.mod.sink)[h]) * SV_LOG2E;
    const float mn = fmaxf(m_run, sink);
    const float c = __builtin_amdgcn_exp2f(m_run - mn);
    inv = c / (l_run * c + __builtin_amdgcn_exp2f(sink - mn));
  }
  if (a.mod.gate)
    inv *= sigmoid_f(bits2f(
        ((const short*)a.mod.gate)[(long)(row0 + my) * a.mod.gst + h]));
  short* dst = a.out + ((long)(row0 + my) * a.H + h) * E;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      const int d = 32 * nb + 8 * rg + 4 * hi;
      if (d < E) {
        float o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = ot[nb][4 * rg + j] * inv;
        if (a.gate) {
          float z[4];
          load4(a.gate + (long)(row0 + my) * a.gst + (long)h * E + d, z);
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] *= sigmoid_f(z[j]);
        }
        uint2 w = {pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
        *(uint2*)(dst + d) = w;
      }
    }
}

// D, DS and E multiples of 8, at most 256; every row 16-byte aligned
extern "C" int sv_attn_tiles(const TilesArgs* a, int n_tiles,
                             hipStream_t stream) {
  if (n_tiles <= 0) return 0;
  const dim3 grid(a->H, n_tiles);
  const int mod = a->mod.cap > 0.f ? 2 : a->mod.slope ? 1 : 0;
  if (a->kr && mod) return 1;
#define ATK(K, V, S, M) \
  attn_tiles_kernel<K, V, 3, S, M><<<grid, 256, 0, stream>>>(*a)
#define AT(K, V)                          \
  do {                                    \
    if (a->kr) ATK(K, V, true, 0);        \
    else if (mod == 2) ATK(K, V, false, 2); \
    else if (mod == 1) ATK(K, V, false, 1); \
    else ATK(K, V, false, 0);             \
  } while (0)
  if (a->D <= 64 && a->E <= 64) AT(64, 64);
  else if (a->D <= 128 && a->E <= 128) AT(128, 128);
  else if (a->D <= 192 && a->E <= 128) AT(192, 128);
  else if (a->D <= 256 && a->E <= 256) AT(256, 256);
  else return 1;
#undef AT
#undef ATK
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// rotary embedding (rotate-half) of the rows of a ragged batch, in place:
// every row has its own position.  cos/sin [positions][D / 2] f32.
// ---------------------------------------------------------------------------
// A thread turns VEC pairs of one head, so that a single token's heads are read
// at once by several workgroups (40 heads of 128, 1 token: 4.4 us; pair after
// pair in one workgroup: 5.4).  Single pairs of many tokens are left to one
// workgroup a token (4096 tokens, 72 heads of 50: 16.8 us, by eight 18.8).
template <typename T, int VEC>
__global__ void __launch_bounds__(256)
rope_rows_kernel(T* __restrict__ q, long qst, int H, T* __restrict__ k,
                 long kst, int G, const float* __restrict__ cosp,
                 const float* __restrict__ sinp, const int* __restrict__ pos,
                 int D) {
  const int t = blockIdx.x, half = D / 2;
  const long row = (long)pos[t] * half;
  auto turn = [&](int i) __attribute__((always_inline)) {
    const int h = i / half, j = i % half;
    T* p = (h < H ? q + t * qst + (long)h * D
                  : k + t * kst + (long)(h - H) * D) + j;
    const long at = row + j;
    float c[VEC], s[VEC], x[VEC], y[VEC], u[VEC], v[VEC];
    if (VEC == 4) {
      load4(p, x);
      load4(p + half, y);
      load4(cosp + at, c);
      load4(sinp + at, s);
    } else {
      x[0] = to_f(p[0]);
      y[0] = to_f(p[half]);
      c[0] = cosp[at];
      s[0] = sinp[at];
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      u[e] = x[e] * c[e] - y[e] * s[e];
      v[e] = y[e] * c[e] + x[e] * s[e];
    }
    if (VEC == 4) {
      store4(p, u);
      store4(p + half, v);
    } else {
      from_f(p[0], u[0]);
      from_f(p[half], v[0]);
    }
  };
  int i = (blockIdx.y * 256 + threadIdx.x) * VEC;
  if (VEC > 1) {
    if (i < (H + G) * half) turn(i);
  } else {
    for (; i < (H + G) * half; i += gridDim.y * 256) turn(i);
  }
}

extern "C" int sv_rope_rows(void* q, long qst, int H, void* k, long kst,
                            int G, const float* cosp, const float* sinp,
                            const int* pos, int T, int D, int f32,
                            hipStream_t stream) {
  if (T <= 0 || H + G <= 0 || D < 2) return 0;
  const size_t size = f32 ? 4 : 2;
  const bool vec = D % 8 == 0 &&
      (((size_t)q | (size_t)k | qst * size | kst * size) & (4 * size - 1)) == 0 &&
      (((size_t)cosp | (size_t)sinp) & 15) == 0;
  const int per = !vec && T > 256
      ? 1 : ((H + G) * (D / 2) / (vec ? 4 : 1) + 255) / 256;
#define ROPE(T_, V)                                                         \
  rope_rows_kernel<T_, V><<<dim3(T, per), 256, 0, stream>>>(                \
      (T_*)q, qst, H, (T_*)k, kst, G, cosp, sinp, pos, D)
  if (f32) { if (vec) ROPE(float, 4); else ROPE(float, 1); }
  else     { if (vec) ROPE(short, 4); else ROPE(short, 1); }
#undef ROPE
  return (int)hipGetLastError();
}
