// Latent attention over a paged cache for ragged batches.
//
// A token keeps one row [latent (R) | rotated shared key (P)] for all heads:
// cache [page][64][R + P].  The key of head h is [W_uk,h c | kr], its value
// W_uv,h c.  Two ways to attend:
//   * absorbed: the query takes W_uk in (q' = W_uk,h^T q), scores and values
//     read the cached rows themselves, W_uv follows; used for single tokens.
//   * expanded: the visible rows are gathered, one GEMM makes keys and values
//     of all heads, and the MFMA prompt kernel of paged_attn.hip runs on them.
//
//   sv_latent_append  norm of the latent, rotation of q and of the shared
//                     key at each row's position, write into the cache
//   sv_latent_gather  cache pages -> contiguous rows
//   sv_head_linear    a small matrix per head (absorption, values), with an
//                     optional sigmoid gate on the result
//   sv_latent_rows    MFMA attention of one absorbed query row over its keys
//
// The denominator of the softmax may hold a sink, a number a head.

#include "serving.h"

#define NEG_BIG (-1e30f)

// ---------------------------------------------------------------------------
// append
// ---------------------------------------------------------------------------
struct LatentAppendArgs {
  void* q;                  // [T] rows; head h's rotated part at h * qh
  long qst, qh;
  void* qr;                 // rotated queries go here (may be q itself)
  long qrst, qrh;
  const void* kv;           // [T] rows of R latents, then P key columns
  long kvst;
  const void* w;            // [R] weight of the latents' norm
  const double* freq;       // [rot / 2] radians a position
  void* cache;
  const int *pos, *seq, *bt;
  int MB, H, R, P, rot;     // rot <= P columns turn, the rest pass
  float eps;
  float amp;                // multiplies cos and sin
  int pairs;                // columns 2i and 2i + 1 turn, not i and i + rot / 2
};

extern __shared__ float dynamic_lds[];

// row t; VEC: words of four elements
template <typename T, int NT, bool VEC>
__device__ __forceinline__ void latent_append(const LatentAppendArgs& a, int t) {
  float* cs = dynamic_lds;               // cos [rot / 2], sin [rot / 2]
  __shared__ float red[16];
  const int tid = threadIdx.x;
  const int half = a.rot / 2, R = a.R, P = a.P;
  const int p = a.pos[t];
  const T* kv = (const T*)a.kv + t * a.kvst;
  const long page = a.bt[(long)a.seq[t] * a.MB + p / SV_PAGE];
  float sq = 0.f;
  if (VEC) {
    for (int i = tid * 4; i < R; i += NT * 4) {
      float v[4];
      load4(kv + i, v);
      sq += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
    }
  } else {
    for (int i = tid; i < R; i += NT) {
      const float v = to_f(kv[i]);
      sq += v * v;
    }
  }
  for (int i = NT - 1 - tid; i < half; i += NT) {      // by the last threads
    float c, s;
    turn(a.freq[i], p, &c, &s);
    cs[i] = c * a.amp;
    cs[half + i] = s * a.amp;
  }
  sq = block_reduce_sum(sq, red);        // its barriers publish cs as well
  const float rstd = 1.f / sqrtf(sq / R + a.eps);
  T* row = (T*)a.cache + (page * SV_PAGE + p % SV_PAGE) * (R + P);
  const T* w = (const T*)a.w;
  if (VEC) {
    for (int i = tid * 4; i < R; i += NT * 4) {
      float v[4], u[4];
      load4(kv + i, v);
      load4(w + i, u);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] *= rstd * u[j];
      store4(row + i, v);
    }
  } else {
    for (int i = tid; i < R; i += NT)
      from_f(row[i], to_f(kv[i]) * rstd * to_f(w[i]));
  }

  // V pairs, or elements past them, from i in [0, P - half) on
  constexpr int V = VEC ? 4 : 1;
  auto rotate = [&](const T* src, T* dst, int i) {
    if (i >= half) {
      if (VEC) {
        float v[4];
        load4(src + i + half, v);
        store4(dst + i + half, v);
      } else {
        dst[i + half] = src[i + half];
      }
      return;
    }
    float x[V], y[V];
    const int u = a.pairs ? 2 * i : i, z = a.pairs ? u + V : i + half;
    if (VEC) {
      load4(src + u, x);
      load4(src + z, y);
    } else {
      x[0] = to_f(src[u]);
      y[0] = to_f(src[z]);
    }
    if (VEC && a.pairs) {                // neighbours: x0 y0 x1 y1 | x2 y2 ...
      const float t[4] = {x[1], x[3], y[1], y[3]};
      x[1] = x[2];
      x[2] = y[0];
      x[3] = y[2];
#pragma unroll
      for (int j = 0; j < V; ++j) y[j] = t[j];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const float c = cs[i + j], s = cs[half + i + j], v = x[j];
      x[j] = v * c - y[j] * s;
      y[j] = y[j] * c + v * s;
    }
    if (VEC && a.pairs) {
      const float t[4] = {x[2], y[2], x[3], y[3]};
      x[2] = x[1];
      x[3] = y[1];
      x[1] = y[0];
#pragma unroll
      for (int j = 0; j < V; ++j) y[j] = t[j];
    }
    if (VEC) {
      store4(dst + u, x);
      store4(dst + z, y);
    } else {
      from_f(dst[u], x[0]);
      from_f(dst[z], y[0]);
    }
  };
  const int items = (P - half) / V;
  for (int i = tid; i < (a.H + 1) * items; i += NT) {
    const int h = i / items, j = i % items * V;
    if (h == a.H)
      rotate(kv + R, row + R, j);
    else
      rotate((const T*)a.q + t * a.qst + h * a.qh,
             (T*)a.qr + t * a.qrst + h * a.qrh, j);
  }
}

template <typename T, int NT, bool VEC>
__global__ void __launch_bounds__(NT)
latent_append_kernel(LatentAppendArgs a) {
  latent_append<T, NT, VEC>(a, blockIdx.x);
}

static bool append_in_words(const LatentAppendArgs* a, size_t size) {
  return ((a->rot / 2 | a->R | a->P | a->qst | a->qh | a->qrst | a->qrh |
           a->kvst) & 3) == 0 &&
      (((size_t)a->q | (size_t)a->qr | (size_t)a->kv | (size_t)a->w |
        (size_t)a->cache) & (4 * size - 1)) == 0;
}

extern "C" int sv_latent_append(const LatentAppendArgs* a, int T, int f32,
                                hipStream_t stream) {
  if (T <= 0) return 0;
  const size_t lds = a->rot * sizeof(float);
  const bool vec = append_in_words(a, f32 ? 4 : 2);
  // few rows: a longer workgroup waits for fewer words one after the other
  // (32 rows of 512 + 64, 32 heads: 7.1 -> 4.3 us; 4096 rows, element after
  // element 21, in words 15)
#define LAV(T_, NT, V)                                                        \
  latent_append_kernel<T_, NT, V><<<T, NT, lds, stream>>>(*a)
#define LA(T_)                                                                \
  do {                                                                        \
    if (T <= 512) { if (vec) LAV(T_, 1024, true); else LAV(T_, 1024, false); } \
    else { if (vec) LAV(T_, 256, true); else LAV(T_, 256, false); }           \
  } while (0)
  if (f32) LA(float); else LA(short);
#undef LAV
#undef LA
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// gather: pages[i] of the cache -> page i of the workspace (16-byte words)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
latent_gather_kernel(const uint4v* __restrict__ cache, uint4v* __restrict__ ws,
                     const int* __restrict__ pages, int words) {
  const uint4v* s = cache + (long)pages[blockIdx.x] * words;
  uint4v* d = ws + (long)blockIdx.x * words;
  for (int i = blockIdx.y * 256 + threadIdx.x; i < words; i += gridDim.y * 256)
    d[i] = s[i];
}

extern "C" int sv_latent_gather(const void* cache, void* ws, const int* pages,
                                int n, int page_bytes, hipStream_t stream) {
  if (n <= 0) return 0;
  const int words = page_bytes / 16;
  const dim3 grid(n, (words + 1023) / 1024);
  latent_gather_kernel<<<grid, 256, 0, stream>>>((const uint4v*)cache,
                                                 (uint4v*)ws, pages, words);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// head linear: out[t, h, n] = sum_k x[t, h, k] w[h, n, k]
// ---------------------------------------------------------------------------
struct HeadLinearArgs {
  const void* x;
  long xst, xh;             // elements between rows, between heads
  const void* w;            // [H][N][K]
  void* out;
  long ost, oh;
  const void* gate;         // out is multiplied by sigmoid(gate), or null
  long gst, gh;
  int T, H, N, K;
};

// 8 elements at p + k, zero from n on: a word is read in either case, since a
// branch a word costs more than the word
__device__ __forceinline__ uint4v word_or_zero(const short* p, int k, int n) {
  const uint4v w = *(const uint4v*)(p + (k < n ? k : 0));
  return k < n ? w : uint4v{0, 0, 0, 0};
}

// One wave of a workgroup's four takes every fourth 64-column block of K for
// 32 outputs and 32 rows; the partial sums meet in LDS.  With SPLIT off each
// wave has 32 outputs of its own.  K, strides and bases in 8 elements.
template <bool SPLIT>
__device__ __forceinline__ void head_linear_mfma(const HeadLinearArgs& a, int nb,
                                                 int h, int t0) {
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int n0 = (SPLIT ? nb : nb * 4 + wid) * 32;
  const int K = a.K;
  const bool vn = n0 + col < a.N, vt = t0 + col < a.T;
  const short* w = (const short*)a.w + ((long)h * a.N + (vn ? n0 + col : 0)) * K;
  const short* x = (const short*)a.x + (long)(vt ? t0 + col : 0) * a.xst + h * a.xh;
  f32x16 acc = {};
  if (n0 < a.N)
    for (int k0 = SPLIT ? wid * 64 : 0; k0 < K; k0 += SPLIT ? 256 : 64) {
      frag_u fw[4], fx[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int k = k0 + 16 * c + 8 * hi;
        fw[c].u4 = word_or_zero(w, k, K);
        fx[c].u4 = word_or_zero(x, k, K);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) acc = mfma_bf16(fw[c].bf, fx[c].bf, acc);
    }
  if (SPLIT) {
    __shared__ float part[4][16][64];
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wid][r][lane] = acc[r];
    __syncthreads();
    // wave w finishes accumulator rows 4 w .. 4 w + 3
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v = 0.f;
#pragma unroll
      for (int s = 0; s < 4; ++s) v += part[s][4 * wid + j][lane];
      acc[j] = v;
    }
  }
  if (!vt) return;
  const int t = t0 + col;
#pragma unroll
  for (int rg = 0; rg < (SPLIT ? 1 : 4); ++rg) {
    const int n = n0 + 8 * (SPLIT ? wid : rg) + 4 * hi;
    if (n + 3 < a.N) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = acc[4 * rg + j];
      if (a.gate) {
        float z[4];
        load4((const short*)a.gate + t * a.gst + h * a.gh + n, z);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] *= sigmoid_f(z[j]);
      }
      store4((short*)a.out + t * a.ost + h * a.oh + n, v);
    }
  }
}

template <bool SPLIT>
__global__ void __launch_bounds__(256)
head_linear_mfma_kernel(HeadLinearArgs a) {
  head_linear_mfma<SPLIT>(a, blockIdx.x, blockIdx.y, blockIdx.z * 32);
}

// What a decoding step does before its attention, in one launch: rows are
// appended by the first `rows` workgroups, the others take the queries into the
// latent space (32 rows, 32 heads of 128 + 64, rank 512: 6 us for 10.5 of two
// launches).
template <bool VEC, bool SPLIT>
__global__ void __launch_bounds__(256)
latent_absorb_kernel(LatentAppendArgs a, HeadLinearArgs l, int rows, int nb) {
  if ((int)blockIdx.x < rows) {
    latent_append<short, 256, VEC>(a, blockIdx.x);
    return;
  }
  const int id = blockIdx.x - rows;
  head_linear_mfma<SPLIT>(l, id % nb, id / nb % l.H, id / nb / l.H * 32);
}

// any size and type: one output a thread
template <typename T>
__global__ void __launch_bounds__(256)
head_linear_kernel(HeadLinearArgs a) {
  const int n = blockIdx.y * 256 + threadIdx.x, h = blockIdx.z;
  const long t = blockIdx.x;
  if (n >= a.N) return;
  const T* x = (const T*)a.x + t * a.xst + h * a.xh;
  const T* w = (const T*)a.w + ((long)h * a.N + n) * a.K;
  float v = 0.f;
  for (int k = 0; k < a.K; ++k) v += to_f(x[k]) * to_f(w[k]);
  if (a.gate) v *= sigmoid_f(to_f(((const T*)a.gate)[t * a.gst + h * a.gh + n]));
  from_f(((T*)a.out)[t * a.ost + h * a.oh + n], v);
}

extern "C" int sv_head_linear(const HeadLinearArgs* a, int mfma, int f32,
                              hipStream_t stream) {
  if (a->T <= 0) return 0;
  if (mfma) {
    const int nt = (a->N + 31) / 32, tt = (a->T + 31) / 32;
    if (a->K >= 256)
      head_linear_mfma_kernel<true><<<dim3(nt, a->H, tt), 256, 0, stream>>>(*a);
    else
      head_linear_mfma_kernel<false><<<dim3((nt + 3) / 4, a->H, tt), 256, 0,
                                       stream>>>(*a);
  } else {
    const dim3 grid(a->T, (a->N + 255) / 256, a->H);
    if (f32) head_linear_kernel<float><<<grid, 256, 0, stream>>>(*a);
    else head_linear_kernel<short><<<grid, 256, 0, stream>>>(*a);
  }
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// rows: MFMA attention of absorbed queries.
//
// One workgroup = 4 waves, one query row, 32 heads, a range of its keys in
// tiles of 32 (half a page, contiguous in the cache).  Per tile:
//   1. S^T = K Q^T, each wave a quarter of the columns; partial sums to LDS
//   2. softmax by all threads (8 lanes a head); the 32-bit weights go to LDS
//      as three bf16 planes that add up to them exactly
//   3. O^T += V^T P^T, each wave a quarter of the latent columns; V^T is the
//      same tile, read through the transposing LDS load
// The columns are padded to EP latents and 64 rotated ones, with zeros.
//
// Several splits: rows * splits workgroups share all rows' tiles, about as many
// each, so that long rows are not waited for (32 rows of 512 to 4096 keys: 33 us
// with as many workgroups for every row, 27 with as many tiles).  A workgroup
// finds its share from the positions.
// ---------------------------------------------------------------------------
struct LatentRowsArgs {
  const short* q;           // [rows][H][R + P]
  const short* cache;
  const int *pos, *seq, *bt;
  float* part;              // sums [rows * splits][H][R], their maxima and
                            //   totals [rows * splits][H][2], of every row its
                            //   first share and their number; null: 1 split
  short* out;               // [rows][H][R]
  int MB, rows, H, R, P, splits, window;
  float scale;
  const short* sink;        // [H] or null
};

__device__ __forceinline__ float2* share_totals(const LatentRowsArgs& a) {
  return (float2*)(a.part + (long)a.rows * a.splits * a.H * a.R);
}
__device__ __forceinline__ int2* row_shares(const LatentRowsArgs& a) {
  return (int2*)(share_totals(a) + (long)a.rows * a.splits * a.H);
}

struct Share { int row, i, n; };         // the i-th of n of a row

#define LATENT_SHARES 512                // most of a group of 32 heads

// The share of workgroup `item`; row is -1 if there is none.  Shares are of at
// most `per` tiles, the least for which there are no more of them than
// workgroups: at least total / items, at most total / (items - rows).  (That bound
// itself left every second workgroup of two a row without work: 46 rows of 3613
// keys, 128 heads 253 us, now 162; as many shares of every row, however long: 191.)
__device__ __forceinline__ Share share_of(const LatentRowsArgs& a, int item) {
  constexpr int B = LATENT_SHARES / 2 / 64;    // rows of two shares, 64 a time
  const int lane = threadIdx.x & 63;
  const int items = a.rows * a.splits;
  auto sum = [](int x) { return __builtin_amdgcn_readlane(scan64(x), 63); };
  int n[B], total = 0;
#pragma unroll
  for (int b = 0; b < B; ++b) {
    n[b] = 0;
    if (64 * b >= a.rows) continue;
    if (64 * b + lane < a.rows) {
      const int p = a.pos[64 * b + lane];
      n[b] = p / 32 - (a.window > 0 ? max(0, p - a.window + 1) / 32 : 0) + 1;
    }
    total += sum(n[b]);
  }
  auto shares = [](int tiles, int per, float inv) {
    const int x = tiles + per - 1;
    int q = (int)(x * inv);              // off by one at most
    q -= q * per > x;
    q += (q + 1) * per <= x;
    return q;
  };
  auto count = [&](int per) {
    const float inv = __builtin_amdgcn_rcpf(per);
    int c = 0;
#pragma unroll
    for (int b = 0; b < B; ++b)
      if (64 * b < a.rows) c += shares(n[b], per, inv);
    return sum(c);
  };
  int per = (total + items - 1) / items;
  for (int most = (total + items - a.rows - 1) / (items - a.rows); per < most;) {
    const int half = (per + most) / 2;
    if (count(half) <= items) most = half; else per = half + 1;
  }
  const float inv = __builtin_amdgcn_rcpf(per);
#pragma unroll
  for (int b = 0; b < B; ++b) {
    if (64 * b >= a.rows) break;
    const int mine = shares(n[b], per, inv);
    const int last = scan64(mine);       // of the shares up to this lane's row
    const int all = __builtin_amdgcn_readlane(last, 63);
    if (item < all) {
      const int l = __ffsll((unsigned long long)__ballot(last > item)) - 1;
      const int k = __builtin_amdgcn_readlane(mine, l);
      return {64 * b + l, item - __builtin_amdgcn_readlane(last, l) + k, k};
    }
    item -= all;
  }
  return {-1, 0, 0};
}

// FULL: R = EP and P = 64, no padding.  ONCE: up to 32 heads, nobody else reads the
// tiles, and no cache keeps them (rank 512, caches that no earlier call has read, us,
// kept | past: 32 heads, 89 rows of 3161 84 | 81, 12 of 402 16.2 | 15.5; 16 heads, 2 of
// up to 2481 14.5 | 13.3).  Of more heads workgroups of 32 read the same ones (128
// heads, 128 rows of 1472 146 | 161, 15 of 504 23.5 | 26.8; 40, 10 of 2057 25.0 | 28.3).
template <int EP, bool FULL, bool ONCE>
__global__ void __launch_bounds__(256, 2)
latent_rows_kernel(LatentRowsArgs a) {
  constexpr int KP = EP + 64;            // columns of a tile row
  constexpr int CPR = KP / 8;            // 16-byte slots of a row
  constexpr int NCW = KP / 64;           // 16-column chunks of a wave
  constexpr int NB = EP >= 128 ? EP / 128 : 1;  // 32-column blocks of a wave
  constexpr int NL = 32 * CPR / 256;     // 16-byte words a thread loads
  constexpr int SP = 36, PP = 40;        // pitches of S and P
  __shared__ __attribute__((aligned(16))) short kt[32 * KP];
  __shared__ __attribute__((aligned(16))) float sp[4][32 * SP];
  __shared__ __attribute__((aligned(16))) short pp[3][32 * PP];
  __shared__ float corr[32], lsum[32], mrow[32];

  const int items = a.rows * a.splits, item = blockIdx.x % items;
  const int h0 = blockIdx.x / items * 32;
  Share my = {item, 0, 1};
  if (a.splits > 1) {
    my = share_of(a, item);
    if (my.row < 0) return;
    if (my.i == 0 && h0 == 0 && threadIdx.x == 0)
      row_shares(a)[my.row] = int2{item, my.n};
  }
  my.i = __builtin_amdgcn_readfirstlane(my.i);
  my.n = __builtin_amdgcn_readfirstlane(my.n);
  const int row = __builtin_amdgcn_readfirstlane(my.row);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int R = FULL ? EP : a.R, P = FULL ? 64 : a.P, RP = R + P;

  // column of a slot in a cached row, -1 for padding
  auto column = [&](int slot) {
    const int c = slot * 8;
    if (FULL) return c;
    return c < EP ? (c < R ? c : -1) : (c - EP < P ? R + c - EP : -1);
  };
  // (read in any case and zeroed behind, words of padding spill 18 registers)
  auto word = [&](const short* src, int k) {
    return k < 0 ? uint4v{0, 0, 0, 0} : *(const uint4v*)(src + k);
  };
  auto swz_slot = [](int r, int slot) {
    return slot ^ (CPR % 16 == 0 ? r & 15 : (r >> 1) & 7);
  };

  frag_u qf[NCW];
  {
    // heads that are none repeat the last one
    const short* src = a.q + ((long)row * a.H + min(h0 + col, a.H - 1)) * RP;
#pragma unroll
    for (int c = 0; c < NCW; ++c)
      qf[c].u4 = word(src, column((wid * NCW + c) * 2 + hi));
  }

  const int i_pos = a.pos[row];
  const int* bt = a.bt + (long)a.seq[row] * a.MB;
  const int lo = a.window > 0 ? max(0, i_pos - a.window + 1) : 0;
  const int t_lo = lo / 32, total = i_pos / 32 - t_lo + 1;
  const int per = (total + my.n - 1) / my.n;   // all of them have some
  const int t0 = t_lo + my.i * per, t1 = min(t_lo + total, t0 + per);

  uint4v reg[NL];
  int page = bt[t0 / 2];                 // of the tile that is asked for next
  auto issue = [&](int t) {
    const short* src = a.cache + ((long)page * SV_PAGE + (t & 1) * 32) * RP;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int it = i * 256 + tid;
      if (FULL && ONCE)                  // a tile is one piece
        reg[i] = __builtin_nontemporal_load((const uint4v*)(src + it * 8u));
      else if (FULL)
        reg[i] = *(const uint4v*)(src + it * 8u);
      else
        reg[i] = word(src + it / CPR * RP, column(it % CPR));
    }
    page = bt[min(t + 1, t1 - 1) / 2];
  };

  f32x16 o[NB] = {};
  const int sh = tid >> 3, sk = tid & 7;   // softmax: head, 4-key group
  float m_run = NEG_BIG, l_run = 0.f;
  if (a.sink && my.i == 0 && h0 + sh < a.H) {    // once for all splits
    m_run = bits2f(a.sink[h0 + sh]) * SV_LOG2E;
    l_run = 1.f;
  }
  const float s2 = a.scale * SV_LOG2E;
  // transposing reads: a group of 16 lanes turns 4 keys x 16 columns
  const int tr_key = (lane & 15) >> 2, tr_col = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;

  if (t0 < t1) issue(t0);
  for (int t = t0; t < t1; ++t) {
    __syncthreads();               // the previous tile has been read
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int it = i * 256 + tid, r = it / CPR;
      *(uint4v*)(kt + r * KP + swz_slot(r, it % CPR) * 8) = reg[i];
    }
    __syncthreads();
    if (t + 1 < t1) issue(t + 1);

    f32x16 acc = {};
#pragma unroll
    for (int c = 0; c < NCW; ++c) {
      frag_u kf;
      kf.u4 = *(const uint4v*)(kt + col * KP +
                               swz_slot(col, (wid * NCW + c) * 2 + hi) * 8);
      acc = mfma_bf16(kf.bf, qf[c].bf, acc);
    }
#pragma unroll
    for (int rg = 0; rg < 4; ++rg)
      *(f32x4*)(sp[wid] + col * SP + 8 * rg + 4 * hi) =
          f32x4{acc[4 * rg], acc[4 * rg + 1], acc[4 * rg + 2], acc[4 * rg + 3]};
    __syncthreads();

    {
      f32x4 s = *(const f32x4*)(sp[0] + sh * SP + 4 * sk);
#pragma unroll
      for (int w = 1; w < 4; ++w) s += *(const f32x4*)(sp[w] + sh * SP + 4 * sk);
      float mt = NEG_BIG;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int key = t * 32 + 4 * sk + j;
        s[j] = key >= lo && key <= i_pos ? s[j] * s2 : NEG_BIG;
        mt = fmaxf(mt, s[j]);
      }
      mt = fold8(mt, MaxOp());
      const float mn = fmaxf(m_run, mt);   // every tile holds a visible key
      const float al = __builtin_amdgcn_exp2f(m_run - mn);
      m_run = mn;
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[j] = __builtin_amdgcn_exp2f(s[j] - mn);
        ps += s[j];
      }
      ps = fold8(ps, SumOp());
      l_run = l_run * al + ps;
      float x[4] = {s[0], s[1], s[2], s[3]};
#pragma unroll
      for (int z = 0; z < 3; ++z) {
        uint2 w = {pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])};
        *(uint2*)(pp[z] + sh * PP + 4 * sk) = w;
        x[0] -= __uint_as_float(w.x << 16);
        x[1] -= __uint_as_float(w.x & 0xffff0000u);
        x[2] -= __uint_as_float(w.y << 16);
        x[3] -= __uint_as_float(w.y & 0xffff0000u);
      }
      if (sk == 0) corr[sh] = al;
    }
    __syncthreads();

    const float al = corr[col];
    if (__ballot(al != 1.f)) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) o[nb] *= al;
    }
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      frag_u pf[3];
#pragma unroll
      for (int z = 0; z < 3; ++z)
        pf[z].u4 = *(const uint4v*)(pp[z] + col * PP + kc * 16 + hi * 8);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int e = (wid * NB + nb) * 32;
        if (EP < 128 && e >= EP) continue;
        union { tr4 h[2]; bf16x8 bf; } vf;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int r = kc * 16 + hi * 8 + u * 4 + tr_key, c = e + tr_col;
          vf.h[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_tr4)(kt + r * KP + swz_slot(r, c >> 3) * 8 + (c & 7)));
        }
#pragma unroll
        for (int z = 0; z < 3; ++z) o[nb] = mfma_bf16(vf.bf, pf[z].bf, o[nb]);
      }
    }
  }

  if (sk == 0) {
    lsum[sh] = l_run;
    mrow[sh] = m_run;
  }
  __syncthreads();
  if (h0 + col >= a.H) return;
  const float inv = 1.f / lsum[col];
  short* out = a.out + ((long)row * a.H + h0 + col) * R;
  float* part = a.part + ((long)item * a.H + h0 + col) * R;
  auto put = [&](auto whole) __attribute__((always_inline)) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int e = (wid * NB + nb) * 32 + 8 * rg + 4 * hi;
        if ((!FULL || EP < 128) && e >= R) continue;
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = o[nb][4 * rg + j];
        if (whole) {
          v *= inv;
          *(uint2*)(out + e) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        } else {
          *(f32x4*)(part + e) = v;
        }
      }
  };
  if (a.splits == 1) put(std::true_type()); else put(std::false_type());
  if (a.splits > 1 && wid == 0 && hi == 0)
    share_totals(a)[(long)item * a.H + h0 + col] = float2{mrow[col], lsum[col]};
}

// ---------------------------------------------------------------------------
// merge: the shares of a row and head, 64 V columns; four waves take every fourth
// share.
// ---------------------------------------------------------------------------
template <int V>
__global__ void __launch_bounds__(256) latent_merge_kernel(LatentRowsArgs a) {
  __shared__ float coef[LATENT_SHARES], sum[4][64][V];
  const int h = blockIdx.x % a.H, row = blockIdx.x / a.H;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int2 sh = row_shares(a)[row];    // first and number
  if (wid == 0) {
    const float2* ml = share_totals(a) + (long)sh.x * a.H + h;
    auto total = [&](int s) {
      return s + lane < sh.y ? ml[(long)(s + lane) * a.H] : float2{NEG_BIG, 0.f};
    };
    const float2 first = total(0);
    float mm = first.x, l = 0.f;
    for (int s = 64; s < sh.y; s += 64) mm = fmaxf(mm, total(s).x);
    mm = fold64(mm, MaxOp());
    for (int s = 0; s < sh.y; s += 64) {
      const float2 v = s ? total(s) : first;
      const float w = __builtin_amdgcn_exp2f(v.x - mm);
      l += w * v.y;
      coef[s + lane] = w;
    }
    l = fold64(l, SumOp());
    for (int s = 0; s < sh.y; s += 64) coef[s + lane] *= 1.f / l;
  }
  __syncthreads();
  const int e = (blockIdx.y * 64 + lane) * V;
  float acc[V] = {};
  if (e < a.R) {
    const long step = (long)a.H * a.R;
    const float* src = a.part + ((long)sh.x * a.H + h) * a.R + e;
#pragma unroll 8
    for (int s = wid; s < sh.y; s += 4) {
      const float c = coef[s];
#pragma unroll
      for (int j = 0; j < V; ++j) acc[j] += c * src[s * step + j];
    }
  }
#pragma unroll
  for (int j = 0; j < V; ++j) sum[wid][lane][j] = acc[j];
  __syncthreads();
  if (wid > 0 || e >= a.R) return;
  short* out = a.out + ((long)row * a.H + h) * a.R + e;
#pragma unroll
  for (int j = 0; j < V; ++j)
    acc[j] = sum[0][lane][j] + sum[1][lane][j] + sum[2][lane][j] + sum[3][lane][j];
#pragma unroll
  for (int j = 0; j < V; j += 2) *(uint*)(out + j) = pack_bf16x2(acc[j], acc[j + 1]);
}

static void launch_latent_merge(const LatentRowsArgs& a, hipStream_t stream) {
  // as many columns a lane as fill a wave (128 rows of 4000 keys, 32 heads, rank 512,
  // a whole step: 115 us in twos, 109 in fours)
  const dim3 grid(a.rows * a.H, a.R <= 128 ? 1 : (a.R + 255) / 256);
  if (a.R <= 128) latent_merge_kernel<2><<<grid, 256, 0, stream>>>(a);
  else latent_merge_kernel<4><<<grid, 256, 0, stream>>>(a);
}

// ---------------------------------------------------------------------------
// values: the shares of four rows of a head, every row by two waves, then the
// head's values of them (and their gate), whose weights are asked for first.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(512)
latent_values_kernel(LatentRowsArgs a, HeadLinearArgs l) {
  constexpr int RB = 4, XP = 512 + 8;    // rows; pitch of merged ones
  __shared__ __attribute__((aligned(16))) float other[4][512];
  __shared__ __attribute__((aligned(16))) short xs[16 * XP];
  __shared__ __attribute__((aligned(16))) float ys[4][2][256];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = wid >> 2;             // of the shares, of the columns
  const int c16 = lane & 15, grp = lane >> 4;
  const int h = blockIdx.x, r0 = blockIdx.y * RB, t = r0 + c16;
  const int R = a.R;
  // 32 outputs a wave, every other 32 columns.  16 rows of 64 bytes a load: as
  // 32 rows of two words each (32 x 32 products) the loads alone took 4 us.
  frag_u fw[2][8];
  s4v gate[2];
  auto weights = [&](int n) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const short* w = (const short*)l.w +
                       ((long)h * l.N + min(n + 16 * i + c16, l.N - 1)) * R;
#pragma unroll
      for (int b = 0; b < 8; ++b)
        fw[i][b].u4 = word_or_zero(w, 32 * (2 * b + part) + 8 * grp, R);
      if (l.gate)
        gate[i] = *(const s4v*)((const short*)l.gate + min(t, a.rows - 1) * l.gst +
                                h * l.gh + min(n + 16 * i + 4 * grp, l.N - 4));
    }
  };
  int n0 = (wid & 3) * 32;
  weights(n0);
  for (int i = threadIdx.x * 8; i < (16 - RB) * XP; i += 512 * 8)  // rows that
    *(uint4v*)(xs + RB * XP + i) = uint4v{0, 0, 0, 0};             //   are none
  const int e = lane * 8;
  const long step = (long)a.H * R;
  {
    const int rr = wid & 3, row = r0 + rr;
    f32x4 acc[2] = {};
    float inv = 0.f;
    if (row < a.rows) {
      const int2 sh = row_shares(a)[row];
      const float2* ml = share_totals(a) + (long)sh.x * a.H + h;
      const float* p = a.part + ((long)sh.x * a.H + h) * R + (e < R ? e : 0);
      auto total = [&](int s) {
        const float2 v = ml[(long)min(s + lane, sh.y - 1) * a.H];
        return s + lane < sh.y ? v : float2{NEG_BIG, 0.f};
      };
      float2 mine = total(0);
      float mm = mine.x, sum = 0.f;
      for (int s = 64; s < sh.y; s += 64) mm = fmaxf(mm, total(s).x);
      mm = fold64(mm, MaxOp());
      for (int b = 0; b < sh.y; b += 64) {
        if (b > 0) mine = total(b);
        const float w = __builtin_amdgcn_exp2f(mine.x - mm);
        sum += w * mine.y;
        const int end = min(64, sh.y - b);
        // eight of this wave's on their way at a time, also the last ones
        for (int s = part; s < end; s += 16) {
          f32x4 v[8][2];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const f32x4* src = (const f32x4*)(p + (b + min(s + 2 * i, end - 1)) * step);
            v[i][0] = src[0];
            v[i][1] = src[1];
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) {  // those past the end weigh nothing
            const float c = __uint_as_float(
                __builtin_amdgcn_readlane(__float_as_uint(w), (s + 2 * i) & 63));
            acc[0] += c * v[i][0];
            acc[1] += c * v[i][1];
          }
        }
      }
      sum = fold64(sum, SumOp());        // by all lanes
      inv = e < R ? 1.f / sum : 0.f;
    }
    f32x4* meet = (f32x4*)(other[wid & 3] + e);
    if (part) {
      meet[0] = acc[0];
      meet[1] = acc[1];
    }
    __syncthreads();
    if (!part) {
      acc[0] = (acc[0] + meet[0]) * inv;
      acc[1] = (acc[1] + meet[1]) * inv;
      const uint4v w = {pack_bf16x2(acc[0][0], acc[0][1]),
                        pack_bf16x2(acc[0][2], acc[0][3]),
                        pack_bf16x2(acc[1][0], acc[1][1]),
                        pack_bf16x2(acc[1][2], acc[1][3])};
      *(uint4v*)(xs + rr * XP + e) = w;  // zeros past R and past the last row
    }
    __syncthreads();
  }
  for (int n1 = 0; n1 < l.N; n1 += 128, n0 += 128) {
    if (n1 > 0) {
      __syncthreads();                   // ys has been read
      weights(n0);
    }
    f32x4 acc[2] = {};
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      frag_u fx;                         // zeros from R on
      fx.u4 = *(const uint4v*)(xs + c16 * XP + 32 * (2 * b + part) + 8 * grp);
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i] = mfma16(fw[i][b].bf, fx.bf, acc[i]);
    }
    if (part)
#pragma unroll
      for (int i = 0; i < 2; ++i) *(f32x4*)(ys[wid & 3][i] + lane * 4) = acc[i];
    __syncthreads();
    if (part || c16 >= RB || t >= a.rows) continue;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int n = n0 + 16 * i + 4 * grp;
      if (n + 3 >= l.N) continue;
      acc[i] += *(const f32x4*)(ys[wid & 3][i] + lane * 4);
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] = l.gate ? acc[i][j] * sigmoid_f(bits2f(gate[i][j])) : acc[i][j];
      store4((short*)l.out + t * l.ost + h * l.oh + n, v);
    }
  }
}

static int launch_latent_rows(const LatentRowsArgs* a, hipStream_t stream) {
  const long grid = (long)a->rows * ((a->H + 31) / 32) * a->splits;
  const bool full = a->P == 64 && (a->R == 64 || a->R == 128 || a->R == 256 ||
                                   a->R == 512);
#define LRK(E, F, O) latent_rows_kernel<E, F, O><<<grid, 256, 0, stream>>>(*a)
#define LR(E)                                           \
  do {                                                  \
    if (full && a->H <= 32) LRK(E, true, true);         \
    else if (full) LRK(E, true, false);                 \
    else LRK(E, false, false);                          \
  } while (0)
  if (a->P > 64 ||
      (a->splits > 1 && (long)a->rows * a->splits > LATENT_SHARES))
    return 1;
  if (a->R <= 64) LR(64);
  else if (a->R <= 128) LR(128);
  else if (a->R <= 256) LR(256);
  else if (a->R <= 512) LR(512);
  else return 1;
#undef LR
#undef LRK
  return 0;
}

// R and P multiples of 8, R <= 512, P <= 64, rows 16-byte aligned; with several
// splits at most LATENT_SHARES workgroups for a group of 32 heads
extern "C" int sv_latent_rows(const LatentRowsArgs* a, hipStream_t stream) {
  if (a->rows <= 0) return 0;
  if (launch_latent_rows(a, stream)) return 1;
  if (a->splits > 1)
    launch_latent_merge(*a, stream);
  return (int)hipGetLastError();
}

struct LatentStepArgs {
  LatentAppendArgs append;
  HeadLinearArgs absorb;
  LatentRowsArgs rows;
  HeadLinearArgs values;    // of rows.out
};

// A decoding step: append and absorb, attend, values.  As sv_latent_rows and the
// form on matrix cores of sv_head_linear.
extern "C" int sv_latent_step(const LatentStepArgs* a, hipStream_t stream) {
  const HeadLinearArgs& l = a->absorb;
  const int T = a->rows.rows;
  if (T <= 0) return 0;
  {
    const bool split = l.K >= 256;
    const int nt = (l.N + 31) / 32, nb = split ? nt : (nt + 3) / 4;
    const long grid = T + (long)nb * l.H * ((T + 31) / 32);
    const size_t lds = a->append.rot * sizeof(float);
#define LA(V, S) \
  latent_absorb_kernel<V, S><<<grid, 256, lds, stream>>>(a->append, l, T, nb)
    if (append_in_words(&a->append, 2)) { if (split) LA(true, true); else LA(true, false); }
    else { if (split) LA(false, true); else LA(false, false); }
#undef LA
  }
  if (launch_latent_rows(&a->rows, stream)) return 1;
  if (a->rows.splits == 1) return sv_head_linear(&a->values, 1, 0, stream);
  // The merge and the values in one launch read a head's weights for every four
  // rows, 16 rows of products of which four are used: only rows of many columns,
  // and one workgroup a CU or less, earn that (us of a step, in brackets in two
  // launches: 32 rows of 4096 keys, 32 heads, rank 512 47.4 (48.2); 11 of 363, 64
  // heads, rank 384 26.1 (27.0); but 5 of 4002, 40 heads, rank 448 33.5 (31.1), 92
  // of 829, 64 heads, rank 128 63.9 (37.3)).
  const int H = a->rows.H, groups = H * ((T + 3) / 4);
  if (a->rows.R > 256 && groups >= 128 && groups <= 256) {
    latent_values_kernel<<<dim3(H, (T + 3) / 4), 512, 0, stream>>>(a->rows, a->values);
  } else {
    launch_latent_merge(a->rows, stream);
    return sv_head_linear(&a->values, 1, 0, stream);
  }
  return (int)hipGetLastError();
}
