// Products of a few rows with a large weight: out[t, n] = sum_k x[t, k] w[n, k].
// Decoding reads every weight once a step and multiplies it with a handful of
// rows, so the time is that of reading the weights.
//
//   sv_stream_linear   bf16 or 32-bit results; or silu(gate) * up of a weight
//                      whose first half of rows are gates, the second the
//                      projections that they multiply
//
// Measured cold, us (library product, with the activation behind it | stream |
// stay), which the rule of ops/serving.py follows:
//   28672 x 4096 gated   1 row 66 | 46 | 44   16 rows 68 | 71 | 47   32: 60 | - | 51
//   28672 x 4096         1 row 63 | 40 | 46    4 rows 64 | 43 | 46   16: 65 | 60 | 49
//   32000 x 4096, 32 bit 1 row 59 | 42 | 48    4 rows 60 | 45 | 48   16: 60 | 64 | 51
//   4096 x 14336         1 row 27 | 22 | -     4 rows 27 | 23 | -
//   4096 x 4096          1 row 14 | 7.5 | 12  16 rows 14 | 10 | 14   32: 13 | 14 | 17
// One row reads 4.1 (with its norm) to 6.4 TB/s of weights, a copy 5.1.  With a branch a load every
// product waited for all loads on their way: 8.5, 23 and 45 us where one row of
// 4096 x 4096, 4096 x 14336 and 28672 gated columns now take 7.5, 22 and 43.5.

#include "serving.h"
#include "words.h"

struct StreamArgs {
  const short* x;           // [T] rows of K
  long xst;
  const short* w;           // [N] rows of K
  long wst;
  void* out;                // [T][N], or [T][N / 2] with GLU
  int T, N, K;
  // instead of x, one row: that of the 32-bit residual (or null: zero) plus
  // `delta`, normed
  const float* res;
  const short* delta;
  float* res_out;           // their sum
  const short* weight;
  float eps;
};

enum Epilogue { PLAIN = 0, F32 = 1, GLU = 2 };

// Accumulator rows are weight rows 4 grp + 0..3, columns rows of x: the results
// of weight rows n ... of row t.  u: what the gates v multiply.
template <int EPI>
__device__ __forceinline__ void store_rows(const StreamArgs& a, int t, int n,
                                           f32x4 v, f32x4 u) {
  const int N = EPI == GLU ? a.N / 2 : a.N;
  if (t >= a.T || n >= N) return;
  if (EPI == GLU)
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = silu_f(v[r]) * u[r];
  if (EPI != GLU && N % 4) {             // no 4 results in a word
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < N) {
        if (EPI == F32) ((float*)a.out)[(long)t * N + n + r] = v[r];
        else ((short*)a.out)[(long)t * N + n + r] = f2bits(v[r]);
      }
    return;
  }
  if (EPI == F32)
    *(f32x4*)((float*)a.out + (long)t * N + n) = v;
  else
    *(uint2*)((short*)a.out + (long)t * N + n) =
        uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

// Words past a row are read as its first ones, and become zeros where they are
// multiplied: a branch a load, or a select behind it, would make every product
// wait for the loads of the next turn.
__device__ __forceinline__ bf16x8 if_there(bool in, frag_u f) {
  if (!in) f.u4 = uint4v{0, 0, 0, 0};
  return f.bf;
}

// The normed row, in LDS, by NT threads.  Every workgroup makes it for itself while
// its first weights are on their way: 32 KB from L2 a workgroup, but no launch
// before this one that all would wait for, and no memory that is idle meanwhile (4
// layers of 4096, one request, 16 steps: 8120 -> 7800 us).  `ask` asks for those weights, behind the
// words of the row, so that these are not waited for with them.  K is at most 4096;
// elements past it are zeros.
template <int NT, typename Ask>
__device__ __forceinline__ void norm_row(const StreamArgs& a, short* row,
                                         float* red, Ask&& ask) {
  constexpr int V = 4096 / NT;           // 4 or 8 elements of a thread
  const int tid = threadIdx.x, i = tid * V, at = min(i, a.K - V);
  f32x4 v[V / 4];
  s4v d[V / 4], u[V / 4];
#pragma unroll
  for (int k = 0; k < V / 4; ++k) {
    v[k] = a.res ? *(const f32x4*)(a.res + at + 4 * k) : f32x4{};
    d[k] = *(const s4v*)(a.delta + at + 4 * k);
    u[k] = *(const s4v*)(a.weight + at + 4 * k);
  }
  __builtin_amdgcn_sched_barrier(0);
  ask();
  __builtin_amdgcn_sched_barrier(0);
  float sq = 0.f;
#pragma unroll
  for (int k = 0; k < V / 4; ++k) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[k][j] += bits2f(d[k][j]);
      sq += i < a.K ? v[k][j] * v[k][j] : 0.f;
    }
    if (blockIdx.x == 0 && i < a.K) *(f32x4*)(a.res_out + i + 4 * k) = v[k];
  }
  sq = fold64(sq, SumOp());
  if ((tid & 63) == 0) red[tid >> 6] = sq;
  __syncthreads();
  float all = 0.f;
#pragma unroll
  for (int k = 0; k < NT / 64; ++k) all += red[k];
  const float rstd = 1.f / sqrtf(all / a.K + a.eps);
#pragma unroll
  for (int k = 0; k < V / 4; ++k) {
    float y[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      y[j] = i < a.K ? v[k][j] * (rstd * bits2f(u[k][j])) : 0.f;
    store4(row + i + 4 * k, y);
  }
  __syncthreads();
}

// One workgroup = 16 weight rows by MT tiles of 16 rows of x; its 16 waves take
// K in turns of 64 columns and meet in LDS.  Weights go from memory straight into registers as fragments (a lane's
// 16 bytes of a row, 64 bytes of 16 rows a load), a turn ahead.  Every workgroup
// reads all of x, as much as its weights at 16 rows.
// FULL: K is a multiple of 64.  NORM: of the normed row.
template <int MT, int EPI, bool FULL, bool NORM>
__global__ void __launch_bounds__(1024) stream_linear_kernel(StreamArgs a) {
  constexpr int U = 2, STEP = 16 * U * 32;
  __shared__ f32x4 part[16][MT][64];
  __shared__ __attribute__((aligned(16))) short row[NORM ? 4096 : 8];
  __shared__ float red[NORM ? 16 : 1];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, grp = lane >> 4;
  const int K = a.K;
  const int n0 = blockIdx.x * 16, t0 = blockIdx.y * 16 * MT;

  // words of column k on are at column(k)
  const int from = FULL ? grp * 8 : 0;
  auto column = [&](int k) __attribute__((always_inline)) {
    return FULL ? k : word_column(k, grp, K);
  };
  const short* w = a.w + (long)min(n0 + c16, a.N - 1) * a.wst + from;
  const short* x[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
    x[i] = NORM ? row + from
                : a.x + (long)min(t0 + i * 16 + c16, a.T - 1) * a.xst + from;

  f32x4 acc[MT] = {};
  auto load_w = [&](int k0, frag_u* fw) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      fw[u].u4 = *(const uint4v*)(w + column(k0 + u * 32));
  };
  auto load_x = [&](int k0, frag_u (*fx)[MT]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int at = column(k0 + u * 32);
#pragma unroll
      for (int i = 0; i < MT; ++i)
        fx[u][i].u4 = *(const uint4v*)(x[i] + at);
    }
  };
  auto load = [&](int k0, frag_u* fw, frag_u (*fx)[MT])
      __attribute__((always_inline)) {
    load_w(k0, fw);
    load_x(k0, fx);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto multiply = [&](int k0, const frag_u* fw, const frag_u (*fx)[MT])
      __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = FULL || k0 + u * 32 + grp * 8 < K;
#pragma unroll
      for (int j = 0; j < MT; ++j)
        acc[j] = mfma16(if_there(in, fw[u]), if_there(in, fx[u][j]), acc[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  frag_u wa[U], xa[U][MT], wb[U], xb[U][MT];
  int k = wid * U * 32;
  if (NORM)
    norm_row<1024>(a, row, red, [&]() __attribute__((always_inline)) {
      load_w(min(k, (K - 1) / 64 * 64), wa);
    });
  if (k < K) {
    if (NORM) load_x(k, xa);
    else load(k, wa, xa);
    // The last turns have no load behind them, in code of their own: where both
    // ways join, a product would wait as for the shorter one.
    for (; k + 2 * STEP < K; k += 2 * STEP) {
      load(k + STEP, wb, xb);
      multiply(k, wa, xa);
      load(k + 2 * STEP, wa, xa);
      multiply(k + STEP, wb, xb);
    }
    if (k + STEP < K) {
      load(k + STEP, wb, xb);
      multiply(k, wa, xa);
      multiply(k + STEP, wb, xb);
    } else {
      multiply(k, wa, xa);
    }
  }
#pragma unroll
  for (int j = 0; j < MT; ++j) part[wid][j][lane] = acc[j];
  __syncthreads();
  if (wid >= MT) return;
  f32x4 v = {}, y[16];
#pragma unroll
  for (int s = 0; s < 16; ++s) y[s] = part[s][wid][lane];
#pragma unroll
  for (int s = 0; s < 16; ++s) v += y[s];
  store_rows<EPI>(a, t0 + wid * 16 + c16, n0 + 4 * grp, v, v);
}

// For weights of many rows: a workgroup stays and takes every so many tiles of
// 16 weight rows (or 16 gates and their projections).  Each of its NW waves
// keeps its 256 PARTS columns of x in registers and reads the same columns of
// one tile after the other, 256 at a time, one such part ahead.
// FULL: K is what they hold.  Otherwise words past it are zeros behind a branch
// each, and a product waits for all loads on their way (zeros made of words that
// are read in any case do not fit the registers).
// NORM: of the normed row.
template <int NW, int PARTS, int MT, int EPI, bool FULL, bool NORM>
__global__ void __launch_bounds__(NW * 64) stay_linear_kernel(StreamArgs a) {
  constexpr int RT = EPI == GLU ? 2 : 1;
  constexpr int UNITS = RT * PARTS;      // parts of a tile
  __shared__ f32x4 part[2][NW][RT * MT][64];
  __shared__ __attribute__((aligned(16))) short row[NORM ? 4096 : 8];
  __shared__ float red[NORM ? 16 : 1];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, grp = lane >> 4;
  const int tiles = a.N / (16 * RT), step = gridDim.x;
  const int k0 = wid * PARTS * 256 + grp * 8;
  auto word = [&](const short* from, int k) __attribute__((always_inline)) {
    return FULL || k0 + k < a.K ? *(const uint4v*)(from + k0 + k)
                                : uint4v{0, 0, 0, 0};
  };

  frag_u fx[PARTS * 8][MT];
  if (!NORM)
#pragma unroll
    for (int c = 0; c < PARTS * 8; ++c)
#pragma unroll
      for (int j = 0; j < MT; ++j)
        fx[c][j].u4 = word(a.x + (long)min(j * 16 + c16, a.T - 1) * a.xst, c * 32);
  const short* w = a.w + (long)c16 * a.wst;
  // unit u of a tile; past the last tile that one again, and not used
  auto load = [&](int tile, int u, frag_u* fw) __attribute__((always_inline)) {
    const int p = u % PARTS;
    const short* src = w +
        (long)(min(tile, tiles - 1) * 16 + (u / PARTS ? a.N / 2 : 0)) * a.wst;
#pragma unroll
    for (int c = 0; c < 8; ++c)
      fw[c].u4 = word(src, p * 256 + c * 32);
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4 acc[MT];
  auto multiply = [&](int u, const frag_u* fw, int buf)
      __attribute__((always_inline)) {
    const int p = u % PARTS;
    if (p == 0)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[j] = f32x4{};
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int j = 0; j < MT; ++j)
        acc[j] = mfma16(fw[c].bf, fx[p * 8 + c][j].bf, acc[j]);
    __builtin_amdgcn_sched_barrier(0);
    if (p == PARTS - 1)
#pragma unroll
      for (int j = 0; j < MT; ++j)
        part[buf][wid][u / PARTS * MT + j][lane] = acc[j];
  };
  // the first waves add up the sums of all; the others go on
  auto finish = [&](int tile, int buf) __attribute__((always_inline)) {
    __syncthreads();
    if (wid >= MT) return;
    f32x4 v = {}, u = {};
    auto sum = [&](int row, f32x4& to) __attribute__((always_inline)) {
      f32x4 y[NW];
#pragma unroll
      for (int s = 0; s < NW; ++s) y[s] = part[buf][s][row][lane];
#pragma unroll
      for (int s = 0; s < NW; ++s) to += y[s];
    };
    sum(wid, v);
    if (EPI == GLU) sum(MT + wid, u);
    store_rows<EPI>(a, wid * 16 + c16, tile * 16 + 4 * grp, v, u);
  };

  frag_u wa[8], wb[8];
  int tile = blockIdx.x;
  auto first = [&]() __attribute__((always_inline)) {
    load(tile, 0, wa);
    load(tile, 1, wb);
  };
  if (NORM) {
    norm_row<NW * 64>(a, row, red, first);
#pragma unroll
    for (int c = 0; c < PARTS * 8; ++c)
#pragma unroll
      for (int j = 0; j < MT; ++j)       // zeros past K
        fx[c][j].u4 = *(const uint4v*)(row + k0 + c * 32);
  } else {
    first();
  }
  for (int buf = 0; tile < tiles; tile += step, buf ^= 1) {
#pragma unroll
    for (int u = 0; u < UNITS; u += 2) {
      const bool last = u + 2 == UNITS;
      multiply(u, wa, buf);
      load(last ? tile + step : tile, last ? 0 : u + 2, wa);
      multiply(u + 1, wb, buf);
      load(last ? tile + step : tile, last ? 1 : u + 3, wb);
    }
    finish(tile, buf);
  }
}

template <int EPI, bool NORM = false>
static int launch(const StreamArgs& a, int stay, hipStream_t stream) {
  constexpr int rows = EPI == GLU ? 32 : 16;
  const int tiles = (a.N + rows - 1) / rows;
  if (stay) {
    if (a.N % rows) return 1;
    const int grid = min(tiles, 256);
    // at most 128 registers of x beside the weights (plain products of 17 to
    // 32 rows by a direct call alone, here and below: the library is faster)
#define STAY(P, M)                                                          \
  do {                                                                      \
    if (a.K == 2048 * P)                                                    \
      stay_linear_kernel<8, P, M, EPI, true, NORM>                          \
          <<<grid, 512, 0, stream>>>(a);                                    \
    else                                                                    \
      stay_linear_kernel<8, P, M, EPI, false, NORM>                         \
          <<<grid, 512, 0, stream>>>(a);                                    \
  } while (0)
    if constexpr (NORM) STAY(2, 1);
    else if (a.T <= 16 && a.K <= 4096) STAY(2, 1);
    else if (a.T <= 16 && a.K <= 8192) STAY(4, 1);
    else if (a.T <= 32 && a.K <= 4096) STAY(2, 2);
    else return 1;
#undef STAY
  } else {
    if constexpr (EPI == GLU) return 1;
    else {
      const bool full = a.K % 64 == 0;
      const dim3 grid(tiles, a.T <= 16 ? 1 : (a.T + 31) / 32);
#define STREAM(M, F) \
  stream_linear_kernel<M, EPI, F, NORM><<<grid, 1024, 0, stream>>>(a)
      if constexpr (NORM) { if (full) STREAM(1, true); else STREAM(1, false); }
      else if (a.T <= 16) { if (full) STREAM(1, true); else STREAM(1, false); }
      else { if (full) STREAM(2, true); else STREAM(2, false); }
#undef STREAM
    }
  }
  return (int)hipGetLastError();
}

// K, strides and bases in 8 elements; GLU stays, on whole tiles
extern "C" int sv_stream_linear(const StreamArgs* a, int epilogue, int stay,
                                hipStream_t stream) {
  if (a->T <= 0 || a->N <= 0) return 0;
  if (a->K % 8) return 1;
  if (a->weight) {
    if (a->T != 1 || a->K > 4096 || epilogue == F32) return 1;
    return epilogue == GLU ? launch<GLU, true>(*a, stay, stream)
                           : launch<PLAIN, true>(*a, stay, stream);
  }
  return epilogue == GLU   ? launch<GLU>(*a, stay, stream)
         : epilogue == F32 ? launch<F32>(*a, stay, stream)
                           : launch<PLAIN>(*a, stay, stream);
}
