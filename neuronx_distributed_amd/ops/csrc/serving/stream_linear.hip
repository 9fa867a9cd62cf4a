// Products of a few rows with a large weight: out[t, n] = sum_k x[t, k] w[n, k].
// Decoding reads every weight once a step and multiplies it with a handful of
// rows, so the time is that of reading the weights.
//
//   sv_stream_linear   bf16 or 32-bit results; or silu(gate) * up of a weight
//                      whose first half of rows are gates, the second the
//                      projections that they multiply
//
// Bound by reading the weights: a read of 235 MB that multiplies nothing takes 36.0 us,
// of 34 MB 7.1, of which 1.7 are a launch.  Measured cold, us (library product, with
// the activation behind it | stream | stay | rings, x kept or flowing), which the rules
// of ops/serving.py follow:
//   28672 x 4096 gated   1 row 62 | - | 45 | 38.5   16 rows 63 | - | 47 | 39.4   32: 51 | - | 52 | 41.1
//   32000 x 4096, 32 bit 1 row 59 | 43 | 48 | 42.5  16 rows 59 | 62 | 52 | 43.3  32: 58 | 93 | 55 | 46.4
//   6144 x 4096          1 row 14 | 12 | 16 | 11.1  16 rows 16 | 17 | 18 | 11.5  32: 16 | 25 | 21 | 13.7
//   4096 x 4096          1 row 15 | 7.7 | 12 | 7.7  16 rows 15 | 10 | 14 | 8.5   32: 14 | 14 | 18 | 11.1
//   4096 x 14336         1 row 27 | 23 | - | 21     16 rows 27 | 32 | - | 25     32: 34 | 43 | - | 33
// A gated product of a normed row: 43.3 us staying, 37.5 through a ring.
// Rings are the faster ones for three reasons, measured by reads alone: loads of whole
// lines (64 of 128 bytes a load: 5.6 TB/s of 235 MB, 128: 6.0), lines that no cache
// keeps (6.5; with halves of a line it reads them twice, 5.5), and as many of them on
// their way as LDS holds instead of registers.
// 64 KB a CU are enough: twice as many cost small weights 10 %.

#include "serving.h"
#include "ring.h"
#include "words.h"

struct StreamArgs {
  const short* x;           // [T] rows of K
  long xst;
  const short* w;           // [N] rows of K
  long wst;
  void* out;                // [T][N], or [T][N / 2] with GLU
  int T, N, K;
  // instead of x, one row: that of the 32-bit residual (or null: zero) plus
  // `delta`, normed; or without residual a row of the table delta
  const float* res;
  const short* delta;
  float* res_out;           // their sum
  const short* weight;
  float eps;
  const int* row;           // which, or null
  long rows;
};

enum Epilogue { PLAIN = 0, F32 = 1, GLU = 2 };

// Accumulator rows are weight rows 4 grp + 0..3, columns rows of x: the results
// of weight rows n ... of row t.  u: what the gates v multiply.
template <int EPI>
__device__ __forceinline__ void store_rows(const StreamArgs& a, int t, int n, int n1,
                                           f32x4 v, f32x4 u) {
  const int N = EPI == GLU ? a.N / 2 : a.N;
  if (t >= a.T || n >= n1) return;
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
  const short* delta = a.delta + at;
  if (a.row) delta += min(max((long)a.row[0], 0L), a.rows - 1) * a.K;
#pragma unroll
  for (int k = 0; k < V / 4; ++k) {
    v[k] = a.res ? *(const f32x4*)(a.res + at + 4 * k) : f32x4{};
    d[k] = *(const s4v*)(delta + 4 * k);
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
  lds_barrier();
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
  lds_barrier();
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
  store_rows<EPI>(a, t0 + wid * 16 + c16, n0 + 4 * grp, a.N, v, v);
}

// For weights of many rows: a workgroup stays and takes every so many tiles of
// 16 weight rows (or 16 gates and their projections).  Each of its NW waves
// keeps its 256 PARTS columns of x in registers and reads the same columns of
// one tile after the other, 256 at a time, one such part ahead.
// Words past K are zeros behind a branch each, and a product waits for all loads on
// their way (zeros made of words that are read in any case do not fit the registers):
// whole blocks of 64 columns come through rings instead.
// NORM: of the normed row.
template <int NW, int PARTS, int MT, int EPI, bool NORM>
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
    return k0 + k < a.K ? *(const uint4v*)(from + k0 + k)
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
    store_rows<EPI>(a, wid * 16 + c16, tile * 16 + 4 * grp, EPI == GLU ? a.N / 2 : a.N, v, u);
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

// Weights through rings: a workgroup takes tiles of 16 weight rows (8 gates and their
// projections), and of what is left over an even share in 8 rows, so that no CU has
// much more than another; each of its 8 waves takes its columns of the tile, 64 at a
// time.  Neighbours take neighbouring tiles: where each had its rows in one piece, all
// read at the same distance, and some distances meet few channels (22016 x 3072: 31
// us, now 24).
template <int R, int EPI>
struct Tiles {
  static constexpr int NW = 8, TR = EPI == GLU ? 8 : 16, UT = TR / 8;
  Ring<R> ring;
  int rows, full, u0, u1, tiles;         // whole tiles, then units of 8 rows of the last
  int first, nb;                         // the wave's blocks of 64 columns
  __amdgpu_buffer_rsrc_t ra, rb;
  int oa, ob, pitch;
  int tile, begin, blk;                  // what is asked for next
  uint ta, tb;

  __device__ __forceinline__ Tiles(const StreamArgs& a, char* lds, int wid,
                                   int rotate = 0)
      : ring(lds + wid * R * 1024) {
    rows = EPI == GLU ? a.N / 2 : a.N;
    const int units = (rows + 7) / 8, G = gridDim.x, b = blockIdx.x;
    full = units / (UT * G);
    const int rest = units - full * UT * G;
    u0 = rest * b / G + full * UT * G;
    u1 = rest * (b + 1) / G + full * UT * G;
    tiles = full + (u1 > u0);
    const int blocks = a.K / 64;
    first = blocks * wid / NW;
    nb = blocks * (wid + 1) / NW - first;
    pitch = (int)a.wst * 2;
    const int end = (rows - 1) * pitch + a.K * 2;
    ra = ring_source(a.w, end);
    rb = ring_source(EPI == GLU ? a.w + rows * a.wst : a.w, end);
    oa = Ring<R>::lane_bytes(pitch, 0) + first * 128;
    ob = Ring<R>::lane_bytes(pitch, 1) + first * 128 + (EPI == GLU ? 0 : 8 * pitch);
    tile = 0;
    blk = begin = rotate ? blockIdx.x / rotate % nb : 0;
    locate();
  }
  // first row of a tile, and past its last one
  __device__ __forceinline__ int row0(int t) const {
    return t < full ? (t * (int)gridDim.x + (int)blockIdx.x) * TR : 8 * u0;
  }
  __device__ __forceinline__ int row1(int t) const {
    return min(rows, t < full ? row0(t) + TR : 8 * u1);
  }
  __device__ __forceinline__ void locate() {
    ta = tile < tiles ? (uint)row0(tile) * pitch : RING_NOWHERE;
    tb = EPI != GLU && tile == full && u1 - u0 < 2 ? RING_NOWHERE : ta;
  }
  __device__ __forceinline__ void ask() {
    ring.ask(ra, oa + ta + blk * 128, rb, ob + tb + blk * 128);
    if (++blk == nb) blk = 0;
    if (blk == begin) {
      ++tile;
      locate();
    }
  }
};

// the sums of a tile's waves meet; the first waves add them up
template <int MT, int EPI>
__device__ __forceinline__ void meet(const StreamArgs& a, f32x4 (*part)[MT][64],
                                     const f32x4* acc, int wid, int n, int n1) {
  constexpr int NW = 8;
  const int lane = threadIdx.x & 63, c16 = lane & 15, grp = lane >> 4;
#pragma unroll
  for (int j = 0; j < MT; ++j) part[wid][j][lane] = acc[j];
  lds_barrier();
  if (wid >= MT) return;
  f32x4 v = {}, p[NW], u;
#pragma unroll
  for (int s = 0; s < NW; ++s) p[s] = part[s][wid][lane];
#pragma unroll
  for (int s = 0; s < NW; ++s) v += p[s];
  if (EPI == GLU)
#pragma unroll
    for (int r = 0; r < 4; ++r) u[r] = __shfl_xor(v[r], 32, 64);
  if (EPI != GLU || grp < 2) store_rows<EPI>(a, wid * 16 + c16, n + 4 * grp, n1, v, u);
}

// this lane's words of rows 16 j on, to be turned
__device__ __forceinline__ const short* row_words(const StreamArgs& a, int j) {
  const int lane = threadIdx.x & 63;
  return a.x + (long)min(j * 16 + (lane >> 2), a.T - 1) * a.xst + (lane & 3) * 8;
}

// The wave's columns of x stay in registers, at most CB blocks of 64.
template <int CB, int MT, int EPI>
__global__ void __launch_bounds__(512) ring_linear_kernel(StreamArgs a) {
  constexpr int R = 8;
  __shared__ __attribute__((aligned(1024))) char ring[8 * R * 1024];
  __shared__ f32x4 part[2][8][MT][64];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Tiles<R, EPI> w(a, ring, wid);
  const int nb = w.nb;
  frag_u fx[CB * 2][MT];
#pragma unroll
  for (int i = 0; i < R / 2; ++i) w.ask();
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const short* x = row_words(a, j) + w.first * 64;
#pragma unroll
    for (int c = 0; c < CB * 2; ++c)     // blocks past the wave's are not used
      fx[c][j].u4 = *(const uint4v*)(x + (c < 2 * nb ? c * 32 : 0));
  }
#pragma unroll
  for (int c = 0; c < CB * 2; ++c)
#pragma unroll
    for (int j = 0; j < MT; ++j) fx[c][j] = turned(fx[c][j]);
  // x, and the ring is full: from here on only pieces (and results) are on their way
  __builtin_amdgcn_s_waitcnt(0x0070);
  for (int t = 0; t < w.tiles; ++t) {
    f32x4 acc[MT] = {};
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      if (c >= nb) continue;
      frag_u f0, f1;
      w.ring.template take<R - 2>(f0, f1);
      w.ask();
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        acc[j] = mfma16(f0.bf, fx[2 * c][j].bf, acc[j]);
        acc[j] = mfma16(f1.bf, fx[2 * c + 1][j].bf, acc[j]);
      }
    }
    meet<MT, EPI>(a, part[t & 1], acc, wid, w.row0(t), w.row1(t));
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // LDS is given back
}

// x flows like the weights, a ring ahead: for few rows, where it is little, and for a
// workgroup's only tile, where there is nothing to keep.  Workgroups of an XCD begin at
// different blocks, so that they do not all ask the same channels of its L2 for x
// (16 rows of 14336: 26.9 us in one order, 23.8).
// NORM: of the normed row, in LDS.
template <int MT, int EPI, bool NORM>
__global__ void __launch_bounds__(512) flow_linear_kernel(StreamArgs a) {
  constexpr int D = 4, R = 2 * D;        // blocks ahead
  __shared__ __attribute__((aligned(1024))) char ring[8 * R * 1024];
  __shared__ f32x4 part[2][8][MT][64];
  __shared__ __attribute__((aligned(16))) short row[NORM ? 4096 : 8];
  __shared__ float red[NORM ? 16 : 1];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Tiles<R, EPI> w(a, ring, wid, 8);
  const int nb = w.nb;
  frag_u fx[D][2][MT];
  const short* x[MT];
  if (!NORM)
#pragma unroll
    for (int j = 0; j < MT; ++j) x[j] = row_words(a, j) + w.first * 64;
  // pieces and words of the wave's next block
  auto ask = [&](int i) __attribute__((always_inline)) {
    if (!NORM) {
      const int k = w.blk * 64;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          fx[i][h][j].u4 = *(const uint4v*)(x[j] + k + h * 32);
    }
    w.ask();
    __builtin_amdgcn_sched_barrier(0);
  };
  int rb = w.begin;                      // block that is multiplied next
  auto fill = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < D; ++i) ask(i);
  };
  if (NORM) norm_row<512>(a, row, red, fill);
  else fill();
  f32x4 acc[MT] = {};
  int c = 0, t = 0;
  const int total = w.tiles * nb;
  for (int s = 0; s < total; s += D) {
#pragma unroll
    for (int i = 0; i < D; ++i) {
      frag_u f0, f1;
      w.ring.template take<(D - 1) * (NORM ? 2 : 2 * MT + 2)>(f0, f1);
      if (NORM) {
        const short* at = row + (w.first + rb) * 64 + ((threadIdx.x & 63) >> 4) * 8;
        fx[i][0][0].u4 = *(const uint4v*)at;
        fx[i][1][0].u4 = *(const uint4v*)(at + 32);
        if (++rb == nb) rb = 0;
      }
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        acc[j] = mfma16(f0.bf, (NORM ? fx[i][0][j] : turned(fx[i][0][j])).bf, acc[j]);
        acc[j] = mfma16(f1.bf, (NORM ? fx[i][1][j] : turned(fx[i][1][j])).bf, acc[j]);
      }
      ask(i);
      if (++c == nb && t < w.tiles) {    // past the last tile nothing counts
        meet<MT, EPI>(a, part[t & 1], acc, wid, w.row0(t), w.row1(t));
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[j] = f32x4{};
        c = 0;
        ++t;
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // LDS is given back
}

template <int EPI, bool NORM = false>
static int launch_ring(const StreamArgs& a, int how, hipStream_t stream) {
  // every wave has a block, all offsets are bytes of 31 bits
  if (a.K % 64 || a.K < 512 || a.wst * 2 * (a.N + 16L) >= 1L << 31 || a.T > 32 ||
      (EPI == GLU && a.N % 8))
    return 1;
  const int units = ((EPI == GLU ? a.N / 2 : a.N) + 7) / 8;
  const int grid = min(units, 256), blocks = (a.K / 64 + 7) / 8;
#define RING(C, M) ring_linear_kernel<C, M, EPI><<<grid, 512, 0, stream>>>(a)
#define FLOW(M) flow_linear_kernel<M, EPI, NORM><<<grid, 512, 0, stream>>>(a)
  if constexpr (NORM) {
    FLOW(1);
  } else if (how == 3) {
    if (a.T <= 16) FLOW(1); else FLOW(2);
  } else {                               // at most 128 registers of x
    if (a.T <= 16 && blocks <= 8) RING(8, 1);
    else if (a.T <= 16 && blocks <= 16) RING(16, 1);
    else if (blocks <= 8) RING(8, 2);
    else return 1;
  }
#undef RING
#undef FLOW
  return (int)hipGetLastError();
}

template <int EPI, bool NORM = false>
static int launch(const StreamArgs& a, int stay, hipStream_t stream) {
  constexpr int rows = EPI == GLU ? 32 : 16;
  const int tiles = (a.N + rows - 1) / rows;
  if (stay) {
    if (a.N % rows) return 1;
    const int grid = min(tiles, 256);
    // at most 128 registers of x beside the weights; for a K that is not whole blocks
    // of 64, and sizes that the rings leave (plain products of 17 to 32 rows by a direct
    // call alone, here and below)
#define STAY(P, M) \
  stay_linear_kernel<8, P, M, EPI, NORM><<<grid, 512, 0, stream>>>(a)
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

// how: 0 stream, 1 stay, 2 and 3 rings (K in blocks of 64, at least 512; 2: at most
// 8192 columns of 16 rows or 4096 of 32).  K, strides and bases in 8 elements; GLU
// not 0, on whole tiles
extern "C" int sv_stream_linear(const StreamArgs* a, int epilogue, int how,
                                hipStream_t stream) {
  if (a->T <= 0 || a->N <= 0) return 0;
  if (a->K % 8) return 1;
  if (a->weight && (a->T != 1 || a->K > 4096 || epilogue == F32)) return 1;
#define TAKE(E, ...)                                              \
  (how >= 2 ? launch_ring<E, ##__VA_ARGS__>(*a, how, stream)      \
            : launch<E, ##__VA_ARGS__>(*a, how, stream))
  if (a->weight) return epilogue == GLU ? TAKE(GLU, true) : TAKE(PLAIN, true);
  return epilogue == GLU   ? TAKE(GLU)
         : epilogue == F32 ? TAKE(F32)
                           : TAKE(PLAIN);
#undef TAKE
}
