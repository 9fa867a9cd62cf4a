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
//   28672 x 4096 gated   1 row 66 | 46 | 45   16 rows 68 | 71 | 48   32: 60 | - | 53
//   28672 x 4096         1 row 63 | 41 | 46    4 rows 64 | 45 | 46   16: 65 | 66 | 50
//   32000 x 4096, 32 bit 1 row 59 | 45 | 50    4 rows 60 | 49 | 51   16: 60 | 72 | 53
//   4096 x 14336         1 row 27 | 25 | -     4 rows 27 | 27 | -
//   4096 x 4096          1 row 15 |  9 | 12   16 rows 15 | 12 | 14   32: 13 | 16 | 18
// One row reads 5.2 to 5.7 TB/s of weights, a copy 5.2.

#include "serving.h"

struct StreamArgs {
  const short* x;           // [T] rows of K
  long xst;
  const short* w;           // [N] rows of K
  long wst;
  void* out;                // [T][N], or [T][N / 2] with GLU
  int T, N, K;
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

// One workgroup = 16 weight rows by MT tiles of 16 rows of x; its 16 waves take
// K in turns of 64 columns and meet in LDS.  Weights go from memory straight into registers as fragments (a lane's
// 16 bytes of a row, 64 bytes of 16 rows a load), a turn ahead.  Every workgroup
// reads all of x, as much as its weights at 16 rows.
template <int MT, int EPI>
__global__ void __launch_bounds__(1024) stream_linear_kernel(StreamArgs a) {
  constexpr int U = 2, STEP = 16 * U * 32;
  __shared__ f32x4 part[16][MT][64];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, grp = lane >> 4;
  const int K = a.K;
  const int n0 = blockIdx.x * 16, t0 = blockIdx.y * 16 * MT;

  const short* w = a.w + (long)min(n0 + c16, a.N - 1) * a.wst + grp * 8;
  const short* x[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
    x[i] = a.x + (long)min(t0 + i * 16 + c16, a.T - 1) * a.xst + grp * 8;

  f32x4 acc[MT] = {};
  const uint4v zero = {0, 0, 0, 0};
  auto load = [&](int k0, frag_u* fw, frag_u (*fx)[MT])
      __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * 32;
      const bool in = k + grp * 8 < K;
      fw[u].u4 = in ? *(const uint4v*)(w + k) : zero;
#pragma unroll
      for (int i = 0; i < MT; ++i)
        fx[u][i].u4 = in ? *(const uint4v*)(x[i] + k) : zero;
    }
  };
  auto multiply = [&](const frag_u* fw, const frag_u (*fx)[MT])
      __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < MT; ++j)
        acc[j] = mfma16(fw[u].bf, fx[u][j].bf, acc[j]);
  };
  frag_u wa[U], xa[U][MT], wb[U], xb[U][MT];
  int k = wid * U * 32;
  if (k < K) load(k, wa, xa);
  for (; k < K; k += 2 * STEP) {
    if (k + STEP < K) load(k + STEP, wb, xb);
    multiply(wa, xa);
    if (k + STEP >= K) break;
    if (k + 2 * STEP < K) load(k + 2 * STEP, wa, xa);
    multiply(wb, xb);
  }
#pragma unroll
  for (int j = 0; j < MT; ++j) part[wid][j][lane] = acc[j];
  __syncthreads();
  if (wid >= MT) return;
  f32x4 v = {};
#pragma unroll
  for (int s = 0; s < 16; ++s) v += part[s][wid][lane];
  store_rows<EPI>(a, t0 + wid * 16 + c16, n0 + 4 * grp, v, v);
}

// For weights of many rows: a workgroup stays and takes every so many tiles of
// 16 weight rows (or 16 gates and their projections).  Each of its NW waves
// keeps its 256 PARTS columns of x in registers and reads the same columns of
// one tile after the other, 256 at a time, one such part ahead.
template <int NW, int PARTS, int MT, int EPI>
__global__ void __launch_bounds__(NW * 64) stay_linear_kernel(StreamArgs a) {
  constexpr int RT = EPI == GLU ? 2 : 1;
  constexpr int UNITS = RT * PARTS;      // parts of a tile
  __shared__ f32x4 part[2][NW][RT * MT][64];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, grp = lane >> 4;
  const int tiles = a.N / (16 * RT), step = gridDim.x;
  const int k0 = wid * PARTS * 256 + grp * 8;
  const uint4v zero = {0, 0, 0, 0};

  frag_u fx[PARTS * 8][MT];
#pragma unroll
  for (int c = 0; c < PARTS * 8; ++c)
#pragma unroll
    for (int j = 0; j < MT; ++j)
      fx[c][j].u4 = k0 + c * 32 < a.K
          ? *(const uint4v*)(a.x + (long)min(j * 16 + c16, a.T - 1) * a.xst +
                             k0 + c * 32)
          : zero;
  const short* w = a.w + (long)c16 * a.wst + k0;
  // unit u of a tile; past the last tile that one again, and not used
  auto load = [&](int tile, int u, frag_u* fw) __attribute__((always_inline)) {
    const int p = u % PARTS;
    const short* src = w + p * 256 +
        (long)(min(tile, tiles - 1) * 16 + (u / PARTS ? a.N / 2 : 0)) * a.wst;
#pragma unroll
    for (int c = 0; c < 8; ++c)
      fw[c].u4 = k0 + p * 256 + c * 32 < a.K ? *(const uint4v*)(src + c * 32)
                                             : zero;
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
#pragma unroll
    for (int s = 0; s < NW; ++s) {
      v += part[buf][s][wid][lane];
      if (EPI == GLU) u += part[buf][s][MT + wid][lane];
    }
    store_rows<EPI>(a, wid * 16 + c16, tile * 16 + 4 * grp, v, u);
  };

  frag_u wa[8], wb[8];
  int tile = blockIdx.x;
  load(tile, 0, wa);
  load(tile, 1, wb);
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

template <int EPI>
static int launch(const StreamArgs& a, int stay, hipStream_t stream) {
  constexpr int rows = EPI == GLU ? 32 : 16;
  const int tiles = (a.N + rows - 1) / rows;
  if (stay) {
    if (a.N % rows) return 1;
    const int grid = min(tiles, 256);
    // at most 128 registers of x beside the weights (plain products of 17 to
    // 32 rows by a direct call alone, here and below: the library is faster)
    if (a.T <= 16 && a.K <= 4096)
      stay_linear_kernel<8, 2, 1, EPI><<<grid, 512, 0, stream>>>(a);
    else if (a.T <= 16 && a.K <= 8192)
      stay_linear_kernel<8, 4, 1, EPI><<<grid, 512, 0, stream>>>(a);
    else if (a.T <= 32 && a.K <= 4096)
      stay_linear_kernel<8, 2, 2, EPI><<<grid, 512, 0, stream>>>(a);
    else
      return 1;
  } else {
    if constexpr (EPI == GLU) return 1;
    else if (a.T <= 16)
      stream_linear_kernel<1, EPI><<<tiles, 1024, 0, stream>>>(a);
    else
      stream_linear_kernel<2, EPI>
          <<<dim3(tiles, (a.T + 31) / 32), 1024, 0, stream>>>(a);
  }
  return (int)hipGetLastError();
}

// K, strides and bases in 8 elements; GLU stays, on whole tiles
extern "C" int sv_stream_linear(const StreamArgs* a, int epilogue, int stay,
                                hipStream_t stream) {
  if (a->T <= 0 || a->N <= 0) return 0;
  if (a->K % 8) return 1;
  return epilogue == GLU   ? launch<GLU>(*a, stay, stream)
         : epilogue == F32 ? launch<F32>(*a, stay, stream)
                           : launch<PLAIN>(*a, stay, stream);
}
