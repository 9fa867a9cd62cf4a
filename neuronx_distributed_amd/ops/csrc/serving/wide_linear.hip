// Products of up to 128 rows with a large weight: out[t, n] = sum_k x[t, k] w[n, k], where
// the rows do not fit the registers of the workgroups that stay with them
// (stream_linear.hip): short prompts, decoding of many requests, long K.
//
//   sv_wide_linear     bf16 or 32-bit results; or silu(gate) * up of a weight whose
//                      first half of rows are gates
//
// Bound by reading the weights up to 64 rows, beside that by LDS (28672 x 4096 gated:
// 36 us to read, 16 us of LDS at 128 rows).  A workgroup has up to 128 weight rows and a
// share of K; few weight rows are shared by K among as many workgroups as there are CUs, and the
// sums of a product meet in a second launch.  us, library (with the activation) | here:
//   28672 x 4096 gated     32 rows 55 | 40.4   64: 56 | 40.7   100: 59 | 48.2   128: 60 | 50.1
//   32000 x 4096, 32 bit   32 rows 57 | 43.7   64: 59 | 44.8   100: 62 | 49.1   128: 62 | 53.2
//   6144 x 4096, by 5      48 rows 17.5 | 16.6  64: 18.1 | 17.9  100: 23.3 | 21.5
//   4096 x 14336, by 8     32 rows 34 | 25.3   64: 40 | 27.1   100: 49 | 31.5   128: 75 | 35.1

#include "ring.h"

struct WideArgs {
  const short* x;           // [T] rows of K
  long xst;
  const short* w;           // [N] rows of K
  long wst;
  void* out;                // [T][N], or [T][N / 2] with GLU; 32-bit sums [splits][T][N]
  int T, N, K, splits;
  int g;                    // rows of a block of 32 (set here)
};

enum Epilogue { PLAIN = 0, F32 = 1, GLU = 2 };

// A stage is here, in all waves, and the one before is read.
template <int BEHIND>
__device__ __forceinline__ void arrive() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(BEHIND) : "memory");
}
// 16 columns of 64 weight rows and of 32 CM rows of x.  Waited for at once: the
// compiler would wait for all loads into LDS as well.
template <int CM>
__device__ __forceinline__ void read_rows(int aw, int ax, frag_u* fw, frag_u* fx) {
  if constexpr (CM == 2)
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:4096\n\t"
                 "ds_read_b128 %2, %5\n\tds_read_b128 %3, %5 offset:4096\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(fw[0].u4), "=&v"(fw[1].u4), "=&v"(fx[0].u4), "=&v"(fx[1].u4)
                 : "v"(aw), "v"(ax) : "memory");
  else
    asm volatile("ds_read_b128 %0, %3\n\tds_read_b128 %1, %3 offset:4096\n\t"
                 "ds_read_b128 %2, %4\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(fw[0].u4), "=&v"(fw[1].u4), "=&v"(fx[0].u4)
                 : "v"(aw), "v"(ax) : "memory");
}

// One workgroup: 128 weight rows (32 gates and their projections by turns; or of every 32
// the first g, for whole rounds of workgroups) by BM rows of x, 64 columns a stage.  Both go straight into LDS, NS - 1 stages ahead, rows of 128 bytes
// whose 16-byte slots s lie at s ^ row % 8.  Waves have 64 weight rows by BM / WM rows of
// x and share the columns of a stage; their sums meet at the end.  Workgroups begin at
// different columns: where all read the same ones, rows of a pitch of 8 KB met few
// channels (28672 x 4096 gated, 64 rows: 49.4 us, now 42.4).
// SPLIT: a share of K, 32-bit sums.
template <int BM, int EPI, bool SPLIT>
__global__ void __launch_bounds__(512) wide_linear_kernel(WideArgs a) {
  constexpr int BN = 128, WN = 2, WM = BM == 32 ? 1 : 2, WK = 8 / (WN * WM);
  constexpr int TM = BM / WM, CM = TM / 32, CN = 2, KC = 4 / WK;
  constexpr int NS = BM == 128 ? 4 : BM == 64 ? 5 : 6;
  constexpr int STAGE = (BN + BM) * 128, LX = BM == 128 ? 2 : 1, LT = 2 + LX;
  __shared__ __attribute__((aligned(1024))) char lds[NS * STAGE + (BM == 32 ? 1024 : 0)];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wid % WN, wm = wid / WN % WM, wk = wid / (WN * WM);
  const int col = lane & 31, hi = lane >> 5;
  const int tile = blockIdx.x, y = blockIdx.y;
  const int blocks = a.K / 64, S = gridDim.y;
  const int b0 = blocks * y / S, steps = blocks * (y + 1) / S - b0;

  const int wp = (int)a.wst * 2, xp = (int)a.xst * 2;
  const auto rw = ring_source(a.w, (a.N - 1) * wp + a.K * 2);
  const auto rx = ring_source(a.x, (a.T - 1) * xp + a.K * 2);
  int ow[2], ox[LX];
  bool held[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = (wid * 2 + i) * 8 + (lane >> 3);
    const int n = (r & 31) +
        (EPI == GLU ? (tile * 2 + (r >> 6)) * a.g + (r & 32 ? a.N / 2 : 0)
                    : (tile * 4 + (r >> 5)) * a.g);
    ow[i] = n * wp + ((lane ^ (lane >> 3)) & 7) * 16 + b0 * 128;
    held[i] = (r & 31) < a.g;
  }
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int r = (wid * LX + i) * 8 + (lane >> 3);
    ox[i] = r * xp + ((lane ^ (lane >> 3)) & 7) * 16 + b0 * 128;
  }
  // (of 32 rows four waves ask for nothing, past all stages, so that they count alike)
  const bool mine = wid * LX * 8 < BM;
  int next = 0, slot = 0, blk = tile % steps;
  auto ask = [&]() __attribute__((always_inline)) {
    char* st = lds + slot * STAGE;
    const uint at = next < steps ? blk * 128 : RING_NOWHERE;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      piece<true>(rw, held[i] ? ow[i] + at : RING_NOWHERE, st + (wid * 2 + i) * 1024);
#pragma unroll
    for (int i = 0; i < LX; ++i)
      piece<false>(rx, mine ? ox[i] + at : RING_NOWHERE,
                   mine ? st + BN * 128 + (wid * LX + i) * 1024 : lds + NS * STAGE);
    ++next;
    if (++blk == steps) blk = 0;
    if (++slot == NS) slot = 0;
  };
#pragma unroll
  for (int i = 0; i < NS - 1; ++i) ask();

  f32x16 acc[CN][CM] = {};
  const int base = (int)(size_t)(lds_ptr)lds;
  // slot 2 (KC wk + c) + hi of row col: rows 32 on are 4096 bytes on
  const int aw = base + wn * 8192 + col * 128, ax = base + BN * 128 + wm * TM * 128 + col * 128;
  int rd = 0;
  for (int i = 0; i < steps; ++i) {
    arrive<(NS - 2) * LT>();
    ask();
    frag_u fw[KC][CN], fx[KC][CM];
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const int s = (((2 * (KC * wk + c) + hi) ^ col) & 7) * 16 + rd;
      read_rows<CM>(aw + s, ax + s, fw[c], fx[c]);
    }
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
      for (int n = 0; n < CN; ++n)
#pragma unroll
        for (int m = 0; m < CM; ++m)
          acc[n][m] = mfma_bf16(fw[c][n].bf, fx[c][m].bf, acc[n][m]);
    rd += STAGE;
    if (rd == NS * STAGE) rd = 0;
  }
  // the sums of the waves that share a tile meet
  arrive<0>();
  float* meet = (float*)lds;
  constexpr int PW = CN * CM * 16 * 64;  // words of a wave
  if (wk > 0) {
    float* to = meet + ((wk - 1) * WN * WM + wm * WN + wn) * PW + lane * 4;
#pragma unroll
    for (int n = 0; n < CN; ++n)
#pragma unroll
      for (int m = 0; m < CM; ++m)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg)
          *(f32x4*)(to + ((n * CM + m) * 4 + rg) * 256) =
              f32x4{acc[n][m][4 * rg], acc[n][m][4 * rg + 1], acc[n][m][4 * rg + 2],
                    acc[n][m][4 * rg + 3]};
  }
  lds_barrier();
  if (wk > 0) return;
  const int N = EPI == GLU && !SPLIT ? a.N / 2 : a.N;
#pragma unroll
  for (int m = 0; m < CM; ++m) {
    const int t = wm * TM + m * 32 + col;
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      f32x4 v[CN];
#pragma unroll
      for (int n = 0; n < CN; ++n) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[n][j] = acc[n][m][4 * rg + j];
#pragma unroll
        for (int k = 1; k < WK; ++k)
          v[n] += *(const f32x4*)(meet + ((k - 1) * WN * WM + wm * WN + wn) * PW +
                                  lane * 4 + ((n * CM + m) * 4 + rg) * 256);
      }
      if (t >= a.T) continue;
      const int r = 8 * rg + 4 * hi;
      if (EPI == GLU && !SPLIT) {
        const int c = (tile * 2 + wn) * a.g + r;
        if (r >= a.g || c >= N) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[0][j] = silu_f(v[0][j]) * v[1][j];
        *(uint2*)((short*)a.out + (long)t * N + c) =
            uint2{pack_bf16x2(v[0][0], v[0][1]), pack_bf16x2(v[0][2], v[0][3])};
      } else {
#pragma unroll
        for (int n = 0; n < CN; ++n) {
          const int c = r + (EPI == GLU ? (tile * 2 + wn) * a.g + n * (N / 2)
                                        : (tile * 4 + wn * 2 + n) * a.g);
          if (r >= a.g || c >= (EPI == GLU && n == 0 ? N / 2 : N)) continue;
          if (SPLIT)
            *(f32x4*)((float*)a.out + ((long)y * a.T + t) * N + c) = v[n];
          else if (EPI == F32)
            *(f32x4*)((float*)a.out + (long)t * N + c) = v[n];
          else
            *(uint2*)((short*)a.out + (long)t * N + c) =
                uint2{pack_bf16x2(v[n][0], v[n][1]), pack_bf16x2(v[n][2], v[n][3])};
        }
      }
    }
  }
}

// [splits][T][N] -> [T][N], or [T][N / 2] with GLU; 4 results a thread
template <int EPI>
__global__ void __launch_bounds__(256)
wide_merge_kernel(const float* __restrict__ part, void* out, int T, int N, int splits) {
  const int NO = EPI == GLU ? N / 2 : N;
  const long i = (blockIdx.x * 256L + threadIdx.x) * 4;
  if (i >= (long)T * NO) return;
  const long t = i / NO, n = i - t * NO;
  const float* p = part + t * N + n;
  const long step = (long)T * N;
  f32x4 v = {}, u = {};
#pragma unroll 8
  for (int s = 0; s < splits; ++s) {
    v += *(const f32x4*)(p + s * step);
    if (EPI == GLU) u += *(const f32x4*)(p + s * step + NO);
  }
  if (EPI == GLU)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = silu_f(v[j]) * u[j];
  if (EPI == F32) *(f32x4*)((float*)out + i) = v;
  else *(uint2*)((short*)out + i) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

// part: [splits][T][N], or null with one split
extern "C" int sv_wide_linear(const WideArgs* a, float* part, int epilogue,
                              hipStream_t stream) {
  if (a->T <= 0 || a->N <= 0) return 0;
  if (a->T > 128 || a->K % 64 || a->N % 8 || a->splits < 1 || a->splits > a->K / 64 ||
      (a->splits > 1) != (part != nullptr) || a->wst * 2 * (a->N + 128L) >= 1L << 31 ||
      a->xst * 2 * 256 >= 1L << 31)
    return 1;
  WideArgs w = *a;
  // Whole rounds of 256 workgroups, each with as many rows: a CU alone reads 25 GB/s
  // (28672 x 4096 gated, 32 rows: 43.3 us by 128, 40.4 by 112; 22016 36.8, 33.9 by 96;
  // 37888 x 3584 64.8, 53.3 by 76; but 57344 x 8192 150.7, 154, an eighth idle).
  const int tiles = (a->N + 127) / 128, all = (tiles + 255) / 256 * 256;
  w.g = 32;
  if (a->splits == 1 && (a->T > 32 || all == 256 || tiles * 5 < all * 4))
    w.g = min(32, (a->N + 16 * all - 1) / (16 * all) * 4);
  const dim3 grid((a->N + 4 * w.g - 1) / (4 * w.g), a->splits);
  if (part) w.out = part;
#define WIDE(M, E, S) wide_linear_kernel<M, E, S><<<grid, 512, 0, stream>>>(w)
#define WIDE_E(M)                                                             \
  do {                                                                        \
    if (part) { if (epilogue == GLU) WIDE(M, GLU, true); else WIDE(M, PLAIN, true); } \
    else if (epilogue == GLU) WIDE(M, GLU, false);                            \
    else if (epilogue == F32) WIDE(M, F32, false);                            \
    else WIDE(M, PLAIN, false);                                               \
  } while (0)
  if (a->T <= 32) WIDE_E(32);
  else if (a->T <= 64) WIDE_E(64);
  else WIDE_E(128);
#undef WIDE
#undef WIDE_E
  if (part) {
    const int NO = epilogue == GLU ? a->N / 2 : a->N;
    const int g = (int)(((long)a->T * NO / 4 + 255) / 256);
#define MERGE(E) wide_merge_kernel<E><<<g, 256, 0, stream>>>(part, a->out, a->T, a->N, a->splits)
    if (epilogue == GLU) MERGE(GLU); else if (epilogue == F32) MERGE(F32); else MERGE(PLAIN);
#undef MERGE
  }
  return (int)hipGetLastError();
}
