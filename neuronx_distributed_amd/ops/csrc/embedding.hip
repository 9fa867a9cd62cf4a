// Gradient of an embedding table: row v is the sum of the gradients of the tokens v, in
// 32 bits and in the order of the tokens, so that it is the same every time.  HBM-bound:
// every row is written once, zeros too.  What a call costs depends little on which
// tokens there are and how far apart: those of a row are linked, few of them are put in
// order where they are summed, many are shared.  8192 tokens, 32000 x 4096, us, torch's
// (sorted, in 18 launches and a wait of the host), with tokens looked for between a row's
// first and last one, and here: evenly spread 331 | 78 | 90 (262 MB written, 67 read),
// as words are 280 | 136 | 125, half of them padding 338 | 472 | 207, all of one row 420 |
// 592 | 257; 32768 tokens of 32000 x 1024, five a row and far apart 210 | 353 | 72.

#include "common.h"

#include <climits>

#define EMB_MANY 8                 // tokens of a row that one wave sums by itself
#define EMB_PART 256               // and one workgroup; more are cut into parts

struct EmbArgs {
  const long* ids;                 // [T]
  const short* dy;                 // [T][W]
  short* out;                      // [V][W]
  int *head, *count;               // [V] tokens of a row: the last one linked; how many
  int *next, *list;                // [T] the one linked before; those of crowded rows
  int* many;                       // [0] of list, [1] crowded rows, [2] parts, [3] rows
                                   //   in parts
  int* rows;                       // [T / (EMB_MANY + 1)] crowded rows
  int2* parts;                     // [T / EMB_PART * 2 + 1] row in parts, part of it
  int4* cut;                       // [T / EMB_PART] its row, parts, first part
  float* sums;                     // [parts][W]
  int T, V, W, skip;               // skip: a row without a gradient, or -1
};

__global__ void __launch_bounds__(256) embedding_clear_kernel(EmbArgs a) {
  const int v = blockIdx.x * 256 + threadIdx.x;
  if (v < 4) a.many[v] = 0;
  if (v < a.V) a.count[v] = 0;
}

__device__ __forceinline__ bool counts(const EmbArgs& a, long v) {
  return v >= 0 && v < a.V && v != a.skip;
}

// (the first one's next is read by nobody: there are as many as the count says)
__global__ void __launch_bounds__(256) embedding_link_kernel(EmbArgs a) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= a.T) return;
  const long v = a.ids[t];
  if (!counts(a, v)) return;
  a.next[t] = atomicExch(a.head + v, t);
  atomicAdd(a.count + v, 1);
}

__device__ __forceinline__ void add8(s8v x, float* acc) {
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] += bits2f(x[j]);
}
__device__ __forceinline__ void put8(short* p, const float* acc) {
  s8v x;
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] = f2bits(acc[j]);
  *(s8v*)p = x;
}

// A wave takes up to 64 rows, `waves` apart (those with tokens may all lie together), and
// sums those of up to EMB_MANY tokens by itself.  Rows of more get room in the list, where
// `head` counts on, or parts.  (2048 tokens, 250000 x 2048: 222 us; a workgroup a row,
// each of which takes 1.2 ns to begin, 321, one for eight rows 361; waves of 1024 columns
// 289.)
__global__ void __launch_bounds__(256, 6) embedding_rows_kernel(EmbArgs a, int waves) {
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int v0 = blockIdx.x * 4 + wid;
  if (v0 >= waves) return;
  const int rows = (a.V - v0 + waves - 1) / waves, held = v0 + lane * waves;
  const int mine = lane < rows ? a.count[held] : 0;
  const int last = lane < rows && mine ? a.head[held] : 0;
  for (int r = 0; r < rows; ++r) {
    const int v = v0 + r * waves, n = __builtin_amdgcn_readlane(mine, r);
    if (n > EMB_MANY) {
      const int parts = (n + EMB_PART - 1) / EMB_PART;
      int first = 0, row = 0;
      if (lane == 0) {
        if (parts == 1) {
          a.head[v] = atomicAdd(a.many, n);
          a.rows[atomicAdd(a.many + 1, 1)] = v;
        } else {
          first = atomicAdd(a.many + 2, parts);
          row = atomicAdd(a.many + 3, 1);
          a.cut[row] = int4{v, parts, first, 0};
        }
      }
      if (parts > 1) {
        first = __builtin_amdgcn_readfirstlane(first);
        row = __builtin_amdgcn_readfirstlane(row);
        for (int i = lane; i < parts; i += 64) a.parts[first + i] = int2{row, i};
      }
      continue;
    }
    short* out = a.out + (long)v * a.W;
    int at[EMB_MANY];
    at[0] = __builtin_amdgcn_readlane(last, r);
    if (n <= 2) {                        // (either one may be first)
      at[1] = n > 1 ? a.next[at[0]] : 0;
      const short *d0 = a.dy + (long)at[0] * a.W, *d1 = a.dy + (long)at[1] * a.W;
      for (int c0 = lane * 8; c0 < a.W; c0 += 1024) {
        s8v x[2], y[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int c = min(c0 + u * 512, a.W - 8);
          if (n > 0) x[u] = *(const s8v*)(d0 + c);
          if (n > 1) y[u] = *(const s8v*)(d1 + c);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          if (c0 + u * 512 >= a.W) break;
          float acc[8] = {};
          if (n > 0) add8(x[u], acc);
          if (n > 1) add8(y[u], acc);
          put8(out + c0 + u * 512, acc);
        }
      }
      continue;
    }
#pragma unroll
    for (int i = 1; i < EMB_MANY; ++i) at[i] = i >= n ? INT_MAX : a.next[at[i - 1]];
#pragma unroll
    for (int y = 0; y < EMB_MANY; ++y)
#pragma unroll
      for (int i = y & 1; i + 1 < EMB_MANY; i += 2) {
        const int lo = min(at[i], at[i + 1]), hi = max(at[i], at[i + 1]);
        at[i] = lo, at[i + 1] = hi;
      }
    for (int c = lane * 8; c < a.W; c += 512) {
      float acc[8] = {};
#pragma unroll
      for (int half = 0; half < EMB_MANY; half += 4) {
        s8v x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (half + i < n) x[i] = *(const s8v*)(a.dy + (long)at[half + i] * a.W + c);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (half + i < n) add8(x[i], acc);
      }
      put8(out + c, acc);
    }
  }
}

// The tokens of crowded rows, in any order within a row's.
__global__ void __launch_bounds__(256) embedding_place_kernel(EmbArgs a) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= a.T) return;
  const long v = a.ids[t];
  if (!counts(a, v)) return;
  const int n = a.count[v];
  if (n > EMB_MANY && n <= EMB_PART) a.list[atomicAdd(a.head + v, 1)] = t;
}

// Crowded rows and parts, one after the other: 512 columns a workgroup, whose 8 waves
// share the tokens; their sums are added in order.  A row's tokens are put in order in
// LDS; a part's are looked for in its share of all tokens.
__global__ void __launch_bounds__(512, 4) embedding_many_kernel(EmbArgs a) {
  __shared__ float sums[8][512];
  __shared__ int at[EMB_PART];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = blockIdx.y * 512 + lane * 8;
  const bool in = c < a.W;
  const short* dy = a.dy + (in ? c : 0);
  const int rows = a.many[1], all = rows + a.many[2];
  for (int i = blockIdx.x; i < all; i += gridDim.x) {
    float acc[8] = {};
    int v;
    if (i < rows) {
      v = a.rows[i];
      const int n = a.count[v];
      const int* list = a.list + a.head[v] - n;
      int size = 16;
      while (size < n) size *= 2;
      if (tid < size) at[tid] = tid < n ? list[tid] : INT_MAX;
      for (int k = 2; k <= size; k *= 2)
        for (int j = k / 2; j > 0; j /= 2) {
          __syncthreads();
          const int o = tid ^ j;
          if (tid < size && o > tid) {
            const int x = at[tid], y = at[o];
            if ((x > y) == ((tid & k) == 0)) at[tid] = y, at[o] = x;
          }
        }
      __syncthreads();
      const int n0 = n * wid / 8, n1 = n * (wid + 1) / 8;
      for (int k = n0; k < n1; k += 8) {   // eight on their way at a time
        s8v x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (k + j < n1) x[j] = *(const s8v*)(dy + (long)at[k + j] * a.W);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (k + j < n1) add8(x[j], acc);
      }
    } else {
      const int2 part = a.parts[i - rows];
      const int4 cut = a.cut[part.x];
      v = cut.x;
      const int t0 = (int)((long)a.T * part.y / cut.y);
      const int span = (int)((long)a.T * (part.y + 1) / cut.y) - t0;
      const int t1 = t0 + (int)((long)span * (wid + 1) / 8);
      for (int t = t0 + (int)((long)span * wid / 8); t < t1; t += 64) {
        unsigned long long which = __ballot(t + lane < t1 && a.ids[t + lane] == v);
        while (which) {
          s8v x[8];
          const int m = min(8, __popcll(which));
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int b = which ? __ffsll(which) - 1 : 0;
            if (j < m) x[j] = *(const s8v*)(dy + (long)(t + b) * a.W);
            which &= which - 1;            // (of none: none)
          }
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (j < m) add8(x[j], acc);
        }
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) sums[wid][lane * 8 + e] = acc[e];
    __syncthreads();
    if (wid == 0 && in) {
      for (int w = 1; w < 8; ++w)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += sums[w][lane * 8 + e];
      if (i < rows) {
        put8(a.out + (long)v * a.W + c, acc);
      } else {
        float* to = a.sums + (long)(i - rows) * a.W + c;
        *(f4v*)to = f4v{acc[0], acc[1], acc[2], acc[3]};
        *(f4v*)(to + 4) = f4v{acc[4], acc[5], acc[6], acc[7]};
      }
    }
    __syncthreads();                       // before the next one's
  }
}

// The parts of a row, in order: 512 columns a workgroup, whose 16 waves share them.
__global__ void __launch_bounds__(1024) embedding_parts_kernel(EmbArgs a) {
  __shared__ float sums[16][512];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = blockIdx.y * 512 + lane * 8;
  const bool in = c < a.W;
  const int rows = a.many[3];
  for (int i = blockIdx.x; i < rows; i += gridDim.x) {
    const int4 cut = a.cut[i];
    const float* from = a.sums + (long)cut.z * a.W + (in ? c : 0);
    float acc[8] = {};
    const int p1 = (int)((long)cut.y * (wid + 1) / 16);
#pragma unroll 4
    for (int p = (int)((long)cut.y * wid / 16); p < p1; ++p) {
      const f4v x = *(const f4v*)(from + (long)p * a.W);
      const f4v y = *(const f4v*)(from + (long)p * a.W + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += x[e], acc[e + 4] += y[e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) sums[wid][lane * 8 + e] = acc[e];
    __syncthreads();
    if (wid == 0 && in) {
      for (int w = 1; w < 16; ++w)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += sums[w][lane * 8 + e];
      put8(a.out + (long)cut.x * a.W + c, acc);
    }
    __syncthreads();                       // before the next one's
  }
}

// Words of 4 bytes that a call needs beside its operands; `work` begins at 16 bytes.
extern "C" long embedding_work(int T, int V, int W) {
  const long p = T / EMB_PART;             // rows in parts, and parts beside one a row
  return 2L * V + 2L * T + 4 + T / (EMB_MANY + 1) + 16 + 2 * (2 * p + 1) + 4 * p +
         2 * p * W;
}

extern "C" int embedding_bwd(const void* ids, const void* dy, void* out, void* work,
                             int T, int V, int W, int skip, hipStream_t stream) {
  // (rows of a workgroup's waves; a grid has fewer than 2^32 threads)
  if (T <= 0 || V <= 0 || V >= 1 << 24 || W <= 0 || W % 8) return 1;
  const long p = T / EMB_PART;
  EmbArgs a = {};
  a.ids = (const long*)ids, a.dy = (const short*)dy, a.out = (short*)out;
  // words of 16 bytes, of 8 and of 4
  a.cut = (int4*)work;
  a.sums = (float*)(a.cut + p);
  a.parts = (int2*)(a.sums + 2 * p * W);
  a.many = (int*)(a.parts + 2 * p + 1);
  a.head = a.many + 4, a.count = a.head + V;
  a.next = a.count + V, a.list = a.next + T, a.rows = a.list + T;
  a.T = T, a.V = V, a.W = W, a.skip = skip;
  embedding_clear_kernel<<<(V + 255) / 256, 256, 0, stream>>>(a);
  embedding_link_kernel<<<(T + 255) / 256, 256, 0, stream>>>(a);
  const int waves = max(min(V, 8192), (V + 63) / 64);
  embedding_rows_kernel<<<(waves + 3) / 4, 256, 0, stream>>>(a, waves);
  const int columns = (W + 511) / 512;
  if (T > EMB_MANY) {
    embedding_place_kernel<<<(T + 255) / 256, 256, 0, stream>>>(a);
    const dim3 grid(min(T / (EMB_MANY + 1), 1024), columns);
    embedding_many_kernel<<<grid, 512, 0, stream>>>(a);
  }
  if (p)
    embedding_parts_kernel<<<dim3(min((int)p, 256), columns), 1024, 0, stream>>>(a);
  return (int)hipGetLastError();
}
