// Gradient of an embedding table: row v is the sum of the gradients of the tokens v, in
// 32 bits and in the order of the tokens, so that it is the same every time.  HBM-bound:
// every row is written once, zeros too.  8192 tokens, 32000 x 4096: 340 us by sorting,
// in torch's 18 launches, with a wait of the host; here 80, 63 of them for the rows
// (262 MB written, 67 read).

#include "common.h"

#define EMB_MANY 8                 // tokens of a row that one workgroup sums by itself

struct EmbArgs {
  const long* ids;                 // [T]
  const short* dy;                 // [T][W]
  short* out;                      // [V][W]
  int *first, *last, *count;       // [V] tokens of a row
  int* many;                       // [0] rows of more than EMB_MANY, [1 ...] which
  int T, V, W, skip;               // skip: a row without a gradient, or -1
};

__global__ void __launch_bounds__(256) embedding_clear_kernel(EmbArgs a) {
  const int v = blockIdx.x * 256 + threadIdx.x;
  if (v == 0) a.many[0] = 0;
  if (v >= a.V) return;
  a.first[v] = a.T;
  a.last[v] = -1;
  a.count[v] = 0;
}

__global__ void __launch_bounds__(256) embedding_count_kernel(EmbArgs a) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= a.T) return;
  const long v = a.ids[t];
  if (v < 0 || v >= a.V || v == a.skip) return;
  atomicMin(a.first + v, t);
  atomicMax(a.last + v, t);
  // the token that makes it too many for one workgroup lists it, whichever that is
  if (atomicAdd(a.count + v, 1) == EMB_MANY) a.many[1 + atomicAdd(a.many, 1)] = v;
}

__device__ __forceinline__ void add8(const short* p, float* acc) {
  const s8v x = *(const s8v*)p;
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] += bits2f(x[j]);
}
__device__ __forceinline__ void put8(short* p, const float* acc) {
  s8v x;
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] = f2bits(acc[j]);
  *(s8v*)p = x;
}

// A row of up to EMB_MANY tokens: of two the first and the last are all, of more one
// wave looks for them between those.
__global__ void __launch_bounds__(256) embedding_rows_kernel(EmbArgs a) {
  __shared__ int at[EMB_MANY];
  const int v = blockIdx.x, n = a.count[v];
  if (n > EMB_MANY) return;
  const int first = a.first[v], last = a.last[v], lane = threadIdx.x & 63;
  if (n > 2) {
    if (threadIdx.x < 64) {
      int found = 0;
      for (int t = first; t <= last; t += 64) {
        const bool here = t + lane <= last && a.ids[t + lane] == v;
        const unsigned long long which = __ballot(here);
        if (here) at[found + __popcll(which & ((1ull << lane) - 1))] = t + lane;
        found += __popcll(which);
      }
    }
    __syncthreads();
  }
  for (int c = threadIdx.x * 8; c < a.W; c += 2048) {
    float acc[8] = {};
    if (n > 2)
      for (int i = 0; i < n; ++i) add8(a.dy + (long)at[i] * a.W + c, acc);
    else {
      if (n) add8(a.dy + (long)first * a.W + c, acc);
      if (n > 1) add8(a.dy + (long)last * a.W + c, acc);
    }
    put8(a.out + (long)v * a.W + c, acc);
  }
}

// Rows of more: 512 columns a workgroup, whose 16 waves share the tokens between the
// first and the last; their sums are added in order.
__global__ void __launch_bounds__(1024) embedding_many_kernel(EmbArgs a) {
  __shared__ float sums[16][512];
  if ((int)blockIdx.x >= a.many[0]) return;
  const int v = a.many[1 + blockIdx.x], lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int first = a.first[v], span = a.last[v] + 1 - first;
  const int t0 = first + (int)((long)span * wid / 16);
  const int t1 = first + (int)((long)span * (wid + 1) / 16);
  const int c = blockIdx.y * 512 + lane * 8;
  const bool in = c < a.W;
  const short* dy = a.dy + (in ? c : 0);
  float acc[8] = {};
  for (int t = t0; t < t1; t += 64) {
    unsigned long long which = __ballot(t + lane < t1 && a.ids[t + lane] == v);
    while (which) {                        // four on their way at a time
      s8v x[4];
      const int n = min(4, __popcll(which));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int b = which ? __ffsll(which) - 1 : 0;
        if (j < n) x[j] = *(const s8v*)(dy + (long)(t + b) * a.W);
        which &= which - 1;                // (of none: none)
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < n)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[e] += bits2f(x[j][e]);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) sums[wid][lane * 8 + e] = acc[e];
  __syncthreads();
  if (wid || !in) return;
  for (int w = 1; w < 16; ++w)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] += sums[w][lane * 8 + e];
  put8(a.out + (long)v * a.W + c, acc);
}

// work: 3 V + 1 + T / (EMB_MANY + 1) ints
extern "C" int embedding_bwd(const void* ids, const void* dy, void* out, int* work,
                             int T, int V, int W, int skip, hipStream_t stream) {
  // (a workgroup of 256 a row: fewer than 2^32 threads)
  if (T <= 0 || V <= 0 || V >= 1 << 24 || W <= 0 || W % 8) return 1;
  const EmbArgs a = {(const long*)ids, (const short*)dy, (short*)out, work, work + V,
                     work + 2 * V, work + 3 * V, T, V, W, skip};
  embedding_clear_kernel<<<(V + 255) / 256, 256, 0, stream>>>(a);
  embedding_count_kernel<<<(T + 255) / 256, 256, 0, stream>>>(a);
  embedding_rows_kernel<<<V, 256, 0, stream>>>(a);
  if (T > EMB_MANY)
    embedding_many_kernel<<<dim3(T / (EMB_MANY + 1), (W + 511) / 512), 1024, 0,
                            stream>>>(a);
  return (int)hipGetLastError();
}
