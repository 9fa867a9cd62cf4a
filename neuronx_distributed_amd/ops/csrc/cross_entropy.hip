// Fused vocab-parallel cross-entropy pieces for CDNA4.
//
// Replaces the torch-op chain of the reference's _ParallelCrossEntropy
// (reference parallel_layers/loss_functions.py:10-129) that eager ROCm
// would run as ~8 elementwise/reduce passes over fp32-materialized logits.
// Two HBM-bound kernels over the bf16 (N, V/tp) logits shard:
//   ce_stats:   per row the shard's max m, sum(exp(l - m)) and, if the shard
//               owns the target, its l - m            [TP all-reduces]
//   ce_bwd:     dlogits = (exp(l-m)/sumexp - onehot) * gout, bf16 out; a row
//               whose gout is zero (ignored, or the last of a sequence) is
//               zero and not read
// The softmax matrix is never materialized (recomputed in bwd).
// One pass for the max and the sum: 8192 x 32000 in 97 us, a pass for each 211;
// a read at the rate of a copy takes 101.

#include "common.h"

#define LOG2E 1.4426950408889634f

extern "C" __global__ void __launch_bounds__(256)
ce_stats_kernel(const short* __restrict__ logits,
                const long* __restrict__ targets, float* __restrict__ rowmax,
                float* __restrict__ sumexp, float* __restrict__ predicted,
                long N, int V, long vocab_start) {
  __shared__ float scratch[16], top[4];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (long row = blockIdx.x; row < N; row += gridDim.x) {
    const short* r = logits + row * V;
    // of the thread's logits: the largest so far, the sum over it
    float m = -3.0e38f, s = 0.f;
    auto add = [&](const s8v* v, int n) __attribute__((always_inline)) {
      float most = m;
      for (int c = 0; c < n; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j) most = fmaxf(most, bits2f(v[c][j]));
      s *= __builtin_amdgcn_exp2f((m - most) * LOG2E);
      m = most;
      for (int c = 0; c < n; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          s += __builtin_amdgcn_exp2f((bits2f(v[c][j]) - m) * LOG2E);
    };
    const int nvec = V >> 3;
    int i = threadIdx.x;
    for (; i + 768 < nvec; i += 1024) {    // four words on their way
      s8v v[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = *(const s8v*)(r + (i + c * 256) * 8);
      add(v, 4);
    }
    for (; i < nvec; i += 256) {
      const s8v v = *(const s8v*)(r + i * 8);
      add(&v, 1);
    }
    const float most = wave_reduce(m, MaxOp());
    if (lane == 0) top[wid] = most;
    __syncthreads();
    const float M = fmaxf(fmaxf(top[0], top[1]), fmaxf(top[2], top[3]));
    s = block_reduce_sum(s * __builtin_amdgcn_exp2f((m - M) * LOG2E), scratch);
    if (threadIdx.x == 0) {
      rowmax[row] = M;
      sumexp[row] = s;
      const long t = targets[row] - vocab_start;
      predicted[row] = (t >= 0 && t < V) ? bits2f(r[t]) - M : 0.f;
    }
    __syncthreads();
  }
}

extern "C" __global__ void __launch_bounds__(256)
ce_bwd_kernel(const short* __restrict__ logits,
              const float* __restrict__ rowmax,
              const float* __restrict__ sumexp,
              const long* __restrict__ targets,
              const float* __restrict__ gout, short* __restrict__ dlogits,
              long N, int V, long vocab_start) {
  for (long row = blockIdx.x; row < N; row += gridDim.x) {
    const short* r = logits + row * V;
    short* d = dlogits + row * V;
    const float m = rowmax[row];
    const float inv = 1.0f / sumexp[row];
    const float g = gout[row];
    const long t = targets[row] - vocab_start;
    int nvec = V >> 3;
    if (g == 0.f) {
      for (int i = threadIdx.x; i < nvec; i += blockDim.x)
        *(s8v*)(d + i * 8) = s8v{0, 0, 0, 0, 0, 0, 0, 0};
      continue;
    }
    for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
      s8v v = *(const s8v*)(r + i * 8);
      s8v o;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float p = __builtin_amdgcn_exp2f((bits2f(v[j]) - m) * LOG2E) * inv;
        long col = i * 8 + j;
        if (col == t) p -= 1.0f;
        o[j] = f2bits(p * g);
      }
      *(s8v*)(d + i * 8) = o;
    }
  }
}

// V a multiple of 8, rows 16-byte aligned
extern "C" void ce_stats(const void* logits, const void* targets, void* rowmax,
                         void* sumexp, void* predicted, long N, int V,
                         long vocab_start, hipStream_t s) {
  if (N <= 0) return;
  int blocks = N < 2048 ? (int)N : 2048;
  ce_stats_kernel<<<blocks, 256, 0, s>>>(
      (const short*)logits, (const long*)targets, (float*)rowmax,
      (float*)sumexp, (float*)predicted, N, V, vocab_start);
}

extern "C" void ce_bwd(const void* logits, const void* rowmax,
                       const void* sumexp, const void* targets,
                       const void* gout, void* dlogits, long N, int V,
                       long vocab_start, hipStream_t s) {
  if (N <= 0) return;
  int blocks = N < 2048 ? (int)N : 2048;
  ce_bwd_kernel<<<blocks, 256, 0, s>>>(
      (const short*)logits, (const float*)rowmax, (const float*)sumexp,
      (const long*)targets, (const float*)gout, (short*)dlogits, N, V,
      vocab_start);
}
