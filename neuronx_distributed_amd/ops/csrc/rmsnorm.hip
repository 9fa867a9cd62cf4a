// Fused RMSNorm forward/backward for CDNA4 (gfx950).
//
// Replaces the reference's torch-level RMSNorm that the Neuron compiler
// fuses (reference modules/rms_norm.py:10-36) — eager ROCm will not fuse,
// so this is a hand-written HBM-bound kernel: one pass, vectorized 16B
// bf16 loads (guide G13), fp32 accumulation, per-row rstd saved for bwd.
//
// Layout: x (N, H) bf16 rows; w (H) bf16; out (N, H) bf16; rstd (N) f32.

#include "common.h"

// ---------------------------------------------------------------------------
// forward: out = x * rsqrt(mean(x^2) + eps) * w
// one block per ROWS_PER_BLOCK rows; vector short8 loads
// ---------------------------------------------------------------------------
extern "C" __global__ void __launch_bounds__(256)
rmsnorm_fwd_kernel(const short* __restrict__ x, const short* __restrict__ w,
                   short* __restrict__ out, float* __restrict__ rstd_out,
                   int H, float eps, int rows) {
  __shared__ float scratch[16];
  int row = blockIdx.x;
  if (row >= rows) return;
  const short* xr = x + (long)row * H;
  short* outr = out + (long)row * H;

  int nvec = H >> 3;  // H % 8 == 0 required
  float ss = 0.f;
  // the first 8192 columns stay in registers between the stats pass and the
  // normalize pass: 2 HBM passes instead of 3
  s8v cache[4];
  auto stats = [&](s8v v) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float f = bits2f(v[j]);
      ss += f * f;
    }
  };
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int i = threadIdx.x + c * 256;
    if (i < nvec) {
      cache[c] = *(const s8v*)(xr + i * 8);
      stats(cache[c]);
    }
  }
  for (int i = threadIdx.x + 1024; i < nvec; i += 256)
    stats(*(const s8v*)(xr + i * 8));
  ss = block_reduce_sum(ss, scratch);
  float rstd = rsqrtf(ss / (float)H + eps);
  if (threadIdx.x == 0 && rstd_out) rstd_out[row] = rstd;

  auto write = [&](int i, s8v v) __attribute__((always_inline)) {
    s8v wv = *(const s8v*)(w + i * 8);
    s8v o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = f2bits(bits2f(v[j]) * rstd * bits2f(wv[j]));
    *(s8v*)(outr + i * 8) = o;
  };
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int i = threadIdx.x + c * 256;
    if (i < nvec) write(i, cache[c]);
  }
  for (int i = threadIdx.x + 1024; i < nvec; i += 256)
    write(i, *(const s8v*)(xr + i * 8));
}

// ---------------------------------------------------------------------------
// backward:
//   dx = rstd * w * dy - rstd^3/H * x * sum(dy * w * x)  [+ dpass]
//   dw = sum_rows(dy * x * rstd)
// dpass != nullptr: the residual fork's pass-through gradient is folded into
// this pass (training fused add+RMSNorm site), replacing a separate 3-pass
// eager add kernel.
//
// HBM-bound.  A workgroup takes every so many rows; a thread owns the same
// columns of all of them, so that its weights and the sums of dw stay in
// registers, and asks for the next row before this one is summed up.  The
// sums of the workgroups go to `part` and are added up by a second kernel, in
// one order.  8192 x 4096 with dpass: 45 us and 5 (rows one after the other, sums in LDS,
// an atomic add a column of 2048 workgroups: 101); its 270 MB take 52 at the
// rate of a copy.
// ---------------------------------------------------------------------------
#define BWD_BLOCKS 512

// VPT: 16-byte words of a row a thread
template <int VPT>
__global__ void __launch_bounds__(256)
rmsnorm_bwd_kernel(const short* __restrict__ x, const short* __restrict__ w,
                   const short* __restrict__ dy,
                   const float* __restrict__ rstd_in,
                   const short* __restrict__ dpass, short* __restrict__ dx,
                   float* __restrict__ part, int H, int rows) {
  __shared__ float scratch[2][4];
  const int tid = threadIdx.x, nvec = H >> 3;
  const s8v zero = {0, 0, 0, 0, 0, 0, 0, 0};
  s8v wv[VPT], xa[VPT], da[VPT], pa[VPT], xb[VPT], db[VPT], pb[VPT];
  float dw[VPT][8] = {};
  auto load = [&](int row, s8v* xv, s8v* dv, s8v* pv)
      __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < VPT; ++c) {
      const int i = tid + c * 256;
      const long at = (long)row * H + i * 8;
      const bool in = i < nvec && row < rows;
      xv[c] = in ? *(const s8v*)(x + at) : zero;
      dv[c] = in ? *(const s8v*)(dy + at) : zero;
      pv[c] = in && dpass ? *(const s8v*)(dpass + at) : zero;
    }
  };
  auto take = [&](int row, int buf, const s8v* xv, const s8v* dv, const s8v* pv)
      __attribute__((always_inline)) {
    const float rstd = rstd_in[row];
    float dot = 0.f;  // sum(dy * w * x)
#pragma unroll
    for (int c = 0; c < VPT; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        dot += bits2f(dv[c][j]) * bits2f(wv[c][j]) * bits2f(xv[c][j]);
    dot = wave_reduce(dot, SumOp());
    if ((tid & 63) == 0) scratch[buf][tid >> 6] = dot;
    __syncthreads();
    dot = scratch[buf][0] + scratch[buf][1] + scratch[buf][2] + scratch[buf][3];
    const float k = rstd * rstd * rstd * dot / (float)H;
#pragma unroll
    for (int c = 0; c < VPT; ++c) {
      const int i = tid + c * 256;
      s8v o;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float xf = bits2f(xv[c][j]), df = bits2f(dv[c][j]);
        float g = rstd * bits2f(wv[c][j]) * df - k * xf;
        if (dpass) g += bits2f(pv[c][j]);
        o[j] = f2bits(g);
        dw[c][j] += df * xf * rstd;
      }
      if (i < nvec) *(s8v*)(dx + (long)row * H + i * 8) = o;
    }
  };
#pragma unroll
  for (int c = 0; c < VPT; ++c) {
    const int i = tid + c * 256;
    wv[c] = i < nvec ? *(const s8v*)(w + i * 8) : zero;
  }
  const int step = gridDim.x;
  int row = blockIdx.x;
  load(row, xa, da, pa);
  for (; row < rows; row += 2 * step) {
    load(row + step, xb, db, pb);
    take(row, 0, xa, da, pa);
    if (row + step >= rows) break;
    load(row + 2 * step, xa, da, pa);
    take(row + step, 1, xb, db, pb);
  }
#pragma unroll
  for (int c = 0; c < VPT; ++c) {
    const int i = tid + c * 256;
    if (i >= nvec) continue;
    f4v* d = (f4v*)(part + (long)blockIdx.x * H + i * 8);
    d[0] = f4v{dw[c][0], dw[c][1], dw[c][2], dw[c][3]};
    d[1] = f4v{dw[c][4], dw[c][5], dw[c][6], dw[c][7]};
  }
}

// rows too long for a workgroup's registers: two passes, sums in LDS
__global__ void __launch_bounds__(256)
rmsnorm_bwd_long_kernel(const short* __restrict__ x, const short* __restrict__ w,
                        const short* __restrict__ dy,
                        const float* __restrict__ rstd_in,
                        const short* __restrict__ dpass,
                        short* __restrict__ dx, float* __restrict__ part,
                        int H, int rows) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float* dw_part = smem;           // [H]
  float* scratch = smem + H;       // [16]
  const int nvec = H >> 3;
  for (int i = threadIdx.x; i < H; i += 256) dw_part[i] = 0.f;
  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    const long at = (long)row * H;
    const float rstd = rstd_in[row];
    float dot = 0.f;
    for (int i = threadIdx.x; i < nvec; i += 256) {
      const s8v xv = *(const s8v*)(x + at + i * 8);
      const s8v dv = *(const s8v*)(dy + at + i * 8);
      const s8v wv = *(const s8v*)(w + i * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        dot += bits2f(dv[j]) * bits2f(wv[j]) * bits2f(xv[j]);
    }
    __syncthreads();               // zeros, and the scratch is free again
    dot = block_reduce_sum(dot, scratch);
    const float k = rstd * rstd * rstd * dot / (float)H;
    for (int i = threadIdx.x; i < nvec; i += 256) {
      const s8v xv = *(const s8v*)(x + at + i * 8);
      const s8v dv = *(const s8v*)(dy + at + i * 8);
      const s8v wv = *(const s8v*)(w + i * 8);
      s8v pv = {0, 0, 0, 0, 0, 0, 0, 0}, o;
      if (dpass) pv = *(const s8v*)(dpass + at + i * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float xf = bits2f(xv[j]), df = bits2f(dv[j]);
        float g = rstd * bits2f(wv[j]) * df - k * xf;
        if (dpass) g += bits2f(pv[j]);
        o[j] = f2bits(g);
        dw_part[i * 8 + j] += df * xf * rstd;  // this thread's own
      }
      *(s8v*)(dx + at + i * 8) = o;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < H; i += 256)
    part[(long)blockIdx.x * H + i] = dw_part[i];
}

// dw = the sum of the workgroups' parts: 32 columns a workgroup, every eighth
// part a row of threads
__global__ void __launch_bounds__(256)
rmsnorm_dw_kernel(const float* __restrict__ part, short* __restrict__ dw, int H,
                  int parts) {
  __shared__ float sum[8][32];
  const int c = blockIdx.x * 32 + (threadIdx.x & 31), g = threadIdx.x >> 5;
  float s = 0.f;
  if (c < H) {
#pragma unroll 16
    for (int p = g; p < parts; p += 8) s += part[(long)p * H + c];
  }
  sum[g][threadIdx.x & 31] = s;
  __syncthreads();
  if (g || c >= H) return;
#pragma unroll
  for (int i = 1; i < 8; ++i) s += sum[i][threadIdx.x];
  dw[c] = f2bits(s);
}

// ---------------------------------------------------------------------------
// fused residual-add + RMSNorm (inference):
//   res_out = res_in + delta;  normed = res_out * rsqrt(mean(res_out^2)+eps) * w
// Collapses the decode path's two elementwise passes per norm site into one
// kernel and reads res/delta exactly once (HBM-bound; decode steps are
// kernel-count-bound inside hipGraph replay).
// ---------------------------------------------------------------------------
extern "C" __global__ void __launch_bounds__(256)
add_rmsnorm_fwd_kernel(const short* __restrict__ res_in,
                       const short* __restrict__ delta,
                       const short* __restrict__ w,
                       short* __restrict__ res_out,
                       short* __restrict__ normed,
                       float* __restrict__ rstd_out, int H, float eps,
                       int rows) {
  __shared__ float scratch[16];
  int row = blockIdx.x;
  if (row >= rows) return;
  const short* rr = res_in + (long)row * H;
  const short* dr = delta + (long)row * H;
  short* ror = res_out + (long)row * H;
  short* nr = normed + (long)row * H;

  int nvec = H >> 3;
  float ss = 0.f;
  // the first 8192 columns of the summed row stay in registers, so the second
  // pass does not read them again (an index known at run time put them into
  // scratch memory: 8192 x 4096 62 us, now 44; 52 at the rate of a copy)
  s8v cache[4];
  auto sum = [&](int i) __attribute__((always_inline)) {
    s8v rv = *(const s8v*)(rr + i * 8);
    s8v dv = *(const s8v*)(dr + i * 8);
    s8v o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float f = bits2f(rv[j]) + bits2f(dv[j]);
      o[j] = f2bits(f);
      f = bits2f(o[j]);  // norm statistics on the ROUNDED bf16 sum so the
                         // result matches an unfused add -> rmsnorm chain
      ss += f * f;
    }
    *(s8v*)(ror + i * 8) = o;
    return o;
  };
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int i = threadIdx.x + c * 256;
    if (i < nvec) cache[c] = sum(i);
  }
  for (int i = threadIdx.x + 1024; i < nvec; i += 256) sum(i);
  ss = block_reduce_sum(ss, scratch);
  float rstd = rsqrtf(ss / (float)H + eps);
  if (rstd_out && threadIdx.x == 0) rstd_out[row] = rstd;

  auto write = [&](int i, s8v v) __attribute__((always_inline)) {
    s8v wv = *(const s8v*)(w + i * 8);
    s8v o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = f2bits(bits2f(v[j]) * rstd * bits2f(wv[j]));
    *(s8v*)(nr + i * 8) = o;
  };
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int i = threadIdx.x + c * 256;
    if (i < nvec) write(i, cache[c]);
  }
  for (int i = threadIdx.x + 1024; i < nvec; i += 256)
    write(i, *(const s8v*)(ror + i * 8));
}

extern "C" void add_rmsnorm_fwd(const void* res_in, const void* delta,
                                const void* w, void* res_out, void* normed,
                                int rows, int H, float eps,
                                hipStream_t stream) {
  if (rows <= 0) return;
  add_rmsnorm_fwd_kernel<<<rows, 256, 0, stream>>>(
      (const short*)res_in, (const short*)delta, (const short*)w,
      (short*)res_out, (short*)normed, nullptr, H, eps, rows);
}

// training variant: also emits per-row rstd for the backward
extern "C" void add_rmsnorm_fwd_train(const void* res_in, const void* delta,
                                      const void* w, void* res_out,
                                      void* normed, void* rstd, int rows,
                                      int H, float eps, hipStream_t stream) {
  if (rows <= 0) return;
  add_rmsnorm_fwd_kernel<<<rows, 256, 0, stream>>>(
      (const short*)res_in, (const short*)delta, (const short*)w,
      (short*)res_out, (short*)normed, (float*)rstd, H, eps, rows);
}

extern "C" void rmsnorm_fwd(const void* x, const void* w, void* out,
                            void* rstd, int rows, int H, float eps,
                            hipStream_t stream) {
  if (rows <= 0) return;
  rmsnorm_fwd_kernel<<<rows, 256, 0, stream>>>(
      (const short*)x, (const short*)w, (short*)out, (float*)rstd, H, eps, rows);
}

// rows of `part` that rmsnorm_bwd fills
extern "C" int rmsnorm_bwd_parts(int rows) {
  return rows < BWD_BLOCKS ? rows : BWD_BLOCKS;
}

// dx and dw of rows of H % 8 == 0; dpass or null is added to dx
extern "C" void rmsnorm_bwd(const void* x, const void* w, const void* dy,
                            const void* rstd, const void* dpass, void* dx,
                            void* part, void* dw, int rows, int H,
                            hipStream_t stream) {
  const int blocks = rmsnorm_bwd_parts(rows);
#define BWD(KERNEL, LDS)                                                     \
  KERNEL<<<blocks, 256, LDS, stream>>>(                                      \
      (const short*)x, (const short*)w, (const short*)dy,                    \
      (const float*)rstd, (const short*)dpass, (short*)dx, (float*)part, H,  \
      rows)
  if (blocks > 0) {
    if (H <= 2048) BWD(rmsnorm_bwd_kernel<1>, 0);
    else if (H <= 4096) BWD(rmsnorm_bwd_kernel<2>, 0);
    else if (H <= 6144) BWD(rmsnorm_bwd_kernel<3>, 0);
    else if (H <= 8192) BWD(rmsnorm_bwd_kernel<4>, 0);
    else BWD(rmsnorm_bwd_long_kernel, (size_t)(H + 16) * sizeof(float));
  }
#undef BWD
  rmsnorm_dw_kernel<<<(H + 31) / 32, 256, 0, stream>>>(
      (const float*)part, (short*)dw, H, blocks);
}
