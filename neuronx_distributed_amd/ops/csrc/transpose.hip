// Rows of 16-bit words turned into columns, for the library's products that read
// both operands along what they contract (weight gradients).  HBM-bound.

#include "common.h"

// x (T, K) rows of pitch xst -> out (K, T) rows of pitch ost >= 8 ceil(T / 8).  A
// lane turns 8 x 8 words in registers; 8 lanes read 128 bytes of a row and write 128
// of a column, four waves 512, so that whole lines move and nothing passes LDS.
extern "C" __global__ void __launch_bounds__(256)
transpose_words_kernel(const short* __restrict__ x, long xst,
                       short* __restrict__ out, long ost, int T, int K) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int k = blockIdx.x * 64 + (lane & 7) * 8;
  const int t = blockIdx.y * 256 + wave * 64 + (lane >> 3) * 8;
  if (k >= K || t >= T) return;
  union { uint4 v[8]; unsigned w[8][4]; } in;
#pragma unroll
  for (int i = 0; i < 8; ++i)                  // past the end: the last row again
    in.v[i] = *(const uint4*)(x + min(t + i, T - 1) * xst + k);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    uint4 o;
    const unsigned sel = j & 1 ? 0x07060302u : 0x05040100u;
    o.x = __builtin_amdgcn_perm(in.w[1][j / 2], in.w[0][j / 2], sel);
    o.y = __builtin_amdgcn_perm(in.w[3][j / 2], in.w[2][j / 2], sel);
    o.z = __builtin_amdgcn_perm(in.w[5][j / 2], in.w[4][j / 2], sel);
    o.w = __builtin_amdgcn_perm(in.w[7][j / 2], in.w[6][j / 2], sel);
    *(uint4*)(out + (k + j) * ost + t) = o;
  }
}

extern "C" int transpose_words(const void* x, long xst, void* out, long ost, int T,
                               int K, hipStream_t stream) {
  if (T <= 0 || K <= 0) return 0;
  if (K % 8 || xst % 8 || ost % 8 || ost < (T + 7) / 8 * 8) return 1;
  const dim3 grid((K + 63) / 64, (T + 255) / 256);
  if (grid.y > 65535) return 1;
  transpose_words_kernel<<<grid, 256, 0, stream>>>((const short*)x, xst,
                                                   (short*)out, ost, T, K);
  return (int)hipGetLastError();
}
