// FlashAttention backward for CDNA4 (gfx950) — FA2-style recompute.
//
// Replaces the reference's NKI flash_attn_bwd (K2; reference
// kernels/flash_attn.py:18,76-88):
//   * fa_bwd_dq:    128-row Q blocks (4 waves x 32 q rows); delta[q] = sum_d
//       dO*O (32-bit) of its rows; sequential kv loop, dQ accumulated in
//       registers.
//   * fa_bwd_dkdv:  128-row KV blocks; a sequential q loop recomputes P^T from
//       (Q,K,lse), forms dS^T = P^T*(dP^T - delta), accumulates dK/dV in
//       registers, for one or several q heads of a kv head.
//   * fa_bwd_reduce: the sum of what is left of them (GQA).
// No atomics anywhere: every output region is written by exactly one
// workgroup.
//
// The accumulator of a product has its rows (the index that the next product
// sums over) in registers and its columns in lanes, so P and dS become operands
// by packing alone; the other operand is read from LDS in the accumulator's
// order of rows by transposing reads.  Results are accumulated transposed
// ([d][row of the lane]).
//
// 8192 tokens, 32/8 heads: dK/dV 2680 -> 1123 us (979 TFLOP/s), dQ 1404 -> 739
// us (1116 TFLOP/s); before, tiles were turned by scattered writes, the halves
// of dK/dV exchanged P and dS through LDS behind a third barrier, and every
// element was masked.  The vector work then stood between the products, beside
// those of another wave at best; cut into pieces, one beside each product of the
// same wave, both directions took 1823 us instead of 1874 (2 x 4096, 32 heads: 986
// for 1021); delta beside the dQ kernel's fragments of dO and the q heads of a kv
// head in one workgroup 1790 (a kernel for delta 22, the sum over heads 31).
// No unit alone bounds them: matrix cores are 57 % busy in dK/dV and 68 % in dQ, LDS 50
// and 34 %, without bank conflicts.  Of the time of a wave of dK/dV 33 % are waits for
// words and barriers (dQ 20 %), 27 % waits for a turn (37 %).

#include "common.h"
#include "flash_attn.h"
#include "mfma.h"
#include "lds.h"

#include <cfloat>

#define FA_D 128
#define LOG2E 1.4426950408889634f

// ---------------------------------------------------------------------------
// dK/dV and dQ.  Tiles go from memory into two LDS buffers as they are and are
// read both as rows and by transposing reads (lds.h).  Masks are applied only
// on tiles that a boundary crosses.
// ---------------------------------------------------------------------------
struct BwdArgs {
  const short *q, *k, *v, *out, *dout;
  const float* lse;
  float* delta;             // [B][Hq][S], written by the dQ kernel
  short *dq, *dk, *dv;      // dk, dv: Hdk heads, each the sum of Hq / Hdk q heads
  int Hq, Hkv, Hdk, S, causal, window;
  float scale;
  // element strides of (batch, head, seq)
  long q_bs, q_hs, q_ss, k_bs, k_hs, k_ss, v_bs, v_hs, v_ss;
  long o_bs, o_hs, o_ss;
  long do_bs, do_hs, do_ss, dq_bs, dq_hs, dq_ss;
  long dk_bs, dk_hs, dk_ss, dv_bs, dv_hs, dv_ss;
};

// N rows of `g` from row r0 on, by NT threads; rows past the last one read that
// again.
template <int N, int NT>
__device__ __forceinline__ void fill_rows(const short* g, long ss, int r0,
                                          int rows, char* lds) {
  constexpr int PASS = NT / 16;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int st_r = threadIdx.x >> 4;
  const int st_c = ((threadIdx.x & 15) ^ row_turn(st_r)) * 16;
  const int pitch = (int)ss * 2;
  if (r0 + N <= rows) {
    const int off = st_r * pitch + st_c;
#pragma unroll
    for (int i = 0; i < N / PASS; ++i)
      words_to_lds(g + (r0 + PASS * i) * ss, off, lds + (i * NT + wid * 64) * 16);
  } else {
#pragma unroll
    for (int i = 0; i < N / PASS; ++i) {
      const int r = min(r0 + PASS * i, rows - 1);
      words_to_lds(g + r * ss, min(st_r, rows - 1 - r) * pitch + st_c,
                   lds + (i * NT + wid * 64) * 16);
    }
  }
}

__device__ __forceinline__ frag_u read_row(const char* lds, int lane_at, int c) {
  frag_u f;
  f.u4 = *(const uint4v*)(lds + (lane_at ^ (c * 32)));
  return f;
}
// rows 16 c ... of columns 32 nb ...
__device__ __forceinline__ bf16x8 read_turned(char* lds, int lane_at, int c,
                                              int nb) {
  union { tr4 t[2]; bf16x8 bf; } f;
#pragma unroll
  for (int u = 0; u < 2; ++u)
    f.t[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_tr4)(lds + (lane_at ^ (nb * 64 + u * 32)) + c * 4096 + u * 2048));
  return f.bf;
}
// [d][lane] accumulators to a row of the lane
__device__ __forceinline__ void store_turned(const f32x16* acc, float scale,
                                             short* dst, int hi) {
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg)
      *(uint2*)(dst + 32 * nb + 8 * rg + 4 * hi) =
          uint2{pack_bf16x2(acc[nb][4 * rg] * scale, acc[nb][4 * rg + 1] * scale),
                pack_bf16x2(acc[nb][4 * rg + 2] * scale,
                            acc[nb][4 * rg + 3] * scale)};
}

// 128 kv rows, 64 q rows a step: wave w takes kv rows 32 (w / 2) ... and every
// other 32 q rows; the two sums of a kv row meet in LDS at the end.  Sums of 32
// kv rows and all of d (128 registers) leave no room for the keys and values,
// which are read from LDS (1.5 KB a product, three quarters of what LDS gives
// at the full matrix rate); with the keys in registers 4 waves of a workgroup
// spilled and took 2840 us.
__global__ void __launch_bounds__(512, 2) fa_bwd_dkdv_kernel(BwdArgs a) {
  constexpr int TILE_B = 64 * FA_D * 2;
  // apart by name, so that a read of one need not wait for the words on their
  // way into the other
  __shared__ __attribute__((aligned(16))) char kb[128 * FA_D * 2];
  __shared__ __attribute__((aligned(16))) char vb[128 * FA_D * 2];
  __shared__ __attribute__((aligned(16))) char q0b[TILE_B], q1b[TILE_B];
  __shared__ __attribute__((aligned(16))) char d0b[TILE_B], d1b[TILE_B];
  // lse * log2(e) and delta of a step's rows
  __shared__ __attribute__((aligned(16))) float ld0[128], ld1[128];
  __shared__ int odd;          // is there a row whose lse is no number?

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int S = a.S, window = a.window;

  // heads on x, kv-blocks on y: causal work DEcreases with kv-block index,
  // so ascending y already dispatches biggest-first
  const int k0 = blockIdx.y * 128, hd = blockIdx.x, b = blockIdx.z;
  const int heads = a.Hq / a.Hdk, h = hd * heads;
  const int hkv = h / (a.Hq / a.Hkv);
  const int g = wid >> 1, half = wid & 1;
  const int kw0 = k0 + g * 32;           // this wave's first kv row
  const int my_k = kw0 + col;
  const short* qg = a.q + b * a.q_bs + h * a.q_hs;
  const short* dg = a.dout + b * a.do_bs + h * a.do_hs;
  const float* lse = a.lse + ((long)b * a.Hq + h) * S;
  const float* delta = a.delta + ((long)b * a.Hq + h) * S;

  f32x16 dv[4] = {}, dk[4] = {};         // [d][kv]
  // a masked score has no weight, whatever the sign of the scale
  const float s2 = a.scale == 0.f ? 1e-37f : a.scale * LOG2E;
  const float gone = s2 > 0.f ? -INFINITY : INFINITY;
  // this lane in the wave's rows of a q tile, of the kv tile
  const int rq = row_lane(col, hi) + half * 8192, tq = tr_lane(lane) + half * 8192;
  const int rk = row_lane(col, hi) + g * 8192;

  const int q_start = a.causal ? k0 : 0;
  // sliding window: q attends k iff k <= q < k + window
  const int q_end = window > 0 ? min(S, k0 + 127 + window) : S;

  // Tiles of the first q head, then of the next ones: what is asked for next
  int next = q_start;
  // (two waves' numbers go into LDS only behind the step: where they are asked for,
  // those two would wait for them, and all others for these two)
  float nl = 0.f;
  // (a row whose lse is no number has no weights in the steps: masked places would
  // get them too, and keys that the row does not see)
  if (tid == 0) odd = 0;
  auto issue = [&](char* qb, char* db) __attribute__((always_inline)) {
    if (wid < 2) nl = (wid ? delta : lse)[min(next + lane, S - 1)];
    fill_rows<64, 512>(qg, a.q_ss, next, S, qb);
    fill_rows<64, 512>(dg, a.do_ss, next, S, db);
  };
  auto leave = [&](float* ld) __attribute__((always_inline)) {
    if (wid == 0) {
      if (!(nl > -INFINITY)) odd = 1;
      ld[tid] = fabsf(nl) < INFINITY ? nl * LOG2E : FLT_MAX;
    }
    if (wid == 1) ld[tid] = nl;
  };
  auto advance = [&]() __attribute__((always_inline)) {
    if ((next += 64) < q_end) return;
    next = q_start;
    qg += a.q_hs;
    dg += a.do_hs;
    lse += S;
    delta += S;
  };

  auto step = [&](int qt, char* qb, char* db, const float* ld_t)
      __attribute__((always_inline)) {
    const int q0 = qt + 32 * half;
    if ((a.causal && q0 + 31 < kw0) || q0 >= S ||
        (window > 0 && q0 >= kw0 + 31 + window))
      return;
    const float* ld = ld_t + half * 32;
    // S^T and dP^T: q in the accumulators' rows, kv in the lanes.  Every product
    // has its own piece of the vector work beside it and reads two ahead.
    f32x16 s = {}, dp = {};
    frag_u f[3][2];
    auto rows_s = [&](int c) __attribute__((always_inline)) {
      f[c % 3][0] = read_row(qb, rq, c);
      f[c % 3][1] = read_row(kb, rk, c);
    };
    auto rows_dp = [&](int c) __attribute__((always_inline)) {
      f[(c + 2) % 3][0] = read_row(db, rq, c);
      f[(c + 2) % 3][1] = read_row(vb, rk, c);
    };
    rows_s(0);
    rows_s(1);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (c < 6) rows_s(c + 2); else rows_dp(c - 6);
      __builtin_amdgcn_sched_barrier(0);
      s = mfma_bf16(f[c % 3][0].bf, f[c % 3][1].bf, s);
      __builtin_amdgcn_sched_barrier(0);
    }
    if ((a.causal && q0 < kw0 + 31) || q0 + 32 > S ||
        (window > 0 && q0 + 31 >= kw0 + window)) {
      asm volatile("");        // a branch: not selects on every tile
      // row r + 4 hi of the tile sees this lane's key if first <= r < last
      const int first = (a.causal ? my_k - q0 : 0) - 4 * hi;
      const int last = min(S, window > 0 ? my_k + window : S) - q0 - 4 * hi;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int j = acc_row(r, 0);
        s[r] = j < first || j >= last ? gone : s[r];
      }
    }
    frag_u pf[2], df[2];
    bf16x8 t[3];
    f4v l[2];
    l[0] = *(const f4v*)(ld + 4 * hi);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (c < 6) rows_dp(c + 2); else t[c - 6] = read_turned(db, tq, 0, c - 6);
      if (c % 2 == 0)            // then delta
        l[(c / 2 + 1) % 2] = *(const f4v*)(
            ld + (c < 6 ? 8 * (c / 2 + 1) : 64) + 4 * hi);
      __builtin_amdgcn_sched_barrier(0);
      dp = mfma_bf16(f[(c + 2) % 3][0].bf, f[(c + 2) % 3][1].bf, dp);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = 2 * c + i;
        s[r] = __builtin_amdgcn_exp2f(s[r] * s2 - l[c / 2 % 2][r % 4]);
      }
      pf[c / 4].u[c % 4] = pack_bf16x2(s[2 * c], s[2 * c + 1]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int n = i + 2;       // fragments of dO, then of Q
      if (n < 16) t[n % 3] = read_turned(n < 8 ? db : qb, tq, n / 4 % 2, n % 4);
      if (i < 6 && i % 2 == 0)
        l[(i / 2 + 1) % 2] = *(const f4v*)(ld + 64 + 8 * (i / 2 + 1) + 4 * hi);
      __builtin_amdgcn_sched_barrier(0);
      f32x16& to = i < 8 ? dv[i % 4] : dk[i % 4];
      to = mfma_bf16(t[i % 3], (i < 8 ? pf : df)[i / 4 % 2].bf, to);
      if (i < 8) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
          s[2 * i + j] *= dp[2 * i + j] - l[i / 2 % 2][(2 * i + j) % 4];
        df[i / 4].u[i % 4] = pack_bf16x2(s[2 * i], s[2 * i + 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  fill_rows<128, 512>(a.k + b * a.k_bs + hkv * a.k_hs, a.k_ss, k0, S, kb);
  fill_rows<128, 512>(a.v + b * a.v_bs + hkv * a.v_hs, a.v_ss, k0, S, vb);
  const int steps = heads * ((q_end - q_start + 63) / 64);
  issue(q0b, d0b);
  leave(ld0);
  __syncthreads();             // also waits for the words on their way
  for (int i = 0; i < steps; i += 2) {
    int q0 = next;
    advance();
    if (i + 1 < steps) issue(q1b, d1b);
    step(q0, q0b, d0b, ld0);
    leave(ld1);
    __syncthreads();
    if (i + 1 >= steps) break;
    q0 = next;
    advance();
    if (i + 2 < steps) issue(q0b, d0b);
    step(q0, q1b, d1b, ld1);
    leave(ld0);
    __syncthreads();
  }

  // 16 accumulators of one wave in 4 KB: the odd wave of a pair hands over dV
  // in kb and vb, then dK
  auto meet = [&](f32x16* acc, char* room) __attribute__((always_inline)) {
    float* m = (float*)room + lane;
    if (half)
#pragma unroll
      for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) m[(nb * 16 + r) * 64] = acc[nb][r];
    __syncthreads();
    if (!half)
#pragma unroll
      for (int nb = 0; nb < 4; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[nb][r] += m[(nb * 16 + r) * 64];
  };
  char* room = (g & 1 ? vb : kb) + (g >> 1) * 16384;   // all have been read
  meet(dv, room);
  __syncthreads();
  meet(dk, room);
  if (half || my_k >= S) return;
  short* to_v = a.dv + b * a.dv_bs + hd * a.dv_hs + my_k * a.dv_ss;
  short* to_k = a.dk + b * a.dk_bs + hd * a.dk_hs + my_k * a.dk_ss;
  store_turned(dv, 1.f, to_v, hi);
  store_turned(dk, a.scale, to_k, hi);
  if (!odd) return;
  // keys that an odd row sees
  lse = a.lse + ((long)b * a.Hq + h) * S;
  bool seen = false;
  for (int n = 0; n < heads; ++n, lse += S)
    for (int q = max(q_start, a.causal ? my_k : 0);
         q < (window > 0 ? min(S, my_k + window) : S); ++q)
      seen |= !(lse[q] > -INFINITY);
  if (!seen) return;
  for (int nb = 0; nb < 4; ++nb) dv[nb] = f32x16{} + NAN;
  store_turned(dv, 1.f, to_v, hi);
  store_turned(dv, 1.f, to_k, hi);
}

__global__ void __launch_bounds__(256, 2) fa_bwd_dq_kernel(BwdArgs a) {
  constexpr int TILE_B = 64 * FA_D * 2;
  __shared__ __attribute__((aligned(16))) char k0b[TILE_B], k1b[TILE_B];
  __shared__ __attribute__((aligned(16))) char v0b[TILE_B], v1b[TILE_B];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int S = a.S, window = a.window;

  // heads on x, q-blocks on y reversed: biggest-causal-work first
  const int q0 = (int)(gridDim.y - 1 - blockIdx.y) * 128;
  const int h = near_head(blockIdx.x, a.Hq), b = blockIdx.z;
  const int hkv = h / (a.Hq / a.Hkv);
  const int qw0 = q0 + wid * 32, my_q = qw0 + col;
  const long q_ld = min(my_q, S - 1);

  // Q, dO fragments in registers (lane: row q=col within wave tile)
  frag_u qf[8], dof[8];
  {
    const short* qs = a.q + b * a.q_bs + h * a.q_hs + q_ld * a.q_ss + hi * 8;
    const short* ds = a.dout + b * a.do_bs + h * a.do_hs + q_ld * a.do_ss + hi * 8;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      qf[c].u4 = *(const uint4v*)(qs + c * 16);
      dof[c].u4 = *(const uint4v*)(ds + c * 16);
    }
  }
  const long at = ((long)b * a.Hq + h) * S + q_ld;
  const float lse2 = a.lse[at] * LOG2E;
  // delta = sum of dO O over the row, half of it in this lane
  float dlt = 0.f;
  {
    const short* os = a.out + b * a.o_bs + h * a.o_hs + q_ld * a.o_ss + hi * 8;
    s8v o[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) o[c] = *(const s8v*)(os + c * 16);
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        dlt += __uint_as_float(dof[c].u[j] << 16) * bits2f(o[c][2 * j]) +
               __uint_as_float(dof[c].u[j] & 0xffff0000u) * bits2f(o[c][2 * j + 1]);
    dlt += __shfl_xor(dlt, 32, 64);
    if (hi == 0 && my_q < S) a.delta[at] = dlt;
  }
  const float s2 = a.scale == 0.f ? 1e-37f : a.scale * LOG2E;
  const float gone = s2 > 0.f ? -INFINITY : INFINITY;

  f32x16 dq[4] = {};                     // [d][q]
  const int rx = row_lane(col, hi), tx = tr_lane(lane);
  const short* kg = a.k + b * a.k_bs + hkv * a.k_hs;
  const short* vg = a.v + b * a.v_bs + hkv * a.v_hs;

  const int kv_end = a.causal ? min(S, q0 + 128) : S;
  // sliding window: this q block's earliest active kv row (tile-aligned)
  const int kv_begin = window > 0 ? max(0, q0 - window + 1) & ~63 : 0;

  auto issue = [&](int k0, char* kb, char* vb) __attribute__((always_inline)) {
    fill_rows<64, 256>(kg, a.k_ss, k0, S, kb);
    fill_rows<64, 256>(vg, a.v_ss, k0, S, vb);
  };
  // 32 keys
  auto step = [&](int k0, char* kb, const char* vb) __attribute__((always_inline)) {
    if ((a.causal && k0 > qw0 + 31) || k0 >= S ||
        (window > 0 && k0 + 31 + window <= qw0))
      return;
    // S^T and dP^T: keys in the accumulators' rows, q in the lanes.  As above,
    // every product has vector work beside it and reads two ahead.
    f32x16 s = {}, dp = {};
    frag_u f[3];
    f[0] = read_row(kb, rx, 0);
    f[1] = read_row(kb, rx, 1);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      f[(c + 2) % 3] = c < 6 ? read_row(kb, rx, c + 2) : read_row(vb, rx, c - 6);
      __builtin_amdgcn_sched_barrier(0);
      s = mfma_bf16(f[c % 3].bf, qf[c].bf, s);
      __builtin_amdgcn_sched_barrier(0);
    }
    if ((a.causal && k0 + 31 > qw0) || k0 + 32 > S ||
        (window > 0 && k0 <= qw0 + 31 - window)) {
      asm volatile("");        // a branch: not selects on every tile
      // key r + 4 hi of the tile is seen if first < r <= last
      const int i0 = my_q - k0;
      const int last = min(a.causal ? i0 : 32, S - 1 - k0) - 4 * hi;
      const int first = (window > 0 ? i0 - window : -1) - 4 * hi;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int j = acc_row(r, 0);
        s[r] = j > last || j <= first ? gone : s[r];
      }
    }
    bf16x8 t[3];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (c < 6) f[(c + 4) % 3] = read_row(vb, rx, c + 2);
      else t[c - 6] = read_turned(kb, tx, 0, c - 6);
      __builtin_amdgcn_sched_barrier(0);
      dp = mfma_bf16(f[(c + 2) % 3].bf, dof[c].bf, dp);
#pragma unroll
      for (int r = 2 * c; r < 2 * c + 2; ++r)
        s[r] = __builtin_amdgcn_exp2f(s[r] * s2 - lse2);
      __builtin_amdgcn_sched_barrier(0);
    }
    frag_u df[2];
    auto weigh = [&](int u) __attribute__((always_inline)) {
      s[2 * u] *= dp[2 * u] - dlt;
      s[2 * u + 1] *= dp[2 * u + 1] - dlt;
      df[u / 4].u[u % 4] = pack_bf16x2(s[2 * u], s[2 * u + 1]);
    };
#pragma unroll
    for (int u = 0; u < 4; ++u) weigh(u);
    // dQ^T[d][q] += K^T dS^T
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int n = i + 2;
      if (n < 8) t[n % 3] = read_turned(kb, tx, n / 4, n % 4);
      __builtin_amdgcn_sched_barrier(0);
      dq[i % 4] = mfma_bf16(t[i % 3], df[i / 4].bf, dq[i % 4]);
      if (i < 4) weigh(4 + i);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto tile = [&](int k0, char* kb, const char* vb) __attribute__((always_inline)) {
    step(k0, kb, vb);
    step(k0 + 32, kb + 8192, vb + 8192);
  };

  issue(kv_begin, k0b, v0b);
  __syncthreads();             // also waits for the words on their way
  for (int k0 = kv_begin; k0 < kv_end; k0 += 128) {
    const bool more = k0 + 64 < kv_end;
    if (more) issue(k0 + 64, k1b, v1b);
    tile(k0, k0b, v0b);
    __syncthreads();
    if (!more) break;
    if (k0 + 128 < kv_end) issue(k0 + 128, k0b, v0b);
    tile(k0 + 64, k1b, v1b);
    __syncthreads();
  }
  if (my_q >= S) return;
  store_turned(dq, a.scale, a.dq + b * a.dq_bs + h * a.dq_hs + my_q * a.dq_ss, hi);
}

// ---------------------------------------------------------------------------
// dK and dV of a kv head: the 32-bit sum of those of its q heads, which are
// [B][Hq][S][128].  Streams at memory rate: 16 lanes a row.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
fa_bwd_reduce_kernel(const short* __restrict__ kq, const short* __restrict__ vq,
                     short* __restrict__ dk, short* __restrict__ dv, long rows,
                     int Hkv, int rep, int S, long dk_bs, long dk_hs,
                     long dk_ss, long dv_bs, long dv_hs, long dv_ss) {
  const bool is_v = blockIdx.y;
  const int sub = threadIdx.x & 15;
  const long step = (long)gridDim.x * 16;
  for (long row = (long)blockIdx.x * 16 + (threadIdx.x >> 4); row < rows;
       row += step) {
    const long bh = row / S, s = row % S;
    const short* src = (is_v ? vq : kq) + (bh * rep * S + s) * FA_D + sub * 8;
    float acc[8] = {};
    for (int r = 0; r < rep; ++r) {
      const s8v x = *(const s8v*)(src + (long)r * S * FA_D);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] += bits2f(x[j]);
    }
    const long b = bh / Hkv, h = bh % Hkv;
    short* dst = (is_v ? dv + b * dv_bs + h * dv_hs + s * dv_ss
                       : dk + b * dk_bs + h * dk_hs + s * dk_ss) + sub * 8;
    uint4v o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = pack_bf16x2(acc[2 * j], acc[2 * j + 1]);
    *(uint4v*)dst = o;
  }
}

extern "C" void flash_attn_bwd_reduce(const void* kq, const void* vq, void* dk,
                                      void* dv, int B, int Hq, int Hkv, int S,
                                      const long* st, hipStream_t stream) {
  // st = 6 longs: (bs, hs, ss) x (dk, dv)
  const long rows = (long)B * Hkv * S, need = (rows + 15) / 16;
  const dim3 grid(need < 8192 ? (unsigned)need : 8192, 2);
  fa_bwd_reduce_kernel<<<grid, 256, 0, stream>>>(
      (const short*)kq, (const short*)vq, (short*)dk, (short*)dv, rows, Hkv,
      Hq / Hkv, S, st[0], st[1], st[2], st[3], st[4], st[5]);
}

// ---------------------------------------------------------------------------
extern "C" void flash_attn_bwd_strided(
    const void* q, const void* k, const void* v, const void* out,
    const void* dout, const void* lse, void* delta, void* dq, void* dk,
    void* dv, int B, int Hq, int Hkv, int Hdk, int S, float scale, int causal,
    int window, const long* st, hipStream_t stream) {
  // st = 24 longs: (bs, hs, ss) x (q, k, v, o, dout, dq, dk, dv); dk and dv of
  // Hdk heads, Hkv <= Hdk <= Hq, each dividing the next
  const BwdArgs a{(const short*)q, (const short*)k, (const short*)v,
                  (const short*)out, (const short*)dout, (const float*)lse,
                  (float*)delta, (short*)dq, (short*)dk, (short*)dv, Hq, Hkv,
                  Hdk, S, causal, window, scale,
                  st[0], st[1], st[2], st[3], st[4], st[5], st[6], st[7], st[8],
                  st[9], st[10], st[11], st[12], st[13], st[14], st[15], st[16],
                  st[17], st[18], st[19], st[20], st[21], st[22], st[23]};
  const int blocks = (S + 127) / 128;
  fa_bwd_dq_kernel<<<dim3(Hq, blocks, B), 256, 0, stream>>>(a);
  fa_bwd_dkdv_kernel<<<dim3(Hdk, blocks, B), 512, 0, stream>>>(a);
}

extern "C" void flash_attn_bwd(const void* q, const void* k, const void* v,
                               const void* out, const void* dout,
                               const void* lse, void* delta, void* dq,
                               void* dk, void* dv, int B, int Hq, int Hkv,
                               int S, float scale, int causal,
                               hipStream_t stream) {
  const long qd[3] = {(long)Hq * S * FA_D, (long)S * FA_D, FA_D};
  const long kd[3] = {(long)Hkv * S * FA_D, (long)S * FA_D, FA_D};
  long st[24];
  for (int i = 0; i < 3; ++i) {
    st[0 + i] = qd[i];            // q
    st[3 + i] = kd[i];            // k
    st[6 + i] = kd[i];            // v
    st[9 + i] = qd[i];            // out
    st[12 + i] = qd[i];           // dout
    st[15 + i] = qd[i];           // dq
    st[18 + i] = qd[i];           // dk (per-Q-head buffers)
    st[21 + i] = qd[i];           // dv
  }
  flash_attn_bwd_strided(q, k, v, out, dout, lse, delta, dq, dk, dv, B, Hq,
                         Hkv, Hq, S, scale, causal, 0, st, stream);
}
