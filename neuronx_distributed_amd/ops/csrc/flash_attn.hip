// FlashAttention forward for CDNA4 (gfx950) — hand-written MFMA kernel.
//
// Replaces the reference's NKI flash kernel K1 (reference
// kernels/flash_attn.py:18,51-63).
//   * 4 waves/WG, each wave owns 32 q rows, two WGs a CU; KV tiles of 64 go
//     straight from memory into two LDS buffers.
//   * swapped QK^T — mfma(A=K, B=Q^T) — so each lane's softmax stats are
//     for ONE q row (l&31): row max / rescale / denom are lane-local
//     (+ one exchange with the partner half-wave).
//   * P never leaves the registers: the accumulator's order of keys is the
//     contraction order of P V, and V^T is read from LDS in that order by
//     transposing reads.
//   * O is accumulated TRANSPOSED (O^T[d][q], q = lane) so the online
//     rescale is a per-lane scalar multiply.
//   * GQA: kv head = q head / (Hq/Hkv); causal masking per element on
//     diagonal tiles only, whole-tile skip below the diagonal.
//
// Bound by the matrix cores together with the exponentials and the rest of
// the vector work: at 8192 tokens, 32/8 heads, the matrix pipes are 51 % busy
// (rocprofv3), LDS 25 %.  845 us before (8 waves, one WG a CU, values turned
// by scattered writes, masks on every tile), 575 us (956 TFLOP/s) now: 600
// with the loads into LDS and masks on the boundary alone, 580 with the next
// tile's scores beside this tile's exponentials, 575 with the order below.
// 64 q rows a wave (half the LDS reads, one wave a SIMD) took 665.  A running
// maximum that lags behind by up to 2^8 took 570, but the largest weight of a
// row is then not exactly one, and the error grows by 5 %.
//
// Layouts: q,k,v,out (B, H, S, D) bf16 contiguous, D = 128; lse (B,Hq,S)
// f32 (natural-log row logsumexp, saved for backward).

#include "common.h"
#include "flash_attn.h"
#include "mfma.h"
#include "lds.h"

#define FA_D 128
#define FA_KV 64       // kv tile
#define LOG2E 1.4426950408889634f
#define NEG_INF (-1e30f)
#define FA_QBLK 128    // q rows of a workgroup: 4 waves of 32
#define FA_TILE_B (FA_KV * FA_D * 2)   // 16 KB: a key or value tile

struct FwdArgs {
  const short *q, *k, *v;
  short* o;
  float* lse;
  int Hq, Hkv, S, causal, window;
  float scale;
  // element strides of (batch, head, seq); the last dim (d) is dense.
  // BHSD contiguous: (H*S*128, S*128, 128).  BSHD transpose views (no-copy
  // model layout): (S*H*128, 128, H*128).
  long q_bs, q_hs, q_ss, k_bs, k_hs, k_ss, v_bs, v_hs, v_ss, o_bs, o_hs, o_ss;
};

// window > 0: Mistral-style sliding window — q row i attends kv rows
// [i - window + 1, i] (causal implied); whole tiles outside the band are
// skipped, boundary tiles masked per element.
__global__ void __launch_bounds__(256, 2) flash_fwd_kernel(FwdArgs a) {
  // two key and two value tiles; apart by name, so that a read of one need
  // not wait for the words on their way into the other
  __shared__ __attribute__((aligned(16))) char k0[FA_TILE_B], k1[FA_TILE_B];
  __shared__ __attribute__((aligned(16))) char v0[FA_TILE_B], v1[FA_TILE_B];

  const int tid = threadIdx.x, lane = tid & 63;
  // readfirstlane: provably wave-uniform -> scalar branches
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int S = a.S, window = a.window;

  // Dispatch mapping (causal LPT): heads on x, q-blocks on y REVERSED so
  // the largest-causal-work blocks launch first and early finishers absorb
  // the small diagonal blocks.
  const int q0 = (int)(gridDim.y - 1 - blockIdx.y) * FA_QBLK;
  const int h = near_head(blockIdx.x, a.Hq), b = blockIdx.z;
  const int hkv = h / (a.Hq / a.Hkv);
  const int qw0 = q0 + wid * 32;         // this wave's first q row
  const int my_q = qw0 + col;            // this lane's q row

  // a negative scale turns the sign of the queries, so that the largest
  // product is the largest score
  const uint flip = a.scale < 0.f ? 0x80008000u : 0u;
  const float s2 = fabsf(a.scale) * LOG2E;
  frag_u qf[8];
  {
    const short* src = a.q + b * a.q_bs + h * a.q_hs +
                       (long)min(my_q, S - 1) * a.q_ss + hi * 8;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      qf[c].u4 = *(const uint4v*)(src + c * 16);
      qf[c].u4 ^= flip;
    }
  }

  f32x16 ot[4] = {};                     // O^T: d-block, rows d, col q
  float m_run = NEG_INF;                 // running max (exp2 domain)
  float l_run = 0.f;                     // sum over this half wave's keys

  const int kv_end = a.causal ? min(S, q0 + FA_QBLK) : S;
  const int ntiles = (kv_end + FA_KV - 1) / FA_KV;
  // the WG starts at its earliest window tile; [w_begin, w_end) are the tiles
  // that a row of this wave sees
  const int t_begin = window > 0 ? max(0, q0 - window + 1) / FA_KV : 0;
  const int w_begin = window > 0 ? max(0, qw0 - window + 1) / FA_KV : 0;
  const int w_end = ((a.causal ? min(S, qw0 + 32) : S) + FA_KV - 1) / FA_KV;

  // Tiles go from memory into LDS as they are, 16 bytes a lane; the rotation
  // of a row's slots (bank conflicts) is done on the source.  Keys are read
  // as rows, values by transposing reads.  Both rotations repeat after 16
  // rows, so the rows st_r + 16 i of a thread have the same.
  const int st_r = tid >> 4, st_s = tid & 15;
  const int st_c = (st_s ^ row_turn(st_r)) * 16;
  const short* kg = a.k + b * a.k_bs + hkv * a.k_hs;
  const short* vg = a.v + b * a.v_bs + hkv * a.v_hs;
  auto issue = [&](const short* g, long ss, int t, char* lds) {
    const int kv0 = t * FA_KV;
    const int pitch = (int)ss * 2;
    if (kv0 + FA_KV <= S) {
      const int off = st_r * pitch + st_c;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        words_to_lds(g + (kv0 + 16 * i) * ss, off, lds + (i * 256 + wid * 64) * 16);
    } else {                   // rows past the end read the last one
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = min(kv0 + 16 * i, S - 1);
        words_to_lds(g + r * ss, min(st_r, S - 1 - r) * pitch + st_c,
                     lds + (i * 256 + wid * 64) * 16);
      }
    }
  };
  const int kx = row_lane(col, hi), vx = tr_lane(lane);

  // S^T[k][q] = K Q^T
  auto scores = [&](f32x16* s, const char* kbuf) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) s[kb] = f32x16{};
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        frag_u kf;
        kf.u4 = *(const uint4v*)(kbuf + (kx ^ (c * 32)) + kb * 8192);
        s[kb] = mfma_bf16(kf.bf, qf[c].bf, s[kb]);
      }
  };
  // masks of tile t (only on a boundary) and the running maximum
  auto level = [&](f32x16* s, int t) {
    const int kv0 = t * FA_KV;
    if ((a.causal && kv0 + FA_KV - 1 > qw0) || kv0 + FA_KV > S ||
        (window > 0 && kv0 <= qw0 + 31 - window)) {
      asm volatile("");        // a branch: not selects on every tile
      // key j + 4 hi of the tile is seen if first < j <= last
      const int i0 = my_q - kv0;
      const int last = min(a.causal ? i0 : FA_KV, S - 1 - kv0) - 4 * hi;
      const int first = (window > 0 ? i0 - window : -1) - 4 * hi;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = 32 * kb + acc_row(r, 0);
          s[kb][r] = j > last || j <= first ? -INFINITY : s[kb][r];
        }
    }
    float mt = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, s[kb][r]);
    mt = max_halves(mt) * s2;
    if (__ballot(mt > m_run)) {
      const float m_new = fmaxf(m_run, mt);
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) ot[nb] *= alpha;
    }
  };
  // weights, as fragments of P^T: the accumulator's order of keys is that in
  // which the transposing reads give the values
  auto weigh = [&](f32x16* s, frag_u* pf) {
    float ps = 0.f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[kb][r] = __builtin_amdgcn_exp2f(s[kb][r] * s2 - m_run);
        ps += s[kb][r];
      }
    l_run += ps;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        pf[c].u[u] = pack_bf16x2(s[c >> 1][8 * (c & 1) + 2 * u],
                                 s[c >> 1][8 * (c & 1) + 2 * u + 1]);
  };
  // O^T[d][q] += V^T P^T
  auto gather = [&](const frag_u* pf, char* vbuf) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        union { tr4 t[2]; bf16x8 bf; } vf;
#pragma unroll
        for (int u = 0; u < 2; ++u)
          vf.t[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (lds_tr4)(vbuf + (vx ^ (nb * 64 + u * 32)) + c * 4096 + u * 2048));
        ot[nb] = mfma_bf16(vf.bf, pf[c].bf, ot[nb]);
      }
  };
  // Tile t's weights and values, while the next tile's scores are made: the
  // products of one run beside the exponentials of the other.
  auto step = [&](int t, f32x16* s, f32x16* next, const char* kbuf, char* vbuf) {
    const bool now = t >= w_begin && t < w_end;
    const bool then = t + 1 >= w_begin && t + 1 < w_end;
    frag_u pf[4];
    if (now) {
      level(s, t);
      scores(next, kbuf);      // past the wave's last tile they are not used
      weigh(s, pf);
      gather(pf, vbuf);
      // four reads ahead; then a product, a read and exponentials in turn;
      // then the products with the values and what is left
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 5, 0);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      }
    } else if (then) {
      scores(next, kbuf);
    }
  };

  f32x16 sa[2], sb[2];
  issue(kg, a.k_ss, t_begin, k0);
  issue(vg, a.v_ss, t_begin, v0);
  if (t_begin + 1 < ntiles) issue(kg, a.k_ss, t_begin + 1, k1);
  __syncthreads();             // also waits for the words on their way
  if (t_begin >= w_begin && t_begin < w_end) scores(sa, k0);
  __syncthreads();
  for (int t = t_begin; t < ntiles; t += 2) {
    // keys of t + 1 and values of t are there
    if (t + 2 < ntiles) issue(kg, a.k_ss, t + 2, k0);
    if (t + 1 < ntiles) issue(vg, a.v_ss, t + 1, v1);
    step(t, sa, sb, k1, v0);
    __syncthreads();
    if (t + 1 >= ntiles) break;
    if (t + 3 < ntiles) issue(kg, a.k_ss, t + 3, k1);
    if (t + 2 < ntiles) issue(vg, a.v_ss, t + 2, v0);
    step(t + 1, sb, sa, k0, v1);
    __syncthreads();
  }

  // ---- epilogue: normalize, store O (transposed back) and LSE ---------
  const float l = l_run + __shfl_xor(l_run, 32, 64);
  if (my_q >= S) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  short* dst = a.o + b * a.o_bs + h * a.o_hs + my_q * a.o_ss;
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg)
      *(uint2*)(dst + 32 * nb + 8 * rg + 4 * hi) =
          uint2{pack_bf16x2(ot[nb][4 * rg] * inv, ot[nb][4 * rg + 1] * inv),
                pack_bf16x2(ot[nb][4 * rg + 2] * inv, ot[nb][4 * rg + 3] * inv)};
  if (hi == 0 && a.lse)        // natural log; scores were in the exp2 domain
    a.lse[((long)b * a.Hq + h) * S + my_q] =
        m_run * 0.6931471805599453f + __logf(l);
}

extern "C" void flash_attn_fwd_strided(
    const void* q, const void* k, const void* v, void* out, void* lse,
    int B, int Hq, int Hkv, int S, float scale, int causal, int window,
    const long* st, hipStream_t stream) {
  // st = 12 longs: (bs, hs, ss) x (q, k, v, o)
  const FwdArgs a{(const short*)q, (const short*)k, (const short*)v,
                  (short*)out, (float*)lse, Hq, Hkv, S, causal, window, scale,
                  st[0], st[1], st[2], st[3], st[4], st[5], st[6], st[7],
                  st[8], st[9], st[10], st[11]};
  const dim3 grid(Hq, (S + FA_QBLK - 1) / FA_QBLK, B);
  flash_fwd_kernel<<<grid, 256, 0, stream>>>(a);
}

static void launch_fwd_dense(const void* q, const void* k, const void* v,
                             void* out, void* lse, int B, int Hq, int Hkv,
                             int S, float scale, int causal, int window,
                             hipStream_t stream) {
  const long h = (long)S * FA_D;
  const long st[12] = {Hq * h, h, FA_D, Hkv * h, h, FA_D,
                       Hkv * h, h, FA_D, Hq * h, h, FA_D};
  flash_attn_fwd_strided(q, k, v, out, lse, B, Hq, Hkv, S, scale, causal,
                         window, st, stream);
}

extern "C" void flash_attn_fwd(const void* q, const void* k, const void* v,
                               void* out, void* lse, int B, int Hq, int Hkv,
                               int S, float scale, int causal,
                               hipStream_t stream) {
  launch_fwd_dense(q, k, v, out, lse, B, Hq, Hkv, S, scale, causal, 0, stream);
}

extern "C" void flash_attn_fwd_window(const void* q, const void* k,
                                      const void* v, void* out, void* lse,
                                      int B, int Hq, int Hkv, int S,
                                      float scale, int window,
                                      hipStream_t stream) {
  launch_fwd_dense(q, k, v, out, lse, B, Hq, Hkv, S, scale, 1, window, stream);
}
