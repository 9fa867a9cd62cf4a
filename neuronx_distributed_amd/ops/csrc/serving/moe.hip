// Mixture of experts for ragged batches: routing, grouping and the grouped
// matrix products.  Every launch has a size that the host knows from the
// number of rows alone, so a decode step can be captured in a graph.
//
//   sv_moe_plan    logits -> chosen experts and weights of each row; (row,
//                  choice) pairs grouped by expert: order and tiles
//   sv_moe_gemm    one grouped product: gate/up with the gated activation in
//                  its epilogue, or down
//
// A pair is row * top + choice.  The order lists the pairs expert by expert;
// a slot is a place in it.  Gate/up reads row pair / top and writes its slot,
// down reads the slot and writes the pair; the weighted sum over a row's
// pairs is taken by the residual norm.

#include "ring.h"

#define MOE_MAX_EXPERTS 512

// ---------------------------------------------------------------------------
// route and plan
// ---------------------------------------------------------------------------
struct MoePlanArgs {
  const float* z;           // [T][E] logits
  const void* bias;         // [E] or null
  int* idx;                 // [T * top] chosen experts
  float* coef;              // [T * top] their weights
  int* order;               // [T * top] slot -> pair
  int* tiles;               // [max_tiles][4]: expert, first slot, slots, number
                            //   of tiles; no slots past it
  int T, E, top, tile_rows, max_tiles;
  int kind;                 // 0: weights are a softmax over the chosen;
                            // 1: scores sigmoid(z), chosen by score + bias;
                            // 2: weights are a softmax over all experts
  int groups, keep;         // experts of the best groups only (groups > 1)
  int best;                 // a group counts the sum of its 1 or 2 largest
};

// Keep the choice scores v of the best groups of neighbours, drop the others.
// `mem` is the wave's own.
template <int NV>
__device__ __forceinline__ void best_groups(const MoePlanArgs& a, float* v,
                                            float* mem) {
  const int lane = threadIdx.x & 63, size = a.E / a.groups;
#pragma unroll
  for (int i = 0; i < NV; ++i) mem[i * 64 + lane] = v[i];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  float score = -INFINITY;
  if (lane < a.groups) {
    float m1 = -INFINITY, m2 = -INFINITY;
    for (int j = 0; j < size; ++j) {
      const float x = mem[lane * size + j];
      m2 = fmaxf(m2, fminf(m1, x));
      m1 = fmaxf(m1, x);
    }
    score = size > 1 && a.best > 1 ? m1 + m2 : m1;
  }
  __builtin_amdgcn_wave_barrier();
  unsigned long long kept = 0;
  for (int k = 0; k < a.keep; ++k) {
    const bool open = lane < a.groups && !(kept >> lane & 1);
    float best = open ? score : -INFINITY;
    int at = open ? lane : 64;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const float ob = __shfl_xor(best, off, 64);
      const int oa = __shfl_xor(at, off, 64);
      if (ob > best || (ob == best && oa < at)) {
        best = ob;
        at = oa;
      }
    }
    kept |= 1ull << (at & 63);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = i * 64 + lane;
    if (e < a.E && !(kept >> (e / size) & 1)) v[i] = -INFINITY;
  }
}

// the largest value of the wave
__device__ __forceinline__ float wave_max(float x) {
#define TURN(n)                                                              \
  x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(                      \
                   __float_as_int(x), 0x120 + n, 0xf, 0xf, true)))
  TURN(8); TURN(4); TURN(2); TURN(1);       // of the 16 lanes of a row
#undef TURN
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x),
                                                  __float_as_uint(x), false,
                                                  false);
  return max_halves(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}

// One wave, one row: the largest choice scores in descending order, the lower
// index first among equals.  Choice scores are the logits with their bias, the
// weights a softmax over the chosen, or over all (then they are not scaled to
// a sum of one); or sigmoids with a bias, the weights the chosen sigmoids over
// their sum.  `chosen`: the experts once more, or null.
template <int NV, typename T>
__device__ __forceinline__ void route_row(const MoePlanArgs& a, int t,
                                          float* mem, int* chosen) {
  const int lane = threadIdx.x & 63;
  const T* bias = (const T*)a.bias;
  float v[NV], own[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = i * 64 + lane;
    v[i] = -INFINITY;
    own[i] = 0.f;
    if (e < a.E) {
      const float z = a.z[(long)t * a.E + e];
      own[i] = a.kind == 1 ? 1.f / (1.f + expf(-z)) : z;
      v[i] = own[i] + (bias ? to_f(bias[e]) : 0.f);
    }
  }
  float first = 0.f, sum = 0.f;
  if (a.kind == 2) {            // the softmax's denominator
    first = -INFINITY;
#pragma unroll
    for (int i = 0; i < NV; ++i) first = fmaxf(first, v[i]);
    first = wave_max(first);
#pragma unroll
    for (int i = 0; i < NV; ++i) sum += expf(v[i] - first);
    sum = wave_reduce(sum, SumOp());
  }
  if (a.groups > 1) best_groups<NV>(a, v, mem);
  float mine = 0.f;
  int mine_e = 0;
  for (int k = 0; k < a.top; ++k) {
    float best = -INFINITY;
    int at = MOE_MAX_EXPERTS;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (v[i] > best) {
        best = v[i];
        at = i * 64 + lane;
      }
    const float most = wave_max(best);
    const unsigned long long have = __ballot(best == most);
    if (__popcll(have) == 1) {
      at = __builtin_amdgcn_readlane(at, __ffsll(have) - 1);
    } else {                     // equals: the lowest index
      if (best != most) at = MOE_MAX_EXPERTS;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) at = min(at, __shfl_xor(at, off, 64));
      at = __builtin_amdgcn_readfirstlane(at);
    }
    best = most;
    at = min(at, a.E - 1);       // logits that are no numbers stay in bounds
    float score = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if (at >> 6 == i) score = own[i];
      if (at == i * 64 + lane) v[i] = -INFINITY;
    }
    if (k == 0 && a.kind != 2) first = best;
    const float w = a.kind == 1
        ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(score), at & 63))
        : expf(best - first);
    if (a.kind != 2) sum += w;
    if (lane == k) {
      mine = w;
      mine_e = at;
    }
  }
  if (a.kind == 1) sum += 1e-20f;
  if (lane < a.top) {
    a.idx[(long)t * a.top + lane] = mine_e;
    a.coef[(long)t * a.top + lane] = mine / sum;
    if (chosen) chosen[t * a.top + lane] = mine_e;
  }
}

template <typename T>
__device__ __forceinline__ void route(const MoePlanArgs& a, int t, float* mem,
                                      int* chosen) {
  if (a.E <= 64) route_row<1, T>(a, t, mem, chosen);
  else if (a.E <= 256) route_row<4, T>(a, t, mem, chosen);
  else route_row<MOE_MAX_EXPERTS / 64, T>(a, t, mem, chosen);
}

template <typename T>
__global__ void __launch_bounds__(256) moe_route_kernel(MoePlanArgs a) {
  __shared__ float mem[4][MOE_MAX_EXPERTS];
  const int wid = threadIdx.x >> 6, t = blockIdx.x * 4 + wid;
  if (t < a.T) route<T>(a, t, mem[wid], nullptr);
}

#define MOE_FUSED_ROWS 16   // a wave each (32 in one kernel 9.4 us, in two 6.6)

// One workgroup; a chain of short steps.  ROUTE: it also routes the (few) rows
// first and keeps their experts in LDS.  Rows to 6 of 64 experts with the routing,
// against maxima and sums by exchanges over LDS, row after row: 64 rows 28 -> 6.5
// us, 8: 9.3 -> 5.6, 4096: 28 -> 21.
template <typename T, bool ROUTE>
__global__ void __launch_bounds__(1024) moe_plan_kernel(MoePlanArgs a) {
  __shared__ int count[MOE_MAX_EXPERTS], wave_slots[8], wave_tiles[8];
  __shared__ float mem[ROUTE ? 16 : 1][MOE_MAX_EXPERTS];
  __shared__ int chosen[ROUTE ? MOE_FUSED_ROWS * 64 : 1];
  const int tid = threadIdx.x, lane = tid & 63, E = a.E, pairs = a.T * a.top;
  for (int e = tid; e < E; e += 1024) count[e] = 0;
  if (ROUTE)
    for (int t = tid >> 6; t < a.T; t += 16)
      route<T>(a, t, mem[tid >> 6], chosen);
  __syncthreads();
  // four experts on their way at a time
  auto each = [&](auto f) __attribute__((always_inline)) {
    for (int p = tid; p < pairs; p += 4096) {
      int e[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (p + j * 1024 < pairs)
          e[j] = ROUTE ? chosen[p + j * 1024] : a.idx[p + j * 1024];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (p + j * 1024 < pairs) f(p + j * 1024, e[j]);
    }
  };
  each([&](int, int e) { atomicAdd(&count[e], 1); });
  __syncthreads();
  // sums of slots and tiles up to each expert: in its wave, then of the waves
  const int n = tid < E ? count[tid] : 0;
  const int nt = (n + a.tile_rows - 1) / a.tile_rows;
  int slots = n, tile_at = nt;
  if (tid < MOE_MAX_EXPERTS) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int x = __shfl_up(slots, off, 64), y = __shfl_up(tile_at, off, 64);
      if (lane >= off) {
        slots += x;
        tile_at += y;
      }
    }
    if (lane == 63) {
      wave_slots[tid >> 6] = slots;
      wave_tiles[tid >> 6] = tile_at;
    }
  }
  __syncthreads();
  int total = 0, s0 = slots - n, t0 = tile_at - nt;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (i < tid >> 6) {
      s0 += wave_slots[i];
      t0 += wave_tiles[i];
    }
    total += wave_tiles[i];
  }
  if (tid < E) {
    for (int i = 0; i < nt; ++i)
      *(int4*)(a.tiles + 4L * (t0 + i)) = int4{
          tid, s0 + i * a.tile_rows, min(a.tile_rows, n - i * a.tile_rows), total};
    count[tid] = s0;
  }
  for (int i = total + tid; i < a.max_tiles; i += 1024) a.tiles[4L * i + 2] = 0;
  __syncthreads();
  each([&](int p, int e) { a.order[atomicAdd(&count[e], 1)] = p; });
}

extern "C" int sv_moe_plan(const MoePlanArgs* a, int f32,
                           hipStream_t stream) {
  if (a->T <= 0) return 0;
  if (a->E > MOE_MAX_EXPERTS || a->top > 64 || a->top > a->E) return 1;
  if (a->groups < 1 || a->groups > 64 || a->E % a->groups || a->keep < 1 ||
      a->keep > a->groups || a->keep * (a->E / a->groups) < a->top ||
      a->best < 1 || a->best > 2)
    return 1;
  const bool fused = a->T <= MOE_FUSED_ROWS;
  if (!fused) {
    const int grid = (a->T + 3) / 4;
    if (f32) moe_route_kernel<float><<<grid, 256, 0, stream>>>(*a);
    else moe_route_kernel<short><<<grid, 256, 0, stream>>>(*a);
    moe_plan_kernel<float, false><<<1, 1024, 0, stream>>>(*a);
  } else if (f32) {
    moe_plan_kernel<float, true><<<1, 1024, 0, stream>>>(*a);
  } else {
    moe_plan_kernel<short, true><<<1, 1024, 0, stream>>>(*a);
  }
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// grouped products
// ---------------------------------------------------------------------------
struct MoeGemmArgs {
  const void* x;            // rows of K
  long xst;
  const void* w;            // [E][2 N or N][K]: gate rows, then up rows
  void* out;                // rows of N
  const int *order, *tiles;
  int top;                  // > 0: x row = pair / top, out row = slot
                            // 0:   x row = slot,       out row = pair
  int N, K, max_tiles;
  float alpha, limit, shift;  // of the gated activation
  int rows;                 // of x
};

// min(g, limit) sigmoid(alpha g) (clamp(u, +-limit) + shift)
__device__ __forceinline__ float glu(const MoeGemmArgs& a, float g, float u) {
  g = fminf(g, a.limit);
  u = fminf(fmaxf(u, -a.limit), a.limit);
  return g * sigmoid_f(a.alpha * g) * (u + a.shift);
}

// -- MFMA tiles ---------------------------------------
// BM slots x BN weight rows, K in steps of 64 through two LDS buffers; the
// next step's words travel while this one is multiplied: straight into LDS
// (DMA, K a multiple of 64; with an address a load, and all LDS reads waited for
// behind them, 36 tiles of 28672 x 4096 and 4096 x 14336 took 2780 us, now 2640) or
// through registers.  With a gated activation
// the weight rows of a tile alternate 32 gate, 32 up, so a lane holds both of
// a column.
// slot0, rows: the tile's; tn: its columns
// PAGED (DMA, top 1): slot s is row s % 64 of page order[s / 64], pages of 64 rows may
// lie anywhere; slot0 and rows are whole pages.
// AHEAD: the weights come two steps ahead, XA: the rows as well
// APART: Where an XCD's 32 workgroups are on several experts, each expert begins
// elsewhere in K and goes round: rows a power of two apart, read at the same place by
// all, meet in few channels.  16 experts of 4096 x 2048, 256 tokens 234 -> 163 us, 1024
// 257 -> 208; 64 of 2048 x 1408, 256 233 -> 221, 1024 311 -> 280 in 256 slots; but where
// matrix cores are the bound, from 224 rows an expert on, not (4096 593 -> 600).  Within
// an expert all keep step, since they share rows and weights (8 of 4096 x 14336, each
// column tile elsewhere: 512 tokens 573 -> 617; each expert, one an XCD: 587).
template <int BM, int BN, int WM, int WN, bool GLU, bool DMA, bool AHEAD, bool XA,
          bool APART, bool PAGED = false>
__device__ __forceinline__ void moe_tile(const MoeGemmArgs& a, int e, int slot0,
                                         int rows, int tn, short* xs0, short* xs1,
                                         short* xs2, short* ws0, short* ws1,
                                         short* ws2) {
  constexpr int NT = BM / WM * BN / WN * 64;
  constexpr int CM = WM / 32, CN = WN / 32;
  constexpr int LX = BM * 8 / NT, LW = BN * 8 / NT;
  constexpr int NOUT = GLU ? BN / 2 : BN;    // columns of a tile's result
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hi = lane >> 5;
  // a SIMD has waves of all slots, so that it gains where some have no rows
  const int wm = wid / (BN / WN) * WM, wn = wid % (BN / WN) * WN;
  const bool idle = DMA && wm >= rows;
  const int K = a.K, N = a.N;
  // 16-byte slot (r, s) of a tile lies at place s ^ (r >> 1); thread tid
  // fills places tid, tid + NT, ... of a buffer, NT / 8 rows apart
  const int kc = ((tid ^ (tid >> 4)) & 7) * 8;

  // DMA: bytes behind bases that all share (buffer loads, which need no address
  // a step and are waited for by count), less than 2^31
  const short* px[DMA ? 1 : LX];
  const short* pw[DMA ? 1 : LW];
  int ox[LX], ow[LW];
  const short* const bx =
      (const short*)a.x + (PAGED || a.top ? 0 : (long)slot0 * a.xst);
  const short* const bw = (const short*)a.w + (long)e * (GLU ? 2 * N : N) * K;
  int page[PAGED ? LX : 1];                // a wave's load is 8 rows of one page
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    if (PAGED) {
      const int r = slot0 + min(i * (NT / 8) + wid * 8, rows - 8);
      page[PAGED ? i : 0] = __builtin_amdgcn_readfirstlane(a.order[r / 64]);
      ox[i] = ((r % 64 + (lane >> 3)) * (int)a.xst + kc) * 2;
      continue;
    }
    const int at = (i * NT + tid) / 8, r = min(at, rows - 1);
    const int row = a.top ? a.order[slot0 + r] / a.top : r;
    // past the last row: out of the buffer, zeros for which nothing is read (64 experts
    // 2048 x 1408, 4096 tokens 595 -> 585 us, 8 of 4096 x 14336, 2048 1563 -> 1541)
    if (DMA) ox[i] = at < rows ? (row * (int)a.xst + kc) * 2 : 0x7fffffff;
    else px[i] = bx + (long)row * a.xst + kc;
  }
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int r = (i * NT + tid) / 8;
    int n = GLU ? tn * NOUT + (r >> 6) * 32 + (r & 31) : tn * NOUT + r;
    n = min(n, N - 1);
    if (GLU && (r & 32)) n += N;
    if (DMA) ow[i] = (n * K + kc) * 2;
    else pw[i] = bw + (long)n * K + kc;
  }

  uint4v rx[LX], rw[LW];
  // a wave's 64 places follow each other
  auto issue_x = [&](int k0, short* xs) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LX; ++i)
      words_to_lds(PAGED ? bx + page[PAGED ? i : 0] * (64 * a.xst) : bx, ox[i],
                   (char*)(xs + (i * NT + wid * 64) * 8), k0 * 2);
  };
  auto issue_w = [&](int k0, short* ws) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LW; ++i)
      words_to_lds(bw, ow[i], (char*)(ws + (i * NT + wid * 64) * 8), k0 * 2);
  };
  auto issue = [&](int k0, short* xs, short* ws) __attribute__((always_inline)) {
    if (DMA) {
      issue_x(k0, xs);
      issue_w(k0, ws);
      return;
    }
    const bool in_k = k0 + kc < K;
    const uint4v zero = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < LX; ++i)
      rx[i] = in_k ? *(const uint4v*)(px[DMA ? 0 : i] + k0) : zero;
#pragma unroll
    for (int i = 0; i < LW; ++i)
      rw[i] = in_k ? *(const uint4v*)(pw[DMA ? 0 : i] + k0) : zero;
  };
  auto commit = [&](short* xs, short* ws) {
    if (DMA) return;
#pragma unroll
    for (int i = 0; i < LX; ++i) *(uint4v*)(xs + (i * NT + tid) * 8) = rx[i];
#pragma unroll
    for (int i = 0; i < LW; ++i) *(uint4v*)(ws + (i * NT + tid) * 8) = rw[i];
  };

  // A step has four chunks of 16 columns.  The fragments of a chunk are read
  // while the one before is multiplied; the last chunk of a step is
  // multiplied after the barrier, while the next step's first is read.
  f32x16 acc[CN][CM] = {};
  frag_u fx[2][CM] = {}, fw[2][CN] = {};
  auto multiply = [&](int c) {
#pragma unroll
    for (int n = 0; n < CN; ++n)
#pragma unroll
      for (int m = 0; m < CM; ++m)
        acc[n][m] = mfma_bf16(fw[c & 1][n].bf, fx[c & 1][m].bf, acc[n][m]);
  };
  auto step = [&](const short* xs, const short* ws) {
    if (idle) return;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      // row 32 m + col, slot 2 c + hi
      const int at = col * 64 + (((2 * c + hi) ^ (col >> 1)) & 7) * 8;
#pragma unroll
      for (int m = 0; m < CM; ++m)
        fx[c & 1][m].u4 = *(const uint4v*)(xs + wm * 64 + at + m * 2048);
#pragma unroll
      for (int n = 0; n < CN; ++n)
        fw[c & 1][n].u4 = *(const uint4v*)(ws + wn * 64 + at + n * 2048);
      multiply(c - 1);             // of the step before, if c is 0
      // two products, the reads, the other products
      __builtin_amdgcn_sched_group_barrier(0x8, CM * CN < 2 ? 1 : 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, CM + CN, 0);
      if (CM * CN > 2) __builtin_amdgcn_sched_group_barrier(0x8, CM * CN - 2, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const int steps = (K + 63) / 64;
  const int skew = APART ? e * 5 % steps : 0;
  // past the last step that one again
  auto place = [&](int i) __attribute__((always_inline)) {
    i = min(i, steps - 1) + skew;
    return (!APART || i < steps ? i : i - steps) * 64;
  };
  if (AHEAD) {
    // step i: its words are here, in all waves, and the weights of i + 1 may be
    // on their way; the step before is read.  Past the last step that one
    // again, so that the words on their way keep their number.
    // The wait counts: it is right only if the loads of i + 1, LW of weights and with
    // XA before them LX of rows, are the last that were asked for, behind the rows and
    // the weights of i.  Nothing else tells the compiler so (they go to different
    // arrays).
    auto in_order = []() __attribute__((always_inline)) {
      asm volatile("" ::: "memory");
    };
    auto turn = [&](int i, short* xs, short* ws, short* xn, short* wn)
        __attribute__((always_inline)) {
      constexpr int AFTER = LW + (XA ? LX : 0);
      static_assert(AFTER < 16, "");
      __builtin_amdgcn_s_waitcnt(0x70 | AFTER);    // vmcnt(AFTER) lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      in_order();
      issue_x(place(i + (XA ? 2 : 1)), xn);
      in_order();
      issue_w(place(i + 2), wn);
      step(xs, ws);
    };
    constexpr int X = XA ? 3 : 2;
    short *const xr[3] = {xs0, xs1, xs2}, *const wr[3] = {ws0, ws1, ws2};
    issue_x(place(0), xs0);
    issue_w(place(0), ws0);
    in_order();
    if (XA) issue_x(place(1), xs1);
    issue_w(place(1), ws1);
    int i = 0;
    for (; i + 6 <= steps; i += 6)
#pragma unroll
      for (int j = 0; j < 6; ++j)
        turn(i + j, xr[j % X], wr[j % 3], xr[(j + X - 1) % X], wr[(j + 2) % 3]);
#pragma unroll
    for (int j = 0; j < 5; ++j)
      if (i + j < steps)
        turn(i + j, xr[j % X], wr[j % 3], xr[(j + X - 1) % X], wr[(j + 2) % 3]);
    __builtin_amdgcn_s_waitcnt(0xf70);             // vmcnt(0): LDS is given back
  } else {
    issue(place(0), xs0, ws0);
    commit(xs0, ws0);
    __syncthreads();                 // also waits for the words on their way
    for (int i = 0; i + 1 < steps; i += 2) {
      issue(place(i + 1), xs1, ws1);
      step(xs0, ws0);
      commit(xs1, ws1);
      __syncthreads();
      issue(place(i + 2), xs0, ws0);   // past the last one not read
      step(xs1, ws1);
      commit(xs0, ws0);
      __syncthreads();
    }
    if (steps & 1) step(xs0, ws0);
  }
  if (idle) return;
  multiply(3);

#pragma unroll
  for (int m = 0; m < CM; ++m) {
    const int r = wm + 32 * m + col;
    if (r >= rows) continue;
    const long orow = PAGED || a.top ? slot0 + r : a.order[slot0 + r];
    short* dst = (short*)a.out + orow * N;
#pragma unroll
    for (int n = 0; n < CN; n += GLU ? 2 : 1)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int c = tn * NOUT + (GLU ? wn / 2 + 16 * n : wn + 32 * n) +
                      8 * rg + 4 * hi;
        if (c >= N) continue;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          v[j] = GLU ? glu(a, acc[n][m][4 * rg + j],
                           acc[n + (GLU ? 1 : 0)][m][4 * rg + j])
                     : acc[n][m][4 * rg + j];
        *(uint2*)(dst + c) = uint2{pack_bf16x2(v[0], v[1]),
                                   pack_bf16x2(v[2], v[3])};
      }
  }
}

// One workgroup a tile.  TAIL: the last tiles, if they leave half of the CUs
// without one, are computed in halves of the slots, or quarters, by all of them
// (36 tiles of 4096 x 14336, 576 workgroups on 256 CUs: 966 us, in whole tiles
// 1128); those of 128 slots, which wait for weights, in halves of the columns (8 tiles
// of 4096 x 14336, 128 workgroups: 250 us, 222).
// PAGED: all rows are one expert's, `rows` of them.
template <int BM, int BN, int WM, int WN, bool GLU, bool DMA, bool TAIL, bool APART,
          bool PAGED = false>
__device__ __forceinline__ void moe_tiles(const MoeGemmArgs& a) {
  constexpr int GROUP = 8;
  constexpr int NOUT = GLU ? BN / 2 : BN;
  // apart by name, so that a read of one buffer need not wait for the words
  // on their way into the other
  __shared__ __attribute__((aligned(16))) short xs0[BM * 64], xs1[BM * 64];
  // weights two steps ahead where one workgroup has the CU anyway (128 slots,
  // 4096 rows of 8 experts 4096 x 14336: 842 -> 741 us, 256 slots 985 -> 965), rows as
  // well where there is room: a step of few rows is shorter than their way (8 experts
  // 4096 x 14336, both products: 256 tokens 563 -> 529 us, 384 589 -> 559; 64 slots by 8
  // waves instead of two workgroups of 4, 128 tokens 580 -> 504)
  constexpr bool AHEAD = DMA && (BM >= 128 || (BM == 64 && BM / WM * BN / WN == 8));
  constexpr bool XA = AHEAD && BM < 256 && !PAGED;
  __shared__ __attribute__((aligned(16))) short xs2[XA ? BM * 64 : 8];
  __shared__ __attribute__((aligned(16))) short ws0[BN * 64], ws1[BN * 64],
      ws2[AHEAD ? BN * 64 : 8];

  // neighbours in the list of tiles run on one XCD: groups of GROUP slot
  // tiles by all column tiles, slot tiles fastest.  The XCDs share the tiles
  // that have rows (all places in the list, the last ones empty: gates of 36
  // tiles of 28672 x 4096 2222 us, now 1789)
  const int ntn = (a.N + NOUT - 1) / NOUT;
  const int live = PAGED ? (a.rows + BM - 1) / BM : a.tiles[3], total = live * ntn;
  const int tail = total % 256;
  const int split =
      !TAIL || tail == 0 || tail > 128 ? 1 : BM < 256 || tail > 64 ? 2 : 4;
  const int whole = split > 1 ? total - tail : total;
  int id = blockIdx.x, piece = 0;
  if (id < whole) {
    const int per = whole / 8, rest = whole % 8, xcd = id % 8;
    id = xcd * per + min(xcd, rest) + id / 8;
  } else {
    piece = (id - whole) % split;
    id = whole + (id - whole) / split;
    if (id >= total) return;
  }
  const int g0 = id / (GROUP * ntn) * GROUP;
  const int gm = min(GROUP, live - g0);
  const int in = id - g0 * ntn;
  const int tn = in / gm;
  const int tile = g0 + in % gm;
  const int* tl = PAGED ? nullptr : a.tiles + 4L * tile;
  const int e = PAGED ? 0 : tl[0], slot0 = PAGED ? tile * BM : tl[1];
  const int rows = PAGED ? min(BM, a.rows - slot0) : tl[2];
  if (!TAIL || id < whole) {
    moe_tile<BM, BN, WM, WN, GLU, DMA, AHEAD, XA, APART, PAGED>(
        a, e, slot0, rows, tn, xs0, xs1, xs2, ws0, ws1, ws2);
    return;
  }
  if constexpr (TAIL && BM < 256) {
    if ((tn * 2 + piece) * (NOUT / 2) < a.N)
      moe_tile<BM, BN / 2, GLU ? WM / 2 : WM, GLU ? WN : WN / 2, GLU, DMA, AHEAD, XA,
               APART, PAGED>(a, e, slot0, rows, tn * 2 + piece, xs0, xs1, xs2, ws0, ws1,
                             ws2);
  } else if constexpr (TAIL) {
    const int s = piece % 2 * (BM / 2);
    if (s >= rows) return;
    if (split == 2)
      moe_tile<BM / 2, BN, WM / 2, WN, GLU, DMA, AHEAD, XA, APART, PAGED>(
          a, e, slot0 + s, min(rows - s, BM / 2), tn, xs0, xs1, xs2, ws0, ws1, ws2);
    else if ((tn * 2 + piece / 2) * (NOUT / 2) < a.N)
      moe_tile<BM / 2, BN / 2, WM / 4, WN, GLU, DMA, AHEAD, XA, APART, PAGED>(
          a, e, slot0 + s, min(rows - s, BM / 2), tn * 2 + piece / 2, xs0, xs1, xs2,
          ws0, ws1, ws2);
  }
}

template <int BM, int BN, int WM, int WN, bool GLU, bool DMA, bool TAIL, bool APART>
__global__ void __launch_bounds__(BM / WM * BN / WN * 64)
moe_tiles_kernel(MoeGemmArgs a) {
  moe_tiles<BM, BN, WM, WN, GLU, DMA, TAIL, APART>(a);
}

// -- a few rows per expert: stream the weights --------------------------------
// Weights meet up to 32 slots of x (16 and less leave the second half out), through
// rings in LDS where K is whole blocks of 64 columns, else from memory straight into
// registers as fragments, a lane's 16 bytes of a row.  A unit is 16 weight rows (8 or
// 16 gates and their up rows) of one slot tile.  Bound by reading the weights, at 6.5
// to 6.7 TB/s through rings (a read alone: 6.9).  Both products, us (through registers
// | rings; 32-slot tiles):
//   64 experts 2048 x 1408, top 6   1 row  30 |  23    8: 108 |  95   32: 199 | 165
//   128: 219 | 175
//   8 experts 4096 x 14336, top 2   1 row 124 | 119    8: 488 | 429   32: 533 | 453
//   16 experts 4096 x 2048, top 2   4 rows 71 |  64    8: 115 | 110   32: 149 | 130

// acc rows 4 grp + 0..3 are the unit's weight rows, columns slots
template <bool GLU>
__device__ __forceinline__ void store_unit(const MoeGemmArgs& a, int slot0,
                                           int rows, int r, int c, f32x4 v,
                                           f32x4 u) {
  if (r >= rows || c >= a.N) return;
  if (GLU)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = glu(a, v[j], u[j]);
  short* dst = (short*)a.out +
      (long)(a.top ? slot0 + r : a.order[slot0 + r]) * a.N + c;
  *(uint2*)dst = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

__device__ __forceinline__ const short* unit_x(const MoeGemmArgs& a, int slot) {
  return (const short*)a.x + (long)(a.top ? a.order[slot] / a.top : slot) * a.xst;
}

template <int N> struct Count { static constexpr int value = N; };

// K up to 512 NW: a workgroup stays.  It takes the same share of all units as
// the others, one after the other, with the columns of its slots in registers:
// wave w those of 64-column blocks w, w + NW, ...  Four blocks of a weight row
// are read at a time, one such part ahead, past the units' borders.
template <int NW, bool GLU>
__global__ void __launch_bounds__(NW * 64, 2) moe_stay_kernel(MoeGemmArgs a) {
  constexpr int RT = GLU ? 2 : 1, PARTS = 2, UNITS = RT * PARTS;
  __shared__ f32x4 part[2][NW][RT * 2][64];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, grp = lane >> 4;
  const int K = a.K, N = a.N, ntn = (N + 15) / 16;
  const long units = (long)a.tiles[3] * ntn;      // all tiles that have rows
  const long first = units * blockIdx.x / gridDim.x;
  int left = (int)(units * (blockIdx.x + 1) / gridDim.x - first);
  if (left == 0) return;
  const uint4v zero = {0, 0, 0, 0};
  const int k0 = wid * 64 + grp * 8;
  // the lane's columns of its chunk c start at k0 + at(c)
  auto at = [](int c) { return (c >> 1) * NW * 64 + (c & 1) * 32; };

  // the unit that is read next
  int tn = (int)(first % ntn);
  const int* tl = a.tiles + 4 * (first / ntn);
  const short* w = (const short*)a.w + (long)tl[0] * RT * N * K;
  auto load = [&](int u, frag_u* fw) __attribute__((always_inline)) {
    const int n = min(tn * 16 + c16, N - 1) + (u / PARTS ? N : 0);
    const short* src = w + (long)n * K + (k0 + at(u % PARTS * 8));
#pragma unroll
    for (int c = 0; c < 8; ++c)
      fw[c].u4 = k0 + at(u % PARTS * 8 + c) < K ? *(const uint4v*)(src + at(c))
                                                : zero;
  };
  auto advance = [&]() __attribute__((always_inline)) {
    if (left == 1) return;         // past the last one that one again, unused
    if (++tn == ntn) {
      tn = 0;
      tl += 4;
      w = (const short*)a.w + (long)tl[0] * RT * N * K;
    }
  };

  frag_u wa[8], wb[8];
  int buf = 0;
  // the units of one slot tile, MT times 16 slots
  auto run = [&](auto tiles_of_16) __attribute__((always_inline)) {
    constexpr int MT = decltype(tiles_of_16)::value;
    const int slot0 = tl[1], rows = tl[2];
    frag_u fx[PARTS * 8][MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const short* x = unit_x(a, slot0 + min(j * 16 + c16, rows - 1)) + k0;
#pragma unroll
      for (int c = 0; c < PARTS * 8; ++c)
        fx[c][j].u4 = k0 + at(c) < K ? *(const uint4v*)(x + at(c)) : zero;
    }
    f32x4 acc[MT];
    auto multiply = [&](int u, const frag_u* fw) __attribute__((always_inline)) {
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
          part[buf][wid][u / PARTS * 2 + j][lane] = acc[j];
    };
    for (int n = min(left, ntn - tn); n > 0; --n, --left, buf ^= 1) {
      const int n0 = tn * 16;
#pragma unroll
      for (int u = 0; u < UNITS; u += 2) {
        const bool last = u + 2 == UNITS;
        if (last) advance();
        multiply(u, wa);
        load(last ? 0 : u + 2, wa);
        multiply(u + 1, wb);
        load(last ? 1 : u + 3, wb);
      }
      // the first waves add up the sums of all; the others go on
      __syncthreads();
      if (wid >= MT) continue;
      f32x4 v = {}, u = {};
#pragma unroll 2
      for (int s = 0; s < NW; ++s) {
        v += part[buf][s][wid][lane];
        if (GLU) u += part[buf][s][2 + wid][lane];
      }
      store_unit<GLU>(a, slot0, rows, wid * 16 + c16, n0 + 4 * grp, v, u);
    }
  };
  load(0, wa);
  load(1, wb);
  while (left > 0) {
    if (tl[2] > 16) run(Count<2>());
    else run(Count<1>());
  }
}

// The same with the weights through rings, for a K in blocks of 64 columns, which the
// waves share evenly.  A unit is 16 weight rows, or 8 gates and their 8 up rows.
template <bool GLU>
struct Units {
  static constexpr int NW = 8, R = 8, TR = GLU ? 8 : 16;
  Ring<R> ring;
  int block, nb;                         // the wave's blocks of 64 columns
  int ntn, left, tn;                     // units of a tile; the workgroup's, and the
  const int* tl;                         //   one that is multiplied next, of its tile
  int asked, blk, to_ask;                // what is asked for next
  const int* from;
  __amdgpu_buffer_rsrc_t ra, rb;
  int oa, ob, pitch;

  __device__ __forceinline__ Units(const MoeGemmArgs& a, char* lds, int wid)
      : ring(lds + wid * R * 1024) {
    ntn = (a.N + TR - 1) / TR;
    const long units = (long)a.tiles[3] * ntn;    // all tiles that have rows
    const long first = units * blockIdx.x / gridDim.x;
    left = (int)(units * (blockIdx.x + 1) / gridDim.x - first);
    block = a.K / 64 * wid / NW;
    nb = a.K / 64 * (wid + 1) / NW - block;
    pitch = a.K * 2;
    oa = Ring<R>::lane_bytes(pitch, 0) + block * 128;
    ob = Ring<R>::lane_bytes(pitch, 1) + block * 128 + (GLU ? 0 : 8 * pitch);
    asked = tn = (int)(first % ntn);
    from = tl = a.tiles + 4 * (first / ntn);
    blk = 0;
    to_ask = left;
  }
  // of the expert of the tile that is asked for
  __device__ __forceinline__ void expert(const MoeGemmArgs& a) {
    const short* w = (const short*)a.w + (long)from[0] * (GLU ? 2 : 1) * a.N * a.K;
    ra = ring_source(w, a.N * pitch);
    rb = ring_source(GLU ? w + (long)a.N * a.K : w, a.N * pitch);
  }
  // the next block; is the one behind it of another tile?
  __device__ __forceinline__ bool ask(const MoeGemmArgs& a) {
    const uint at = to_ask > 0 ? (uint)(asked * TR) * pitch + blk * 128 : RING_NOWHERE;
    ring.ask(ra, oa + at, rb, ob + at);
    if (++blk < nb) return false;
    blk = 0;
    if (--to_ask <= 0 || ++asked < ntn) return false;
    asked = 0;
    from += 4;
    expert(a);
    return true;
  }
  // on to the next unit
  __device__ __forceinline__ void advance() {
    --left;
    if (++tn < ntn) return;
    tn = 0;
    tl += 4;
  }
};

// The sums of a unit's waves meet, and the first waves add them up.  `out`: where
// this lane's row starts, if it is one.
template <int MT, bool GLU>
__device__ __forceinline__ void meet(const MoeGemmArgs& a, f32x4 (*part)[2][64],
                                     const f32x4* acc, int wid, int tn, bool in,
                                     short* out) {
  constexpr int NW = 8;
  const int lane = threadIdx.x & 63, grp = lane >> 4;
#pragma unroll
  for (int j = 0; j < MT; ++j) part[wid][j][lane] = acc[j];
  lds_barrier();
  if (wid >= MT) return;
  f32x4 v = {}, p[NW];
#pragma unroll
  for (int s = 0; s < NW; ++s) p[s] = part[s][wid][lane];
#pragma unroll
  for (int s = 0; s < NW; ++s) v += p[s];
  const int col = tn * Units<GLU>::TR + 4 * grp;
  if (GLU)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = glu(a, v[i], __shfl_xor(v[i], 32, 64));
  if (in && col < a.N && (!GLU || grp < 2))
    *(uint2*)(out + col) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

// K up to 512 CB: a workgroup stays, with the columns of its slots in registers.
template <int CB, bool GLU>
__global__ void __launch_bounds__(512) moe_ring_kernel(MoeGemmArgs a) {
  using U = Units<GLU>;
  __shared__ __attribute__((aligned(1024))) char lds[U::NW * U::R * 1024];
  __shared__ f32x4 part[2][U::NW][2][64];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  U w(a, lds, wid);
  if (w.left == 0) return;
  w.expert(a);
#pragma unroll
  for (int i = 0; i < U::R / 2; ++i) w.ask(a);
  const int nb = w.nb;
  int buf = 0;
  // the units of one slot tile, MT times 16 slots
  auto run = [&](auto tiles_of_16) __attribute__((always_inline)) {
    constexpr int MT = decltype(tiles_of_16)::value;
    const int slot0 = w.tl[1], rows = w.tl[2];
    frag_u fx[CB * 2][MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const short* x = unit_x(a, slot0 + min(j * 16 + (lane >> 2), rows - 1)) +
                       w.block * 64 + (lane & 3) * 8;
#pragma unroll
      for (int c = 0; c < CB * 2; ++c)   // blocks past the wave's are not used
        fx[c][j].u4 = *(const uint4v*)(x + (c < 2 * nb ? c * 32 : 0));
    }
#pragma unroll
    for (int c = 0; c < CB * 2; ++c)
#pragma unroll
      for (int j = 0; j < MT; ++j) fx[c][j] = turned(fx[c][j]);
    const int r = wid * 16 + (lane & 15);  // the row that this lane stores
    const int slot = slot0 + min(r, rows - 1);
    short* const out = (short*)a.out + (long)(a.top ? slot : a.order[slot]) * a.N;
    // from here on only pieces (and results) are on their way
    __builtin_amdgcn_s_waitcnt(0x0070);
    for (int n = min(w.left, w.ntn - w.tn); n > 0; --n, buf ^= 1) {
      f32x4 acc[MT] = {};
#pragma unroll
      for (int c = 0; c < CB; ++c) {
        if (c >= nb) continue;
        frag_u f0, f1;
        w.ring.template take<U::R - 2>(f0, f1);
        w.ask(a);
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          acc[j] = mfma16(f0.bf, fx[2 * c][j].bf, acc[j]);
          acc[j] = mfma16(f1.bf, fx[2 * c + 1][j].bf, acc[j]);
        }
      }
      meet<MT, GLU>(a, part[buf], acc, wid, w.tn, r < rows, out);
      w.advance();
    }
  };
  while (w.left > 0) {
    if (w.tl[2] > 16) run(Count<2>());
    else run(Count<1>());
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // LDS is given back
}

// Longer rows: x flows too, a ring ahead.
template <bool GLU>
__global__ void __launch_bounds__(512) moe_flow_kernel(MoeGemmArgs a) {
  using U = Units<GLU>;
  constexpr int D = U::R / 2;            // blocks ahead
  __shared__ __attribute__((aligned(1024))) char lds[U::NW * U::R * 1024];
  __shared__ f32x4 part[2][U::NW][2][64];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  U w(a, lds, wid);
  if (w.left == 0) return;
  w.expert(a);
  bool two = false;
  for (int i = 0; i <= (w.tn + w.left - 1) / w.ntn; ++i) two |= w.tl[4 * i + 2] > 16;
  const int total = w.left * w.nb;
  auto run = [&](auto tiles_of_16) __attribute__((always_inline)) {
    constexpr int MT = decltype(tiles_of_16)::value;
    const short* x[MT];
    auto rows_of = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < MT; ++j)
        x[j] = unit_x(a, w.from[1] + min(j * 16 + (lane >> 2), w.from[2] - 1)) +
               w.block * 64 + (lane & 3) * 8;
    };
    frag_u fx[D][2][MT];
    auto ask = [&](int i) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          fx[i][h][j].u4 = *(const uint4v*)(x[j] + w.blk * 64 + h * 32);
      if (w.ask(a)) rows_of();
      __builtin_amdgcn_sched_barrier(0);
    };
    // The row that this lane stores.  Waited for at once: where ways with and
    // without it join, every product would wait for all loads.
    const int r = wid * 16 + (lane & 15);
    short* out;
    bool in;
    auto row_of = [&]() __attribute__((always_inline)) {
      const int rows = w.tl[2], slot = w.tl[1] + min(r, rows - 1);
      in = r < rows;
      out = (short*)a.out + (long)(a.top ? slot : a.order[slot]) * a.N;
      __builtin_amdgcn_s_waitcnt(0x0f70);
    };
    row_of();
    rows_of();
#pragma unroll
    for (int i = 0; i < D; ++i) ask(i);
    f32x4 acc[MT] = {};
    int c = 0, buf = 0;
    for (int s = 0; s < total; s += D) {
#pragma unroll
      for (int i = 0; i < D; ++i) {
        frag_u f0, f1;
        w.ring.template take<(D - 1) * (2 * MT + 2)>(f0, f1);
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          acc[j] = mfma16(f0.bf, turned(fx[i][0][j]).bf, acc[j]);
          acc[j] = mfma16(f1.bf, turned(fx[i][1][j]).bf, acc[j]);
        }
        ask(i);
        if (++c == w.nb && w.left > 0) {  // past the last unit nothing counts
          meet<MT, GLU>(a, part[buf], acc, wid, w.tn, in, out);
#pragma unroll
          for (int j = 0; j < MT; ++j) acc[j] = f32x4{};
          c = 0;
          buf ^= 1;
          w.advance();
          if (w.tn == 0 && w.left > 0) row_of();
        }
      }
    }
  };
  if (two) run(Count<2>());
  else run(Count<1>());
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // LDS is given back
}

// Longer rows: a workgroup a unit; its 16 waves take turns of 64 columns of
// the weight rows and of x, a turn ahead.
template <bool GLU>
__global__ void __launch_bounds__(1024) moe_stream_kernel(MoeGemmArgs a) {
  constexpr int RT = GLU ? 2 : 1, U = 2, STEP = 16 / RT * U * 32;
  __shared__ f32x4 part[16][2][64];
  const int* tl = a.tiles + 4L * blockIdx.y;
  const int rows = tl[2];
  if (rows == 0) return;
  const int slot0 = tl[1];
  const bool two = rows > 16;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, grp = lane >> 4;
  const int K = a.K, N = a.N, n0 = blockIdx.x * 16;
  const short* w = (const short*)a.w + grp * 8 +
      ((long)tl[0] * RT * N + min(n0 + c16, N - 1) + (wid % RT ? N : 0)) * K;
  const short* x[2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
    x[j] = unit_x(a, slot0 + min(j * 16 + c16, rows - 1)) + grp * 8;

  f32x4 acc[2] = {};
  const uint4v zero = {0, 0, 0, 0};
  auto load = [&](int k0, frag_u* fw, frag_u (*fx)[2])
      __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * 32;
      const bool in = k + grp * 8 < K;
      fw[u].u4 = in ? *(const uint4v*)(w + k) : zero;
      fx[u][0].u4 = in ? *(const uint4v*)(x[0] + k) : zero;
      fx[u][1].u4 = in && two ? *(const uint4v*)(x[1] + k) : zero;
    }
  };
  auto multiply = [&](const frag_u* fw, const frag_u (*fx)[2])
      __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[j] = mfma16(fw[u].bf, fx[u][j].bf, acc[j]);
  };
  frag_u wa[U], xa[U][2], wb[U], xb[U][2];
  int k = wid / RT * U * 32;
  if (k < K) load(k, wa, xa);
  for (; k < K; k += 2 * STEP) {
    if (k + STEP < K) load(k + STEP, wb, xb);
    multiply(wa, xa);
    if (k + STEP >= K) break;
    if (k + 2 * STEP < K) load(k + 2 * STEP, wa, xa);
    multiply(wb, xb);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) part[wid][j][lane] = acc[j];
  __syncthreads();
  if (wid >= 2 || (wid == 1 && !two)) return;
  f32x4 v = {}, u = {};
#pragma unroll
  for (int s = 0; s < 16; s += RT) {
    v += part[s][wid][lane];
    if (GLU) u += part[s + 1][wid][lane];
  }
  store_unit<GLU>(a, slot0, rows, wid * 16 + c16, n0 + 4 * grp, v, u);
}

// -- any size and type -------------------------------------------------------
template <typename T, bool GLU>
__global__ void __launch_bounds__(256) moe_plain_kernel(MoeGemmArgs a) {
  constexpr int B = 32;
  __shared__ float xs[B][B + 1], gs[B][B + 1], us[GLU ? B : 1][B + 1];
  const int* tl = a.tiles + 4L * blockIdx.y;
  const int rows = tl[2];
  if (rows == 0) return;
  const int e = tl[0], slot0 = tl[1], n0 = blockIdx.x * B;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int K = a.K, N = a.N;
  const T* w = (const T*)a.w + (long)e * (GLU ? 2 * N : N) * K;
  float g[2][2] = {}, u[2][2] = {};
  for (int k0 = 0; k0 < K; k0 += B) {
    for (int i = threadIdx.x; i < B * B; i += 256) {
      const int r = i / B, k = k0 + i % B;
      const int s = slot0 + r;
      float xv = 0.f, gv = 0.f, uv = 0.f;
      if (k < K) {
        if (r < rows)
          xv = to_f(((const T*)a.x)[(long)(a.top ? a.order[s] / a.top : s) *
                                    a.xst + k]);
        if (n0 + r < N) {
          gv = to_f(w[(long)(n0 + r) * K + k]);
          if (GLU) uv = to_f(w[(long)(N + n0 + r) * K + k]);
        }
      }
      xs[r][i % B] = xv;
      gs[r][i % B] = gv;
      if (GLU) us[r][i % B] = uv;
    }
    __syncthreads();
    for (int k = 0; k < B; ++k)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float xv = xs[ty + 16 * i][k];
          g[i][j] += xv * gs[tx + 16 * j][k];
          if (GLU) u[i][j] += xv * us[tx + 16 * j][k];
        }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = ty + 16 * i, c = n0 + tx + 16 * j;
      if (r >= rows || c >= N) continue;
      const long orow = a.top ? slot0 + r : a.order[slot0 + r];
      from_f(((T*)a.out)[orow * N + c], GLU ? glu(a, g[i][j], u[i][j]) : g[i][j]);
    }
}

// BN2, WM2, WN2: through registers
template <int BM, int BN, int WM, int WN, bool GLU, int BN2 = BN, int WM2 = WM,
          int WN2 = WN>
static void launch_tiles(const MoeGemmArgs& a, hipStream_t stream) {
  // halves of 64 slots' gates are too few for 8 waves
  constexpr bool TAIL = BM >= 128 || (BM == 64 && !GLU && BN / WN == 4);
  auto launch = [&](auto kernel, int nout, int nt, int more) {
    const long grid = (long)a.max_tiles * ((a.N + nout - 1) / nout) + more;
    kernel<<<grid, nt, 0, stream>>>(a);
  };
  constexpr int NOUT = GLU ? BN / 2 : BN, NT = BM / WM * BN / WN * 64;
  // a plan has a tile for every BM pairs and one for every expert
  const long pairs = (long)a.rows * (a.top ? a.top : 1);
  const bool apart = !(a.K & (a.K - 1)) && a.N < 32 * NOUT &&
                     pairs < 224 * (a.max_tiles - pairs / BM);
  // offsets of a tile's rows, and of an expert's weights, are bytes of 31 bits
  const bool near = (a.top ? a.rows : 256) * a.xst < 1L << 30 &&
                    (GLU ? 2L : 1L) * a.N * a.K < 1L << 30;
  if (a.K % 64 || !near)
    launch(moe_tiles_kernel<BM, BN2, WM2, WN2, GLU, false, false, false>,
           GLU ? BN2 / 2 : BN2, BM / WM2 * BN2 / WN2 * 64, 0);
  else if (apart)                        // at most 3 * 64 or 128 pieces more
    launch(moe_tiles_kernel<BM, BN, WM, WN, GLU, true, TAIL, true>, NOUT, NT,
           TAIL ? 192 : 0);
  else
    launch(moe_tiles_kernel<BM, BN, WM, WN, GLU, true, TAIL, false>, NOUT, NT,
           TAIL ? 192 : 0);
}

template <bool GLU>
static void launch_stream(const MoeGemmArgs& a, hipStream_t stream) {
  const int units = (a.N + 15) / 16;
  const long all = (long)units * a.max_tiles;
  // Rings: a workgroup of 8 waves a CU (of 4 waves, two or three a CU: 168 and 184 us
  // where one takes 165).  They share whole units, so they need a few (6 tiles of
  // 2048 x 1408, 528 units: 23 us, a workgroup a unit 30; 16 experts 4096 x 2048, 1
  // row, 256 and 512 units: 24, 22.5).  The host knows the most tiles there can be:
  // rows that share few experts stay as well.
  // every wave has a block, an expert's offsets are bytes of 31 bits
  if (a.K % 64 == 0 && a.K >= 512 && (GLU ? 2L : 1L) * a.N * a.K < 1L << 30 &&
      all > 512) {
    if (a.K <= 2048) moe_ring_kernel<4, GLU><<<256, 512, 0, stream>>>(a);
    else if (a.K <= 4096) moe_ring_kernel<8, GLU><<<256, 512, 0, stream>>>(a);
    else moe_flow_kernel<GLU><<<256, 512, 0, stream>>>(a);
    return;
  }
  // through registers, as many workgroups as are resident: with twice as many, 2% to
  // 30% longer
  const int grid = a.K <= 2048 ? 512 : 256;
  if (a.K > 4096 || all < 2 * grid)
    moe_stream_kernel<GLU><<<dim3(units, a.max_tiles), 1024, 0, stream>>>(a);
  else if (a.K <= 2048)
    moe_stay_kernel<4, GLU><<<grid, 256, 0, stream>>>(a);
  else
    moe_stay_kernel<8, GLU><<<grid, 512, 0, stream>>>(a);
}

// how: 0 any size and type, 1 stream, 2 to 5 tiles (1 to 5: bf16, N, K, xst
// and bases in 8 elements).  The plan's tile_rows: 32, 32, 32, 64, 128, 256.
extern "C" int sv_moe_gemm(const MoeGemmArgs* a, int how, int gated, int f32,
                           hipStream_t stream) {
  if (a->max_tiles <= 0) return 0;
  if (how == 5) {
    if (gated) launch_tiles<256, 256, 128, 64, true>(*a, stream);
    else launch_tiles<256, 256, 128, 64, false>(*a, stream);
  } else if (how == 4) {
    if (gated) launch_tiles<128, 256, 64, 64, true>(*a, stream);
    else launch_tiles<128, 256, 64, 64, false>(*a, stream);
  } else if (how == 3) {
    if (gated) launch_tiles<64, 256, 32, 64, true, 256, 64, 64>(*a, stream);
    else launch_tiles<64, 256, 32, 64, false, 128, 64, 32>(*a, stream);
  } else if (how == 2) {
    if (gated) launch_tiles<32, 256, 32, 64, true>(*a, stream);
    else launch_tiles<32, 128, 32, 32, false>(*a, stream);
  } else if (how == 1) {
    if (gated) launch_stream<true>(*a, stream);
    else launch_stream<false>(*a, stream);
  } else {
    const dim3 grid((a->N + 31) / 32, a->max_tiles);
#define PK(T, G) moe_plain_kernel<T, G><<<grid, 256, 0, stream>>>(*a)
    if (f32) { if (gated) PK(float, true); else PK(float, false); }
    else     { if (gated) PK(short, true); else PK(short, false); }
#undef PK
  }
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// Keys and values of a latent cache: rows of `pages` (R latents, P shared columns)
// times w (N, R), page after page, and their shared columns beside them.  The tiles
// above, with rows that are read where they lie, of 128 x 128 with two workgroups a CU,
// since R is short: one works while the other's first words come and its results go.
// As a copy of the pages and a library product it took, us, then and now (R 512, within
// a call): N 8192: 128 rows 13.2 | 8.6, 704 20.2 | 16.0; N 4096: 1600 rows 25.8 | 17.4,
// 6656 72.8 | 49.2.  (5120 x 8192 over and over: 70.7 | 63.1, in 256 x 256, one workgroup a
// CU, 77.5, in 128 x 256 67.5; but within a call 63.1 | 70.4, and so left to the library.)
// 64 x 128 is for what does not fill the chip otherwise.
// ---------------------------------------------------------------------------
template <int BM, int BN, int WM, int WN>
__global__ void __launch_bounds__(BM / WM * BN / WN * 64)
latent_expand_kernel(MoeGemmArgs a, uint4v* rot, int P, int tiles) {
  constexpr int NT = BM / WM * BN / WN * 64;
  if ((int)blockIdx.x < tiles) {
    moe_tiles<BM, BN, WM, WN, false, true, false, false, true>(a);
    return;
  }
  const int page = blockIdx.x - tiles, words = P / 8;    // its shared columns
  const short* src = (const short*)a.x + a.order[page] * (64 * a.xst) + a.K;
  for (int i = threadIdx.x; i < 64 * words; i += NT)
    rot[(long)page * 64 * words + i] =
        *(const uint4v*)(src + i / words * a.xst + i % words * 8);
}

// R a multiple of 64, P and N of 8; rot [n][64][P]
extern "C" int sv_latent_expand(const void* cache, const int* pages, int n, const void* w,
                                void* out, void* rot, int R, int P, int N,
                                hipStream_t stream) {
  if (n <= 0) return 0;
  if (R % 64 || R <= 0 || P % 8 || P < 0 || N % 8 || N <= 0 || (long)N * R >= 1L << 30)
    return 1;
  MoeGemmArgs a = {};
  a.x = cache;
  a.xst = R + P;
  a.w = w;
  a.out = out;
  a.order = pages;
  a.top = 1;
  a.N = N;
  a.K = R;
  a.rows = n * 64;
#define LE(BM, BN, WM, WN)                                                          \
  do {                                                                              \
    const long tiles = (a.rows + BM - 1L) / BM * ((N + BN - 1) / BN);               \
    latent_expand_kernel<BM, BN, WM, WN>                                            \
        <<<tiles + (P ? n : 0), BM / WM * BN / WN * 64, 0, stream>>>(               \
            a, (uint4v*)rot, P, (int)tiles);                                        \
  } while (0)
  // as many workgroups as are resident (N 8192: 640 rows 13.6 | 14.0 in the larger
  // tiles, 896 17.8 | 15.1; N 2048: 2688 12.9 | 13.9, 3200 17.1 | 14.1)
  if (n * ((N + 127L) / 128) <= 768) LE(64, 128, 64, 32);
  else LE(128, 128, 64, 64);
#undef LE
  return (int)hipGetLastError();
}
