// Weights that stream through rings in LDS: blocks of 16 weight rows by 64 columns, in
// two pieces of 8 rows by 128 bytes, that a wave asks for one after the other and takes
// as fragments.  Loads that hold no register and wait for nobody fill a ring, whole
// cache lines of a row at a time: results are summed and stored, and the ring goes on.
#pragma once

#include "serving.h"

// A piece: 16 bytes a lane from `off` on, to where the wave's 1 KB begins.  ONCE: no
// cache keeps it.
template <bool ONCE>
__device__ __forceinline__ void piece(__amdgpu_buffer_rsrc_t src, uint off, char* lds) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_ptr)lds, 16, off, 0, 0, ONCE ? 2 : 0);
}

// One wave's ring of R pieces of 1 KB.
template <int R>
struct Ring {
  char* mine;
  int slot, rd, src;                     // what is asked for and taken next

  __device__ __forceinline__ explicit Ring(char* at) : mine(at), slot(0), rd(0) {
    const int lane = threadIdx.x & 63, r = lane & 7, b = lane >> 3 & 1;
    src = (int)(size_t)(lds_ptr)mine + b * 1024 + r * 128 +
          (((lane >> 4) ^ r ^ b) & 7) * 16;
  }
  // This lane's bytes of a first or second piece of rows `pitch` bytes apart.  Slot s
  // (of 16 bytes) of row r of a piece lies at place s ^ r, of a second one at s ^ r ^
  // 1, so that 16 rows of one slot touch every bank once.
  static __device__ __forceinline__ int lane_bytes(int pitch, int second) {
    const int lane = threadIdx.x & 63, r = lane >> 3;
    return r * pitch + ((lane ^ r ^ second) & 7) * 16;
  }
  // The next block: bytes oa behind a, ob behind b; those past their ends are not
  // read.  No cache keeps them (each is read once: 235 MB in 40.0 us, so 36.0).
  __device__ __forceinline__ void ask(__amdgpu_buffer_rsrc_t a, uint oa,
                                      __amdgpu_buffer_rsrc_t b, uint ob) {
    piece<true>(a, oa, mine + slot);
    piece<true>(b, ob, mine + slot + 1024);
    slot = (slot + 2048) & (R * 1024 - 1);
  }
  // The oldest block, when no more than AFTER loads are on their way behind it:
  // columns 8 grp of its first and second 32.
  template <int AFTER>
  __device__ __forceinline__ void take(frag_u& f0, frag_u& f1) {
    asm volatile("s_waitcnt vmcnt(%4)\n\t"
                 "ds_read_b128 %0, %2\n\t"
                 "ds_read_b128 %1, %3\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(f0.u4), "=&v"(f1.u4)
                 : "v"(src + rd), "v"((src ^ 64) + rd), "n"(AFTER)
                 : "memory");
    rd = (rd + 2048) & (R * 1024 - 1);
  }
};

// `bytes` that pieces are asked of
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ring_source(const void* base,
                                                              int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00027000);
}
#define RING_NOWHERE (1u << 31)          // past every end

// A barrier for what is in LDS: it waits for no load.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Rows that meet them, as fragments.  A fragment's neighbouring lanes have different
// rows, and a load of it would look up a cache line a lane (28672 x 4096 gated, 32
// rows: 44.5 us, now 41.1); neighbours in fours read 64 bytes of a row instead, row
// lane / 4 from column 8 (lane % 4) on, and hand them on.
__device__ __forceinline__ frag_u turned(frag_u f) {
  const int lane = threadIdx.x & 63, from = ((lane & 15) * 4 + (lane >> 4)) * 4;
#pragma unroll
  for (int i = 0; i < 4; ++i) f.u[i] = __builtin_amdgcn_ds_bpermute(from, f.u[i]);
  return f;
}
