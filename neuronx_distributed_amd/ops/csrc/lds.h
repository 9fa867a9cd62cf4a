// Tiles that go straight from memory into LDS, 16 bytes a lane, and transposing
// reads of them.
#pragma once

#include "common.h"

// operands of direct loads into LDS and of transposing LDS loads
typedef __attribute__((address_space(1))) const void* global_ptr;
typedef __attribute__((address_space(3))) void* lds_ptr;
typedef short tr4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) tr4* lds_tr4;

// 16 bytes a lane from `off` + `at` bytes (less than 2^31; the wave shares `at`)
// behind a base that the wave shares, to where the wave's 1 KB begins.  A buffer load: behind other loads into
// LDS the compiler waits for everything on its way, loads and LDS reads, wherever it
// needs a value that came from either.
__device__ __forceinline__ void words_to_lds(const void* base, int off, char* lds,
                                             int at = 0) {
  const auto src = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0x7fffffff,
                                                     0x00027000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_ptr)lds, 16, off, at, 0, 0);
}

// The 16-byte slots of a key row are rotated, so that consecutive rows of one
// column spread over the banks: all 16 of a row of 256 bytes (16 lanes are
// served at once), else within groups of eight; those of a value row in pieces
// of four, which a transposing read takes from four rows at once.
template <int SLOTS>
__device__ __forceinline__ int key_turn(int row) {
  return SLOTS == 16 ? row & 15 : (SLOTS % 16 == 0 ? row : row >> 1) & 7;
}
// after how many fragments of two slots the rotation repeats
template <int SLOTS> struct KeySlots { static constexpr int steps = 4; };
template <> struct KeySlots<16> { static constexpr int steps = 8; };
template <int SLOTS>
__device__ __forceinline__ int value_turn(int row) {
  return (SLOTS % 16 == 0 ? row & 3 : (row >> 1) & 1) << 2;
}

// Rows of 256 bytes (16 slots) that are read both as rows, 16 lanes taking the
// same slot of 16 rows at once, and by transposing reads, 32 lanes taking four
// slots of 4 rows: each touches every bank once.
__device__ __forceinline__ int row_turn(int row) {
  return (row & 3) << 2 | (row >> 2 & 3);
}
// This lane's part of the address of a fragment of rows: slot 2 c + hi of row
// col is at row_lane(col, hi) ^ 32 c, rows col + 16 n follow 4096 n bytes on.
__device__ __forceinline__ int row_lane(int col, int hi) {
  return col * 256 + (hi ^ row_turn(col)) * 16;
}
// The same of a transposing read, where 16 lanes turn 4 rows by 16 columns:
// columns 32 nb ... of rows 16 c + 8 u + 4 hi ... are at (tr_lane() ^ 64 nb ^
// 32 u) + 4096 c + 2048 u.  Lane col gets column col, rows in the order in
// which an accumulator holds them.
__device__ __forceinline__ int tr_lane(int lane) {
  const int hi = lane >> 5, r = (lane & 15) >> 2;
  const int slot = (lane >> 4 & 1) * 2 + (lane >> 1 & 1);
  return (4 * hi + r) * 256 + ((4 * r) ^ slot ^ hi) * 16 + (lane & 1) * 8;
}
