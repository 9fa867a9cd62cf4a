// Which words of a row a lane reads.  No device code: a host compiler can check
// that every one of them lies in the row.
#pragma once

// Of columns k .. k + 31 of a row of K (a multiple of 8), the first of the 8 that
// lanes of group `grp` of four read: theirs, or where the row has ended its first
// ones, which every row has.
constexpr int word_column(int k, int grp, int K) {
  return k + grp * 8 < K ? k + grp * 8 : 0;
}
