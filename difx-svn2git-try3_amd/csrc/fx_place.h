// fx_place.h — which blocks a workgroup of the F stage takes and which rows of V
// one of the cross-multiply stores, shared by the kernels and host-side tests.
#pragma once
#include "fx_bits.h"

namespace fxg {

// A launch has rows (a band, or a pair) of groups of blocks, each group for PW
// workgroups.  Workgroups are dealt to the 8 XCDs round-robin, x first, and a
// grid's x is a multiple of 8 PW; the PW of a group lie on one XCD, whose L2
// merges the lines that they write.
//   8 groups and more: a grid row is a row, and each XCD takes an eighth of its
// groups (neighbouring blocks share lines in the grouped layout).  Below 64
// groups the eighths may be far from even, so which XCD has the first moves on
// with the row (nine blocks of 40 bands of 65536 8-bit points 191 -> 116 us); from
// there on it stays, and finds in its L2 what the row before read of the same
// blocks (112 bands of 512 points 1.22 ms, with the move 1.24).
//   Fewer than 8: a grid row is a group and the rows go to the XCDs in turn.  A
// grid of rows starts eight workgroups for each of one block's that has work, and
// without the move all on one XCD (144 bands of 8192 points, one block: 26 us, with
// the move 16, now 10; 40 bands of 65536 8-bit points 97, 24, 24).
struct FsGrid { unsigned x, y; };
FXG_HD FsGrid fstage_grid(unsigned groups, unsigned rows, unsigned PW) {
  return groups < 8 ? FsGrid{(rows + 7) / 8 * 8 * PW, groups} : FsGrid{(groups + 7) / 8 * 8 * PW, rows};
}
struct FsPlace { unsigned row, grp, pw; };      // row or group may lie past the last: no work
FXG_HD FsPlace fstage_place(unsigned x, unsigned y, unsigned gx, unsigned groups, unsigned PW) {
  const unsigned k = x / (8 * PW), pw = x / 8 % PW;
  return groups < 8 ? FsPlace{8 * k + x % 8, y, pw} : FsPlace{y, (groups < 64 ? x + y : x) % 8 * (gx / (8 * PW)) + k, pw};
}

// The turns of 8 rows in which a 32-row tile of V is stored, with `left` inputs
// from its first row on: 2 inputs, 32768 channels, one block 38 us a launch with
// all four turns, 29 with one.
FXG_HD int tile_turns(int left) { return left <= 0 ? 0 : left < 32 ? (left + 7) / 8 : 4; }

}  // namespace fxg
