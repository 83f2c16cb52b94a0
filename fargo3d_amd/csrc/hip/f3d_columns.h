// f3d_columns.h -- which cells of a ring the lanes of a one-pass source wave
// hold (kd_src_fused2).  Plain C++, so that the host can go through the indexes.
#pragma once

// cells a wave updates: its 64 stress columns but for the first and the last
constexpr int kSrcCols = 62;

// the stress column of lane `lane` of the ring's wave `wave`, counted from the
// ring's first cell: -1 is the ring's last cell, nx its first again
constexpr int src_position(int wave, int lane) { return kSrcCols * wave - 1 + lane; }

// its cell on a ring of nx cells.  Of the positions past the ring's end, up to 62
// of them, only the first is a neighbour that an updated cell reads; all take
// the first cell, which lies on a ring of any length.
constexpr int src_cell(int is, int nx) { return is < 0 ? is + nx : (is >= nx ? 0 : is); }

// whether the lane updates its cell
constexpr bool src_updates(int is, int lane, int nx) { return lane >= 1 && lane <= kSrcCols && is < nx; }
