// column_types.h -- plain types of the column layout, shared by the sweep
// body (column_sweep.h), its host launchers (kernels.h) and its CPU emulation
// (tests/emu/column_emu.cpp).
//
// A column is 16 x 8 (j, k) lines along i, two lines per lane of a wave: lane
// j%16 + 16*(k%8/2) holds lines k and k+1.  Its slots are numbered by
// hyperplane h = i + j + k first, lane second and line last: one slice of 128
// slots per hyperplane between the lowest and the highest one that holds a
// pressure row of the column.  A wave that follows the hyperplanes then reads
// and writes whole slices of consecutive addresses, and every neighbour of a
// slot is at a fixed place of the next or the previous hyperplane's slice.
// Slots without a row hold zeros in every array.
#pragma once

namespace ff {

constexpr int COL_R = 2;                      // lines (along k) of a lane
constexpr int COL_J = 16, COL_K = 4 * COL_R;  // lines along j and k
constexpr int COL_LANES = 64;
constexpr int COL_SLICE = COL_LANES * COL_R;  // slots per slice
constexpr int COL_SKEW = COL_J + COL_K - 2;   // a column spans up to ni + COL_SKEW hyperplanes
constexpr int COL_WAVES = 2;                  // columns of a tile, along k

// place in a slice of line (j, k) of its column
constexpr int columnPlace(int j, int k) { return (j % COL_J + COL_J * (k % COL_K / COL_R)) * COL_R + k % COL_R; }
// and the line of a place
constexpr int columnLineJ(int place) { return place / COL_R % COL_J; }
constexpr int columnLineK(int place) { return place / COL_R / COL_J * COL_R + place % COL_R; }

// first slot of h's slice = base + COL_SLICE*h for lo <= h <= hi; no rows: lo > hi
struct ColumnRange {
    int lo, hi, base, pad;
};

// per slice: first slot of the neighbouring slices (hyperplane h-1 of the
// column itself and of its -j and -k neighbours, h+1 of itself, +j and +k),
// -1 where that slice does not exist; then the column and h
struct SliceLinks {
    int im, ip, jm, jp, km, kp, col, h;
};

}  // namespace ff
