// Where int4_head_rows_kernel keeps its rows in LDS (plain arithmetic, no HIP).  SETS > 0 (up to eight rows): sets of four rows; 0: up to sixteen rows.
#pragma once
#include <algorithm>
#include <cstddef>

constexpr int HR_AHEAD = 8;  // scale groups of a tile on their way at a time
constexpr int HR_KQ = 272;   // sets: bytes between the runs of eight k: sixteen rows of 16 bytes, and 16 against bank conflicts

constexpr int hr_sets(int rows) { return rows <= 8 ? (rows + 3) / 4 : 0; }
constexpr int hr_batches(int groups) { return (groups + HR_AHEAD - 1) / HR_AHEAD; }
constexpr size_t hr_rows_bytes(int rows, int K) {
    return hr_sets(rows) > 0 ? (size_t)hr_sets(rows) * 4 * HR_AHEAD * hr_batches(K / 32) * HR_KQ : (size_t)(K / 32) * 3 * 1024;
}

// Where eight k of a row are put.  SETS > 0: [set][run of eight k, padded to whole batches][4 sequence + piece]; 0: [group][piece][run][row], rows moved about by
// the run against bank conflicts.
template <int SETS>
constexpr int hr_piece_at(int groups, int run, int row, int piece) {
    if (SETS > 0) return ((row >> 2) * 4 * HR_AHEAD * hr_batches(groups) + run) * HR_KQ + (4 * (row & 3) + piece) * 16;
    return (((run >> 2) * 3 + piece) * 4 + (run & 3)) * 256 + ((row ^ (run & 15)) << 4);
}

// Where the operand of group g + u, g a multiple of HR_AHEAD, is read by lane (c16, kq).  The last batch asks for all of its places; those behind the last group are
// not multiplied: padding where there are sets, the row's first group again where there is no room for padding.
template <int SETS>
constexpr int hr_operand_at(int groups, int g, int u, int set, int piece, int kq, int c16) {
    if (SETS > 0) return (4 * g + kq) * HR_KQ + c16 * 16 + (4 * HR_AHEAD * set * hr_batches(groups) + 4 * u) * HR_KQ;
    return kq * 256 + ((c16 ^ ((4 * u + kq) & 15)) << 4) + (g + u < groups ? g + u : 0) * 3072 + piece * 1024;
}
