// Address arithmetic of the kernels that holds only within limits, as plain
// functions that the kernels and host checks share.
#pragma once

#include <cstddef>
#include <cstdint>

namespace hn {

// lines per FFT workgroup: n * L elements held 16 per thread, plus the
// twiddle table (8 bytes per entry), within 64 KiB of LDS
constexpr int lines_per_wg(int64_t n, int max_elems) {
  int L = 16;
  while (L > 1 && (n * L > max_elems || (size_t)n * (L + 2) * 8 > 65536)) L >>= 1;
  return L;
}

// Lines per workgroup of a pass over `lines` lines: the axis's L, or a
// quarter of it where that leaves CUs without any workgroup.  A single 2D
// image has a few dozen workgroups of L lines, whose threads then walk 12 to
// 16 elements each with most of the chip idle (256^2, one image: the four
// passes 33.5 -> 21.9 us).  min_l: fewer lines are not allowed (line masks).
constexpr int lines_of(int L, int64_t lines, int min_l = 1) {
  return L >= 4 && L / 4 >= min_l && lines < 256 * (int64_t)L ? L / 4 : L;
}

// Strided FFT pass.  Position pos of a line of n, column c of its workgroup's
// adjacent lines, stands at pos * lstride + c cells from the first line's
// first cell.  Thread (e0, l) of E = threads / L rows takes positions
// e0 + i * E: slot i.  Of M kept positions (M > 0; hin = M / 2), the e-th
// stands at e - hin, + n if that is negative.

// every cell of the lines is within 32-bit byte offsets of the first
constexpr bool strided_fits_32(int64_t n, int64_t lstride, int64_t nx) {
  return (n * lstride + nx) * 8 < ((int64_t)1 << 32);
}

// byte offset of position e0, column c (right for every cell of lines that
// fit 32 bits, and for the threads' first positions of any)
constexpr uint32_t strided_thread_offset(int e0, int64_t lstride, int c) {
  return ((uint32_t)e0 * (uint32_t)lstride + (uint32_t)c) * 8u;
}

// byte offset that slot i adds for every thread (negative ones wrap)
constexpr uint32_t strided_slot_offset(int i, int E, int hin, int64_t lstride) {
  return (uint32_t)(i * E - hin) * (uint32_t)lstride * 8u;
}

// byte offset of the cell of position e = e0 + i * E, where the lines fit 32
// bits: the terms wrap, their sum is the offset of a cell and does not
constexpr uint32_t strided_cell_offset(uint32_t thread, uint32_t slot, int e, int hin,
                                       uint32_t line) {
  return thread + slot + (e < hin ? line : 0u);
}

// bytes from the first cell of `cols` lines to the end of their last.  A wave
// loads its slot as one, also the lanes past the last position: the loads are
// bounded by this length, past it they return zero without an access.
constexpr uint32_t strided_line_bytes(int64_t n, int64_t lstride, int cols) {
  return (uint32_t)(((n - 1) * lstride + cols) * 8);
}

// k_interp_pairs: the region's cells from 0, planes apart by a stride, the row
// table (a cell per region row) behind them.  Before the region, its cells
// hold the points' weights, kPairWRow floats each (axis 1 at 0, axis 2 at 8).
constexpr int kStreamRows = 256;  // region rows that row tables hold
constexpr int kPairNT = 512;
constexpr int kPairCells = 9216;  // two workgroups per CU
constexpr int kPairTrips = 2;
constexpr int kPairPoints = kPairTrips * kPairNT / 8;
constexpr int kPairWRow = 20;
constexpr int kPairWeightCells = kPairPoints * kPairWRow / 2;

// cells between the region's planes: at least the plane, 4 modulo 8
constexpr int pair_plane_stride(int plane) { return plane + ((12 - plane % 8) % 8); }

// the row table's first cell, behind a region of `cells` and the weights
constexpr int pair_row_table(int cells) {
  return cells > kPairWeightCells ? cells : kPairWeightCells;
}

}  // namespace hn
