// sac_common.h -- device-side layout and parameter blocks shared by the
// HIP kernels of the SAC perturbation-MHD stage.
//
// Layout: every field is a 3-D array over the grid (mesh + 2 ghost layers
// per active axis, src/vacdef.t:23), index 1 fastest as in the reference's
// w(ixG^T,nw), with the row pitch padded for coalescing.  Indices here are
// 0-based: grid 0..G-1, mesh Mlo..Mhi with Mlo=2, Mhi=G-3.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sac {

constexpr int kMaxDim = 3;
constexpr int kMaxDir = 3;
constexpr int kMaxEvolve = 2 + 2 * kMaxDir;  // rho, m(3), e, b(3)
constexpr int kMaxBg = 2 + kMaxDir;          // eb, rhob, bg(3)
constexpr int kMaxPairs = 21;                // setnu (variable, direction) pairs
constexpr int kRedSlots = 8;                 // reduction values per buffer

// Cell widths come as four tables, dxs elements apart: dx, 1/dx, (1/dx)/12 and
// 0.5/dx, so that a cell's work starts with a load instead of an FP64 division
constexpr int kDxInv = 1, kDxInv12 = 2, kDxHalf = 3, kDxTables = 4;

// the tables of n widths dx, at t, t + dxs, ...
inline void fill_dx_tables(double* t, long long dxs, const double* dx, long long n) {
  for (long long i = 0; i < n; i++) {
    t[i] = dx[i];
    t[kDxInv * dxs + i] = 1.0 / dx[i];
    t[kDxInv12 * dxs + i] = (1.0 / dx[i]) / 12.0;
    t[kDxHalf * dxs + i] = 0.5 / dx[i];
  }
}

// storage precision of the evolving fields
enum PrecCode : int { PREC_FP64 = 0, PREC_MIXED = 1 };

// boundary codes (typeB strings, src/vacgrid.t:257-464)
enum BcCode : int {
  BC_CONT = 1,
  BC_FIXED = 2,
  BC_PERIODIC = 3,
  BC_SYMM = 4,
  BC_SYMM0 = 5,
  BC_ASYMM = 6,
  BC_CONT1 = 7,
  BC_FIXED1 = 8,
  BC_GRAD1 = 9,
  BC_CONTCD4 = 10,
  BC_ZERO = 11
};

// Fields start kFieldPad elements into their allocation, so that the first
// mesh cell of every row (grid index 2, rows padded to 16 elements, 32 where
// elements are FP32) lies on a 128-byte line: tiles that start at the mesh
// fill whole lines, or halves of one with their neighbour in FP32.  (Tiles
// that start at the row start to be aligned cover two ghost columns: 9 tiles
// for 128 cells, 3 for 31; the 128^3 stage took 8 % longer with them.)
constexpr int kFieldPad = 30, kFieldPadEnd = 2;

struct GridDesc {
  int ndim, ndir;
  int G[3];        // grid extents (1 on inactive axes)
  int Mlo[3];      // first mesh index (2 on active axes, 0 otherwise)
  int Mhi[3];      // last mesh index
  long long st[3]; // element strides per axis
  long long fs;    // field stride (elements)
  int per_lo[3];   // 1 if the lower boundary of axis d is periodic (for var 1)
  int per_hi[3];
};

// Reductions (as uint64 bit patterns of non-negative doubles), per register:
// [d] = max over the mesh of cmax_d (c_tot of setnu) and [ndim+d] = max over
// the mesh of cmax_d/dx_d (getdt_courant), d<ndim; maxviscoef is a word of
// its own.
//
// The blocks of a stage add their maxima to kRedLines lines of 128 bytes
// (block b to line b % kRedLines; words as above, maxviscoef in word
// kRedVisc), and the kernel after the stage takes the maximum over the lines
// into the register's words and clears them (red_combine).  Maxima of one
// word are served one after another, about 3-4 ns each: the 65536 blocks x 6
// words of an update of 256^3 cells queued for longer than its memory
// traffic takes.
constexpr int kRedLines = 16;
constexpr int kRedWords = 16;  // words per line
constexpr int kRedVisc = 6;

// What red_combine does with the lines: red[k] = max over the lines of word
// k (k < kRedVisc); *visc = that of word kRedVisc, or the larger of it and
// *visc (visc_keep); both also to host memory if given.
struct RedCombine {
  unsigned long long* acc;   // null: nothing to combine
  unsigned long long* red;
  unsigned long long* visc;  // null: leave maxviscoef
  unsigned long long* host;  // pinned, kRedSlots words
  int visc_keep;
};

}  // namespace sac
