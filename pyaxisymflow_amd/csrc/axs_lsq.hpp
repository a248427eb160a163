// Least-squares extrapolation of the soft-body steps.
#pragma once

#include "axs_common.hpp"

namespace axs {

struct LsqEntry {
  int cell, level;
};

// Buffers of one case's extrapolation over its doubled (2 nr, nz) grid.  The
// pass before it (the mirror) writes every cell's flags and the values of
// the target cells; the values are extrapolated in place.
struct LsqWork {
  // bit rows of wstride words, 32 cells a word: cells known before the
  // extrapolation (a walk outside LDS adds those it finds), and target cells
  // (the known ones among them)
  unsigned *kb, *tb;
  unsigned* kb2;  // the known cells after every other front of the launches
  unsigned* cnt;  // cells of each front of the launches (cleared by the step's dt pass)
  // a box that does not fit in LDS: the words with cells to find (row << 16 |
  // word of the row), their cells not found yet and found by this front
  unsigned *wl, *tw, *fw;
  int wstride;
  int* lev;       // 0 known, else the front that fits the cell; kLsqNever: none has yet
  LsqEntry* list; // cells to fit, front after front
  int* off;       // list end of each front (off[0] = 0)
  unsigned* head; // listed cells, fronts
  unsigned* win;  // packed windows of the listed cells
  double* fac;    // factors of the first fcap of them, nine arrays of fcap
  int fcap;
};

constexpr int kLsqNever = 0x7fffffff;

// A solid whose radius is this many cells or more is large: the first
// kLsqFrontLaunches fronts of a step (a stiff solid's loop takes 9 to 13) are
// found, and fitted, by launches of many workgroups, the others by one.  About
// there one workgroup's walk no longer fits in LDS; us a step, one workgroup /
// the launches: radius 205 cells (512 x 256) walk 52 / -, fits 71 / -; 410
// (1024 x 512) 129 (380 on the whole box) / 92, 123 / 62; 1638 (4096 x 2048)
// 511 (4918) / 136, 684 / 70.
constexpr double kLsqLargeRadius = 224.0;
constexpr int kLsqFrontLaunches = 12;
static_assert(kLsqFrontLaunches % 2 == 0, "the known cells end in kb");
__host__ __device__ constexpr bool lsq_large(double r_ball, double dx) {
  return r_ball >= kLsqLargeRadius * dx;
}

// Words per bit row: whole 256-column workgroups of the mirror pass.
__host__ __device__ constexpr int lsq_words(int nz) { return (nz + 255) / 256 * 8; }
// Most fronts of a doubled grid of n cells (both sizes even): a shortest
// path between 8-neighbours holds at most two cells of a 2 x 2 block.
__host__ __device__ constexpr int64_t lsq_max_fronts(int64_t n) { return n / 2; }
// Factors kept per case: a sixteenth of the doubled grid's n (a band a few
// cells wide is 2% of it at 256 rows).
__host__ __device__ constexpr int lsq_factor_cap(int64_t n) { return int(n / 16 + 1); }

// Extrapolates (e1d, e2d) of a case whose known cells are all targets: the
// reference's loop (core/src/extrapolate_using_least_squares.hpp:142-446),
// bit for bit, in three launches (and 2 kLsqFrontLaunches more of a large
// solid).  z: coordinates of both axes.  zone[1]:
// the last physical row with a target cell, -1 if none.
hipError_t launch_lsq_fronts(const LsqWork& w, double* e1d, double* e2d, const double* z, int nr,
                             int nz, const int* zone, bool large, hipStream_t s);

}  // namespace axs
