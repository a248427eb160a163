// Least-squares extrapolation of the reference map (row A14):
// core/src/extrapolate_using_least_squares.hpp:142-446 as instantiated by
// extrapolate_using_least_squares_till_first_order<short, double> (:450-467).
//
// Each sweep of the reference scans every cell, collects the cells with
// current ^ target set and at least one known 3x3 neighbour, fits
// eta = c0 + c1 x + c2 y on a shifted 3x3 window of known cells and only
// then marks the collected cells known (:441-444).  A sweep is therefore
// data-parallel: here one thread per cell fits into side buffers, and a
// second pass commits values and flags.  The arithmetic follows the
// reference's order with FMA contraction off, so results match it bit for
// bit.  Out-of-range cells read as flag 0 (the reference has no bounds
// checks there, :205-219, 276-280).
#include "axs_lsq.hpp"
#include "axs_softbatch.hpp"

#include <vector>

namespace axs {

__device__ __forceinline__ short lsq_flag(const int16_t* f, int n0, int n1, int j, int i) {
  return (j < 0 || j >= n0 || i < 0 || i >= n1) ? short(0) : short(f[(int64_t)j * n1 + i]);
}

// ExtrapolationConfig.hpp:17-19, 131-158 (grid size 3: start = code - 3).
__device__ __forceinline__ short lsq_start_code(short positional_sum, short total_sum) {
  float temp = (positional_sum > short(4)) ? float(ceil(0.5 * float(positional_sum)) * 2.0)
                                           : float(positional_sum);
  short code = short(2.0 * double(temp) / double(total_sum));
  return short(short(2 * code - short(6)) / short(2));
}

template <typename V>
__device__ __forceinline__ void lsq_swap(bool take, V& a, V& b) {
  const V t = a;
  a = take ? b : a;
  b = take ? t : b;
}

// least_squares.hpp:10-59 for 3 coefficients and 2 right-hand sides, split
// into what depends on the known cells alone (the elimination of the normal
// matrix with its pivots) and what depends on the values (the right-hand
// sides); the two parts together run the reference's operations in its
// order.  Rows are exchanged by selects: a row index known only at run time
// would send the matrix to scratch memory.
struct LsqFactor {
  // multipliers of rows 1 and 2 (after the first exchange) and of row 2
  // (after the second), then the upper triangle
  double c1, c2, c3, u00, u01, u02, u11, u12, u22;
  int m0;  // row exchanged with row 0
  int m1;  // rows 1 and 2 exchanged (0 or 1)
};

__device__ __forceinline__ LsqFactor lsq_factor_3x3(double a00, double a01, double a02,
                                                    double a10, double a11, double a12,
                                                    double a20, double a21, double a22) {
  LsqFactor f;
  f.m0 = 0;
  double best = fabs(a00);
  if (fabs(a10) > best) {
    best = fabs(a10);
    f.m0 = 1;
  }
  if (fabs(a20) > best) f.m0 = 2;
  lsq_swap(f.m0 == 1, a00, a10);
  lsq_swap(f.m0 == 1, a01, a11);
  lsq_swap(f.m0 == 1, a02, a12);
  lsq_swap(f.m0 == 2, a00, a20);
  lsq_swap(f.m0 == 2, a01, a21);
  lsq_swap(f.m0 == 2, a02, a22);
  f.c1 = -a10 / a00;
  a11 += f.c1 * a01;
  a12 += f.c1 * a02;
  f.c2 = -a20 / a00;
  a21 += f.c2 * a01;
  a22 += f.c2 * a02;
  f.m1 = fabs(a21) > fabs(a11) ? 1 : 0;
  lsq_swap(f.m1 == 1, a11, a21);
  lsq_swap(f.m1 == 1, a12, a22);
  f.c3 = -a21 / a11;
  a22 += f.c3 * a12;
  f.u00 = a00;
  f.u01 = a01;
  f.u02 = a02;
  f.u11 = a11;
  f.u12 = a12;
  f.u22 = a22;
  return f;
}

// The fit's value at (px, py) for one right-hand side (b0, b1, b2).
__device__ __forceinline__ double lsq_eval(const LsqFactor& f, double b0, double b1, double b2,
                                           double px, double py) {
  lsq_swap(f.m0 == 1, b0, b1);
  lsq_swap(f.m0 == 2, b0, b2);
  b1 += f.c1 * b0;
  b2 += f.c2 * b0;
  lsq_swap(f.m1 == 1, b1, b2);
  b2 += f.c3 * b1;
  const double s2 = b2 / f.u22;
  b1 -= f.u12 * s2;
  b0 -= f.u02 * s2;
  const double s1 = b1 / f.u11;
  b0 -= f.u01 * s1;
  const double s0 = b0 / f.u00;
  double e = 0.0;
  e += s0 * 1.0;
  e += s1 * (1.0 * px);
  e += s2 * (1.0 * py);
  return e;
}

// Normal matrix of the window at (s_y, s_x) from its cells' flags m (row
// major, 0 or 1), factored.
__device__ __forceinline__ LsqFactor lsq_window_factor(const double m[9],
                                                       const double* __restrict__ gx,
                                                       const double* __restrict__ gy, int n0,
                                                       int n1, int s_y, int s_x) {
  double L1[9], L2[9];
#pragma unroll
  for (int n = 0; n < 9; ++n) {
    const int jl = s_y + n / 3, il = s_x + n % 3;
    L1[n] = m[n] * ((il >= 0 && il < n1) ? gx[il] : 0.0);
    L2[n] = m[n] * ((jl >= 0 && jl < n0) ? gy[jl] : 0.0);
  }
  double b00 = 0.0, b01 = 0.0, b02 = 0.0, b11 = 0.0, b12 = 0.0, b22 = 0.0;
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    b00 += m[q] * m[q];
    b01 += m[q] * L1[q];
    b02 += m[q] * L2[q];
    b11 += L1[q] * L1[q];
    b12 += L1[q] * L2[q];
    b22 += L2[q] * L2[q];
  }
  return lsq_factor_3x3(b00, b01, b02, b01, b11, b12, b02, b12, b22);
}

// Fit of cell (j, i) from the known cells around it
// (extrapolate_using_least_squares.hpp:190-305); false when no 3x3
// neighbour is known (the cell waits for a later sweep).
__device__ __forceinline__ bool lsq_fit_cell(const int16_t* __restrict__ cur,
                                             const double* __restrict__ ex,
                                             const double* __restrict__ ey,
                                             const double* __restrict__ gx,
                                             const double* __restrict__ gy, int n0, int n1,
                                             int j, int i, double& vx, double& vy) {
  short local_sum = 0, lx = 0, ly = 0;
#pragma unroll
  for (int jl = -1; jl <= 1; ++jl)
#pragma unroll
    for (int il = -1; il <= 1; ++il) {
      const short f = lsq_flag(cur, n0, n1, j + jl, i + il);
      local_sum += (jl == 0 && il == 0) ? short(0) : f;
      lx += f * short(il + 1);
      ly += f * short(jl + 1);
    }
  if (!local_sum) return false;
  const int s_x = i + lsq_start_code(lx, local_sum);
  const int s_y = j + lsq_start_code(ly, local_sum);
  double m[9], r0[9], r1[9];
#pragma unroll
  for (int n = 0; n < 9; ++n) {
    const int jl = s_y + n / 3, il = s_x + n % 3;
    const bool in = (jl >= 0 && jl < n0 && il >= 0 && il < n1);
    const int64_t g = (int64_t)jl * n1 + il;
    m[n] = in ? double(cur[g]) : 0.0;
    r0[n] = m[n] * (in ? ex[g] : 0.0);
    r1[n] = m[n] * (in ? ey[g] : 0.0);
  }
  const LsqFactor f = lsq_window_factor(m, gx, gy, n0, n1, s_y, s_x);
  double bx[3] = {0.0, 0.0, 0.0}, by[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int n = 0; n < 9; ++n) {
    const int jl = s_y + n / 3, il = s_x + n % 3;
    const double l1 = m[n] * ((il >= 0 && il < n1) ? gx[il] : 0.0);
    const double l2 = m[n] * ((jl >= 0 && jl < n0) ? gy[jl] : 0.0);
    bx[0] += m[n] * r0[n];
    bx[1] += l1 * r0[n];
    bx[2] += l2 * r0[n];
    by[0] += m[n] * r1[n];
    by[1] += l1 * r1[n];
    by[2] += l2 * r1[n];
  }
  vx = lsq_eval(f, bx[0], bx[1], bx[2], gx[i], gy[j]);
  vy = lsq_eval(f, by[0], by[1], by[2], gx[i], gy[j]);
  return true;
}

// One sweep, phase 1: select + fit.  pend[c] = 1 when cell c is extrapolated
// this sweep (new values in nx/ny), else 0.
__global__ void __launch_bounds__(256) lsq_fit_kernel(const int16_t* __restrict__ cur, const int16_t* __restrict__ tgt,
                               const double* __restrict__ ex, const double* __restrict__ ey,
                               const double* __restrict__ gx, const double* __restrict__ gy,
                               int n0, int n1, double* __restrict__ nx, double* __restrict__ ny,
                               int8_t* __restrict__ pend, unsigned* __restrict__ counter,
                               const unsigned* __restrict__ prev_counter) {
  // A sweep after one that fitted nothing does nothing (the reference loop
  // has ended); its commit sees a zero counter and exits too.
  if (prev_counter && *prev_counter == 0u) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;  // column (x)
  const int j = blockIdx.y;                              // row (y)
  if (i >= n1) return;
  const int64_t c = (int64_t)j * n1 + i;
  pend[c] = 0;
  if (!(cur[c] ^ tgt[c])) return;
  double vx, vy;
  if (!lsq_fit_cell(cur, ex, ey, gx, gy, n0, n1, j, i, vx, vy)) return;
  nx[c] = vx;
  ny[c] = vy;
  pend[c] = 1;
  atomicAdd(counter, 1u);
}

// Phase 2: commit values and flags of the cells fitted in phase 1.
__global__ void lsq_commit_kernel(int16_t* __restrict__ cur, double* __restrict__ ex,
                                  double* __restrict__ ey, const double* __restrict__ nx,
                                  const double* __restrict__ ny, const int8_t* __restrict__ pend,
                                  int64_t n, const unsigned* __restrict__ counter) {
  if (*counter == 0u) return;  // nothing fitted (or the loop has ended)
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n || !pend[c]) return;
  ex[c] = nx[c];
  ey[c] = ny[c];
  cur[c] = 1;
}

__global__ void fill_u32_kernel(unsigned* p, int n, unsigned v) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) p[k] = v;
}

// Scratch of the drop-in entry point's sweeps.
struct LsqSweepWork {
  double* nx;          // fitted eta_x of this sweep, (n0, n1)
  double* ny;          // fitted eta_y of this sweep, (n0, n1)
  int8_t* pend;        // 1 where a cell was fitted this sweep
  unsigned* counters;  // cells fitted per sweep (one slot per sweep)
};

// One sweep (fit + commit).  Sweep `sweep` exits at once when
// counters[sweep - 1] is zero, so many sweeps can be queued without a sync.
static hipError_t launch_lsq_sweep(int16_t* cur, const int16_t* tgt, double* ex, double* ey,
                            const double* gx, const double* gy, int n0, int n1, const LsqSweepWork& w,
                            int sweep, hipStream_t s) {
  dim3 grid(ceil_div(n1, 256), n0);
  lsq_fit_kernel<<<grid, 256, 0, s>>>(cur, tgt, ex, ey, gx, gy, n0, n1, w.nx, w.ny, w.pend,
                                      w.counters + sweep,
                                      sweep > 0 ? w.counters + sweep - 1 : nullptr);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t n = (int64_t)n0 * n1;
  lsq_commit_kernel<<<ceil_div(n, 256), 256, 0, s>>>(cur, ex, ey, w.nx, w.ny, w.pend, n,
                                                      w.counters + sweep);
  return hipGetLastError();
}

static hipError_t launch_fill_u32(unsigned* p, int n, unsigned v, hipStream_t s) {
  fill_u32_kernel<<<ceil_div(n, 256), 256, 0, s>>>(p, n, v);
  return hipGetLastError();
}

// -------------------------------------------------- soft steps: by fronts
//
// In the soft steps every known cell is a target (known: phi > 0, target:
// phi > -extrap_zone), so a sweep of the reference fits exactly the unknown
// target cells next to a cell known before it: the sweep that fits a cell
// is its 8-neighbour distance from the known set within the target set,
// whatever the values are.  The loop then splits into three launches:
//   levels  one workgroup per case walks the fronts on bit rows in LDS and
//           lists the cells front by front (the first fronts of a large solid
//           are launches of their own: kLsqLargeRadius);
//   factor  one thread per listed cell: its window, the cells of it known
//           before its front, and the factored normal matrix, none of which
//           depends on the values;
//   solve   one workgroup per case and component takes the fronts in order
//           (a block barrier between them): window values in, right-hand
//           side, back substitution, value out (a large solid's first
//           fronts by many workgroups, a launch each).
// One launch per sweep was bound by a fit's latency (flags, window, a 3 x 3
// elimination with nine divisions, its pivoted rows in scratch memory): 17
// us a sweep for twelve cases of 130 to 490 rows, paid for every queued
// sweep.  Now a front pays only the value-dependent part: on those cases 125
// us a step (levels 46, factor 19, solve 61) instead of 273, and 52 instead
// of 163 for one 256 x 128 case (19, 10, 24).  The solve pass is bound by the
// rate of its gathers (nine window values per cell, each lane another line:
// about a line per cycle from the CU's L1), so the two components run on two
// CUs; the levels pass by the list stores and barriers of each front.
// Every fit runs the same operations in the same order as lsq_fit_cell on
// the flags and values its sweep saw, so the results are the same bits.

// The fronts' known-cell bit rows in LDS: words of 32 cells, at most
// kLsqOwn per thread.
constexpr int kLsqThreads = 1024, kLsqOwn = 7;
constexpr int kLsqLdsWords = kLsqThreads * kLsqOwn;  // 28 KiB

// 8-neighbour dilation at word (row, c) of `known` (rows x wc words).
__device__ __forceinline__ unsigned lsq_dilate(const unsigned* known, int row, int c, int rows,
                                               int wc) {
  unsigned d = 0u;
#pragma unroll
  for (int rr = -1; rr <= 1; ++rr) {
    const int r = row + rr;
    if (r < 0 || r >= rows) continue;
    const unsigned* k = known + (r * wc + c);
    const unsigned m = k[0];
    d |= m | (m << 1) | (m >> 1);
    if (c > 0) d |= k[-1] >> 31;
    if (c + 1 < wc) d |= k[1] << 31;
  }
  return d;
}

// The same on words in global memory, every load issued at once (a word outside
// the rows reads its neighbour and counts as 0).
__device__ __forceinline__ unsigned lsq_dilate_at(const unsigned* known, int row, int c, int rows,
                                                  int wc) {
  unsigned m[9];
#pragma unroll
  for (int n = 0; n < 9; ++n) {
    const int r = min(max(row + n / 3 - 1, 0), rows - 1), q = min(max(c + n % 3 - 1, 0), wc - 1);
    m[n] = known[(int64_t)r * wc + q];
  }
  unsigned d = 0u;
#pragma unroll
  for (int n = 0; n < 3; ++n) {
    const int r = row + n - 1;
    const unsigned mid = m[3 * n + 1];
    const unsigned left = c > 0 ? m[3 * n] >> 31 : 0u, right = c + 1 < wc ? m[3 * n + 2] << 31 : 0u;
    if (r >= 0 && r < rows) d |= mid | (mid << 1) | (mid >> 1) | left | right;
  }
  return d;
}

// Lists the cells of `bits`, whose lowest is cell `base`, as front `level`,
// from entry `pos` on.
__device__ __forceinline__ void lsq_list_bits(const LsqWork& w, unsigned bits, unsigned base,
                                              int level, unsigned pos) {
  while (bits) {
    const unsigned cell = base + (unsigned)__ffs((int)bits) - 1u;
    bits &= bits - 1u;
    w.list[pos++] = LsqEntry{(int)cell, level};
    w.lev[cell] = level;
  }
}
__device__ __forceinline__ void lsq_emit(const LsqWork& w, unsigned bits, unsigned base, int level,
                                         unsigned* s_n) {
  // the counter's address made to look divergent: on a uniform address the
  // compiler adds the lanes up one by one in a loop before its one atomic
  int zero;
  asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
  lsq_list_bits(w, bits, base, level, atomicAdd(s_n + zero, (unsigned)__popc(bits)));
}

// Block barrier that orders LDS accesses alone: the global stores of a
// front's list entries stay in flight (nothing in the walk reads them), where
// __syncthreads would wait for each front's to land.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The fronts of one case, by one workgroup of kLsqThreads, after the first
// `done` of them (0 or kLsqFrontLaunches: lsq_front_levels_body has listed
// those).  zone[1]: the last physical row with a target cell (-1: none); the
// doubled rows with target cells are nr - 1 - zone[1] .. nr + zone[1].
__device__ __forceinline__ void lsq_levels_body(const LsqWork& w, int nr, int nz,
                                                const int* __restrict__ zone, int done) {
  __shared__ unsigned sk[kLsqLdsWords];
  __shared__ int s_w0, s_w1;
  __shared__ unsigned s_n, s_m;
  const int tid = threadIdx.x;
  unsigned n = 0u;
  int level = 0;
  for (; level < done; ++level) {  // uniform
    const unsigned c = w.cnt[level];
    if (!c) break;
    n += c;
    if (tid == 0) w.off[level + 1] = (int)n;
  }
  if (tid == 0) w.off[0] = 0;
  if (level < done) {  // a front of the launches found nothing: all are listed
    if (tid == 0) {
      w.head[0] = n;
      w.head[1] = (unsigned)level;
    }
    return;
  }
  const int z1 = zone[1];
  const int W = (nz + 31) / 32, r0 = nr - 1 - z1, rows = 2 * (z1 + 1);
  if (tid == 0) {
    s_w0 = W;
    s_w1 = -1;
    s_n = n;
    s_m = 0u;
  }
  __syncthreads();
  // word columns with target cells: a word per thread, or, of more rows than
  // fit in LDS whole, groups of four words as they lie (a row's words beyond
  // nz are 0)
  const int G = w.wstride / 4, ng = rows * G;
  const uint4* tb4 = reinterpret_cast<const uint4*>(w.tb + (int64_t)r0 * w.wstride);
  const uint4* kb4 = reinterpret_cast<const uint4*>(w.kb + (int64_t)r0 * w.wstride);
  int lo = W, hi = -1;
  if (rows * W <= kLsqLdsWords) {
    for (int q = tid; q < rows * W; q += kLsqThreads) {
      const int r = (int)((unsigned)q / (unsigned)W), c = q - r * W;
      if (w.tb[(int64_t)(r0 + r) * w.wstride + c]) {
        lo = min(lo, c);
        hi = max(hi, c);
      }
    }
  } else {
#pragma unroll 4
    for (int q = tid; q < ng; q += kLsqThreads) {
      const uint4 t = tb4[q];
      const int c = (int)((unsigned)q % (unsigned)G) * 4;
      const unsigned any = (t.x ? 1u : 0u) | (t.y ? 2u : 0u) | (t.z ? 4u : 0u) | (t.w ? 8u : 0u);
      lo = any ? min(lo, c + __ffs((int)any) - 1) : lo;
      hi = any ? max(hi, c + 31 - __clz((int)any)) : hi;
    }
  }
  if (hi >= 0) {
    atomicMin(&s_w0, lo);
    atomicMax(&s_w1, hi);
  }
  __syncthreads();
  const int w0 = s_w0, wc = max(0, s_w1 - s_w0 + 1), nw = rows * wc;
  // A front's cells join the known ones only after every thread has read
  // the known words (first barrier), and are read by the next front after
  // all have joined (second barrier); s_n moves between the second and the
  // first alone, so every thread reads the same count and leaves together.
  if (nw <= kLsqLdsWords) {
    const int own = (nw + kLsqThreads - 1) / kLsqThreads;  // uniform
    unsigned todo[kLsqOwn], f[kLsqOwn];
    int rc[kLsqOwn];  // row << 16 | column (rows <= 8192)
#pragma unroll
    for (int u = 0; u < kLsqOwn; ++u) {
      todo[u] = 0u;
      rc[u] = 0;
      const int q = tid + u * kLsqThreads;
      if (u < own && q < nw) {
        const int r = (int)((unsigned)q / (unsigned)wc), c = q - r * wc;
        const int64_t g = (int64_t)(r0 + r) * w.wstride + w0 + c;
        const unsigned k = w.kb[g];
        rc[u] = r << 16 | c;
        sk[q] = k;
        todo[u] = w.tb[g] & ~k;
      }
    }
    lds_barrier();
    for (;;) {
#pragma unroll
      for (int u = 0; u < kLsqOwn; ++u) {
        f[u] = 0u;
        if (u >= own || !todo[u]) continue;
        const int r = rc[u] >> 16, c = rc[u] & 0xffff;
        f[u] = lsq_dilate(sk, r, c, rows, wc) & todo[u];
        if (f[u])
          lsq_emit(w, f[u], (unsigned)(r0 + r) * (unsigned)nz + (unsigned)(w0 + c) * 32u, level + 1,
                   &s_n);
      }
      lds_barrier();
      const unsigned now = s_n;
      if (now == n) break;
      n = now;
      ++level;
      if (tid == 0) w.off[level] = (int)n;
#pragma unroll
      for (int u = 0; u < kLsqOwn; ++u) {
        if (u >= own || !f[u]) continue;
        sk[tid + u * kLsqThreads] |= f[u];
        todo[u] &= ~f[u];
      }
      lds_barrier();
    }
  } else {
    // A box too large for LDS: the same walk over a list of the words that
    // hold cells to find, and the known words in global memory (kb itself:
    // the next step's mirror writes these rows again).  A front costs the
    // band's words instead of the box's: 129 us a step instead of 380 for a
    // solid of radius 410 cells on 1024 x 512.  Four list entries at a time,
    // so that their loads are in flight together.  A word's entries of tw and
    // fw belong to one thread.
#pragma unroll 4
    for (int q = tid; q < ng; q += kLsqThreads) {
      const uint4 t = tb4[q], k = kb4[q];
      const int r = (int)((unsigned)q / (unsigned)G), c = (q - r * G) * 4;
      const unsigned todo[4] = {t.x & ~k.x, t.y & ~k.y, t.z & ~k.z, t.w & ~k.w};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (!todo[u]) continue;
        const unsigned i = atomicAdd(&s_m, 1u);
        w.wl[i] = (unsigned)(r0 + r) << 16 | (unsigned)(c + u);  // 2 nr <= 8192
        w.tw[i] = todo[u];
      }
    }
    __syncthreads();
    const int m = (int)s_m;
    constexpr int kU = 4;
    for (;;) {
      for (int b = tid; b < m; b += kU * kLsqThreads) {
        unsigned at[kU], todo[kU], f[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const int i = min(b + u * kLsqThreads, m - 1);
          at[u] = w.wl[i];
          todo[u] = w.tw[i];
        }
#pragma unroll
        for (int u = 0; u < kU; ++u)
          f[u] = lsq_dilate_at(w.kb + (int64_t)r0 * w.wstride, (int)(at[u] >> 16) - r0,
                               (int)(at[u] & 0xffffu), rows, w.wstride) & todo[u];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const int i = b + u * kLsqThreads;
          if (i >= m) continue;
          w.fw[i] = f[u];
          if (f[u])
            lsq_emit(w, f[u], (at[u] >> 16) * (unsigned)nz + (at[u] & 0xffffu) * 32u, level + 1,
                     &s_n);
        }
      }
      __syncthreads();
      const unsigned now = s_n;
      if (now == n) break;
      n = now;
      ++level;
      if (tid == 0) w.off[level] = (int)n;
#pragma unroll 4
      for (int i = tid; i < m; i += kLsqThreads) {
        const unsigned f = w.fw[i];
        if (!f) continue;
        const unsigned at = w.wl[i];
        w.kb[(int64_t)(at >> 16) * w.wstride + (at & 0xffffu)] |= f;
        w.tw[i] &= ~f;
      }
      __syncthreads();
    }
  }
  if (tid == 0) {
    w.head[0] = n;
    w.head[1] = (unsigned)level;
  }
}

// Front `front` (from 0) of a case by many workgroups of 256 threads, four
// words each, this one the blk-th: from one buffer of known words into the
// other, the cells found listed after the fronts before it.  cnt[i] holds the
// cells of front i (cleared before the step's first); a front after one that
// found nothing does nothing.
__device__ __forceinline__ void lsq_front_levels_body(const LsqWork& w, int nr, int nz,
                                                      const int* __restrict__ zone, int front,
                                                      int blk) {
  __shared__ unsigned s_n, s_at;
  const int tid = threadIdx.x;
  const int z1 = zone[1], r0 = nr - 1 - z1, rows = 2 * (z1 + 1);
  const int G = w.wstride / 4, ng = rows * G;
  if (blk * 256 >= ng || (front > 0 && w.cnt[front - 1] == 0u)) return;  // uniform
  unsigned base = 0u;
  for (int i = 0; i < front; ++i) base += w.cnt[i];
  const int64_t o = (int64_t)r0 * w.wstride;
  const unsigned* in = ((front & 1) ? w.kb2 : w.kb) + o;
  unsigned* out = ((front & 1) ? w.kb : w.kb2) + o;
  if (tid == 0) s_n = 0u;
  __syncthreads();
  const int q = blk * 256 + tid;
  const int r = (int)((unsigned)q / (unsigned)G), c = (q - r * G) * 4;
  unsigned f[4] = {0u, 0u, 0u, 0u};
  unsigned n = 0u, pos = 0u;
  if (q < ng) {
    const uint4 k = reinterpret_cast<const uint4*>(in)[q];
    const uint4 t = reinterpret_cast<const uint4*>(w.tb + o)[q];
    const unsigned kw[4] = {k.x, k.y, k.z, k.w}, tw[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const unsigned todo = tw[u] & ~kw[u];
      if (todo) f[u] = lsq_dilate_at(in, r, c + u, rows, w.wstride) & todo;
      n += (unsigned)__popc(f[u]);
    }
    reinterpret_cast<uint4*>(out)[q] =
        make_uint4(kw[0] | f[0], kw[1] | f[1], kw[2] | f[2], kw[3] | f[3]);
  }
  if (n) pos = atomicAdd(&s_n, n);
  __syncthreads();
  if (tid == 0 && s_n) s_at = base + atomicAdd(w.cnt + front, s_n);
  __syncthreads();
  if (!n) return;
  pos += s_at;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    lsq_list_bits(w, f[u], (unsigned)(r0 + r) * (unsigned)nz + (unsigned)(c + u) * 32u, front + 1,
                  pos);
    pos += (unsigned)__popc(f[u]);
  }
}

// A listed cell's window: flags (bit n: window cell n, row major, known
// before the cell's front), origin relative to the cell, and whether an
// unknown window cell holds a non-finite value (the reference multiplies
// it by its zero flag, which makes the fit NaN).
struct LsqWindow {
  unsigned mask;
  int dy, dx;  // [-3, 1]
  bool nan_x, nan_y;
};
__device__ __forceinline__ unsigned lsq_pack(const LsqWindow& v, int m0, int m1) {
  return v.mask | (unsigned)(v.dy + 3) << 9 | (unsigned)(v.dx + 3) << 12 | (v.nan_x ? 1u : 0u) << 15 |
         (v.nan_y ? 1u : 0u) << 16 | (unsigned)m0 << 17 | (unsigned)m1 << 19;
}
__device__ __forceinline__ LsqWindow lsq_unpack(unsigned p, int& m0, int& m1) {
  m0 = (int)(p >> 17) & 3;
  m1 = (int)(p >> 19) & 1;
  return LsqWindow{p & 511u, (int)(p >> 9 & 7u) - 3, (int)(p >> 12 & 7u) - 3, (p >> 15 & 1u) != 0u,
                   (p >> 16 & 1u) != 0u};
}

// Window and factor of cell c = (j, i) of front `level` (a cell is known
// before it when its level is lower).
__device__ __forceinline__ LsqWindow lsq_window_of(const LsqWork& w, const double* __restrict__ ex,
                                                   const double* __restrict__ ey,
                                                   const double* __restrict__ g, int n0, int n1,
                                                   int j, int i, int level, LsqFactor& f) {
  short local_sum = 0, lx = 0, ly = 0;
#pragma unroll
  for (int jl = -1; jl <= 1; ++jl)
#pragma unroll
    for (int il = -1; il <= 1; ++il) {
      const int jj = j + jl, ii = i + il;
      const bool in = jj >= 0 && jj < n0 && ii >= 0 && ii < n1;
      const short k = (in && w.lev[(int64_t)jj * n1 + ii] < level) ? short(1) : short(0);
      local_sum += k;  // the cell itself is unknown
      lx += k * short(il + 1);
      ly += k * short(jl + 1);
    }
  LsqWindow v{0u, lsq_start_code(ly, local_sum), lsq_start_code(lx, local_sum), false, false};
  double m[9];
#pragma unroll
  for (int n = 0; n < 9; ++n) {
    const int jl = j + v.dy + n / 3, il = i + v.dx + n % 3;
    const bool in = (jl >= 0 && jl < n0 && il >= 0 && il < n1);
    const int64_t c = (int64_t)jl * n1 + il;
    const bool known = in && w.lev[c] < level;
    m[n] = known ? 1.0 : 0.0;
    if (known) {
      v.mask |= 1u << n;
    } else if (in) {
      v.nan_x = v.nan_x || !isfinite(ex[c]);
      v.nan_y = v.nan_y || !isfinite(ey[c]);
    }
  }
  f = lsq_window_factor(m, g, g, n0, n1, j + v.dy, i + v.dx);
  return v;
}

// Windows of listed cells idx, idx + stride, ..., and the factors of the
// first fcap (the solve pass factors the rest itself).
__device__ __forceinline__ void lsq_factor_body(const LsqWork& w, const double* __restrict__ ex,
                                                const double* __restrict__ ey,
                                                const double* __restrict__ g, int n0, int n1,
                                                int idx, int stride) {
  const int n = (int)w.head[0];
  const size_t cap = (size_t)w.fcap;
  for (int k = idx; k < n; k += stride) {
    const LsqEntry t = w.list[k];
    const int j = t.cell / n1, i = t.cell - j * n1;
    LsqFactor f;
    const LsqWindow v = lsq_window_of(w, ex, ey, g, n0, n1, j, i, t.level, f);
    w.win[k] = lsq_pack(v, f.m0, f.m1);
    if (k >= w.fcap) continue;
    w.fac[k] = f.c1;
    w.fac[cap + k] = f.c2;
    w.fac[2 * cap + k] = f.c3;
    w.fac[3 * cap + k] = f.u00;
    w.fac[4 * cap + k] = f.u01;
    w.fac[5 * cap + k] = f.u02;
    w.fac[6 * cap + k] = f.u11;
    w.fac[7 * cap + k] = f.u12;
    w.fac[8 * cap + k] = f.u22;
  }
}

// Value-dependent part of one component's fit of cell (j, i): right-hand
// side from the window's known cells (an unknown one adds +-0 to a sum that
// began at +0), back substitution, value in place.
__device__ __forceinline__ void lsq_fit_window(const LsqWindow& v, bool nan, const LsqFactor& f,
                                               double* e, const double* __restrict__ g, int n0,
                                               int n1, int j, int i) {
  const int c = j * n1 + i, o = c + v.dy * n1 + v.dx;
  double x[9], l1[3], l2[3];
#pragma unroll
  for (int n = 0; n < 9; ++n)
    x[n] = e[(v.mask >> n & 1u) ? o + (n / 3) * n1 + n % 3 : c];
#pragma unroll
  for (int n = 0; n < 3; ++n) {  // clamped: a window cell off the grid is unknown
    l1[n] = g[min(max(i + v.dx + n, 0), n1 - 1)];
    l2[n] = g[min(max(j + v.dy + n, 0), n0 - 1)];
  }
  const double px = g[i], py = g[j];
  double b0 = 0.0, b1 = 0.0, b2 = 0.0;
#pragma unroll
  for (int n = 0; n < 9; ++n) {
    const bool known = (v.mask >> n & 1u) != 0u;
    b0 = known ? b0 + x[n] : b0;
    b1 = known ? b1 + l1[n % 3] * x[n] : b1;
    b2 = known ? b2 + l2[n / 3] * x[n] : b2;
  }
  if (nan) b0 = b1 = b2 = __longlong_as_double(0x7ff8000000000000LL);
  e[c] = lsq_eval(f, b0, b1, b2, px, py);
}

// A listed cell whose factor was not kept (out of line: its registers would
// spill those of the common path).
__device__ __attribute__((noinline)) void lsq_fit_unfactored(const LsqWindow& v, bool nan,
                                                             double* e, const double* g, int n0,
                                                             int n1, int j, int i) {
  double m[9];
#pragma unroll
  for (int n = 0; n < 9; ++n) m[n] = (v.mask >> n & 1u) ? 1.0 : 0.0;
  const LsqFactor f = lsq_window_factor(m, g, g, n0, n1, j + v.dy, i + v.dx);
  lsq_fit_window(v, nan, f, e, g, n0, n1, j, i);
}

// A listed cell's window and factor as the factor pass left them (the
// factor of the last kept one when the cell's own was not).
struct LsqRecord {
  int cell;
  unsigned win;
  LsqFactor f;
};
__device__ __forceinline__ LsqRecord lsq_record(const LsqWork& w, int k) {
  const size_t cap = (size_t)w.fcap, q = (size_t)min(k, w.fcap - 1);
  LsqRecord r;
  r.cell = w.list[k].cell;
  r.win = w.win[k];
  r.f.c1 = w.fac[q];
  r.f.c2 = w.fac[cap + q];
  r.f.c3 = w.fac[2 * cap + q];
  r.f.u00 = w.fac[3 * cap + q];
  r.f.u01 = w.fac[4 * cap + q];
  r.f.u02 = w.fac[5 * cap + q];
  r.f.u11 = w.fac[6 * cap + q];
  r.f.u12 = w.fac[7 * cap + q];
  r.f.u22 = w.fac[8 * cap + q];
  return r;
}

// One component's fits of one case (e: its values; second: the second
// component), front by front, in place: a fit reads only cells known before
// its front (the value it loads for another window cell is its own cell's,
// and is not used) and writes its own cell.  A thread's first record of the
// next front is loaded before this front's barrier, so that the front after
// starts with its window's values.
// The first `done` fronts are those of lsq_front_solve_body.
__device__ __forceinline__ void lsq_solve_body(const LsqWork& w, double* e, bool second,
                                               const double* __restrict__ g, int n0, int n1,
                                               int done) {
  const int levels = (int)w.head[1], total = (int)w.head[0];
  const int tid = threadIdx.x, nth = blockDim.x;
  if (levels <= done) return;
  int begin = w.off[done], end = w.off[done + 1], next = levels > done + 1 ? w.off[done + 2] : end;
  LsqRecord r = lsq_record(w, min(begin + tid, total - 1));
  for (int level = done + 1; level <= levels; ++level) {
    const LsqRecord r1 = lsq_record(w, min(end + tid, total - 1));
    const int after = level + 2 <= levels ? w.off[level + 2] : next;
    for (int k = begin + tid; k < end; k += nth) {
      if (k != begin + tid) r = lsq_record(w, k);
      const int j = r.cell / n1, i = r.cell - j * n1;
      const LsqWindow v = lsq_unpack(r.win, r.f.m0, r.f.m1);
      const bool nan = second ? v.nan_y : v.nan_x;
      if (k < w.fcap)
        lsq_fit_window(v, nan, r.f, e, g, n0, n1, j, i);
      else
        lsq_fit_unfactored(v, nan, e, g, n0, n1, j, i);
    }
    __syncthreads();
    r = r1;
    begin = end;
    end = next;
    next = after;
  }
}

// One component's fits of front `front` (from 0) by many workgroups: cells
// idx, idx + stride, ... of it.
__device__ __forceinline__ void lsq_front_solve_body(const LsqWork& w, double* e, bool second,
                                                     const double* __restrict__ g, int n0, int n1,
                                                     int front, int idx, int stride) {
  if ((int)w.head[1] <= front) return;
  const int end = w.off[front + 1];
  for (int k = w.off[front] + idx; k < end; k += stride) {
    LsqRecord r = lsq_record(w, k);
    const int j = r.cell / n1, i = r.cell - j * n1;
    const LsqWindow v = lsq_unpack(r.win, r.f.m0, r.f.m1);
    const bool nan = second ? v.nan_y : v.nan_x;
    if (k < w.fcap)
      lsq_fit_window(v, nan, r.f, e, g, n0, n1, j, i);
    else
      lsq_fit_unfactored(v, nan, e, g, n0, n1, j, i);
  }
}

__global__ void __launch_bounds__(kLsqThreads) lsq_levels_kernel(LsqWork w, int nr, int nz,
                                                                 const int* __restrict__ zone,
                                                                 int done) {
  lsq_levels_body(w, nr, nz, zone, done);
}
__global__ void __launch_bounds__(256) lsq_front_levels_kernel(LsqWork w, int nr, int nz,
                                                               const int* __restrict__ zone,
                                                               int front) {
  lsq_front_levels_body(w, nr, nz, zone, front, blockIdx.x);
}
__global__ void __launch_bounds__(256) lsq_factor_kernel(LsqWork w, const double* __restrict__ ex,
                                                         const double* __restrict__ ey,
                                                         const double* __restrict__ g, int n0,
                                                         int n1) {
  lsq_factor_body(w, ex, ey, g, n0, n1, blockIdx.x * blockDim.x + threadIdx.x,
                  gridDim.x * blockDim.x);
}
// 512 threads: a front has a few hundred cells, and the barrier after it
// costs more with 1024 (256 x 128: 19 us a step, 23 with 1024; the widest
// fronts that are left to it, a solid of 205 cells' radius: 74, 71).
constexpr int kLsqSolveThreads = 512;
__global__ void __launch_bounds__(kLsqSolveThreads) lsq_solve_kernel(LsqWork w, double* ex,
                                                                     double* ey,
                                                                     const double* __restrict__ g,
                                                                     int n0, int n1, int done) {
  lsq_solve_body(w, blockIdx.x ? ey : ex, blockIdx.x != 0, g, n0, n1, done);
}
__global__ void __launch_bounds__(256) lsq_front_solve_kernel(LsqWork w, double* ex, double* ey,
                                                              const double* __restrict__ g, int n0,
                                                              int n1, int front) {
  lsq_front_solve_body(w, blockIdx.y ? ey : ex, blockIdx.y != 0, g, n0, n1, front,
                       blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// A band's cells, one per thread at a time (a 256-row case lists about
// 5,000).  The factor pass takes 238 registers, one wave per SIMD: a
// workgroup has its CU alone, and twelve cases' 768 run three to a CU in turn.
constexpr int kLsqFactorBlocks = 64;

// Workgroups of a front of lsq_front_levels_body over a doubled grid.
static int lsq_front_blocks(int nr, int nz) {
  return (int)ceil_div((int64_t)2 * nr * (lsq_words(nz) / 4), 256);
}

hipError_t launch_lsq_fronts(const LsqWork& w, double* e1d, double* e2d, const double* z, int nr,
                             int nz, const int* zone, bool large, hipStream_t s) {
  const int done = large ? kLsqFrontLaunches : 0;
  hipError_t e;
  for (int k = 0; k < done; ++k) {
    lsq_front_levels_kernel<<<lsq_front_blocks(nr, nz), 256, 0, s>>>(w, nr, nz, zone, k);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  lsq_levels_kernel<<<1, kLsqThreads, 0, s>>>(w, nr, nz, zone, done);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  lsq_factor_kernel<<<kLsqFactorBlocks, 256, 0, s>>>(w, e1d, e2d, z, 2 * nr, nz);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  for (int k = 0; k < done; ++k) {
    lsq_front_solve_kernel<<<dim3(kLsqFactorBlocks, 2), 256, 0, s>>>(w, e1d, e2d, z, 2 * nr, nz, k);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  lsq_solve_kernel<<<2, kLsqSolveThreads, 0, s>>>(w, e1d, e2d, z, 2 * nr, nz, done);
  return hipGetLastError();
}

// Soft batches: the same passes, one workgroup (levels, solve) or
// kLsqFactorBlocks workgroups (factor) per case.
template <typename B>
__global__ void __launch_bounds__(kLsqThreads) soft_batch_lsq_levels_kernel(
    const SoftCaseT<B>* __restrict__ cs, int done) {
  const SoftCaseT<B>& C = cs[blockIdx.x];
  lsq_levels_body(C.lw, C.nr, C.nz, C.zone, done);
}
template <typename B>
__global__ void __launch_bounds__(256) soft_batch_lsq_front_levels_kernel(
    const SoftCaseT<B>* __restrict__ cs, int front) {
  const SoftCaseT<B>& C = cs[blockIdx.y];
  lsq_front_levels_body(C.lw, C.nr, C.nz, C.zone, front, blockIdx.x);
}
template <typename B>
__global__ void __launch_bounds__(256) soft_batch_lsq_factor_kernel(
    const SoftCaseT<B>* __restrict__ cs) {
  const SoftCaseT<B>& C = cs[blockIdx.y];
  lsq_factor_body(C.lw, C.e1d, C.e2d, C.z, 2 * C.nr, C.nz, blockIdx.x * blockDim.x + threadIdx.x,
                  gridDim.x * blockDim.x);
}
template <typename B>
__global__ void __launch_bounds__(kLsqSolveThreads) soft_batch_lsq_solve_kernel(
    const SoftCaseT<B>* __restrict__ cs, int done) {
  const SoftCaseT<B>& C = cs[blockIdx.y];
  lsq_solve_body(C.lw, blockIdx.x ? C.e2d : C.e1d, blockIdx.x != 0, C.z, 2 * C.nr, C.nz, done);
}
template <typename B>
__global__ void __launch_bounds__(256) soft_batch_lsq_front_solve_kernel(
    const SoftCaseT<B>* __restrict__ cs, int front) {
  const SoftCaseT<B>& C = cs[blockIdx.z];
  lsq_front_solve_body(C.lw, blockIdx.y ? C.e2d : C.e1d, blockIdx.y != 0, C.z, 2 * C.nr, C.nz,
                       front, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

template <typename B>
hipError_t launch_soft_batch_lsq(const SoftCaseT<B>* cases, const SoftBatchDims& d,
                                 hipStream_t s) {
  const int done = d.large_solid ? kLsqFrontLaunches : 0;
  hipError_t e;
  for (int k = 0; k < done; ++k) {
    soft_batch_lsq_front_levels_kernel<B>
        <<<dim3(lsq_front_blocks(d.max_nr, d.max_nz), d.ncase), 256, 0, s>>>(cases, k);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  soft_batch_lsq_levels_kernel<B><<<d.ncase, kLsqThreads, 0, s>>>(cases, done);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  soft_batch_lsq_factor_kernel<B><<<dim3(kLsqFactorBlocks, d.ncase), 256, 0, s>>>(cases);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  for (int k = 0; k < done; ++k) {
    soft_batch_lsq_front_solve_kernel<B>
        <<<dim3(kLsqFactorBlocks, 2, d.ncase), 256, 0, s>>>(cases, k);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  soft_batch_lsq_solve_kernel<B><<<dim3(2, d.ncase), kLsqSolveThreads, 0, s>>>(cases, done);
  return hipGetLastError();
}

template hipError_t launch_soft_batch_lsq<double>(const SoftCaseT<double>*, const SoftBatchDims&,
                                                  hipStream_t);
template hipError_t launch_soft_batch_lsq<float>(const SoftCaseT<float>*, const SoftBatchDims&,
                                                 hipStream_t);

}  // namespace axs

using namespace axs;

extern "C" {

axs_status axs_extrapolate_lsq_first_order_f64(int16_t* current_flag, const int16_t* target_flag,
                                               double* eta_x, double* eta_y,
                                               const double* grid_x, const double* grid_y,
                                               int n0, int n1, int max_sweeps,
                                               int* sweeps_done_host, void* stream) {
  AXS_CHECK_ARG(current_flag && target_flag && eta_x && eta_y && grid_x && grid_y,
                "null pointer");
  AXS_CHECK_ARG(n0 >= 1 && n1 >= 1, "bad shape");
  AXS_CHECK_ARG(max_sweeps >= 1 && max_sweeps <= 1 << 20, "bad max_sweeps");
  hipStream_t s = as_stream(stream);
  const int64_t n = (int64_t)n0 * n1;
  // Sweeps are issued in batches; a sweep whose predecessor found nothing
  // exits at once, so the host only reads the counters once per batch.
  constexpr int kBatch = 8;
  LsqSweepWork w{};
  AXS_HIP(hipMalloc(reinterpret_cast<void**>(&w.nx), sizeof(double) * n));
  hipError_t e = hipMalloc(reinterpret_cast<void**>(&w.ny), sizeof(double) * n);
  if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(&w.pend), n);
  if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(&w.counters), sizeof(unsigned) * kBatch);
  int done = 0;
  bool finished = false;
  std::vector<unsigned> h(kBatch);
  while (e == hipSuccess && !finished && done < max_sweeps) {
    e = launch_fill_u32(w.counters, kBatch, 0u, s);
    const int nb = std::min(kBatch, max_sweeps - done);
    for (int q = 0; q < nb && e == hipSuccess; ++q)
      e = launch_lsq_sweep(current_flag, target_flag, eta_x, eta_y, grid_x, grid_y, n0, n1, w,
                           q, s);
    if (e == hipSuccess)
      e = hipMemcpyAsync(h.data(), w.counters, sizeof(unsigned) * kBatch, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    for (int q = 0; q < nb && e == hipSuccess; ++q) {
      if (h[q] == 0) {
        finished = true;
        break;
      }
      ++done;
    }
  }
  (void)hipFree(w.nx);
  (void)hipFree(w.ny);
  (void)hipFree(w.pend);
  (void)hipFree(w.counters);
  if (e != hipSuccess) {
    set_error(std::string("lsq extrapolation: ") + hipGetErrorString(e));
    return AXS_ERR_HIP;
  }
  if (sweeps_done_host) *sweeps_done_host = done;
  return AXS_OK;
}

}  // extern "C"
