// Row transforms for any nz: the DCT-II / DCT-III pair of the Neumann
// Stokes and potential plans, the real DFT pair of the periodic-z plans, and
// the DST-I of the implicit diffusion plan, each one row per workgroup with
// the row's DFT in LDS (axs_anydft.hpp: Stockham when the length factors
// into primes up to 13, Bluestein's chirp-z form otherwise).  The grids of the
// drivers (nz = 256 .. 4096, nz / 2 a power of two) keep the faster
// half-length transforms of axs_stokes.hip; these cover every other nz the
// reference's dense eig route accepts (kernels/FastDiagonalisationStokesSolver.py:41-128,
// kernels/implicit_diffusion_solver.py:74-106), up to the LDS bound.
//
// DCT-II of x[0..N) by one length-N DFT (J. Makhoul, "A fast cosine
// transform in one and two dimensions", IEEE Trans. ASSP 28(1), 1980):
//   v_n = x_{2n}, v_{N-1-n} = x_{2n+1},  V = DFT_N(v),
//   X_k = Re(e^{-i pi k / (2N)} V_k)      (X_k = sum_n x_n cos(pi k (2n+1) / (2N)))
// and its inverse V_k = e^{i pi k / (2N)} (X_k - i X_{N-k}) (X_N = 0),
// v = DFT_N^{-1}(V) / N, x unshuffled; valid for odd N too.  For even N the
// real sequence v is packed as z_m = v_{2m} + i v_{2m+1} and V comes from
// one length-N/2 DFT of z (the split of dct2_post_at / dct3_pre_at, as the
// half-length transforms of the smooth lengths do): half the DFT length,
// half the LDS.
// DST-I of x[0..N) (S_k = sum_j x_j sin(pi (j+1)(k+1) / (N+1))) through the
// odd extension y of length 2M, M = N + 1 (y_0 = y_M = 0, y_m = x_{m-1},
// y_{2M-m} = -x_{m-1}), packed as z_p = y_{2p} + i y_{2p+1}:
//   Z = DFT_M(z),  Y_k = (Z_k + conj Z_{M-k}) / 2 - i e^{-i pi k / M} (Z_k - conj Z_{M-k}) / 2,
//   S_{k-1} = -Im(Y_k) / 2.
#pragma clang fp contract(fast)

#include "axs_anydft.hpp"
#include "axs_fused.hpp"
#include "axs_softbatch.hpp"
#include "axs_stokes.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

namespace axs {

// ------------------------------------------------------------------ plan

// Radices of an M-point FFT: fours, a two, threes and fives; for M with a
// factor 7, 11 or 13 (primes = 13 allows them) the power of two in the fewest
// stages (two fours, not an eight and a two).
static bool radices_of(int M, int primes, FftPlanArgs* p) {
  p->M = M;
  p->nstages = 0;
  int m = M;
  const auto stages = [&](int r, int most) {
    for (int i = 0; i < most && m % r == 0 && p->nstages < kMaxFftStages; ++i) {
      p->radix[p->nstages++] = r;
      m /= r;
    }
  };
  if (primes > 5 && (M % 7 == 0 || M % 11 == 0 || M % 13 == 0)) {
    const int e2 = __builtin_ctz(M), rest = e2 % 3;
    stages(4, rest == 2 ? 1 : (rest == 1 && e2 > 1 ? 2 : 0));
    stages(8, kMaxFftStages);
  }
  for (int r : {4, 2, 3, 5, 7, 11, 13})
    if (r <= primes) stages(r, kMaxFftStages);
  return m == 1;
}

// The FFT twiddles are staged in LDS only while the doubled footprint still
// lets two workgroups share a CU (longer rows lose more to occupancy than the
// LDS twiddles save).
static int stages_twiddles(int L) { return 2 * sizeof(Cplx<double>) * (size_t)L <= 65536 ? 1 : 0; }

// Threads of a row of more than 1920 points when there are many: the PER that
// keeps the most threads in flight on a CU (rows by its 160 KiB of LDS and by
// the waves per SIMD that the registers of PER = 1, 2, 4 and of the wide
// radices allow; the inverse cosine rows at PER = 2 hold four, not six), the
// smallest where that is equal, but PER = 4 where it holds more rows than
// PER = 2.  Whole multiples of 256 threads: a row's
// waves spread evenly over the four SIMDs, where 5 or 6 waves leave room for
// one row less than their number says.  us per step of 1024 rows, sine rows
// of L points (a quarter, half, three quarters, all of 1024 threads): 2160
// (chirp-z) 134 / 134 / 134 / 138, 384 threads 137; 2560 (direct) - / 106 / 96 /
// 120, 320 threads 136; 2880 123 / 104 / 105 / 105; 3456 - / 140 / 168 / 153;
// cosine rows of 1250 points (chirp-z, 2500) 169 / 160 / 139 / 179, 384
// threads 192.
struct LongRow {
  int nth, rows;  // threads; rows in flight on a CU
};
static LongRow long_row(const AnyDftArgs& a, bool wide) {
  const size_t lds = sizeof(Cplx<double>) * (size_t)a.L * (a.stage ? 2 : 1);
  const int in_lds = (int)((size_t)160 * 1024 / lds);
  int nth = 0, rows = 0;
  for (int p : {1, 2, 4}) {
    const int t = (fft_threads(a, p, wide) + 255) / 256 * 256;
    if (t > 1024) continue;
    const int waves = wide || p == 4 ? 4 : p == 2 ? 6 : 7;  // per SIMD
    const int r = std::min(in_lds, waves / (t / 256));
    const int n = r == 1 ? 1024 : t;
    if (r * n > rows * nth || (p == 4 && r * n == rows * nth && r > rows)) {
      nth = n;
      rows = r;
    }
  }
  return {nth, rows};
}

// Whether chirp-z rows of l points, a length without a lone radix 2, are
// faster than rows of the L < l that is the shortest.  A stage costs about the
// same in any radix, so a length with fewer stages is, if its waves spread
// over the four SIMDs as well (us per implicit step of 1024 rows: 1125 points
// 71, 1080 79; 1875 108, 1800 121; but 1280 94, 1250 83, equal stages, and
// 1600 128, 1536 120, thirteen waves for twelve).  Of more than 1920 points
// the radix 2 also sets the butterflies per thread and the rows in flight:
// 2160 points 134, 2048 167; 3375 182, 3200 203; 5120 280, 5000 343; but 6912
// 485, 6750 444, equal in all three.
static bool better_length(int l, int L) {
  AnyDftArgs a, b;
  a.L = l;
  b.L = L;
  a.stage = stages_twiddles(l);
  b.stage = stages_twiddles(L);
  radices_of(l, 5, &a.fp);
  radices_of(L, 5, &b.fp);
  const bool fewer = a.fp.nstages < b.fp.nstages;
  if (L <= 1920) {
    const int wl = (l / 2 + 63) / 64, wL = (L / 2 + 63) / 64;
    return fewer && (wl == wL || wl % 4 == 0);
  }
  const LongRow A = long_row(a, false), B = long_row(b, false);
  return fewer || A.rows > B.rows || fft_per(a, A.nth, false) < fft_per(b, B.nth, false);
}

// The chirp-z length is the smallest smooth one, or one up to 1 / 16 longer
// without its lone radix 2 (that stage has the most butterflies and does the
// least) where that is faster: 4500 points instead of 4320 for N = 2049, 284 ->
// 202 us per implicit step at 2048 x 1024; 1125 instead of 1080 for 513, 33 ->
// 31 us at 512 x 256.  Factors 7, 11 and 13 are radices of
// their own where the chirp-z form would do too (rows of 770, 385 = 5 x 7 x 11
// points instead of two FFTs of 800: 68.6 -> 62.3 us per step of 770 x 386;
// 113 -> 72 us at 1001 x 500); the longest rows stay those it holds.  A
// batch's rows of many lengths run in one kernel, which the wide radices of
// one would slow for all, so they keep to primes = 5 and the smallest
// chirp-z length (twelve FP32 cases: 110 us of rows per step with the wide
// radices, 119 without, inside the noise of the 960 us step).
int any_dft_length(int N, bool* bluestein, int primes) {
  FftPlanArgs p;
  if (bluestein) *bluestein = false;
  if (radices_of(N, 5, &p)) return N;
  int L = 2 * N - 1;
  while (!radices_of(L, 5, &p)) ++L;
  if (L <= kAnyMaxL && radices_of(N, primes, &p)) return N;
  if (bluestein) *bluestein = true;
  if (primes == 5) return L;
  for (int l = L; l <= std::min(L + L / 16, kAnyMaxL); ++l)
    if (radices_of(l, 5, &p) && __builtin_ctz(l) % 2 == 0 && (l == L || better_length(l, L)))
      return l;
  return L;
}

template <typename V>
static hipError_t upload_table(V** dev, const std::vector<V>& host) {
  hipError_t e = hipMalloc(reinterpret_cast<void**>(dev), sizeof(V) * host.size());
  if (e != hipSuccess) return e;
  return hipMemcpy(*dev, host.data(), sizeof(V) * host.size(), hipMemcpyHostToDevice);
}

// bhat = FFT_L(b) / L in place, one workgroup
template <int PER>
__global__ void __launch_bounds__(1024) any_bhat_kernel(Cplx<double>* __restrict__ b,
                                                        AnyDftArgs a) {
  extern __shared__ unsigned char smem_raw[];
  Cplx<double>* work = reinterpret_cast<Cplx<double>*>(smem_raw);
  for (int k = threadIdx.x; k < a.L; k += blockDim.x) work[k] = b[k];
  any_dft_stage(work, a, threadIdx.x, blockDim.x);
  __syncthreads();
  any_fft<double, PER>(work, a, -1, threadIdx.x, blockDim.x);
  const double inv = 1.0 / (double)a.L;
  for (int k = threadIdx.x; k < a.L; k += blockDim.x)
    b[k] = Cplx<double>{work[k].x * inv, work[k].y * inv};
}

static void allow_large_lds();
// bytes of dynamic LDS every any-kernel may take (raised by allow_large_lds)
static int g_any_lds_limit = 65536;

hipError_t AnyDft::init(int N, int primes) {
  allow_large_lds();
  bool blue = false;
  const int L = any_dft_length(N, &blue, primes);
  if (L > kAnyMaxL || sizeof(Cplx<double>) * (size_t)L > (size_t)g_any_lds_limit)
    return hipErrorInvalidValue;
  args.N = N;
  args.L = L;
  args.bluestein = blue ? 1 : 0;
  args.stage = stages_twiddles(L);
  radices_of(L, primes, &args.fp);
  const bool wide = fft_wide(args);
  many.nth = std::max(64, (L / (wide ? 4 : 2) + 63) / 64 * 64);
  if (many.nth >= 1024) many.nth = long_row(args, wide).nth;
  if (!many.nth) return hipErrorInvalidValue;
  many.nth = std::max(many.nth, fft_threads(args, 4, wide));
  many.per = fft_per(args, many.nth, wide);
  few = many;
  if (L > 1920 && !wide) {
    // a row alone on its CU: the fewest butterflies per thread (160 rows:
    // sine rows of 3456 points 51 us with 512 threads by 4, 45 with 1024 by
    // 2; of 2880 points 41 and 38)
    for (int p : {4, 2, 1}) {
      const int t = (fft_threads(args, p, false) + 255) / 256 * 256;
      if (t <= 1024) few = Shape{p == 2 ? t : 1024, p};
    }
  }
  if (wide) many.per |= kFftWide;
  if (wide) few.per |= kFftWide;
  std::vector<Cplx<double>> tw(L);
  for (int t = 0; t < L; ++t) {
    const double ang = -2.0 * M_PI * (double)t / (double)L;
    tw[t] = {std::cos(ang), std::sin(ang)};
  }
  Cplx<double>* d_tw = nullptr;
  hipError_t e = upload_table(&d_tw, tw);
  if (e != hipSuccess) return e;
  owned.push_back(d_tw);
  args.tw = d_tw;
  if (!blue) return hipSuccess;
  // w_n = e^{-i pi (n^2 mod 2N) / N}
  std::vector<Cplx<double>> chirp(N), b(L, Cplx<double>{0.0, 0.0});
  const int64_t two_n = 2 * (int64_t)N;
  for (int n = 0; n < N; ++n) {
    const int64_t m = ((int64_t)n * n) % two_n;
    const double ang = -M_PI * (double)m / (double)N;
    chirp[n] = {std::cos(ang), std::sin(ang)};
  }
  b[0] = {chirp[0].x, -chirp[0].y};
  for (int m = 1; m < N; ++m) {
    b[m] = {chirp[m].x, -chirp[m].y};
    b[L - m] = b[m];
  }
  Cplx<double>*d_chirp = nullptr, *d_bhat = nullptr;
  if ((e = upload_table(&d_chirp, chirp)) != hipSuccess) return e;
  owned.push_back(d_chirp);
  if ((e = upload_table(&d_bhat, b)) != hipSuccess) return e;
  owned.push_back(d_bhat);
  const size_t shm = lds_bytes<double>();
  // chirp-z lengths hold radices up to 5 only
  if (many.per == 1)
    any_bhat_kernel<1><<<1, many.nth, shm, 0>>>(d_bhat, args);
  else if (many.per == 2)
    any_bhat_kernel<2><<<1, many.nth, shm, 0>>>(d_bhat, args);
  else
    any_bhat_kernel<4><<<1, many.nth, shm, 0>>>(d_bhat, args);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if ((e = hipDeviceSynchronize()) != hipSuccess) return e;
  args.chirp = d_chirp;
  args.bhat = d_bhat;
  return hipSuccess;
}

AnyDft::~AnyDft() {
  for (void* p : owned) (void)hipFree(p);
}

// ------------------------------------------------------------------ kernels

// Forward DCT-II of row i of one field (src, tapered, dst at the case):
// x = rscale_i * src row (with the kill taper of
// kill_boundary_vorticity_sine.py:4-27 applied on the fly when TAPER, as
// taper_dct2_row does; the tapered row also goes to `tapered` when not
// null), dst row = X.  Threads tid of nth, work of a.L entries in LDS; every
// thread of the block calls it (block barriers).
// The tables of one plan's DCT rows: a = the DFT (length nz, or nz / 2
// when half), ge2[k] = e^{-i pi k / (2 nz)} for k < nz (full form), e1[k] =
// e^{-2 pi i k / nz} and e2[k] = e^{-i pi k / (2 nz)} for k <= nz / 2 (half
// form).
struct AnyDctTables {
  AnyDftArgs a;
  const Cplx<double>* ge2;
  const Cplx<double>* e1;
  const Cplx<double>* e2;
  int half;
};

template <typename T, int PER, bool TAPER>
__device__ void any_dct2_row(const T* __restrict__ src, T* __restrict__ tapered,
                             T* __restrict__ dst, const double* __restrict__ rscale,
                             const double* __restrict__ wz, const double* __restrict__ wr, int nr,
                             int nz, int w, const AnyDctTables& tb, int i, Cplx<T>* work, int tid,
                             int nth) {
  const int srow = (TAPER && i >= nr - w) ? nr - w : i;
  const T* row = src + (int64_t)srow * nz;
  const T rs = rscale ? T(rscale[i]) : T(1);
  T left = T(0), right = T(0), rowf = T(1);
  if constexpr (TAPER) {
    left = row[w - 1];
    right = row[nz - w];
    rowf = (i == 0) ? T(0) : ((i >= nr - w) ? T(wr[i - (nr - w)]) : T(1));
  }
  T* out_t = (TAPER && tapered) ? tapered + (int64_t)i * nz : nullptr;
  any_dft_stage(work, tb.a, tid, nth);
  for (int j = tid; j < nz; j += nth) {
    T t = row[j];
    if constexpr (TAPER) {
      if (j < w)
        t = T(wz[j]) * left;
      else if (j >= nz - w)
        t = T(wz[w + (j - (nz - w))]) * right;
      if (i >= nr - w) t = rowf * t;
      if (i == 0) t = T(0);
      if (out_t) out_t[j] = t;
    }
    if (tb.half)
      packed_component(work, dct_dst_index(j, nz)) = rs * t;
    else
      work[dct_dst_index(j, nz)] = Cplx<T>{rs * t, T(0)};
  }
  __syncthreads();
  any_dft<T, PER>(work, tb.a, -1, tid, nth);
  T* out = dst + (int64_t)i * nz;
  if (tb.half) {
    const int M = nz / 2;
    for (int k = tid; k <= M / 2; k += nth)
      dct2_post_at<T>(work, M, k, tb.e1[k], tb.e1[M - k], tb.e2[k], tb.e2[M - k],
                      [&](int q, T val) { out[q] = val; });
    return;
  }
  for (int k = tid; k < nz; k += nth) {
    const Cplx<double> e = tb.ge2[k];
    const Cplx<T> v = work[k];
    out[k] = T(e.x) * v.x - T(e.y) * v.y;
  }
}

// Inverse (DCT-III scaled by 1 / N) of row i of one field.
template <typename T, int PER>
__device__ void any_dct3_row(const T* __restrict__ src, T* __restrict__ dst, int nz,
                             const AnyDctTables& tb, int i, Cplx<T>* work, int tid, int nth) {
  const T* row = src + (int64_t)i * nz;
  const T invN = T(1) / T(nz);
  T* out = dst + (int64_t)i * nz;
  any_dft_stage(work, tb.a, tid, nth);
  if (tb.half) {
    const int M = nz / 2;
    for (int k = tid; k < M; k += nth) {
      const int mk = M - k;  // in [1, M]
      const T xk = row[k], xnk = (k == 0) ? T(0) : row[nz - k];
      const T xm = row[mk], xnm = row[nz - mk];
      work[k] = dct3_pre_at<T>(xk, xnk, xm, xnm, tb.e2[k], tb.e2[mk], tb.e1[k]);
    }
    __syncthreads();
    any_dft<T, PER>(work, tb.a, +1, tid, nth);
    for (int j = tid; j < nz; j += nth)
      out[j] = packed_component(work, dct_dst_index(j, nz)) * invN;
    return;
  }
  const Cplx<double>* __restrict__ e2 = tb.ge2;
  for (int k = tid; k < nz; k += nth) {
    const T xk = row[k];
    const T xn = (k == 0) ? T(0) : row[nz - k];
    const Cplx<double> e = e2[k];
    work[k] = cmul(Cplx<T>{T(e.x), T(-e.y)}, Cplx<T>{xk, -xn});
  }
  __syncthreads();
  any_dft<T, PER>(work, tb.a, +1, tid, nth);
  for (int j = tid; j < nz; j += nth) out[j] = work[dct_dst_index(j, nz)].x * invN;
}

// Forward DCT-II rows; case blockIdx.y of a batch; workgroup nr completes the
// previous step when fin is given.
template <typename T, int PER, bool TAPER>
__global__ void __launch_bounds__(1024) any_dct2_rows_kernel(
    const T* __restrict__ src, T* __restrict__ tapered, T* __restrict__ dst,
    const double* __restrict__ rscale, const double* __restrict__ wz,
    const double* __restrict__ wr, int nr, int nz, int w, AnyDctTables tb, StepFinalize fin) {
  if (fin.partials && blockIdx.x == nr) {  // completes the previous step
    __shared__ double fin_red[1024];  // one entry per thread (finalize_pending)
    const int cb = blockIdx.y;
    const RigidConfig& cfg = fin.cfgs[cb];
    finalize_pending(fin.partials + (int64_t)cb * fin.count, fin.count,
                     fin.slots + (int64_t)cb * kSlotsPerCase, fin.sc + (int64_t)cb * AXS_RIGID_SCALARS,
                     fin.drag ? fin.drag + (int64_t)cb * cfg.history : nullptr, cfg, fin_red);
    return;
  }
  extern __shared__ unsigned char smem_raw[];
  const int64_t cs = (int64_t)blockIdx.y * nr * nz;
  any_dct2_row<T, PER, TAPER>(src + cs, (TAPER && tapered) ? tapered + cs : nullptr, dst + cs,
                              rscale, wz, wr, nr, nz, w, tb, blockIdx.x,
                              reinterpret_cast<Cplx<T>*>(smem_raw), threadIdx.x, blockDim.x);
}

template <typename T, int PER>
__global__ void __launch_bounds__(1024) any_dct3_rows_kernel(
    const T* __restrict__ src, T* __restrict__ dst, int nr, int nz, AnyDctTables tb) {
  extern __shared__ unsigned char smem_raw[];
  const int64_t cs = (int64_t)blockIdx.y * nr * nz;
  any_dct3_row<T, PER>(src + cs, dst + cs, nz, tb, blockIdx.x,
                       reinterpret_cast<Cplx<T>*>(smem_raw), threadIdx.x, blockDim.x);
}

// Soft batches: row blockIdx.x of case blockIdx.y (tapered omega -> w0,
// r omega -> spectrum; the spectrum -> psi), in the batch's storage type.
template <typename B, int PER>
__global__ void __launch_bounds__(1024) soft_batch_dct2_kernel(
    const SoftCaseT<B>* __restrict__ cs) {
  const SoftCaseT<B>& C = cs[blockIdx.y];
  if ((int)blockIdx.x >= C.nr) return;
  extern __shared__ unsigned char smem_raw[];
  const AnyDctTables tb{C.any, C.ge2, C.te1, C.te2, C.any_half};
  any_dct2_row<B, PER, true>(C.vorticity, C.w0, C.spec, C.rvec, C.kill_wz, C.kill_wr, C.nr,
                             C.nz, C.kill_width, tb, blockIdx.x,
                             reinterpret_cast<Cplx<B>*>(smem_raw), threadIdx.x, blockDim.x);
}

template <typename B, int PER>
__global__ void __launch_bounds__(1024) soft_batch_dct3_kernel(
    const SoftCaseT<B>* __restrict__ cs) {
  const SoftCaseT<B>& C = cs[blockIdx.y];
  if ((int)blockIdx.x >= C.nr) return;
  extern __shared__ unsigned char smem_raw[];
  const AnyDctTables tb{C.any, C.ge2, C.te1, C.te2, C.any_half};
  any_dct3_row<B, PER>(C.spec, C.psi, C.nz, tb, blockIdx.x, reinterpret_cast<Cplx<B>*>(smem_raw),
                       threadIdx.x, blockDim.x);
}

// Real DFT rows of any length into the packed real layout of the periodic
// plans: [X_0, Re X_1, Im X_1, ..., Re X_h, Im X_h (, X_{N/2} when N is
// even)], h = (N - 1) / 2; every entry one real unknown of its mode.
template <int PER>
__global__ void __launch_bounds__(1024) any_rfft_rows_kernel(
    const double* __restrict__ src, double* __restrict__ dst, const double* __restrict__ rscale,
    int nz, AnyDftArgs a) {
  extern __shared__ unsigned char smem_raw[];
  Cplx<double>* work = reinterpret_cast<Cplx<double>*>(smem_raw);
  const int i = blockIdx.x, tid = threadIdx.x, nth = blockDim.x;
  const double* row = src + (int64_t)i * nz;
  const double sc = rscale ? rscale[i] : 1.0;
  any_dft_stage(work, a, tid, nth);
  for (int j = tid; j < nz; j += nth) work[j] = Cplx<double>{sc * row[j], 0.0};
  __syncthreads();
  any_dft<double, PER>(work, a, -1, tid, nth);
  double* out = dst + (int64_t)i * nz;
  for (int p = tid; p < nz; p += nth) {
    double v;
    if (p == 0)
      v = work[0].x;
    else if (p == nz - 1 && nz % 2 == 0)
      v = work[nz / 2].x;
    else
      v = (p & 1) ? work[(p + 1) / 2].x : work[p / 2].y;
    out[p] = v;
  }
}

template <int PER>
__global__ void __launch_bounds__(1024) any_irfft_rows_kernel(const double* __restrict__ src,
                                                              double* __restrict__ dst, int nz,
                                                              AnyDftArgs a) {
  extern __shared__ unsigned char smem_raw[];
  Cplx<double>* work = reinterpret_cast<Cplx<double>*>(smem_raw);
  const int i = blockIdx.x, tid = threadIdx.x, nth = blockDim.x;
  const double* row = src + (int64_t)i * nz;
  any_dft_stage(work, a, tid, nth);
  for (int k = tid; k < nz; k += nth) {
    Cplx<double> v;
    if (k == 0) {
      v = {row[0], 0.0};
    } else if (2 * k == nz) {
      v = {row[nz - 1], 0.0};
    } else if (2 * k < nz) {
      v = {row[2 * k - 1], row[2 * k]};
    } else {  // conjugate of mode nz - k
      const int m = nz - k;
      v = {row[2 * m - 1], -row[2 * m]};
    }
    work[k] = v;
  }
  __syncthreads();
  any_dft<double, PER>(work, a, +1, tid, nth);
  const double invN = 1.0 / (double)nz;
  double* out = dst + (int64_t)i * nz;
  for (int j = tid; j < nz; j += nth) out[j] = work[j].x * invN;
}

// Real component m of the packed sequence z_p = y_{2p} + i y_{2p+1}.
__device__ __forceinline__ double& packed_y(Cplx<double>* z, int m) {
  return (m & 1) ? z[m >> 1].y : z[m >> 1].x;
}

// Orthonormal DST-I rows (sqrt(2 / (N + 1)) S), its own inverse; a has
// length M = nz + 1, em[k] = e^{-i pi k / M} for k <= nz.
template <int PER>
__device__ __forceinline__ void any_dst1_rows_body(
    const double* __restrict__ src, double* __restrict__ dst, int nz, AnyDftArgs a,
    const Cplx<double>* __restrict__ em, double norm) {
  extern __shared__ unsigned char smem_raw[];
  Cplx<double>* work = reinterpret_cast<Cplx<double>*>(smem_raw);
  const int i = blockIdx.x, tid = threadIdx.x, nth = blockDim.x;
  const int M = nz + 1;
  const double* row = src + (int64_t)i * nz;
  any_dft_stage(work, a, tid, nth);
  for (int j = tid; j < nz; j += nth) {
    const double x = row[j];
    packed_y(work, j + 1) = x;
    packed_y(work, 2 * M - 1 - j) = -x;
  }
  if (tid == 0) {
    packed_y(work, 0) = 0.0;
    packed_y(work, M) = 0.0;
  }
  __syncthreads();
  any_dft<double, PER>(work, a, -1, tid, nth);
  double* out = dst + (int64_t)i * nz;
  for (int k = tid + 1; k <= nz; k += nth) {
    const Cplx<double> zk = work[k], zc = cconj(work[M - k]);
    const Cplx<double> s = cadd(zk, zc), d = csub(zk, zc);
    const Cplx<double> ed = cmul(em[k], d);
    // -Im(Y_k) / 2 with Y_k = s / 2 - i ed / 2
    out[k - 1] = (ed.x - s.y) * norm;
  }
}
template <int PER>
__global__ void __launch_bounds__(1024) any_dst1_rows_kernel(
    const double* __restrict__ src, double* __restrict__ dst, int nz, AnyDftArgs a,
    const Cplx<double>* __restrict__ em, double norm) {
  any_dst1_rows_body<PER>(src, dst, nz, a, em, norm);
}
// At most 80 scalar registers: a SIMD has 800, and a wave takes them in
// steps of 16 with 16 more for the trap handler, so 81 leave seven waves
// instead of eight and a CU one row of 1024 threads instead of two (a step at
// 2000 x 1024: 37 us a row pass with 81, 29 with 80).
template <>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_num_sgpr(80)))
any_dst1_rows_kernel<1>(const double* __restrict__ src, double* __restrict__ dst, int nz,
                        AnyDftArgs a, const Cplx<double>* __restrict__ em, double norm) {
  any_dst1_rows_body<1>(src, dst, nz, a, em, norm);
}

// Every kernel above may take more than the default 64 KiB of dynamic LDS
// (a length-8192 FP64 row is 128 KiB of the CU's 160 KiB): each is allowed
// the device's opt-in maximum per workgroup less its own static LDS.  A
// refused request leaves the default limit (a launch above it then fails
// with a launch error); the error it records is cleared here so that the
// next launch check does not report it.
static void allow_large_lds() {
  static std::once_flag once;
  std::call_once(once, [] {
    int dev = 0, optin = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&optin, hipDeviceAttributeSharedMemPerBlockOptin, dev) !=
            hipSuccess ||
        optin <= 0) {
      (void)hipGetLastError();
      return;
    }
#define AXS_ANY_KERNELS(P)                                                                       \
  (const void*)any_dct2_rows_kernel<double, P, false>,                                           \
      (const void*)any_dct2_rows_kernel<double, P, true>,                                        \
      (const void*)any_dct2_rows_kernel<float, P, false>,                                        \
      (const void*)any_dct2_rows_kernel<float, P, true>,                                         \
      (const void*)any_dct3_rows_kernel<double, P>, (const void*)any_dct3_rows_kernel<float, P>, \
      (const void*)any_rfft_rows_kernel<P>, (const void*)any_irfft_rows_kernel<P>,               \
      (const void*)any_dst1_rows_kernel<P>
#define AXS_ANY_BATCH_KERNELS(P)                                                                  \
  (const void*)soft_batch_dct2_kernel<double, P>, (const void*)soft_batch_dct3_kernel<double, P>, \
      (const void*)soft_batch_dct2_kernel<float, P>, (const void*)soft_batch_dct3_kernel<float, P>
    const void* ks[] = {(const void*)any_bhat_kernel<1>,  (const void*)any_bhat_kernel<2>,
                        (const void*)any_bhat_kernel<4>,  AXS_ANY_KERNELS(1),
                        AXS_ANY_KERNELS(2),               AXS_ANY_KERNELS(4),
                        AXS_ANY_KERNELS(1 | kFftWide),    AXS_ANY_KERNELS(2 | kFftWide),
                        AXS_ANY_KERNELS(4 | kFftWide),    AXS_ANY_BATCH_KERNELS(1),
                        AXS_ANY_BATCH_KERNELS(2),         AXS_ANY_BATCH_KERNELS(4)};
#undef AXS_ANY_KERNELS
#undef AXS_ANY_BATCH_KERNELS
    int limit = optin;
    for (const void* k : ks) {
      hipFuncAttributes fa{};
      int allowed = 65536;
      if (hipFuncGetAttributes(&fa, k) == hipSuccess) {
        const int want = optin - (int)fa.sharedSizeBytes;
        if (want > 65536 &&
            hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, want) == hipSuccess)
          allowed = want;
      }
      (void)hipGetLastError();
      limit = std::min(limit, allowed);
    }
    g_any_lds_limit = limit;
  });
}

// ------------------------------------------------------------------ launchers

#define AXS_ANY_P(V, CALL) \
  case V: {                \
    constexpr int P = V;   \
    CALL;                  \
    break;                 \
  }
#define AXS_ANY_BATCH_PER(PERV, CALL) \
  do {                                \
    switch (PERV) {                   \
      AXS_ANY_P(1, CALL)              \
      AXS_ANY_P(2, CALL)              \
      AXS_ANY_P(4, CALL)              \
      default:                        \
        return hipErrorInvalidValue;  \
    }                                 \
  } while (0)
#define AXS_ANY_PER(PERV, CALL)      \
  do {                               \
    switch (PERV) {                  \
      AXS_ANY_P(1, CALL)             \
      AXS_ANY_P(2, CALL)             \
      AXS_ANY_P(4, CALL)             \
      AXS_ANY_P((1 | kFftWide), CALL) \
      AXS_ANY_P((2 | kFftWide), CALL) \
      AXS_ANY_P((4 | kFftWide), CALL) \
      default:                       \
        return hipErrorInvalidValue; \
    }                                \
  } while (0)

template <typename T>
hipError_t launch_any_dct2_rows(const StokesPlan& pl, const T* src, T* tapered, T* dst,
                                const double* rscale, const double* wz, const double* wr, int w,
                                bool taper, int batch, const StepFinalize* fin, hipStream_t s) {
  const AnyDft& D = *pl.any;
  const AnyDctTables tb{D.args, pl.ge2, pl.e1, pl.e2, pl.any_half ? 1 : 0};
  const StepFinalize f = fin ? *fin : StepFinalize{};
  const dim3 grid(pl.nr + (f.partials ? 1 : 0), batch);
  const size_t shm = D.lds_bytes<T>();
  const AnyDft::Shape h = D.shape(pl.nr);
  if (taper)
    AXS_ANY_PER(h.per, (any_dct2_rows_kernel<T, P, true><<<grid, h.nth, shm, s>>>(
                       src, tapered, dst, rscale, wz, wr, pl.nr, pl.nz, w, tb, f)));
  else
    AXS_ANY_PER(h.per, (any_dct2_rows_kernel<T, P, false><<<grid, h.nth, shm, s>>>(
                       src, nullptr, dst, rscale, nullptr, nullptr, pl.nr, pl.nz, 0, tb, f)));
  return hipGetLastError();
}

template <typename T>
hipError_t launch_any_dct3_rows(const StokesPlan& pl, const T* src, T* dst, int rows, int batch,
                                hipStream_t s) {
  const AnyDft& D = *pl.any;
  const AnyDctTables tb{D.args, pl.ge2, pl.e1, pl.e2, pl.any_half ? 1 : 0};
  const AnyDft::Shape h = D.shape(rows);
  AXS_ANY_PER(h.per, (any_dct3_rows_kernel<T, P><<<dim3(rows, batch), h.nth, D.lds_bytes<T>(), s>>>(
                     src, dst, rows, pl.nz, tb)));
  return hipGetLastError();
}

hipError_t launch_any_rfft_rows(const StokesPlan& pl, const double* src, double* dst,
                                const double* rscale, int rows, bool inverse, hipStream_t s) {
  const AnyDft& D = *pl.any;
  const size_t shm = D.lds_bytes<double>();
  const AnyDft::Shape h = D.shape(rows);
  if (inverse)
    AXS_ANY_PER(h.per, (any_irfft_rows_kernel<P><<<rows, h.nth, shm, s>>>(src, dst, pl.nz, D.args)));
  else
    AXS_ANY_PER(h.per, (any_rfft_rows_kernel<P><<<rows, h.nth, shm, s>>>(src, dst, rscale, pl.nz,
                                                                      D.args)));
  return hipGetLastError();
}

hipError_t launch_any_dst1_rows(const AnyDft& D, const Cplx<double>* em, const double* src,
                                double* dst, int rows, int batch, int nz, hipStream_t s) {
  const double norm = std::sqrt(2.0 / (double)(nz + 1)) / 4.0;
  const AnyDft::Shape h = D.shape(rows);
  AXS_ANY_PER(h.per, (any_dst1_rows_kernel<P><<<rows * batch, h.nth, D.lds_bytes<double>(), s>>>(
                     src, dst, nz, D.args, em, norm)));
  return hipGetLastError();
}

template <typename B>
hipError_t launch_soft_batch_dct2(const SoftCaseT<B>* cases, const SoftBatchDims& d,
                                  hipStream_t s) {
  const dim3 grid(d.max_nr, d.ncase);
  AXS_ANY_BATCH_PER(
      d.any_per, (soft_batch_dct2_kernel<B, P><<<grid, d.any_nth, d.any_lds, s>>>(cases)));
  return hipGetLastError();
}

template <typename B>
hipError_t launch_soft_batch_dct3(const SoftCaseT<B>* cases, const SoftBatchDims& d,
                                  hipStream_t s) {
  const dim3 grid(d.max_nr, d.ncase);
  AXS_ANY_BATCH_PER(
      d.any_per, (soft_batch_dct3_kernel<B, P><<<grid, d.any_nth, d.any_lds, s>>>(cases)));
  return hipGetLastError();
}

template hipError_t launch_soft_batch_dct2<double>(const SoftCaseT<double>*, const SoftBatchDims&,
                                                   hipStream_t);
template hipError_t launch_soft_batch_dct2<float>(const SoftCaseT<float>*, const SoftBatchDims&,
                                                  hipStream_t);
template hipError_t launch_soft_batch_dct3<double>(const SoftCaseT<double>*, const SoftBatchDims&,
                                                   hipStream_t);
template hipError_t launch_soft_batch_dct3<float>(const SoftCaseT<float>*, const SoftBatchDims&,
                                                  hipStream_t);

#undef AXS_ANY_PER
#undef AXS_ANY_BATCH_PER
#undef AXS_ANY_P

template hipError_t launch_any_dct2_rows<double>(const StokesPlan&, const double*, double*,
                                                 double*, const double*, const double*,
                                                 const double*, int, bool, int,
                                                 const StepFinalize*, hipStream_t);
template hipError_t launch_any_dct2_rows<float>(const StokesPlan&, const float*, float*, float*,
                                                const double*, const double*, const double*, int,
                                                bool, int, const StepFinalize*, hipStream_t);
template hipError_t launch_any_dct3_rows<double>(const StokesPlan&, const double*, double*, int,
                                                 int, hipStream_t);
template hipError_t launch_any_dct3_rows<float>(const StokesPlan&, const float*, float*, int,
                                                int, hipStream_t);

}  // namespace axs
