// mpsa_factor.hip -- batched thin SVD of many small charge-sector matrices on
// gfx950, one workgroup per sector: the SVD behind prepareSite / prepareBlock
// (src/MPSfunctions.hpp:21-140, BoostSVD + FixPhase blas/lapack_routines.cpp:
// 614-634) for MPS canonicalisation and truncation, where a site tensor splits
// into hundreds of sectors of tens of rows each.
//
// Method: X = M (m >= n) or X = M^H (m < n), p x r with p >= r, is reduced
// by Householder QR, X = Q R, and one-sided Jacobi (Hestenes) runs on the
// columns of A = R^H (r x r; the Drmac-Veselic preconditioning without
// pivoting).  Column pairs are visited in the round-robin order of a
// tournament (r/2 disjoint pairs per round, r - 1 rounds per sweep), one wave
// per pair, so a wave needs no barrier inside a rotation; the workgroup
// synchronises between rounds.  A pair is rotated when
// |a_i^H a_j| > tol sqrt(|a_i|^2 |a_j|^2) with tol = sqrt(r) eps; sweeps stop
// when a whole sweep rotates nothing.  The 2 x 2 Hermitian Jacobi rotation
// with gamma = |gamma| e^{i phi}, zeta = (b - a) / (2 |gamma|),
// t = sign(zeta) / (|zeta| + sqrt(1 + zeta^2)), c = 1 / sqrt(1 + t^2), s = c t:
//   a_i' = c a_i - s e^{-i phi} a_j,   a_j' = s e^{i phi} a_i + c a_j
// makes the pair orthogonal; Wm accumulates the same rotations.  Then
// sigma_j = |a_j|, sorted descending (ties by column index), Z = A / sigma,
// and X = (Q Wm) Sigma Z^H:
//   m >= n: U = Q Wm, V^dagger = Z^H;   m < n: U = Z, V^dagger = (Q Wm)^H.
// Singular vectors of exactly zero singular values (on the Z side; Q Wm is
// orthonormal by construction) are completed to an orthonormal basis
// (Gram-Schmidt of unit vectors, twice), as a LAPACK thin SVD returns them.
// A sector whose matrix holds a value that is not finite, or that still rotates
// after max_sweeps sweeps, has NaN in every output.
// Real data: FixPhase makes the first largest-|.| entry of every row of
// V^dagger positive (the column of U flips with it).
//
// Complex data is planar (real parts, then imaginary parts at a plane offset),
// like every complex buffer of the library.
#include <hip/hip_runtime.h>

#include <cfloat>

#include "mpsa_internal.h"

namespace mpsa {

namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;

// Sum over the 64 lanes of a wave (all active), in every lane: moves inside
// the vector unit (rows of 16 lanes, then across rows) instead of six trips
// through the LDS crossbar, which a Jacobi rotation or reflection waits for
// one after another.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, ROWS, 0xf, false);
  return x + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum(double x) {
  x = dpp_add<0x111, 0xf>(x);  // row_shr 1, 2, 4, 8: lane 15 of a row holds its sum
  x = dpp_add<0x112, 0xf>(x);
  x = dpp_add<0x114, 0xf>(x);
  x = dpp_add<0x118, 0xf>(x);
  x = dpp_add<0x142, 0xa>(x);  // row_bcast 15: rows 0 and 2 into rows 1 and 3
  x = dpp_add<0x143, 0xc>(x);  // row_bcast 31: row 1 into rows 2 and 3
  const int lo = __builtin_amdgcn_readlane(__double2loint(x), 63);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(x), 63);
  return __hiloint2double(hi, lo);
}

// High word of |x|: ordered as the values are, kNotFinite and above for Inf
// and NaN.  The loads of a sector collect its maximum, since NaN fails every
// comparison that the reflections and rotations make and would be left out.
constexpr int kNotFinite = 0x7ff00000;
__device__ __forceinline__ int magnitude(double x) { return __double2hiint(x) & 0x7fffffff; }
// Maximum of x over the workgroup, in every thread; red: one int per wave
// (LDS).  All LDS written before is visible after.
template <int NT>
__device__ __forceinline__ int group_max(int x, int* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = max(x, __shfl_xor(x, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) x = max(x, red[w]);
  return x;
}
// What a sector's values are multiplied by at the outputs (its loads by 1 /
// scale).  A power of two near its largest entry where that lies outside
// 2^-300 .. 2^300, so that the squares of its entries stay in the range of
// doubles; else 1.  NaN where its matrix holds a value that is not finite (or
// the sweeps reach their limit), so that no caller takes the factors for a
// result.
__device__ __forceinline__ double sector_scale(int mx) {
  if (mx >= kNotFinite) return __longlong_as_double(0x7ff8000000000000ll);
  const int e = mx >> 20;  // exponent + 1023
  return e > 723 && e < 1323 ? 1.0 : __hiloint2double(min(max(e, 1), 2045) << 20, 0);
}
// Columns of squared norm below this count as zero: with the largest entry at
// 2^-300 or above they are less than 2^-140 of it, and their reciprocal
// squares and products would leave the range of doubles.
constexpr double kTinySq = 0x1p-880;
// A column's head of |x|^2 below this has phase 1 in its reflection: its
// square has lost bits, and it is less than 2^-60 of a column that is not zero.
constexpr double kPhaseSq = 0x1p-1000;
// |x| and the unit phase of a column's head, for its reflection
template <bool C>
__device__ __forceinline__ double head_phase(double xr, double xi, double& er, double& ei) {
  const double s = xr * xr + xi * xi;
  const double a = C ? sqrt(s) : fabs(xr);
  const bool ok = C ? s >= kPhaseSq : a > 0.0;
  er = ok ? xr / a : 1.0;
  ei = C && ok ? xi / a : 0.0;
  return a;
}

// Column j of a p-row matrix with leading dimension ld, planar complex.
template <bool C>
struct Mat {
  double* re;
  double* im;  // unused when !C
  int64_t ld;
  __device__ __forceinline__ double& r(int i, int j) const { return re[i + (int64_t)j * ld]; }
  __device__ __forceinline__ double& m(int i, int j) const { return im[i + (int64_t)j * ld]; }
};

// Rotate columns (i, j) of a p-row matrix by the Jacobi rotation (c, s, phase
// er + i ei): x_i' = c x_i - s conj(e) x_j, x_j' = s e x_i + c x_j.
template <bool C>
__device__ __forceinline__ void rotate_cols(const Mat<C>& X, int p, int i, int j, double c, double s, double er,
                                            double ei, int lane) {
  for (int row = lane; row < p; row += 64) {
    const double xir = X.r(row, i), xjr = X.r(row, j);
    if (C) {
      const double xii = X.m(row, i), xji = X.m(row, j);
      // conj(e) x_j = (er - i ei)(xjr + i xji) = (er xjr + ei xji) + i (er xji - ei xjr)
      const double cjr = er * xjr + ei * xji, cji = er * xji - ei * xjr;
      // e x_i = (er + i ei)(xir + i xii) = (er xir - ei xii) + i (er xii + ei xir)
      const double eir = er * xir - ei * xii, eii = er * xii + ei * xir;
      X.r(row, i) = c * xir - s * cjr;
      X.m(row, i) = c * xii - s * cji;
      X.r(row, j) = s * eir + c * xjr;
      X.m(row, j) = s * eii + c * xji;
    } else {
      X.r(row, i) = c * xir - s * er * xjr;
      X.r(row, j) = s * er * xir + c * xjr;
    }
  }
}

// The Jacobi rotation (c, sn, phase er + i ei) that makes columns of squared
// norms a and b and inner product gr + i gi orthogonal, in every lane; false
// when |g| <= tol sqrt(a b) (nothing to rotate).  t = h / (|d| + sqrt(d^2 + h^2))
// with d = b - a, h = 2 |g| is the smaller root of the rotation's quadratic; two
// square roots and one division, where the quotient form takes three of each
// in a chain that a whole round waits for.  Columns whose products could leave
// the range of doubles take that form; those below kTinySq are not rotated.
template <bool C>
__device__ __forceinline__ bool jacobi_rotation(double a, double b, double gr, double gi, double tol, double& c,
                                                double& sn, double& er, double& ei) {
  if (!(a >= kTinySq && b >= kTinySq)) return false;
  if (a > 1e-120 && b > 1e-120 && a < 1e120 && b < 1e120) {
    const double g2 = gr * gr + (C ? gi * gi : 0.0);
    if (!(g2 > tol * tol * (a * b))) return false;
    double g;
    if (C) {
      const double ig = rsqrt(g2);
      er = gr * ig;
      ei = gi * ig;
      g = g2 * ig;
    } else {
      er = gr < 0.0 ? -1.0 : 1.0;
      ei = 0.0;
      g = fabs(gr);
    }
    const double d = b - a, h = 2.0 * g;
    const double t = (d >= 0.0 ? h : -h) / (fabs(d) + sqrt(d * d + h * h));
    c = rsqrt(1.0 + t * t);
    sn = c * t;
    return true;
  }
  const double g = C ? hypot(gr, gi) : fabs(gr);
  if (!(g > tol * (sqrt(a) * sqrt(b)))) return false;
  er = gr / g;
  ei = C ? gi / g : 0.0;
  const double zeta = (b - a) / (2.0 * g);
  const double t = fabs(zeta) > 1e100 ? 0.5 / zeta  // zeta^2 may overflow
                                      : (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
  c = 1.0 / sqrt(1.0 + t * t);
  sn = c * t;
  return true;
}

// Rows per lane of the register-held column paths: a column of up to
// 64 * kRpl rows lives in registers of one wave while it is reduced and
// updated (one global read and one write instead of two reads and a write),
// and a reflection vector of up to kRpl * 64 rows sits in LDS.
constexpr int kRpl = 16;
constexpr int kVecRows = 64 * kRpl;
static_assert(kSvdMaxR <= kVecRows, "a Jacobi column of r <= kSvdMaxR rows fits the register path");

// y <- y - f v for one column y (rows from..p-1) held by one wave, with
// f = beta (v^H y) and v at vl (LDS, planar at + kVecRows, v[0] at row from).
template <bool C>
__device__ __forceinline__ void reflect_col_regs(const Mat<C>& Y, int c, int from, int p, const double* vl,
                                                 double b, int lane) {
  double yr[kRpl], yi[kRpl];
  double wr_ = 0.0, wi_ = 0.0;
#pragma unroll
  for (int q = 0; q < kRpl; ++q) {
    const int i = from + lane + 64 * q;
    yr[q] = yi[q] = 0.0;
    if (i < p) {
      yr[q] = Y.r(i, c);
      if (C) yi[q] = Y.m(i, c);
      const double v_r = vl[i - from];
      wr_ += v_r * yr[q];
      if (C) {
        const double v_i = vl[kVecRows + i - from];
        wr_ += v_i * yi[q];
        wi_ += v_r * yi[q] - v_i * yr[q];  // conj(v) y
      }
    }
  }
  wr_ = wave_sum(wr_);
  if (C) wi_ = wave_sum(wi_);
  const double fr = b * wr_, fi = b * wi_;
#pragma unroll
  for (int q = 0; q < kRpl; ++q) {
    const int i = from + lane + 64 * q;
    if (i < p) {
      const double v_r = vl[i - from];
      const double v_i = C ? vl[kVecRows + i - from] : 0.0;
      Y.r(i, c) = yr[q] - (fr * v_r - fi * v_i);
      if (C) Y.m(i, c) = yi[q] - (fr * v_i + fi * v_r);
    }
  }
}

// The same update with v read from its global column (any p).
template <bool C>
__device__ __forceinline__ void reflect_col_global(const Mat<C>& Y, int c, int from, int p, const Mat<C>& Hv, int j,
                                                   double b, int lane) {
  double wr_ = 0.0, wi_ = 0.0;
  for (int i = from + lane; i < p; i += 64) {
    const double v_r = Hv.r(i, j), y_r = Y.r(i, c);
    wr_ += v_r * y_r;
    if (C) {
      const double v_i = Hv.m(i, j), y_i = Y.m(i, c);
      wr_ += v_i * y_i;
      wi_ += v_r * y_i - v_i * y_r;
    }
  }
  wr_ = wave_sum(wr_);
  if (C) wi_ = wave_sum(wi_);
  const double fr = b * wr_, fi = b * wi_;
  for (int i = from + lane; i < p; i += 64) {
    const double v_r = Hv.r(i, j);
    const double v_i = C ? Hv.m(i, j) : 0.0;
    Y.r(i, c) -= fr * v_r - fi * v_i;
    if (C) Y.m(i, c) -= fr * v_i + fi * v_r;
  }
}

// Householder reflections of X (p x r, planar, ld p) in place, one per
// column j < k = min(p, r): H_j = I - beta_j v_j v_j^H with v_j = x - alpha e_j,
// alpha = -e^{i arg x_j} |x| (x = rows j.. of column j), beta_j = 2 / |v_j|^2
// (0 for a zero column, below kTinySq: H_j = I, alpha = 0).  Column j becomes (alpha, 0, ...), the
// columns after it are reflected (one wave per column, the column in
// registers and v_j in LDS when p - j <= kVecRows); v_j goes to rows j.. of
// column j of Hv, beta_j to beta[j].  NT threads; red holds NT / 64 doubles,
// hv 3, vl 2 kVecRows (LDS).
template <bool C, int NT>
__device__ void house_reflect(const Mat<C>& X, const Mat<C>& Hv, double* beta, int p, int r, double* red,
                              double* hv, double* vl) {
  const int k = p < r ? p : r;
  constexpr int NW = NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int j = 0; j < k; ++j) {
    double a = 0.0;
    for (int i = j + tid; i < p; i += NT) {
      const double x = X.r(i, j);
      a += x * x;
      if (C) {
        const double y = X.m(i, j);
        a += y * y;
      }
    }
    a = wave_sum(a);
    if (lane == 0) red[wave] = a;
    __syncthreads();
    if (tid == 0) {
      double nn = 0.0;
      for (int w = 0; w < NW; ++w) nn += red[w];
      const double x0r = X.r(j, j), x0i = C ? X.m(j, j) : 0.0;
      const double nrm = sqrt(nn);
      double ar = 0.0, ai = 0.0, b = 0.0;
      if (nn >= kTinySq) {
        double er, ei;
        const double a0 = head_phase<C>(x0r, x0i, er, ei);
        ar = -er * nrm;
        ai = -ei * nrm;
        const double v0r = x0r - ar, v0i = x0i - ai;
        const double vn = nn - a0 * a0 + v0r * v0r + v0i * v0i;
        b = vn > 0.0 ? 2.0 / vn : 0.0;
      }
      hv[0] = ar;
      hv[1] = ai;
      hv[2] = b;
      beta[j] = b;
    }
    __syncthreads();
    const double ar = hv[0], ai = hv[1], b = hv[2];
    const bool in_lds = p - j <= kVecRows;
    for (int i = j + tid; i < p; i += NT) {
      double v_r = X.r(i, j), v_i = C ? X.m(i, j) : 0.0;
      if (i == j) {
        v_r -= ar;
        v_i -= ai;
      }
      Hv.r(i, j) = v_r;
      if (C) Hv.m(i, j) = v_i;
      if (in_lds) {
        vl[i - j] = v_r;
        if (C) vl[kVecRows + i - j] = v_i;
      }
    }
    __syncthreads();
    for (int c = j + 1 + wave; c < r; c += NW) {
      if (in_lds) reflect_col_regs<C>(X, c, j, p, vl, b, lane);
      else reflect_col_global<C>(X, c, j, p, Hv, j, b, lane);
    }
    for (int i = j + tid; i < p; i += NT) {
      X.r(i, j) = i == j ? ar : 0.0;
      if (C) X.m(i, j) = i == j ? ai : 0.0;
    }
    __syncthreads();
  }
}

// Y <- H_0 H_1 ... H_{k-1} Y for the ncols columns of Y (p rows), applying
// H_j for j = k-1 .. 0; with from_j only columns >= j (Y = [I; 0] there, as
// LAPACK's xORGQR forms Q).  vl: 2 kVecRows doubles of LDS.
template <bool C, int NT>
__device__ void house_apply(const Mat<C>& Y, int ncols, bool from_j, const Mat<C>& Hv, const double* beta, int p,
                            int k, double* vl) {
  constexpr int NW = NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int j = k - 1; j >= 0; --j) {
    const double b = beta[j];
    if (b == 0.0) continue;  // uniform across the workgroup
    const bool in_lds = p - j <= kVecRows;
    if (in_lds) {
      for (int i = j + tid; i < p; i += NT) {
        vl[i - j] = Hv.r(i, j);
        if (C) vl[kVecRows + i - j] = Hv.m(i, j);
      }
      __syncthreads();
    }
    for (int c = (from_j ? j : 0) + wave; c < ncols; c += NW) {
      if (in_lds) reflect_col_regs<C>(Y, c, j, p, vl, b, lane);
      else reflect_col_global<C>(Y, c, j, p, Hv, j, b, lane);
    }
    __syncthreads();
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Householder QR of a small sector (p <= kSmallRows rows) held in LDS.  The
// factorisation is a serial chain of short reflections, each of which the
// general path above takes through memory with four barriers; here a
// reflection costs one barrier and no memory: X stays in LDS with v_j in place
// in column j (its head in v0, R's diagonal in alpha), every thread computes
// the reflection's scalars itself, and the wave that updates column j + 1
// leaves its norm for the next reflection.  Q's columns are then formed in
// registers, one wave per column, without any barrier.  A 60 x 20 complex
// sector and its like: 47 us by the general path, 28 us here (mean launch of
// three Chebyshev moments, Hubbard L = 20, D = 192, 4 vectors; with the sectors
// of 32 to 64 columns in the same launches, 45 us).
// ---------------------------------------------------------------------------
constexpr int kSmallRpl = 8;
constexpr int kSmallRows = 64 * kSmallRpl;
constexpr int kSmallCols = 64;

template <bool C>
struct SmallQr {
  double *xr, *xi;          // X, column-major, ld p (LDS)
  double (*s)[kSmallCols];  // rows: beta, alpha re / im, v0 re / im, norms (LDS)
  int p, r, k;
  __device__ __forceinline__ double& re(int i, int j) const { return xr[i + j * p]; }
  __device__ __forceinline__ double& im(int i, int j) const { return xi[i + j * p]; }
  // X = Q R in place, X complete behind a barrier; ends with one
  template <int NT>
  __device__ __forceinline__ void factor() const {
    constexpr int NW = NT / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (wave == 0) {
      double a = 0.0;
      for (int i = lane; i < p; i += 64) {
        a += re(i, 0) * re(i, 0);
        if (C) a += im(i, 0) * im(i, 0);
      }
      a = wave_sum(a);
      if (lane == 0) s[5][0] = a;
    }
    __syncthreads();
    for (int j = 0; j < k; ++j) {
      const double nn = s[5][j & 1];
      const double x0r = re(j, j), x0i = C ? im(j, j) : 0.0;
      const double nrm = sqrt(nn);
      double ar = 0.0, ai = 0.0, b = 0.0;
      if (nn >= kTinySq) {
        double er, ei;
        const double a0 = head_phase<C>(x0r, x0i, er, ei);
        ar = -er * nrm;
        ai = -ei * nrm;
        const double v0r = x0r - ar, v0i = x0i - ai;
        const double vn = nn - a0 * a0 + v0r * v0r + v0i * v0i;
        b = vn > 0.0 ? 2.0 / vn : 0.0;
      }
      const double hr = x0r - ar, hi = x0i - ai;
      if (threadIdx.x == 0) {
        s[0][j] = b;
        s[1][j] = ar;
        s[2][j] = ai;
        s[3][j] = hr;
        s[4][j] = hi;
      }
      for (int c = j + 1 + wave; c < r; c += NW) {
        double yr[kSmallRpl], yi[kSmallRpl], vr[kSmallRpl], vi[kSmallRpl];
        double wr = 0.0, wi = 0.0;
#pragma unroll
        for (int q = 0; q < kSmallRpl; ++q) {
          yr[q] = yi[q] = vr[q] = vi[q] = 0.0;
          if (j + 64 * q >= p) continue;  // uniform
          const int i = j + lane + 64 * q;
          if (i < p) {
            yr[q] = re(i, c);
            vr[q] = q == 0 && lane == 0 ? hr : re(i, j);
            if (C) {
              yi[q] = im(i, c);
              vi[q] = q == 0 && lane == 0 ? hi : im(i, j);
            }
          }
          wr += vr[q] * yr[q];
          if (C) {
            wr += vi[q] * yi[q];
            wi += vr[q] * yi[q] - vi[q] * yr[q];  // conj(v) y
          }
        }
        wr = b * wave_sum(wr);
        if (C) wi = b * wave_sum(wi);
        double a = 0.0;
#pragma unroll
        for (int q = 0; q < kSmallRpl; ++q) {
          if (j + 64 * q >= p) continue;
          const int i = j + lane + 64 * q;
          if (i < p) {
            yr[q] -= wr * vr[q] - wi * vi[q];
            re(i, c) = yr[q];
            if (C) {
              yi[q] -= wr * vi[q] + wi * vr[q];
              im(i, c) = yi[q];
            }
            if (i > j) a += yr[q] * yr[q] + (C ? yi[q] * yi[q] : 0.0);
          }
        }
        if (c == j + 1) {
          a = wave_sum(a);
          if (lane == 0) s[5][(j + 1) & 1] = a;
        }
      }
      __syncthreads();
    }
  }
  // R(i, c) of the factored X
  __device__ __forceinline__ double r_re(int i, int c) const { return i < c ? re(i, c) : (i == c ? s[1][i] : 0.0); }
  __device__ __forceinline__ double r_im(int i, int c) const { return i < c ? im(i, c) : (i == c ? s[2][i] : 0.0); }
  // y <- H_0 .. H_{j1 - 1} y for the register-held column y (rows lane + 64 q)
  __device__ __forceinline__ void apply(double (&yr)[kSmallRpl], double (&yi)[kSmallRpl], int j1) const {
    const int lane = threadIdx.x & 63;
    for (int j = j1 - 1; j >= 0; --j) {
      const double b = s[0][j], hr = s[3][j], hi = s[4][j];
      if (b == 0.0) continue;
      double vr[kSmallRpl], vi[kSmallRpl], wr = 0.0, wi = 0.0;
#pragma unroll
      for (int q = 0; q < kSmallRpl; ++q) {
        vr[q] = vi[q] = 0.0;
        if (64 * q >= p) continue;  // uniform
        const int i = lane + 64 * q;
        if (i >= j && i < p) {
          vr[q] = i == j ? hr : re(i, j);
          if (C) vi[q] = i == j ? hi : im(i, j);
        }
        wr += vr[q] * yr[q];
        if (C) {
          wr += vi[q] * yi[q];
          wi += vr[q] * yi[q] - vi[q] * yr[q];
        }
      }
      wr = b * wave_sum(wr);
      if (C) wi = b * wave_sum(wi);
#pragma unroll
      for (int q = 0; q < kSmallRpl; ++q) {
        if (64 * q >= p) continue;
        yr[q] -= wr * vr[q] - wi * vi[q];
        if (C) yi[q] -= wr * vi[q] + wi * vr[q];
      }
    }
  }
};

// One-sided Jacobi sweeps on the r <= 64 columns of A (r x r, ld r) with the
// rotations accumulated in w, all in LDS: the pairing, rotation and stopping
// rule of svd_jacobi_kernel's sweeps, one row per lane.  Starts and ends with
// a barrier; flag: one LDS integer.  False when the last sweep still rotated.
template <bool C, int NT>
__device__ __forceinline__ bool jacobi_small(double* ar, double* ai, double* wr, double* wi, int r, int max_sweeps,
                                             int* flag) {
  constexpr int NW = NT / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double tol = sqrt((double)r) * DBL_EPSILON;
  const int rr = r + (r & 1);
  __syncthreads();
  if (r <= 1) return true;
  for (int sweep = 0; sweep < max_sweeps; ++sweep) {
    if (threadIdx.x == 0) *flag = 0;
    __syncthreads();
    for (int round = 0; round < rr - 1; ++round) {
      for (int q = wave; q < rr / 2; q += NW) {
        int i = (round + q) % (rr - 1);
        int j = q == 0 ? rr - 1 : (round + rr - 1 - q) % (rr - 1);
        if (i > j) {
          const int x = i;
          i = j;
          j = x;
        }
        if (j >= r) continue;
        double xir = 0.0, xii = 0.0, xjr = 0.0, xji = 0.0;
        if (lane < r) {
          xir = ar[i * r + lane];
          xjr = ar[j * r + lane];
          if (C) {
            xii = ai[i * r + lane];
            xji = ai[j * r + lane];
          }
        }
        const double a = wave_sum(xir * xir + xii * xii), b = wave_sum(xjr * xjr + xji * xji);
        const double gr = wave_sum(xir * xjr + xii * xji);
        const double gi = C ? wave_sum(xir * xji - xii * xjr) : 0.0;  // a_i^H a_j
        double c, sn, er, ei;
        if (!jacobi_rotation<C>(a, b, gr, gi, tol, c, sn, er, ei)) continue;
        // x_i' = c x_i - s conj(e) x_j, x_j' = s e x_i + c x_j (as rotate_cols)
        if (lane < r) {
          const double yir = wr[i * r + lane], yjr = wr[j * r + lane];
          if (C) {
            const double yii = wi[i * r + lane], yji = wi[j * r + lane];
            ar[i * r + lane] = c * xir - sn * (er * xjr + ei * xji);
            ai[i * r + lane] = c * xii - sn * (er * xji - ei * xjr);
            ar[j * r + lane] = sn * (er * xir - ei * xii) + c * xjr;
            ai[j * r + lane] = sn * (er * xii + ei * xir) + c * xji;
            wr[i * r + lane] = c * yir - sn * (er * yjr + ei * yji);
            wi[i * r + lane] = c * yii - sn * (er * yji - ei * yjr);
            wr[j * r + lane] = sn * (er * yir - ei * yii) + c * yjr;
            wi[j * r + lane] = sn * (er * yii + ei * yir) + c * yji;
          } else {
            ar[i * r + lane] = c * xir - sn * er * xjr;
            ar[j * r + lane] = sn * er * xir + c * xjr;
            wr[i * r + lane] = c * yir - sn * er * yjr;
            wr[j * r + lane] = sn * er * yir + c * yjr;
          }
        }
        if (lane == 0) *flag = 1;
      }
      __syncthreads();
    }
    const int any = *flag;
    __syncthreads();
    if (!any) return true;
  }
  return false;
}

static_assert(kSmallRows == 512 && kSmallCols == 64 && kQrLds + 6 * kSmallCols <= 8192, "qr_in_lds states these limits");
// LDS doubles of X: p r elements (both planes) of at most cap
__device__ __forceinline__ bool small_fits(int p, int r, bool cplx, int64_t cap) {
  return p <= kSmallRows && r <= kSmallCols && (int64_t)p * r * (cplx ? 2 : 1) <= cap;
}

template <bool C>
__global__ __launch_bounds__(kThreads) void svd_jacobi_kernel(const SvdTask* __restrict__ tasks,
                                                              const double* __restrict__ M, int64_t m_plane,
                                                              double* __restrict__ U, int64_t u_plane,
                                                              double* __restrict__ Vt, int64_t vt_plane,
                                                              double* __restrict__ S, double* __restrict__ W,
                                                              int64_t w_plane, int max_sweeps, int phases) {
  __shared__ double sig[kSvdMaxR];
  __shared__ int rank[kSvdMaxR];
  __shared__ int rotated, mxw[kWaves];
  __shared__ double red[kWaves], redc[kWaves];
  __shared__ double hv[3];
  // X, A and Wm of a small sector, or the general path's reflection vector
  constexpr int kCap = 12288;
  __shared__ double buf[kCap];
  __shared__ double scal[6][kSmallCols];
  static_assert(2 * kVecRows <= kCap, "the reflection vector fits");
  double* const vl = buf;
  const SvdTask t = tasks[blockIdx.x];
  const int m = t.m, n = t.n;
  if (m <= 0 || n <= 0) return;
  const bool wide = m < n;
  const int p = wide ? n : m, r = wide ? m : n, k = r;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // X = Q R (Householder), then the rotations run on the columns of
  // A = R^H (r x r), accumulated in Wm: A Wm = Z Sigma, so R = Wm Sigma Z^H
  // and X = (Q Wm) Sigma Z^H.  On R^H the sweeps of a graded or rank-deficient
  // sector are a third of those on R or X itself (the rows of a triangular
  // factor are closer to orthogonal than its columns).  The p-side singular
  // vectors Q Wm are orthonormal by construction; the r-side ones are the
  // rotated columns of A divided by sigma.  Workspace: X (p x r), Wm (r x r),
  // the reflection vectors (p x r), A (r x r), betas (r), the scale.
  Mat<C> X{W + t.w_off, W + t.w_off + w_plane, p};
  Mat<C> Wm{W + t.w_off + (int64_t)p * r, W + t.w_off + (int64_t)p * r + w_plane, r};
  const int64_t o_hv = (int64_t)p * r + (int64_t)r * r, o_a = 2 * (int64_t)p * r + (int64_t)r * r;
  Mat<C> Hv{W + t.w_off + o_hv, W + t.w_off + o_hv + w_plane, p};
  Mat<C> A{W + t.w_off + o_a, W + t.w_off + o_a + w_plane, r};
  double* const beta = W + t.w_off + o_a + (int64_t)r * r;
  double* const state = beta + r;  // the sector's scale, for the phases
  double scale = 1.0;
  // A small sector: reflections, sweeps and back-transform in LDS, A and
  // X = Q [Wm; 0] then in the workspace for the outputs below.  (A sweep of 30
  // columns is 30 rounds, each of which waits for memory on the general path.)
  const bool small = phases == kPhAll && small_fits(p, r, C, kCap - (C ? 4 : 2) * r * r);
  if (small) {
    constexpr int NP = C ? 2 : 1;
    double* const la = buf + NP * p * r;
    double* const lw = la + NP * r * r;
    const SmallQr<C> f{buf, buf + p * r, scal, p, r, r};
    int mx = 0;
    for (int e = tid; e < p * r; e += kThreads) {
      const int i = wide ? e / r : e % p, j = wide ? e % r : e / p;
      const int64_t src = t.a_off + (wide ? j + (int64_t)i * t.lda : i + (int64_t)j * t.lda);
      const double x = M[src], y = C ? M[m_plane + src] : 0.0;
      mx = max(mx, max(magnitude(x), magnitude(y)));
      f.re(i, j) = x;
      if (C) f.im(i, j) = wide ? -y : y;
    }
    scale = sector_scale(group_max<kThreads>(mx, mxw));
    if (scale != 1.0) {  // uniform
      for (int e = tid; e < p * r; e += kThreads) {
        const int i = wide ? e / r : e % p, j = wide ? e % r : e / p;
        f.re(i, j) /= scale;
        if (C) f.im(i, j) /= scale;
      }
      __syncthreads();
    }
    f.template factor<kThreads>();
    for (int e = tid; e < r * r; e += kThreads) {  // A = R^H, Wm = I
      const int i = e % r, j = e / r;
      la[e] = f.r_re(j, i);
      lw[e] = i == j ? 1.0 : 0.0;
      if (C) {
        la[r * r + e] = -f.r_im(j, i);
        lw[r * r + e] = 0.0;
      }
    }
    if (!jacobi_small<C, kThreads>(la, la + r * r, lw, lw + r * r, r, max_sweeps, &rotated))
      scale = sector_scale(kNotFinite);
    for (int c = wave; c < r; c += kWaves) {
      double yr[kSmallRpl], yi[kSmallRpl];
#pragma unroll
      for (int q = 0; q < kSmallRpl; ++q) {
        const int i = lane + 64 * q;
        yr[q] = i < r ? lw[c * r + i] : 0.0;
        yi[q] = C && i < r ? lw[r * r + c * r + i] : 0.0;
      }
      f.apply(yr, yi, r);
#pragma unroll
      for (int q = 0; q < kSmallRpl; ++q) {
        const int i = lane + 64 * q;
        if (i >= p) continue;
        X.r(i, c) = yr[q];
        if (C) X.m(i, c) = yi[q];
      }
      if (lane < r) {
        A.r(lane, c) = la[c * r + lane];
        if (C) A.m(lane, c) = la[r * r + c * r + lane];
      }
    }
    __syncthreads();
    phases = kPhOut;
  }
  // phases (kPh* bits; kPhAll: the whole SVD): the multi-workgroup path runs
  // the load, then house_panel/update kernels for the reflections, the init,
  // block rounds for the sweeps, the back-transform's init, house_apply_kernel,
  // and the outputs, each phase reading what the previous left in the workspace
  // X = M or M^H
  if (phases & kPhLoad) {
    int mx = 0;
    for (int64_t e = tid; e < (int64_t)p * r; e += kThreads) {
      const int i = (int)(e % p), j = (int)(e / p);
      const int64_t src = t.a_off + (wide ? (j + (int64_t)i * t.lda) : (i + (int64_t)j * t.lda));
      const double x = M[src], y = C ? M[m_plane + src] : 0.0;
      mx = max(mx, max(magnitude(x), magnitude(y)));
      X.r(i, j) = x;
      if (C) X.m(i, j) = wide ? -y : y;
    }
    scale = sector_scale(group_max<kThreads>(mx, mxw));
    if (scale != 1.0) {  // uniform
      for (int64_t e = tid; e < (int64_t)p * r; e += kThreads) {
        X.re[e] /= scale;
        if (C) X.im[e] /= scale;
      }
      __syncthreads();
    }
    if (tid == 0) *state = scale;
  } else if (!small) {
    scale = *state;
  }
  if (phases & kPhReflect) house_reflect<C, kThreads>(X, Hv, beta, p, r, red, hv, vl);
  // A = R^H (lower triangular), Wm = identity
  if (phases & kPhInit) {
    for (int64_t e = tid; e < (int64_t)r * r; e += kThreads) {
      const int i = (int)(e % r), j = (int)(e / r);
      A.r(i, j) = i >= j ? X.r(j, i) : 0.0;
      if (C) A.m(i, j) = i >= j ? -X.m(j, i) : 0.0;
      Wm.r(i, j) = i == j ? 1.0 : 0.0;
      if (C) Wm.m(i, j) = 0.0;
    }
    __syncthreads();
  }
  if (phases & kPhSweep) {
  const double tol = sqrt((double)r) * DBL_EPSILON;
  const int rr = r + (r & 1);
  bool ended = r <= 1;
  for (int sweep = 0; sweep < max_sweeps && !ended; ++sweep) {
    if (tid == 0) rotated = 0;
    __syncthreads();
    for (int round = 0; round < rr - 1; ++round) {
      for (int q = wave; q < rr / 2; q += kWaves) {
        int i = (round + q) % (rr - 1);
        int j = q == 0 ? rr - 1 : (round + rr - 1 - q) % (rr - 1);
        if (i > j) {
          const int x = i;
          i = j;
          j = x;
        }
        if (j >= r) continue;
        // the pair's columns stay in registers (r <= kSvdMaxR = 64 kRpl rows)
        double xir[kRpl], xii[kRpl], xjr[kRpl], xji[kRpl];
        double a = 0.0, b = 0.0, gr = 0.0, gi = 0.0;
#pragma unroll
        for (int q = 0; q < kRpl; ++q) {
          const int row = lane + 64 * q;
          xir[q] = xii[q] = xjr[q] = xji[q] = 0.0;
          if (row < r) {
            xir[q] = A.r(row, i);
            xjr[q] = A.r(row, j);
            a += xir[q] * xir[q];
            b += xjr[q] * xjr[q];
            gr += xir[q] * xjr[q];
            if (C) {
              xii[q] = A.m(row, i);
              xji[q] = A.m(row, j);
              a += xii[q] * xii[q];
              b += xji[q] * xji[q];
              gr += xii[q] * xji[q];
              gi += xir[q] * xji[q] - xii[q] * xjr[q];  // a_i^H a_j = sum conj(a_i) a_j
            }
          }
        }
        a = wave_sum(a);
        b = wave_sum(b);
        gr = wave_sum(gr);
        if (C) gi = wave_sum(gi);
        double c, s, er, ei;
        if (!jacobi_rotation<C>(a, b, gr, gi, tol, c, s, er, ei)) continue;
        // a_i' = c a_i - s conj(e) a_j, a_j' = s e a_i + c a_j (as rotate_cols)
#pragma unroll
        for (int q = 0; q < kRpl; ++q) {
          const int row = lane + 64 * q;
          if (row < r) {
            if (C) {
              const double cjr = er * xjr[q] + ei * xji[q], cji = er * xji[q] - ei * xjr[q];
              const double eir = er * xir[q] - ei * xii[q], eii = er * xii[q] + ei * xir[q];
              A.r(row, i) = c * xir[q] - s * cjr;
              A.m(row, i) = c * xii[q] - s * cji;
              A.r(row, j) = s * eir + c * xjr[q];
              A.m(row, j) = s * eii + c * xji[q];
            } else {
              A.r(row, i) = c * xir[q] - s * er * xjr[q];
              A.r(row, j) = s * er * xir[q] + c * xjr[q];
            }
          }
        }
        rotate_cols<C>(Wm, r, i, j, c, s, er, ei, lane);
        if (lane == 0) rotated = 1;
      }
      __syncthreads();
    }
    ended = !rotated;
    __syncthreads();
  }
  if (!ended) {
    scale = sector_scale(kNotFinite);
    if (tid == 0) *state = scale;
  }
  }
  // X = Q [Wm; 0]: the accumulated rotations back through the reflections
  if (phases & kPhBackInit) {
    for (int64_t e = tid; e < (int64_t)p * r; e += kThreads) {
      const int i = (int)(e % p), j = (int)(e / p);
      X.r(i, j) = i < r ? Wm.r(i, j) : 0.0;
      if (C) X.m(i, j) = i < r ? Wm.m(i, j) : 0.0;
    }
    __syncthreads();
  }
  if (phases & kPhApply) house_apply<C, kThreads>(X, r, false, Hv, beta, p, r, vl);
  if (!(phases & kPhOut)) return;
  // singular values (column norms of the rotated A) and their descending order
  if (tid == 0) rotated = r;  // from here: the rank of the first zero singular value
  for (int j = wave; j < r; j += kWaves) {
    double a = 0.0;
    for (int row = lane; row < r; row += 64) {
      const double x = A.r(row, j);
      a += x * x;
      if (C) {
        const double y = A.m(row, j);
        a += y * y;
      }
    }
    a = wave_sum(a);
    a = a < kTinySq ? 0.0 : sqrt(a);
    if (lane == 0) sig[j] = a;
    if (!(a <= DBL_MAX)) scale = a;
  }
  if (__syncthreads_or(!(scale <= DBL_MAX))) {  // no factors: every output NaN
    const double none = sector_scale(kNotFinite);
    for (int i = tid; i < k; i += kThreads) S[t.s_off + i] = none;
    for (int64_t e = tid; e < (int64_t)m * k; e += kThreads) {
      U[t.u_off + e] = none;
      if (C) U[t.u_off + u_plane + e] = none;
    }
    for (int64_t e = tid; e < (int64_t)k * n; e += kThreads) {
      Vt[t.vt_off + e] = none;
      if (C) Vt[t.vt_off + vt_plane + e] = none;
    }
    return;
  }
  for (int j = tid; j < r; j += kThreads) {
    int rk = 0;
    const double sj = sig[j];
    for (int i = 0; i < r; ++i) rk += (sig[i] > sj || (sig[i] == sj && i < j)) ? 1 : 0;
    rank[j] = rk;
    if (sj == 0.0) atomicMin(&rotated, rk);
    S[t.s_off + rk] = sj * scale;
  }
  __syncthreads();
  // U (m x k, ld m) and V^dagger (k x n, ld k): the p side from Q Wm, the r
  // side from A / sigma
  double* Ur = U + t.u_off;
  double* Ui = U + t.u_off + u_plane;
  double* Vr = Vt + t.vt_off;
  double* Vi = Vt + t.vt_off + vt_plane;
  for (int64_t e = tid; e < (int64_t)p * r; e += kThreads) {
    const int row = (int)(e % p), j = (int)(e / p);
    const int rk = rank[j];
    if (!wide) {  // U[:, rk] = (Q Wm)[:, j]
      Ur[row + (int64_t)rk * m] = X.r(row, j);
      if (C) Ui[row + (int64_t)rk * m] = X.m(row, j);
    } else {  // V^dagger[rk, :] = (Q Wm)[:, j]^H
      Vr[rk + (int64_t)row * k] = X.r(row, j);
      if (C) Vi[rk + (int64_t)row * k] = -X.m(row, j);
    }
  }
  for (int64_t e = tid; e < (int64_t)r * r; e += kThreads) {
    const int row = (int)(e % r), j = (int)(e / r);
    const int rk = rank[j];
    const double sj = sig[j];
    const double zr = sj > 0.0 ? A.r(row, j) / sj : 0.0;
    const double zi = (C && sj > 0.0) ? A.m(row, j) / sj : 0.0;
    if (!wide) {  // V^dagger[rk, row] = conj(Z[row, j])
      Vr[rk + (int64_t)row * k] = zr;
      if (C) Vi[rk + (int64_t)row * k] = -zi;
    } else {  // U[row, rk] = Z[row, j]
      Ur[row + (int64_t)rk * m] = zr;
      if (C) Ui[row + (int64_t)rk * m] = zi;
    }
  }
  __syncthreads();
  // orthonormal completion of the r-side vectors of zero singular values
  // (descending order puts them last, from rank `first` on): vectors of length
  // r stored at base + idx * vs with stride es between elements (V^dagger rows:
  // es = k, vs = 1; U columns: es = 1, vs = m).  The conjugate of a V^dagger
  // row is the vector.  Each starts from a unit vector e_c and loses its
  // components along the vectors before it, twice; c is the first index whose
  // residual 1 - sum |u_i[c]|^2 is above 1/4, or the one of the largest
  // residual (at least 1 / r).  All components of a pass are taken at once, so
  // a vector costs seven barriers, where unit vectors tried one after another,
  // component by component, cost r^2 of them: the zero sector of 160 x 160
  // took 2.7 million (and a null space whose residuals are all below 1/4 got
  // no vector).  60 x 60 zeros: 73.5 ms so, 0.9 ms here; a sector of nothing
  // but zeros takes the unit vectors as they are.
  const int first = rotated;
  const int64_t es = wide ? 1 : k, vs = wide ? m : 1;
  double* Br = wide ? Ur : Vr;
  double* Bi = wide ? Ui : Vi;
  if (first == 0) {
    for (int64_t e = tid; e < (int64_t)r * r; e += kThreads) {
      const int i = (int)(e / r), c = (int)(e % r);
      Br[i * vs + c * es] = i == c ? 1.0 : 0.0;
      if (C) Bi[i * vs + c * es] = 0.0;
    }
    __syncthreads();
  } else if (first < k) {
    const double csign = wide ? 1.0 : -1.0;  // stored imaginary part = csign * vector imaginary part
    double *const wr = buf, *const wi = buf + kSvdMaxR;                     // the vector
    double *const dr = buf + 2 * kSvdMaxR, *const di = buf + 3 * kSvdMaxR;  // its components
    static_assert(4 * kSvdMaxR <= kCap, "the completion's vectors fit");
    double* const rho = sig;  // residual of e_c
    for (int c = tid; c < r; c += kThreads) {
      double x = 1.0;
      for (int i = 0; i < first; ++i) {
        const double ur = Br[i * vs + c * es], ui = C ? Bi[i * vs + c * es] : 0.0;
        x -= ur * ur + ui * ui;
      }
      rho[c] = x;
    }
    __syncthreads();
    for (int rk = first; rk < k; ++rk) {
      // the start
      int c = r;
      double top = -1.0;
      for (int x = tid; x < r; x += kThreads)
        if (rho[x] > 0.25 ? top < 2.0 : rho[x] > top) {
          c = x;
          top = rho[x] > 0.25 ? 2.0 : rho[x];
        }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const double ot = __shfl_xor(top, o, 64);
        const int oc = __shfl_xor(c, o, 64);
        if (ot > top || (ot == top && oc < c)) {
          top = ot;
          c = oc;
        }
      }
      if (lane == 0) {
        red[wave] = top;
        mxw[wave] = c;
      }
      __syncthreads();
      c = mxw[0];
      top = red[0];
      for (int w = 1; w < kWaves; ++w)
        if (red[w] > top || (red[w] == top && mxw[w] < c)) {
          top = red[w];
          c = mxw[w];
        }
      double nn = 0.0;
      for (int pass = 0; pass < 2; ++pass) {
        // components u_i^H w; those of e_c are conj(u_i[c])
        if (pass == 0) {
          for (int i = tid; i < rk; i += kThreads) {
            dr[i] = Br[i * vs + c * es];
            if (C) di[i] = -csign * Bi[i * vs + c * es];
          }
        } else {
          for (int i = wave; i < rk; i += kWaves) {
            double ar = 0.0, ai = 0.0;
            for (int row = lane; row < r; row += 64) {
              const double ur = Br[i * vs + row * es];
              ar += ur * wr[row];
              if (C) {
                const double ui = csign * Bi[i * vs + row * es];
                ar += ui * wi[row];
                ai += ur * wi[row] - ui * wr[row];
              }
            }
            ar = wave_sum(ar);
            if (C) ai = wave_sum(ai);
            if (lane == 0) {
              dr[i] = ar;
              if (C) di[i] = ai;
            }
          }
        }
        __syncthreads();
        nn = 0.0;
        for (int row = tid; row < r; row += kThreads) {
          double xr = pass ? wr[row] : (row == c ? 1.0 : 0.0), xi = C && pass ? wi[row] : 0.0;
          for (int i = 0; i < rk; ++i) {
            const double ur = Br[i * vs + row * es];
            xr -= dr[i] * ur;
            if (C) {
              const double ui = csign * Bi[i * vs + row * es];
              xr += di[i] * ui;
              xi -= dr[i] * ui + di[i] * ur;
            }
          }
          wr[row] = xr;
          if (C) wi[row] = xi;
          nn += xr * xr + xi * xi;
        }
        __syncthreads();
      }
      nn = wave_sum(nn);
      if (lane == 0) redc[wave] = nn;
      __syncthreads();
      nn = 0.0;
      for (int w = 0; w < kWaves; ++w) nn += redc[w];
      const double inv = 1.0 / sqrt(nn);
      for (int row = tid; row < r; row += kThreads) {
        const double xr = wr[row] * inv, xi = C ? wi[row] * inv : 0.0;
        Br[rk * vs + row * es] = xr;
        if (C) Bi[rk * vs + row * es] = csign * xi;
        rho[row] -= xr * xr + xi * xi;
      }
      __syncthreads();
    }
  }
  // FixPhase (real data): first index of the largest |V^dagger[i, c]|; flip
  // row i of V^dagger and column i of U unless that entry is > 0
  if (!C) {
    for (int i = wave; i < k; i += kWaves) {
      double best = 0.0;
      int bi = 0;
      for (int c = lane; c < n; c += 64) {
        const double a = fabs(Vr[i + (int64_t)c * k]);
        if (a > best) {
          best = a;
          bi = c;
        }
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const double ob = __shfl_xor(best, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (ob > best || (ob == best && oi < bi)) {
          best = ob;
          bi = oi;
        }
      }
      const double phi = Vr[i + (int64_t)bi * k] > 0.0 ? 1.0 : -1.0;
      if (phi < 0.0) {
        for (int c = lane; c < n; c += 64) Vr[i + (int64_t)c * k] = -Vr[i + (int64_t)c * k];
        for (int row = lane; row < m; row += 64) Ur[row + (int64_t)i * m] = -Ur[row + (int64_t)i * m];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Block Jacobi rounds for large sectors, several workgroups per sector.
// After the reduction and init phases the r columns of A = R^H are
// split into blocks of kBj columns; one launch runs one round of the block
// tournament over every large sector at once, one workgroup per block pair
// (I, J) (svd_block_across_kernel): it rotates every pair (i in I, j in J)
// once with the scalar kernel's rotation and threshold, writes the columns
// back and applies the accumulated 2 kBj x 2 kBj rotation to the same columns
// of Wm.  The launch with round < 0 (svd_block_inner_kernel) does the pairs
// inside each block (a tournament over its columns, one workgroup per block),
// so a sweep (that launch, then the rounds) visits every pair of columns once.  Sectors have
// their block pairs at pair_base[s] .. pair_base[s + 1] of the grid (twice
// that for the intra-block launch); rotated[s] is set when any pair of the
// sector rotated (the host repeats sweeps until none does, then the
// back-transform and output phases finish).  r <= kBjMaxR.
constexpr int kBj = 8;
constexpr int kBjMaxR = 512;
static_assert(kBj == kWaves, "one wave per column of block I in the rounds across blocks");

template <bool C>
__global__ __launch_bounds__(kThreads) void svd_block_inner_kernel(const SvdTask* __restrict__ tasks, int ntasks,
                                                                   const int* __restrict__ pair_base,
                                                                   double* __restrict__ W, int64_t w_plane,
                                                                   double* __restrict__ rotated, int rmax) {
  // the block's columns: kBj x rmax per plane of dynamic LDS (rmax: the
  // launch's largest r, so that small launches fit several workgroups per CU)
  extern __shared__ double blk_lds[];
  double* const Lr = blk_lds;
  double* const Li = blk_lds + kBj * rmax;
  __shared__ double Vr[kBj * kBj], Vi[kBj * kBj];
  __shared__ int any;
  // sector of this workgroup: pair_base is ascending, pair_base[0] = 0; two
  // workgroups per block pair slot
  int lo = 0, hi = ntasks - 1;
  const int b = blockIdx.x, bs = b >> 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (pair_base[mid] <= bs) lo = mid;
    else hi = mid - 1;
  }
  const int sidx = lo;
  const SvdTask t = tasks[sidx];
  const int q = b - 2 * pair_base[sidx];
  const int m = t.m, n = t.n;
  const int p = m < n ? n : m, r = m < n ? m : n;
  const int nb = (r + kBj - 1) / kBj;
  if (r > rmax || q >= nb) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i0 = q * kBj, w = min(kBj, r - i0);
  auto colof = [&](int c) { return i0 + c; };
  const int64_t o_wm = (int64_t)p * r, o_a = 2 * (int64_t)p * r + (int64_t)r * r;
  Mat<C> Wm{W + t.w_off + o_wm, W + t.w_off + o_wm + w_plane, r};
  Mat<C> A{W + t.w_off + o_a, W + t.w_off + o_a + w_plane, r};
  // the block's columns of A into LDS (column c at c * r), V = identity
  for (int e = tid; e < w * r; e += kThreads) {
    const int c = e / r, row = e - c * r;
    Lr[c * r + row] = A.r(row, colof(c));
    if (C) Li[c * r + row] = A.m(row, colof(c));
  }
  for (int e = tid; e < w * w; e += kThreads) {
    Vr[e] = (e % w) == (e / w) ? 1.0 : 0.0;
    Vi[e] = 0.0;
  }
  if (tid == 0) any = 0;
  __syncthreads();
  const double tol = sqrt((double)r) * DBL_EPSILON;
  const int ww = w + (w & 1);
  // a tournament over the block's columns
  for (int sub = 0; sub < ww - 1; ++sub) {
    for (int pq = wave; pq < ww / 2; pq += kWaves) {
      int i = (sub + pq) % (ww - 1);
      int j = pq == 0 ? ww - 1 : (sub + ww - 1 - pq) % (ww - 1);
      if (i > j) {
        const int x = i;
        i = j;
        j = x;
      }
      if (j >= w) continue;
      double a = 0.0, bb = 0.0, gr = 0.0, gi = 0.0;
      for (int row = lane; row < r; row += 64) {
        const double xir = Lr[i * r + row], xjr = Lr[j * r + row];
        a += xir * xir;
        bb += xjr * xjr;
        gr += xir * xjr;
        if (C) {
          const double xii = Li[i * r + row], xji = Li[j * r + row];
          a += xii * xii;
          bb += xji * xji;
          gr += xii * xji;
          gi += xir * xji - xii * xjr;
        }
      }
      a = wave_sum(a);
      bb = wave_sum(bb);
      gr = wave_sum(gr);
      if (C) gi = wave_sum(gi);
      double c, sn, er, ei;
      if (!jacobi_rotation<C>(a, bb, gr, gi, tol, c, sn, er, ei)) continue;
      // a_i' = c a_i - s conj(e) a_j, a_j' = s e a_i + c a_j (as rotate_cols), on the columns and on V
      for (int row = lane; row < r; row += 64) {
        const double xir = Lr[i * r + row], xjr = Lr[j * r + row];
        if (C) {
          const double xii = Li[i * r + row], xji = Li[j * r + row];
          const double cjr = er * xjr + ei * xji, cji = er * xji - ei * xjr;
          const double eir = er * xir - ei * xii, eii = er * xii + ei * xir;
          Lr[i * r + row] = c * xir - sn * cjr;
          Li[i * r + row] = c * xii - sn * cji;
          Lr[j * r + row] = sn * eir + c * xjr;
          Li[j * r + row] = sn * eii + c * xji;
        } else {
          Lr[i * r + row] = c * xir - sn * er * xjr;
          Lr[j * r + row] = sn * er * xir + c * xjr;
        }
      }
      if (lane < w) {
        const int row = lane;
        const double vir = Vr[i * w + row], vjr = Vr[j * w + row];
        if (C) {
          const double vii = Vi[i * w + row], vji = Vi[j * w + row];
          const double cjr = er * vjr + ei * vji, cji = er * vji - ei * vjr;
          const double eir = er * vir - ei * vii, eii = er * vii + ei * vir;
          Vr[i * w + row] = c * vir - sn * cjr;
          Vi[i * w + row] = c * vii - sn * cji;
          Vr[j * w + row] = sn * eir + c * vjr;
          Vi[j * w + row] = sn * eii + c * vji;
        } else {
          Vr[i * w + row] = c * vir - sn * er * vjr;
          Vr[j * w + row] = sn * er * vir + c * vjr;
        }
      }
      if (lane == 0) any = 1;
    }
    __syncthreads();
  }
  if (!any) return;  // uniform: read after the last barrier; nothing changed
  // columns back to A; Wm[:, cols] <- Wm[:, cols] V (V column c: entries c * w + row)
  for (int e = tid; e < w * r; e += kThreads) {
    const int c = e / r, row = e - c * r;
    A.r(row, colof(c)) = Lr[c * r + row];
    if (C) A.m(row, colof(c)) = Li[c * r + row];
  }
  for (int row = tid; row < r; row += kThreads) {
    double orr[kBj], oi[kBj];
#pragma unroll
    for (int c = 0; c < kBj; ++c) {
      orr[c] = c < w ? Wm.r(row, colof(c)) : 0.0;
      oi[c] = (C && c < w) ? Wm.m(row, colof(c)) : 0.0;
    }
    for (int c = 0; c < w; ++c) {
      double sr = 0.0, si = 0.0;
#pragma unroll
      for (int c2 = 0; c2 < kBj; ++c2) {
        if (c2 >= w) break;
        const double vr = Vr[c * w + c2], vi = Vi[c * w + c2];  // V[c2, c]
        sr += orr[c2] * vr - (C ? oi[c2] * vi : 0.0);
        if (C) si += orr[c2] * vi + oi[c2] * vr;
      }
      Wm.r(row, colof(c)) = sr;
      if (C) Wm.m(row, colof(c)) = si;
    }
  }
  if (tid == 0) rotated[sidx] = 1.0;
}

// A barrier that waits for this wave's LDS accesses only: global loads stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The rounds across blocks (round >= 0): wave a keeps column a of block I in
// registers through all kBj sub-rounds and meets column (a + sub) mod kBj of
// block J, which is in LDS, so a sub-round reads one column and writes one
// where columns of both blocks in LDS cost two of each.  Latency bounds it:
// every launch waits for the one before, so the sector is found by one wave
// read, the columns of A and Wm are requested together before the first
// wait, and for columns of at most 64 NQ rows (zero beyond r) no sub-round
// has a branch on the row.  Mean launch: real, r up to 256: 13.0 us against
// 20 with both blocks in LDS and the quotient form of the rotation; complex,
// r up to 128 (Hubbard L = 20, D = 192, 4 vectors): 15.5 us against 20.
template <bool C, int NQ>
__global__ __launch_bounds__(kThreads) void svd_block_across_kernel(const SvdTask* __restrict__ tasks, int ntasks,
                                                                    const int* __restrict__ pair_base, int round,
                                                                    double* __restrict__ W, int64_t w_plane,
                                                                    double* __restrict__ rotated) {
  constexpr int kRows = 64 * NQ, kPairs = 2 * kBj;
  extern __shared__ double blk_lds[];  // block J: kBj columns of kRows, per plane
  double* const Lr = blk_lds;
  double* const Li = blk_lds + kBj * kRows;
  __shared__ double Vr[kPairs * kPairs], Vi[kPairs * kPairs];  // column c at c * kPairs
  __shared__ int any;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // sector of this workgroup: pair_base is ascending, pair_base[0] = 0
  int s = 0;
  for (int n = ntasks; n > 1;) {
    const int step = (n + 63) >> 6, i = lane * step;
    const bool ok = i < n && pair_base[s + (i < n ? i : 0)] <= (int)blockIdx.x;
    const int c = __popcll(__ballot(ok)) - 1;
    s += c * step;
    n = min(step, n - c * step);
  }
  s = __builtin_amdgcn_readfirstlane(s);
  const SvdTask t = tasks[s];
  const int q = (int)blockIdx.x - pair_base[s];
  const int p = t.m < t.n ? t.n : t.m, r = t.m < t.n ? t.m : t.n;
  const int nb = (r + kBj - 1) / kBj, nbb = nb + (nb & 1);
  if (r > kRows || round >= nbb - 1 || q >= nbb / 2) return;
  int I = (round + q) % (nbb - 1);
  int J = q == 0 ? nbb - 1 : (round + nbb - 1 - q) % (nbb - 1);
  if (I > J) {
    const int x = I;
    I = J;
    J = x;
  }
  if (J >= nb) return;  // the bye of an odd block count
  const int i0 = I * kBj, j0 = J * kBj, w = kBj + min(kBj, r - j0);  // J > I: block I is whole
  const int64_t o_wm = (int64_t)p * r, o_a = 2 * (int64_t)p * r + (int64_t)r * r;
  Mat<C> Wm{W + t.w_off + o_wm, W + t.w_off + o_wm + w_plane, r};
  Mat<C> A{W + t.w_off + o_a, W + t.w_off + o_a + w_plane, r};
  // column c of the pair's 2 kBj; those past the sector read its last one
  auto colof = [&](int c) { return c < kBj ? i0 + c : min(j0 + c - kBj, r - 1); };
  const bool has = kBj + wave < w;
  double xr[NQ], xi[NQ];
  {
    double jr[NQ], ji[NQ];
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const int row = min(lane + 64 * k, r - 1);
      xr[k] = A.r(row, i0 + wave);
      jr[k] = A.r(row, colof(kBj + wave));
      if (C) {
        xi[k] = A.m(row, i0 + wave);
        ji[k] = A.m(row, colof(kBj + wave));
      }
    }
    if (tid < kPairs * kPairs) {
      Vr[tid] = tid % kPairs == tid / kPairs ? 1.0 : 0.0;
      Vi[tid] = 0.0;
    }
    if (tid == 0) any = 0;
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const bool in = lane + 64 * k < r;
      xr[k] = in ? xr[k] : 0.0;
      Lr[wave * kRows + lane + 64 * k] = in && has ? jr[k] : 0.0;
      if (C) {
        xi[k] = in ? xi[k] : 0.0;
        Li[wave * kRows + lane + 64 * k] = in && has ? ji[k] : 0.0;
      }
    }
  }
  // this thread's row of Wm's columns: kThreads / kRows threads share a row and
  // write kNc columns each
  constexpr int kNc = kPairs * kRows / kThreads;
  const int wrow = tid % kRows, c_lo = __builtin_amdgcn_readfirstlane(tid / kRows) * kNc;
  double wr[kPairs], wi[kPairs];
#pragma unroll
  for (int c = 0; c < kPairs; ++c) {
    const double re = Wm.r(min(wrow, r - 1), colof(c)), im = C ? Wm.m(min(wrow, r - 1), colof(c)) : 0.0;
    wr[c] = c < w ? re : 0.0;
    wi[c] = c < w ? im : 0.0;
  }
  lds_barrier();
  const double tol = sqrt((double)r) * DBL_EPSILON;
  for (int sub = 0; sub < kBj; ++sub) {
    const int j = (wave + sub) % kBj;
    double* const yjr = Lr + j * kRows + lane;
    double* const yji = Li + j * kRows + lane;
    double yr[NQ], yi[NQ], a = 0.0, bb = 0.0, gr = 0.0, gi = 0.0;
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      yr[k] = yjr[64 * k];
      if (C) yi[k] = yji[64 * k];
    }
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      a += xr[k] * xr[k];
      bb += yr[k] * yr[k];
      gr += xr[k] * yr[k];
      if (C) {
        a += xi[k] * xi[k];
        bb += yi[k] * yi[k];
        gr += xi[k] * yi[k];
        gi += xr[k] * yi[k] - xi[k] * yr[k];
      }
    }
    a = wave_sum(a);
    bb = wave_sum(bb);
    gr = wave_sum(gr);
    if (C) gi = wave_sum(gi);
    double c, sn, er, ei;
    if (jacobi_rotation<C>(a, bb, gr, gi, tol, c, sn, er, ei)) {
      // x' = c x - s conj(e) y, y' = s e x + c y (as rotate_cols), on the columns and on V
#pragma unroll
      for (int k = 0; k < NQ; ++k) {
        if (C) {
          const double ujr = er * yr[k] + ei * yi[k], uji = er * yi[k] - ei * yr[k];
          const double uir = er * xr[k] - ei * xi[k], uii = er * xi[k] + ei * xr[k];
          xr[k] = c * xr[k] - sn * ujr;
          xi[k] = c * xi[k] - sn * uji;
          yjr[64 * k] = sn * uir + c * yr[k];
          yji[64 * k] = sn * uii + c * yi[k];
        } else {
          const double x0 = xr[k];
          xr[k] = c * x0 - sn * er * yr[k];
          yjr[64 * k] = sn * er * x0 + c * yr[k];
        }
      }
      if (lane < kPairs) {
        const int ci = wave * kPairs + lane, cj = (kBj + j) * kPairs + lane;
        const double vir = Vr[ci], vjr = Vr[cj];
        if (C) {
          const double vii = Vi[ci], vji = Vi[cj];
          Vr[ci] = c * vir - sn * (er * vjr + ei * vji);
          Vi[ci] = c * vii - sn * (er * vji - ei * vjr);
          Vr[cj] = sn * (er * vir - ei * vii) + c * vjr;
          Vi[cj] = sn * (er * vii + ei * vir) + c * vji;
        } else {
          Vr[ci] = c * vir - sn * er * vjr;
          Vr[cj] = sn * er * vir + c * vjr;
        }
      }
      if (lane == 0) any = 1;
    }
    lds_barrier();
  }
  if (!any) return;  // uniform: read after the last barrier; nothing changed
  // every thread's row of Wm has arrived before the threads that share it write
#pragma unroll
  for (int c = 0; c < kPairs; ++c) {
    asm volatile("" : "+v"(wr[c]));
    if (C) asm volatile("" : "+v"(wi[c]));
  }
  lds_barrier();
  // columns back to A; Wm[:, cols] <- Wm[:, cols] V
#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    const int row = lane + 64 * k;
    if (row >= r) continue;
    A.r(row, i0 + wave) = xr[k];
    if (C) A.m(row, i0 + wave) = xi[k];
    if (has) {
      A.r(row, j0 + wave) = Lr[wave * kRows + row];
      if (C) A.m(row, j0 + wave) = Li[wave * kRows + row];
    }
  }
  if (wrow < r)
    for (int c = c_lo; c < min(w, c_lo + kNc); ++c) {
      double sr = 0.0, si = 0.0;
#pragma unroll
      for (int c2 = 0; c2 < kPairs; ++c2) {
        const double vr = Vr[c * kPairs + c2], vi = C ? Vi[c * kPairs + c2] : 0.0;
        sr += wr[c2] * vr - (C ? wi[c2] * vi : 0.0);
        if (C) si += wr[c2] * vi + wi[c2] * vr;
      }
      Wm.r(wrow, colof(c)) = sr;
      if (C) Wm.m(wrow, colof(c)) = si;
    }
  if (tid == 0) rotated[s] = 1.0;
}

// ---------------------------------------------------------------------------
// Batched Householder QR of the same sector matrices, for the gauge steps
// that need an isometry but no Schmidt values: left (right = 0) M = Q R with
// Q (m x k) orthonormal columns, R (k x n) upper trapezoidal; right
// (right = 1) M = L Q' from the QR of M^H = Q R: L = R^H (m x k), Q' = Q^H
// (k x n) orthonormal rows; k = min(m, n).  Written in the SVD's output
// format with S = 1: U = Q (left) or L (right), V^dagger = R (left) or Q'
// (right), so that U S V^dagger = M as for the SVD.
//
// X = M or M^H (p x r) in the workspace; for j < k the reflection
// H_j = I - beta_j v_j v_j^H (v_j at rows j.. of column j of the vector
// store, beta_j = 2 / |v_j|^2, v_j = x - alpha e_j with alpha = -e^{i arg x_j}
// |x|) zeroes column j below the diagonal, applied to columns j+1.. one wave
// per column; then Q = H_0 ... H_{k-1} [I; 0] is accumulated backwards
// (columns j.. of the partial product, as LAPACK's xORGQR does).
// Workspace per task (qr_workspace): X (p r), the vectors (p k), the betas (k)
// and the scale, per plane.  A matrix with a value that is not finite gives an
// R of NaN.
constexpr int kQrThreads = 512;
constexpr int kQrWaves = kQrThreads / 64;

template <bool C>
__global__ __launch_bounds__(kQrThreads) void qr_householder_kernel(const SvdTask* __restrict__ tasks, int right,
                                                                    const double* __restrict__ M, int64_t m_plane,
                                                                    double* __restrict__ U, int64_t u_plane,
                                                                    double* __restrict__ Vt, int64_t vt_plane,
                                                                    double* __restrict__ S, double* __restrict__ W,
                                                                    int64_t w_plane, int phases) {
  __shared__ double red[kQrWaves];
  __shared__ double hv[3];
  __shared__ int mxw[kQrWaves];
  // X of a small sector, or the general path's reflection vector
  constexpr int kCap = kQrLds;
  __shared__ double buf[kCap];
  __shared__ double scal[6][kSmallCols];
  static_assert(2 * kVecRows <= kCap, "the reflection vector fits");
  double* const vl = buf;
  const SvdTask t = tasks[blockIdx.x];
  const int m = t.m, n = t.n;
  if (m <= 0 || n <= 0) return;
  const int p = right ? n : m, r = right ? m : n, k = p < r ? p : r;
  const int tid = threadIdx.x;
  if (phases == kPhAll && qr_in_lds(m, n, right, C)) {
    const SmallQr<C> f{buf, buf + p * r, scal, p, r, k};
    int mx = 0;
    for (int e = tid; e < p * r; e += kQrThreads) {
      // neighbouring threads read neighbouring elements of M
      const int i = right ? e / r : e % p, j = right ? e % r : e / p;
      const int64_t src = t.a_off + (right ? j + (int64_t)i * t.lda : i + (int64_t)j * t.lda);
      const double x = M[src], y = C ? M[m_plane + src] : 0.0;
      mx = max(mx, max(magnitude(x), magnitude(y)));
      f.re(i, j) = x;
      if (C) f.im(i, j) = right ? -y : y;
    }
    const double scale = sector_scale(group_max<kQrThreads>(mx, mxw));
    if (scale != 1.0) {  // uniform
      for (int e = tid; e < p * r; e += kQrThreads) {
        const int i = right ? e / r : e % p, j = right ? e % r : e / p;
        f.re(i, j) /= scale;
        if (C) f.im(i, j) /= scale;
      }
      __syncthreads();
    }
    f.template factor<kQrThreads>();
    for (int e = tid; e < k * r; e += kQrThreads) {
      const int i = right ? e / r : e % k, c = right ? e % r : e / k;
      // V^dagger (k x n) = R, or U (m x k) = R^H: U[c, i] = conj(R[i, c])
      double* const o = right ? U + t.u_off + c + (int64_t)i * m : Vt + t.vt_off + i + (int64_t)c * k;
      o[0] = scale * f.r_re(i, c);
      if (C) o[right ? u_plane : vt_plane] = scale * (right ? -f.r_im(i, c) : f.r_im(i, c));
    }
    for (int i = tid; i < k; i += kQrThreads) S[t.s_off + i] = 1.0;
    const int lane = tid & 63;
    for (int c = tid >> 6; c < k; c += kQrWaves) {  // Q[:, c] = H_0 .. H_c e_c
      double yr[kSmallRpl], yi[kSmallRpl];
#pragma unroll
      for (int q = 0; q < kSmallRpl; ++q) {
        yr[q] = lane + 64 * q == c ? 1.0 : 0.0;
        yi[q] = 0.0;
      }
      f.apply(yr, yi, c + 1);
#pragma unroll
      for (int q = 0; q < kSmallRpl; ++q) {
        const int i = lane + 64 * q;
        if (i >= p) continue;
        // U (m x k) = Q, or V^dagger (k x n) = Q^H
        double* const o = right ? Vt + t.vt_off + c + (int64_t)i * k : U + t.u_off + i + (int64_t)c * m;
        o[0] = yr[q];
        if (C) o[right ? vt_plane : u_plane] = right ? -yi[q] : yi[q];
      }
    }
    return;
  }
  // X (p x r) at 0, vectors (p x k) at p r, betas at p r + p k (real plane)
  Mat<C> X{W + t.w_off, W + t.w_off + w_plane, p};
  Mat<C> Hv{W + t.w_off + (int64_t)p * r, W + t.w_off + (int64_t)p * r + w_plane, p};
  double* const beta = W + t.w_off + (int64_t)p * r + (int64_t)p * k;
  double* const state = beta + k;  // the sector's scale, for the phases
  double scale = 1.0;
  // phases: kPhLoad, kPhReflect, kPhInit (R out, Q := [I; 0]), kPhApply, kPhOut
  // (the multi-workgroup path runs the reflections and the apply in
  // house_panel/update_kernel and house_apply_kernel between them)
  if (phases & kPhLoad) {
    int mx = 0;
    for (int64_t e = tid; e < (int64_t)p * r; e += kQrThreads) {
      const int i = (int)(e % p), j = (int)(e / p);
      const int64_t src = t.a_off + (right ? (j + (int64_t)i * t.lda) : (i + (int64_t)j * t.lda));
      const double x = M[src], y = C ? M[m_plane + src] : 0.0;
      mx = max(mx, max(magnitude(x), magnitude(y)));
      X.r(i, j) = x;
      if (C) X.m(i, j) = right ? -y : y;
    }
    scale = sector_scale(group_max<kQrThreads>(mx, mxw));
    if (scale != 1.0) {  // uniform
      for (int64_t e = tid; e < (int64_t)p * r; e += kQrThreads) {
        X.re[e] /= scale;
        if (C) X.im[e] /= scale;
      }
      __syncthreads();
    }
    if (tid == 0) *state = scale;
  } else {
    scale = *state;
  }
  if (phases & kPhReflect) house_reflect<C, kQrThreads>(X, Hv, beta, p, r, red, hv, vl);
  // R (k x r) = the upper trapezoid of X; written before X is reused for Q
  double* Ur = U + t.u_off;
  double* Ui = U + t.u_off + u_plane;
  double* Vr = Vt + t.vt_off;
  double* Vi = Vt + t.vt_off + vt_plane;
  if (phases & kPhInit) {
  for (int64_t e = tid; e < (int64_t)k * r; e += kQrThreads) {
    const int i = (int)(e % k), c = (int)(e / k);
    const double rr = scale * (i <= c ? X.r(i, c) : 0.0);
    const double ri = (C && i <= c) ? scale * X.m(i, c) : 0.0;
    if (!right) {  // V^dagger (k x n) = R
      Vr[i + (int64_t)c * k] = rr;
      if (C) Vi[i + (int64_t)c * k] = ri;
    } else {  // U (m x k) = R^H: U[c, i] = conj(R[i, c])
      Ur[c + (int64_t)i * m] = rr;
      if (C) Ui[c + (int64_t)i * m] = -ri;
    }
  }
  for (int i = tid; i < k; i += kQrThreads) S[t.s_off + i] = 1.0;
  __syncthreads();
  // Q (p x k) in X's storage: [I; 0], then H_{k-1} .. H_0 applied to columns j..
  for (int64_t e = tid; e < (int64_t)p * k; e += kQrThreads) {
    const int i = (int)(e % p), c = (int)(e / p);
    X.r(i, c) = i == c ? 1.0 : 0.0;
    if (C) X.m(i, c) = 0.0;
  }
  __syncthreads();
  }
  if (phases & kPhApply) house_apply<C, kQrThreads>(X, k, true, Hv, beta, p, k, vl);
  if (!(phases & kPhOut)) return;
  for (int64_t e = tid; e < (int64_t)p * k; e += kQrThreads) {
    const int i = (int)(e % p), c = (int)(e / p);
    if (!right) {  // U (m x k) = Q
      Ur[i + (int64_t)c * m] = X.r(i, c);
      if (C) Ui[i + (int64_t)c * m] = X.m(i, c);
    } else {  // V^dagger (k x n) = Q^H: Vt[c, i] = conj(Q[i, c])
      Vr[c + (int64_t)i * k] = X.r(i, c);
      if (C) Vi[c + (int64_t)i * k] = -X.m(i, c);
    }
  }
}

// ---------------------------------------------------------------------------
// Multi-workgroup Householder reflections for large sectors (p <= kVecRows).
// The one-workgroup kernels above keep a sector on one CU for its whole
// factorisation; here the reflections run in panels of kHp: per panel one
// launch factors the panel's columns (one workgroup per sector,
// house_panel_kernel) and one applies its reflections to the later columns,
// one column per wave held in registers through the kHp reflections, the
// panel's vectors in LDS (house_update_kernel); house_apply_kernel forms
// H_0 ... H_{k-1} Y column by column the same way, every column through all
// reflections in one launch.  Workspace layouts (layout): 0 the SVD's (X, Wm,
// vectors, A, betas; p = max(m, n)), 1 / 2 the QR's left / right (X, vectors,
// betas; p = m / n).  Sector s has its 8-column chunks at
// col_base[s] .. col_base[s + 1] of the grid.
constexpr int kHp = 8;
constexpr int kHcols = kThreads / 64;  // columns per workgroup, one per wave
static_assert(kVecRows == kVecRowsMax, "the host routes sectors of at most kVecRowsMax rows to these kernels");

template <bool C>
struct HView {
  int p, r, k;
  Mat<C> X, Hv;
  double* beta;
};

template <bool C>
__device__ __forceinline__ HView<C> house_view(const SvdTask& t, int layout, double* W, int64_t w_plane) {
  HView<C> v;
  const bool sw = layout == 0 ? t.m < t.n : layout == 2;
  v.p = sw ? t.n : t.m;
  v.r = sw ? t.m : t.n;
  v.k = v.p < v.r ? v.p : v.r;
  const int64_t o_hv = layout == 0 ? (int64_t)v.p * v.r + (int64_t)v.r * v.r : (int64_t)v.p * v.r;
  const int64_t o_b = layout == 0 ? 2 * (int64_t)v.p * v.r + 2 * (int64_t)v.r * v.r
                                  : (int64_t)v.p * v.r + (int64_t)v.p * v.k;
  v.X = Mat<C>{W + t.w_off, W + t.w_off + w_plane, v.p};
  v.Hv = Mat<C>{W + t.w_off + o_hv, W + t.w_off + o_hv + w_plane, v.p};
  v.beta = W + t.w_off + o_b;
  return v;
}

__device__ __forceinline__ int task_of(const int* __restrict__ base, int ntasks, int b) {
  int lo = 0, hi = ntasks - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (base[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// vectors j0 .. j1 - 1 into LDS, rows 0 .. p - 1, zero above row j
template <bool C>
__device__ __forceinline__ void panel_to_lds(const HView<C>& v, int j0, int j1, double* pl) {
  for (int e = threadIdx.x; e < (j1 - j0) * v.p; e += kThreads) {
    const int jj = e / v.p, i = e - jj * v.p, j = j0 + jj;
    pl[jj * kVecRows + i] = i >= j ? v.Hv.r(i, j) : 0.0;
    if (C) pl[(kHp + jj) * kVecRows + i] = i >= j ? v.Hv.m(i, j) : 0.0;
  }
}

// y <- H_j y for the register-held column y (rows lane + 64 q), v_j in LDS
template <bool C>
__device__ __forceinline__ void reflect_regs_full(double* yr, double* yi, const double* pl, int jj, double b, int p,
                                                  int lane) {
  double wr_ = 0.0, wi_ = 0.0;
#pragma unroll
  for (int q = 0; q < kRpl; ++q) {
    const int i = lane + 64 * q;
    if (i < p) {
      const double v_r = pl[jj * kVecRows + i];
      wr_ += v_r * yr[q];
      if (C) {
        const double v_i = pl[(kHp + jj) * kVecRows + i];
        wr_ += v_i * yi[q];
        wi_ += v_r * yi[q] - v_i * yr[q];
      }
    }
  }
  wr_ = wave_sum(wr_);
  if (C) wi_ = wave_sum(wi_);
  const double fr = b * wr_, fi = b * wi_;
#pragma unroll
  for (int q = 0; q < kRpl; ++q) {
    const int i = lane + 64 * q;
    if (i < p) {
      const double v_r = pl[jj * kVecRows + i];
      const double v_i = C ? pl[(kHp + jj) * kVecRows + i] : 0.0;
      yr[q] -= fr * v_r - fi * v_i;
      if (C) yi[q] -= fr * v_i + fi * v_r;
    }
  }
}

template <bool C>
__device__ __forceinline__ void col_load(const HView<C>& v, int c, double* yr, double* yi, int lane) {
#pragma unroll
  for (int q = 0; q < kRpl; ++q) {
    const int i = lane + 64 * q;
    yr[q] = i < v.p ? v.X.r(i, c) : 0.0;
    yi[q] = (C && i < v.p) ? v.X.m(i, c) : 0.0;
  }
}

template <bool C>
__device__ __forceinline__ void col_store(const HView<C>& v, int c, const double* yr, const double* yi, int lane) {
#pragma unroll
  for (int q = 0; q < kRpl; ++q) {
    const int i = lane + 64 * q;
    if (i < v.p) {
      v.X.r(i, c) = yr[q];
      if (C) v.X.m(i, c) = yi[q];
    }
  }
}

// Reflections j0 .. j1 - 1 of the panel's own columns, X's rows j0 .. p - 1
// (at most 64 NQ).  Wave w holds column j0 + w in registers; wave j forms v_j
// and its scalars by itself and leaves v_j in LDS (zero above row j and
// beyond p), so a reflection costs one barrier and no memory.  The chain of
// reflections bounds it: 8 complex columns of up to 128 rows take 8.4 us, 17.8
// when every reflection went through memory with four barriers.
// vl: 2 x 2 planes of 64 NQ doubles, sb: 2.
template <bool C, int NQ>
__device__ __forceinline__ void panel_regs(const HView<C>& v, int j0, int j1, double* vl, double* sb) {
  constexpr int kRows = 64 * NQ;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = j0 + wave, cc = min(c, j1 - 1);  // waves past the panel read its last column
  double xr[NQ], xi[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int i = j0 + lane + 64 * q, ii = min(i, v.p - 1);
    xr[q] = v.X.r(ii, cc);
    xi[q] = C ? v.X.m(ii, cc) : 0.0;
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q)
    if (j0 + lane + 64 * q >= v.p) xr[q] = xi[q] = 0.0;
  for (int j = j0; j < j1; ++j) {
    const int h = j - j0, buf = h & 1;  // buf: read until the barrier after the next one
    double* const wr = vl + buf * 2 * kRows;
    double* const wi = wr + kRows;
    if (c == j) {
      double nn = 0.0;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const double x = q == 0 && lane < h ? 0.0 : xr[q], y = C ? (q == 0 && lane < h ? 0.0 : xi[q]) : 0.0;
        nn += x * x;
        if (C) nn += y * y;
      }
      nn = wave_sum(nn);
      const double x0r = __shfl(xr[0], h, 64), x0i = C ? __shfl(xi[0], h, 64) : 0.0;
      const double nrm = sqrt(nn);
      double ar = 0.0, ai = 0.0, b = 0.0;
      if (nn >= kTinySq) {
        double er, ei;
        const double a0 = head_phase<C>(x0r, x0i, er, ei);
        ar = -er * nrm;
        ai = -ei * nrm;
        b = 1.0 / (nn + a0 * nrm);  // 2 / |v|^2, v = x + e |x| e_0
      }
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const bool above = q == 0 && lane < h, head = q == 0 && lane == h;
        const int i = j0 + lane + 64 * q;
        const double vr = above ? 0.0 : xr[q] - (head ? ar : 0.0), vi = above ? 0.0 : xi[q] - (head ? ai : 0.0);
        wr[lane + 64 * q] = vr;
        if (C) wi[lane + 64 * q] = vi;
        if (!above && i < v.p) {
          v.Hv.r(i, j) = vr;
          v.X.r(i, j) = head ? ar : 0.0;
          if (C) {
            v.Hv.m(i, j) = vi;
            v.X.m(i, j) = head ? ai : 0.0;
          }
        } else if (above) {
          v.X.r(i, j) = xr[q];
          if (C) v.X.m(i, j) = xi[q];
        }
      }
      if (lane == 0) {
        sb[buf] = b;
        v.beta[j] = b;
      }
    }
    lds_barrier();
    if (c > j && c < j1) {
      double dr = 0.0, di = 0.0;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const double vr = wr[lane + 64 * q], vi = C ? wi[lane + 64 * q] : 0.0;
        dr += vr * xr[q];
        if (C) {
          dr += vi * xi[q];
          di += vr * xi[q] - vi * xr[q];  // conj(v) x
        }
      }
      const double b = sb[buf];
      dr = b * wave_sum(dr);
      if (C) di = b * wave_sum(di);
      if (C && NQ > 8) asm volatile("" ::: "memory");  // v read again: held, it would spill
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const double vr = wr[lane + 64 * q], vi = C ? wi[lane + 64 * q] : 0.0;
        xr[q] -= dr * vr - (C ? di * vi : 0.0);
        if (C) xi[q] -= dr * vi + di * vr;
      }
    }
  }
}

template <bool C>
__global__ __launch_bounds__(kThreads) void house_panel_kernel(const SvdTask* __restrict__ tasks, int layout, int j0,
                                                               double* __restrict__ W, int64_t w_plane) {
  __shared__ double vl[4 * kVecRows];
  __shared__ double sb[2];
  const HView<C> v = house_view<C>(tasks[blockIdx.x], layout, W, w_plane);
  if (j0 >= v.k) return;
  const int j1 = min(j0 + kHp, v.k), rows = v.p - j0;
  if (rows <= 128) panel_regs<C, 2>(v, j0, j1, vl, sb);
  else if (rows <= 256) panel_regs<C, 4>(v, j0, j1, vl, sb);
  else panel_regs<C, kRpl>(v, j0, j1, vl, sb);
}

template <bool C>
__global__ __launch_bounds__(kThreads) void house_update_kernel(const SvdTask* __restrict__ tasks, int ntasks,
                                                                const int* __restrict__ col_base, int layout, int j0,
                                                                double* __restrict__ W, int64_t w_plane) {
  __shared__ double pl[(C ? 2 : 1) * kHp * kVecRows];
  const int s = task_of(col_base, ntasks, blockIdx.x);
  const HView<C> v = house_view<C>(tasks[s], layout, W, w_plane);
  const int c0 = (blockIdx.x - col_base[s]) * kHcols;
  if (j0 >= v.k) return;
  const int j1 = min(j0 + kHp, v.k);
  if (c0 + kHcols <= j1 || c0 >= v.r) return;  // no column of this workgroup is after the panel
  panel_to_lds<C>(v, j0, j1, pl);
  __syncthreads();
  const int lane = threadIdx.x & 63, c = c0 + (threadIdx.x >> 6);
  if (c < j1 || c >= v.r) return;
  double yr[kRpl], yi[kRpl];
  col_load<C>(v, c, yr, yi, lane);
  for (int j = j0; j < j1; ++j) {
    const double b = v.beta[j];
    if (b != 0.0) reflect_regs_full<C>(yr, yi, pl, j - j0, b, v.p, lane);
  }
  col_store<C>(v, c, yr, yi, lane);
}

// Y <- H_0 ... H_{k-1} Y on X's first ncols columns (layout 0: all r,
// columns from 0; QR layouts: the k columns of [I; 0], reflection j skipped on
// columns before j, which it leaves unchanged, as LAPACK's xORGQR)
template <bool C>
__global__ __launch_bounds__(kThreads) void house_apply_kernel(const SvdTask* __restrict__ tasks, int ntasks,
                                                               const int* __restrict__ col_base, int layout,
                                                               double* __restrict__ W, int64_t w_plane) {
  __shared__ double pl[(C ? 2 : 1) * kHp * kVecRows];
  const int s = task_of(col_base, ntasks, blockIdx.x);
  const HView<C> v = house_view<C>(tasks[s], layout, W, w_plane);
  const bool from_j = layout != 0;
  const int ncols = from_j ? v.k : v.r;
  const int c0 = (blockIdx.x - col_base[s]) * kHcols;
  if (c0 >= ncols) return;
  const int lane = threadIdx.x & 63, c = c0 + (threadIdx.x >> 6);
  const bool mine = c < ncols;
  double yr[kRpl], yi[kRpl];
  if (mine) col_load<C>(v, c, yr, yi, lane);
  const int cmax = min(c0 + kHcols, ncols) - 1;
  for (int j0 = ((v.k - 1) / kHp) * kHp; j0 >= 0; j0 -= kHp) {
    if (from_j && cmax < j0) continue;  // uniform: every column here is before the panel
    const int j1 = min(j0 + kHp, v.k);
    __syncthreads();  // the previous panel's vectors are no longer read
    panel_to_lds<C>(v, j0, j1, pl);
    __syncthreads();
    if (mine)
      for (int j = j1 - 1; j >= j0; --j) {
        const double b = v.beta[j];
        if (b != 0.0 && !(from_j && c < j)) reflect_regs_full<C>(yr, yi, pl, j - j0, b, v.p, lane);
      }
  }
  if (mine) col_store<C>(v, c, yr, yi, lane);
}

hipError_t launch_qr_batched(int cplx, int right, const SvdTask* tasks, int ntasks, const double* M, int64_t m_plane,
                             double* U, int64_t u_plane, double* Vt, int64_t vt_plane, double* S, double* W,
                             int64_t w_plane, hipStream_t st) {
  if (ntasks <= 0) return hipSuccess;
  if (cplx)
    qr_householder_kernel<true><<<ntasks, kQrThreads, 0, st>>>(tasks, right, M, m_plane, U, u_plane, Vt, vt_plane, S,
                                                               W, w_plane, kPhAll);
  else
    qr_householder_kernel<false><<<ntasks, kQrThreads, 0, st>>>(tasks, right, M, m_plane, U, u_plane, Vt, vt_plane,
                                                                S, W, w_plane, kPhAll);
  return hipGetLastError();
}

hipError_t launch_qr_phase(int cplx, int right, int phases, const SvdTask* tasks, int ntasks, const double* M,
                           int64_t m_plane, double* U, int64_t u_plane, double* Vt, int64_t vt_plane, double* S,
                           double* W, int64_t w_plane, hipStream_t st) {
  if (ntasks <= 0) return hipSuccess;
  if (cplx)
    qr_householder_kernel<true><<<ntasks, kQrThreads, 0, st>>>(tasks, right, M, m_plane, U, u_plane, Vt, vt_plane, S,
                                                               W, w_plane, phases);
  else
    qr_householder_kernel<false><<<ntasks, kQrThreads, 0, st>>>(tasks, right, M, m_plane, U, u_plane, Vt, vt_plane,
                                                                S, W, w_plane, phases);
  return hipGetLastError();
}

hipError_t launch_svd_phase(int cplx, int phases, const SvdTask* tasks, int ntasks, const double* M, int64_t m_plane,
                            double* U, int64_t u_plane, double* Vt, int64_t vt_plane, double* S, double* W,
                            int64_t w_plane, hipStream_t st) {
  if (ntasks <= 0) return hipSuccess;
  if (cplx)
    svd_jacobi_kernel<true><<<ntasks, kThreads, 0, st>>>(tasks, M, m_plane, U, u_plane, Vt, vt_plane, S, W, w_plane,
                                                          kSvdSweeps, phases);
  else
    svd_jacobi_kernel<false><<<ntasks, kThreads, 0, st>>>(tasks, M, m_plane, U, u_plane, Vt, vt_plane, S, W,
                                                           w_plane, kSvdSweeps, phases);
  return hipGetLastError();
}

namespace {
// NQ: the smallest that holds the launch's longest column (an unused column
// segment costs LDS traffic and registers, a branch on it a wait)
template <bool C>
hipError_t block_round(const SvdTask* tasks, int ntasks, const int* pair_base, int npairs, int round, double* W,
                       int64_t w_plane, double* rotated, int rmax, hipStream_t st) {
  static bool attr = false;  // the dynamic LDS limit, raised once
  constexpr size_t kCol = sizeof(double) * (C ? 2 : 1) * kBj;  // bytes of a block's row
  if (!attr) {
    const void* k[2] = {(const void*)svd_block_inner_kernel<C>, (const void*)svd_block_across_kernel<C, 8>};
    for (const void* f : k) {
      const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kCol * kBjMaxR));
      if (e != hipSuccess) return e;
    }
    attr = true;
  }
  if (round < 0)
    svd_block_inner_kernel<C><<<2 * npairs, kThreads, kCol * rmax, st>>>(tasks, ntasks, pair_base, W, w_plane, rotated,
                                                                         rmax);
  else if (rmax <= 64)
    svd_block_across_kernel<C, 1><<<npairs, kThreads, kCol * 64, st>>>(tasks, ntasks, pair_base, round, W, w_plane,
                                                                       rotated);
  else if (rmax <= 128)
    svd_block_across_kernel<C, 2><<<npairs, kThreads, kCol * 128, st>>>(tasks, ntasks, pair_base, round, W, w_plane,
                                                                        rotated);
  else if (rmax <= 256)
    svd_block_across_kernel<C, 4><<<npairs, kThreads, kCol * 256, st>>>(tasks, ntasks, pair_base, round, W, w_plane,
                                                                        rotated);
  else
    svd_block_across_kernel<C, 8><<<npairs, kThreads, kCol * 512, st>>>(tasks, ntasks, pair_base, round, W, w_plane,
                                                                        rotated);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_svd_block_round(int cplx, const SvdTask* tasks, int ntasks, const int* pair_base, int npairs,
                                  int round, double* W, int64_t w_plane, double* rotated, int rmax, hipStream_t st) {
  if (ntasks <= 0 || npairs <= 0) return hipSuccess;
  if (rmax < 1 || rmax > kBjMaxR) return hipErrorInvalidValue;
  if (cplx) return block_round<true>(tasks, ntasks, pair_base, npairs, round, W, w_plane, rotated, rmax, st);
  return block_round<false>(tasks, ntasks, pair_base, npairs, round, W, w_plane, rotated, rmax, st);
}

hipError_t launch_house_panels(int cplx, int layout, const SvdTask* tasks, int ntasks, const int* col_base,
                               int nchunks, int kmax, double* W, int64_t w_plane, hipStream_t st) {
  if (ntasks <= 0 || nchunks <= 0) return hipSuccess;
  for (int j0 = 0; j0 < kmax; j0 += kHp) {
    if (cplx) {
      house_panel_kernel<true><<<ntasks, kThreads, 0, st>>>(tasks, layout, j0, W, w_plane);
      house_update_kernel<true><<<nchunks, kThreads, 0, st>>>(tasks, ntasks, col_base, layout, j0, W, w_plane);
    } else {
      house_panel_kernel<false><<<ntasks, kThreads, 0, st>>>(tasks, layout, j0, W, w_plane);
      house_update_kernel<false><<<nchunks, kThreads, 0, st>>>(tasks, ntasks, col_base, layout, j0, W, w_plane);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_house_apply(int cplx, int layout, const SvdTask* tasks, int ntasks, const int* col_base,
                              int nchunks, double* W, int64_t w_plane, hipStream_t st) {
  if (ntasks <= 0 || nchunks <= 0) return hipSuccess;
  if (cplx)
    house_apply_kernel<true><<<nchunks, kThreads, 0, st>>>(tasks, ntasks, col_base, layout, W, w_plane);
  else
    house_apply_kernel<false><<<nchunks, kThreads, 0, st>>>(tasks, ntasks, col_base, layout, W, w_plane);
  return hipGetLastError();
}

int house_chunks(int m, int n, int layout) {
  const int r = layout == 0 ? (m < n ? m : n) : (layout == 1 ? n : m);
  return (r + kHcols - 1) / kHcols;
}

int svd_block_pairs(int m, int n) {
  const int r = m < n ? m : n;
  const int nb = (r + kBj - 1) / kBj;
  return (nb + (nb & 1)) / 2;
}
int svd_block_rounds(int m, int n) {
  const int r = m < n ? m : n;
  const int nb = (r + kBj - 1) / kBj;
  return nb + (nb & 1) - 1;
}

hipError_t launch_svd_batched(int cplx, const SvdTask* tasks, int ntasks, const double* M, int64_t m_plane,
                              double* U, int64_t u_plane, double* Vt, int64_t vt_plane, double* S, double* W,
                              int64_t w_plane, hipStream_t st, int max_sweeps) {
  if (ntasks <= 0) return hipSuccess;
  if (cplx)
    svd_jacobi_kernel<true><<<ntasks, kThreads, 0, st>>>(tasks, M, m_plane, U, u_plane, Vt, vt_plane, S, W, w_plane,
                                                          max_sweeps, kPhAll);
  else
    svd_jacobi_kernel<false><<<ntasks, kThreads, 0, st>>>(tasks, M, m_plane, U, u_plane, Vt, vt_plane, S, W,
                                                           w_plane, max_sweeps, kPhAll);
  return hipGetLastError();
}

}  // namespace mpsa
