// mfc_pairs.h — the cell window of a particle and the FP64 terms of one pair, shared by the step
// kernels and the reverse mode.
#pragma once

#include "mfc_kernels.h"

namespace mfc {

constexpr int REC_DOUBLES = 16;  // doubles per FP64 neighbour record

// patches of the grid: patch p holds the cell rows [r patch_s, (r + 1) patch_s) and the columns
// [c patch_w, (c + 1) patch_w) with p = c patch_rows + r; the number of them is also the patch of the
// particles sorted past the grid's cells (an adaptive grid's blanked ones)
template <class K>  // dev_consts or kconst
__device__ inline int patch_rows(K &k) { return (k.gny + k.patch_s - 1) / k.patch_s; }
template <class K>
__device__ inline int patch_total(K &k) { return ((k.gnx + k.patch_w - 1) / k.patch_w) * patch_rows(k); }

// a tag: the index of a neighbour's record (storage order) and its flags
constexpr int TAG_BITS = 4;  // FIXED, BLANKED, TOOL, NONFINITE
__device__ inline int make_tag(int index, int flags) { return (int)(((unsigned)index << TAG_BITS) | (unsigned)flags); }
__device__ inline unsigned tag_index(int tag) { return (unsigned)tag >> TAG_BITS; }

// The 5 x 5 cell window around the cell of a particle (interactions_gpu.cu:219-229): up to 5
// columns of the cell grid (clipped to the grid), each a contiguous range of the sorted order.
// The candidates are numbered 0..total-1 column by column in ascending sorted index, which is
// the reference's visiting order; at(t) is the sorted index of candidate t. The ten range
// bounds are loaded together, before any candidate.
struct window {
  int total;
  int c1, c2, c3, c4;      // number of the first candidate of columns 1..4
  int d0;                  // sorted index minus candidate number in column 0
  int e1, e2, e3, e4;      // its change from column r - 1 to column r
  __device__ inline int at(int t) const {
    // sums of selected increments (not a select among the five offsets, which the compiler
    // may turn into an indexed load from private memory)
    return t + d0 + (t >= c1 ? e1 : 0) + (t >= c2 ? e2 : 0) + (t >= c3 ? e3 : 0) + (t >= c4 ? e4 : 0);
  }
};

// the up to 5 column ranges [b, e) of the window of a particle in cell column gi and row gj;
// at(column, row) is the first index of a cell (the last one past the column's end for row gny)
template <class K, class AT>
__device__ inline void window_ranges(K &k, int gi, int gj, const AT &at, int b[5], int e[5]) {
  const int li = gi - 2 < 0 ? 0 : gi - 2;
  const int lj = gj - 2 < 0 ? 0 : gj - 2;
  const int hi = gi + 3 > k.gnx ? k.gnx : gi + 3;
  const int hj = gj + 3 > k.gny ? k.gny : gj + 3;
#pragma unroll
  for (int r = 0; r < 5; r++) {
    const bool in = li + r < hi;
    const int ii = in ? li + r : hi - 1;
    b[r] = at(ii, lj);
    e[r] = at(ii, hj);
    if (!in) e[r] = b[r];
  }
}

// its candidates numbered through the ranges
__device__ inline window window_of(const int b[5], const int e[5]) {
  window w;
  // d_r = b[r] - c_r with c_r the candidates before column r; e_r = d_r - d_(r-1)
  int c = e[0] - b[0];
  w.d0 = b[0];
  w.c1 = c; w.e1 = b[1] - c - w.d0; c += e[1] - b[1];
  w.c2 = c; w.e2 = b[2] - c - (b[1] - w.c1); c += e[2] - b[2];
  w.c3 = c; w.e3 = b[3] - c - (b[2] - w.c2); c += e[3] - b[3];
  w.c4 = c; w.e4 = b[4] - c - (b[3] - w.c3); c += e[4] - b[4];
  w.total = c;
  return w;
}

template <class K, class AT>
__device__ inline window make_window_at(K &k, int gi, int gj, const AT &at) {
  int b[5], e[5];
  window_ranges(k, gi, gj, at, b, e);
  return window_of(b, e);
}


// the window of a particle with cell id hsh over the cell ranges in memory
template <class K>
__device__ inline window make_window(K &k, const int *__restrict__ offsets, int hsh) {
  const int gi = hsh / k.gny, gj = hsh - gi * k.gny;
  return make_window_at(k, gi, gj, [&](int col, int row) { return offsets[col * k.gny + row]; });
}

__device__ inline double bits_to_double(int f) { return __longlong_as_double((long long)f); }
__device__ inline int double_to_bits(double d) { return (int)__double_as_longlong(d); }
__device__ inline bool finite_d(double v) { return !mfcm::is_nan(v) && !mfcm::is_inf(v); }

struct pair_acc {
  double vd0, vd1, vd2, vd3;   // v_der (vx,x vx,y vy,x vy,y)
  double sd0, sd1, sd2, sd3;   // S_der
  double vt0, vt1, xt0, xt1;   // vel_t, pos_t (XSPH)
  double tl;                   // Brookshaw sum
};

// neighbour sums stored per particle as ACC_N arrays of N doubles (structure of arrays, in
// the order vd0..vd3, sd0..sd3, vt0, vt1, xt0, xt1, tl, PSE sum)

__device__ inline void store_acc(double *__restrict__ acc, size_t N, int i, const pair_acc &a, double tpse) {
  acc[0 * N + i] = a.vd0; acc[1 * N + i] = a.vd1; acc[2 * N + i] = a.vd2; acc[3 * N + i] = a.vd3;
  acc[4 * N + i] = a.sd0; acc[5 * N + i] = a.sd1; acc[6 * N + i] = a.sd2; acc[7 * N + i] = a.sd3;
  acc[8 * N + i] = a.vt0; acc[9 * N + i] = a.vt1; acc[10 * N + i] = a.xt0; acc[11 * N + i] = a.xt1;
  acc[12 * N + i] = a.tl; acc[13 * N + i] = tpse;
}

__device__ inline void load_acc(const double *__restrict__ acc, size_t N, int i, pair_acc &a, double &tpse) {
  a.vd0 = acc[0 * N + i]; a.vd1 = acc[1 * N + i]; a.vd2 = acc[2 * N + i]; a.vd3 = acc[3 * N + i];
  a.sd0 = acc[4 * N + i]; a.sd1 = acc[5 * N + i]; a.sd2 = acc[6 * N + i]; a.sd3 = acc[7 * N + i];
  a.vt0 = acc[8 * N + i]; a.vt1 = acc[9 * N + i]; a.xt0 = acc[10 * N + i]; a.xt1 = acc[11 * N + i];
  a.tl = acc[12 * N + i]; tpse = acc[13 * N + i];
}

// a particle's FP64 record as the pair terms read it
struct rec64 {
  double x, y, u, v, rho, vol, Axx, Axy, Ayy, Rxx, Rxy, Ryy, c, T, h;
};

// sqrt of x far from the ends of the exponent range: Goldschmidt's iterations from the hardware's
// estimate of 1 / sqrt(x) and corrections by the exact remainder (P. Markstein, Software division and
// square root using Goldschmidt's algorithms, RNC6, 2004), without scaling and special cases
// around them (correctly rounded)
__device__ inline double root(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double s = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, s, 0.5);
  s = __builtin_fma(s, r, s);
  h = __builtin_fma(h, r, h);
  s = __builtin_fma(__builtin_fma(-s, s, x), h, s);
  return __builtin_fma(__builtin_fma(-s, s, x), h, s);
}
// the same in single precision: the hardware's value (within one unit in the last place), or its
// neighbour where x is beyond the midpoint to it by the sign of the exact remainder (P. Markstein,
// Computation of elementary functions on the IBM RISC System/6000 processor, IBM J. Res. Dev. 34, 1990)
__device__ inline float root32(float x) {
  const float s = __builtin_amdgcn_sqrtf(x);
  const float lo = __uint_as_float(__float_as_uint(s) - 1u), hi = __uint_as_float(__float_as_uint(s) + 1u);
  float t = __builtin_fmaf(-lo, s, x) <= 0.0f ? lo : s;
  return __builtin_fmaf(-hi, s, x) > 0.0f ? hi : t;
}

// the terms of one pair in the body of the neighbour loop of do_interactions_monaghan
// (interactions_gpu.cu:249-326 with cubic_spline kernels.cuh:30-70), in the order and with the
// operations of the reference's sums, given to add (pair_sums adds them up, pair_row keeps them).
// A term that the reference does not add is left out, or 0 in a row: a sum starts at +0 and adding +0
// leaves every value it can take unchanged. FINITE: both records are finite and the pair is in support, so
// the quotients by the same divisor can share its reciprocal (div_by), and quotients and roots of
// kernel values and distances need no scaling. inv_wd = 1 / wdeltap.
template <bool FINITE, class ADD>
__device__ inline void pair_terms(kconst &k, const rec64 &a, bool tool_i, double ta, double h1,
                                  double fourh2, double fac, double inv_wd, const rec64 &b, bool tool_j, ADD &add) {
  const double mass = k.mass;
  auto over = [](double n, double d) { return FINITE ? mfcm::quotient(n, d) : n / d; };
  // cubic spline with h_i
  double w = 0., w_x = 0., w_y = 0.;
  const double xij = a.x - b.x, yij = a.y - b.y;
  const double rr2 = xij * xij + yij * yij;
  if (FINITE || !(rr2 >= fourh2 || rr2 < 1e-8)) {
    double der, val;
    double rad;
    if constexpr (FINITE) rad = k.promote ? root(rr2) : (double)root32((float)rr2);
    else rad = tsqrt(k, rr2);
    double q = rad * h1;
    double num;  // of der: one division for both pieces of the spline
    if (q > 1) {
      double m = 2 - q, m2 = m * m;
      val = 0.25 * m2 * m2 * m2;
      num = -0.75 * m2 * h1;
    } else {
      val = 1 - 1.5 * q * q * (1 - 0.5 * q);
      num = -3.0 * q * (1 - 0.75 * q) * h1;
    }
    der = over(num, rad);
    w = val * fac;
    w_x = der * xij * fac;
    w_y = der * yij * fac;
  }
  if (!tool_i && !tool_j) {
    double fab = FINITE ? div_by(w, k.wdeltap, inv_wd) : w / k.wdeltap;
    fab *= fab;
    fab *= fab;
    const double Rx = fab * (a.Rxx + b.Rxx), Ry = fab * (a.Rxy + b.Rxy), Rz = fab * (a.Ryy + b.Ryy);
    add.strain((b.u - a.u) * w_x * b.vol, (b.u - a.u) * w_y * b.vol, (b.v - a.v) * w_x * b.vol,
               (b.v - a.v) * w_y * b.vol);
    add.stress(mass * (a.Axx + b.Axx + Rx) * w_x, mass * (a.Axy + b.Axy + Ry) * w_y,
               mass * (a.Axy + b.Axy + Ry) * w_x, mass * (a.Ayy + b.Ayy + Rz) * w_y);
    const double vijx = a.u - b.u, vijy = a.v - b.v;
    const double vijposij = vijx * xij + vijy * yij;
    const double rhoij = 0.5 * (a.rho + b.rho);
    if (vijposij < 0.) {
      const double cij = 0.5 * (a.c + b.c);
      const double hij = 0.5 * (a.h + b.h);
      const double muij = (hij * vijposij) / (rr2 + k.av_eta * k.av_eta * hij * hij);
      const double piij = (-k.av_alpha * cij * muij + k.av_beta * muij * muij) / rhoij;
      add.viscosity(-mass * piij * w_x, -mass * piij * w_y);
    }
    const double xs = over(-k.xsph_eps * w * mass, rhoij);
    add.advection(xs * vijx, xs * vijy);
  }
  if (ta != 0.) {  // Brookshaw
    const double rij = FINITE ? root(rr2) : sqrt(rr2);
    if (rij > 1e-8) {
      const double rij1 = over(1., rij);
      const double eijx = FINITE ? div_by(xij, rij, rij1) : xij / rij, eijy = FINITE ? div_by(yij, rij, rij1) : yij / rij;
      add.conduction(2.0 * b.vol * (a.T - b.T) * rij1 * (eijx * w_x + eijy * w_y));
    }
  }
}

// the terms added to a particle's sums
struct pair_sums : pair_acc {
  __device__ inline void strain(double a, double b, double c, double d) { vd0 += a; vd1 += b; vd2 += c; vd3 += d; }
  __device__ inline void stress(double a, double b, double c, double d) { sd0 += a; sd1 += b; sd2 += c; sd3 += d; }
  __device__ inline void viscosity(double a, double b) { vt0 += a; vt1 += b; }
  __device__ inline void advection(double a, double b) { xt0 += a; xt1 += b; }
  __device__ inline void conduction(double a) { tl += a; }
};
// the terms of a pair by themselves
struct pair_row {
  double t[14] = {};  // in the order of ACC_N
  __device__ inline void strain(double a, double b, double c, double d) { t[0] = a; t[1] = b; t[2] = c; t[3] = d; }
  __device__ inline void stress(double a, double b, double c, double d) { t[4] = a; t[5] = b; t[6] = c; t[7] = d; }
  __device__ inline void viscosity(double a, double b) { t[8] = a; t[9] = b; }
  __device__ inline void advection(double a, double b) { t[10] = a; t[11] = b; }
  __device__ inline void conduction(double a) { t[12] = a; }
};

}  // namespace mfc
