// Seismic x-shift registration (matchSeismicSeries): the displacement has an x component only (the
// y component of the field stays zero); the data term is the mean over the image rows of the 1-D
// normalised cross-correlation of the template row shifted by that row of phi_x against the reference
// row (FELineShiftRegisEnergy, registration.h:2137-2193, over NormalizedCrossCorrelationEnergy on the
// row's 1-D grid, registration.h:1909-2018); the regulariser is lambda/2 phi_x^T (K_xx + y K_yy) phi_x
// with y = yRegFactor (findXShift, matchSeries.h:805-868).
//
// One workgroup per (pair, row), each thread a run of consecutive nodes in registers; the template's row
// goes to LDS for the interpolation, and the ends of the warped runs for their neighbours. FP64 arithmetic: the assembled 1-D mass matrix of the 2-point Gauss rule, FastDeformImage with clamping, the
// mass-weighted mean and centred moments. Two reductions per row, whatever the number of candidates: the
// means, then the centred moments and the stiffness forms. The rows' values are summed by the control in a
// fixed order.
#pragma once

#include "ms_kernels.h"

namespace msg {

// Local 1-D mass matrix of one element (2-point rule, weights 1/2) times h: l[0] = L00 = L11, l[1] = L01.
__device__ __forceinline__ void xs_mass_local(double h, double &l00, double &l01, double &l11) {
  double L[2][2] = {{0, 0}, {0, 0}};
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const double xi = q ? MSG_QP1 : MSG_QP0;
    const double b[2] = {1.0 - xi, xi};
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int c = 0; c < 2; ++c) L[a][c] += 0.5 * b[a] * b[c];
  }
  l00 = L[0][0] * h;
  l01 = L[0][1] * h;
  l11 = L[1][1] * h;
}

// (M v)_i of the assembled 1-D mass matrix from the node's value and its neighbours' (unused at the ends)
__device__ __forceinline__ double xs_mass_row(double vl, double v, double vr, int i, int n, double l00, double l01,
                                              double l11) {
  double s = 0, dg = 0;
  if (i > 0) {
    dg += l11;
    s += l01 * vl;
  }
  if (i < n - 1) dg += l00;
  s += dg * v;
  if (i < n - 1) s += l01 * vr;
  return s;
}

// aol::Vector::interpolate (vec.h:461-471)
__device__ __forceinline__ double xs_interp(const double *v, int n, double pos) {
  const int p = (int)pos;
  const double pf = pos - p;
  if (p == n - 1) return v[p];
  return (1 - pf) * v[p] + pf * v[p + 1];
}

// Sums of NV values over a workgroup of TH threads, for every thread; red holds TH / 64 * NV doubles and is
// not reused by the caller.
template <int NV, int TH>
__device__ __forceinline__ void xs_sums(double (&v)[NV], double *red) {
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) red[(threadIdx.x >> 6) * NV + k] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double a = red[k];
#pragma unroll
    for (int w = 1; w < TH / 64; ++w) a += red[w * NV + k];
    v[k] = a;
  }
}

// ================================================================================================
// Energy pass: per (pair, row) and candidate step size, the row's NCC energy (term 0) and the
// regulariser of the element row below it (term 1; psi = phi + tau d at the stored positions), the
// element's form psi^T (K_xx + y K_yy) psi from its differences a, b along x and c, d along y as
// (a^2 + ab + b^2 + y (c^2 + cd + d^2)) / 3. Dynamic LDS: n doubles.
// Two FP64 pairs of 1024^2, three step sizes: 95 us with four reductions per candidate and a division
// per node, 48 us so (FP64 arithmetic and the reductions' latency).
// ================================================================================================
template <typename S, int TH, int PN>
__global__ void __launch_bounds__(TH)
k_energy_xshift(const S *__restrict__ R, const S *__restrict__ T, const S *__restrict__ phi, const S *__restrict__ z,
                const S *__restrict__ dold, int n, double h, double yreg, const PairState *st, double *__restrict__ part,
                int npairs) {
  const int pair = blockIdx.x / n, line = blockIdx.x - pair * n;
  const int nc = st[pair].ncand;
  if (nc == 0) return;  // uniform across the workgroup
  constexpr int NC = PLAN_CAND;
  const int dm = st[pair].dirmode;
  const bool cg = (dm == DIR_CG), use_old = st[pair].cg_old != 0, use_dir = (dm != DIR_NONE);
  const double beta = st[pair].beta;
  extern __shared__ double xs_lds[];
  double *tl = xs_lds;
  __shared__ double ends[NC][2][TH];  // first and last node of every thread's warped run
  __shared__ double red1[TH / 64 * (1 + NC)], red2[TH / 64 * (1 + 3 * NC)];
  const size_t nn = (size_t)n * n, row = (size_t)line * n;
  const S *Rr = R + pair * nn + row, *Tr = T + pair * nn + row;
  const S *px = phi + pair * 2 * nn, *zx = z + pair * 2 * nn, *ox = dold + pair * 2 * nn;
  const bool skip = (Rr[0] != Rr[0]) || (Tr[0] != Tr[0]);  // a row starting with NaN is left out
  const Div hd = make_div(h);
  double l00, l01, l11;
  xs_mass_local(h, l00, l01, l11);
  const int i0 = (int)threadIdx.x * PN;
  const bool below = line < n - 1;
  double tau[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) tau[k] = st[pair].cand[k < nc ? k : 0];

  // this thread's nodes (and the next one's first) of phi and the direction on the two rows, and of R
  S f[2][PN + 1], d[2][PN + 1];
  double r[PN + 2];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int j = 0; j <= PN; ++j) {
      const size_t g = (size_t)min(line + q, n - 1) * n + min(i0 + j, n - 1);
      f[q][j] = px[g];
      d[q][j] = use_dir ? search_dir<S>(zx, ox, g, cg, use_old, beta) : (S)0;
    }
#pragma unroll
  for (int j = 0; j < PN + 2; ++j) r[j] = (double)Rr[min(max(i0 + j - 1, 0), n - 1)];
#pragma unroll
  for (int j = 0; j < PN; ++j)
    if (i0 + j < n) tl[i0 + j] = (double)Tr[i0 + j];
  __syncthreads();

  double s1[1 + NC];  // 1'M r, 1'M t of the candidates
#pragma unroll
  for (int k = 0; k <= NC; ++k) s1[k] = 0;
  double w[NC][PN + 2] = {}, reg[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    reg[k] = 0;
    if (k < nc) {
      double p[2][PN + 1];
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int j = 0; j <= PN; ++j)
          p[q][j] = use_dir ? (double)step_at<S>(f[q][j], tau[k], d[q][j]) : (double)f[q][j];
#pragma unroll
      for (int j = 0; j < PN; ++j) {
        const int i = i0 + j;
        if (i < n) {
          double ds = i + p[0][j] / hd;
          ds = ds < 0 ? 0 : (ds > (double)(n - 1) ? (double)(n - 1) : ds);
          w[k][j + 1] = skip ? 0. : xs_interp(tl, n, ds);
        }
        if (below && i < n - 1) {
          const double a = p[0][j + 1] - p[0][j], b = p[1][j + 1] - p[1][j];
          const double c = p[1][j] - p[0][j], e = p[1][j + 1] - p[0][j + 1];
          reg[k] += ((a * a + a * b + b * b) + yreg * (c * c + c * e + e * e)) * (1.0 / 6.0);
        }
      }
      ends[k][0][threadIdx.x] = w[k][1];
      ends[k][1][threadIdx.x] = w[k][PN];
    }
  }
  // the sums of M v over all nodes: v times the column sums of M
#pragma unroll
  for (int j = 0; j < PN; ++j) {
    const int i = i0 + j;
    if (i < n) {
      const double cs = xs_mass_row(1.0, 1.0, 1.0, i, n, l00, l01, l11);
      s1[0] += cs * r[j + 1];
#pragma unroll
      for (int k = 0; k < NC; ++k)
        if (k < nc) s1[1 + k] += cs * w[k][j + 1];
    }
  }
  xs_sums<1 + NC, TH>(s1, red1);  // its barrier also completes the runs' ends
#pragma unroll
  for (int j = 0; j < PN + 2; ++j) r[j] += -s1[0];
  double s2[1 + 3 * NC];  // u'Mu; per candidate w'Mw, w'Mu, the regulariser
  s2[0] = 0;
#pragma unroll
  for (int j = 0; j < PN; ++j)
    if (i0 + j < n) s2[0] += r[j + 1] * xs_mass_row(r[j], r[j + 1], r[j + 2], i0 + j, n, l00, l01, l11);
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    s2[1 + 3 * k] = s2[2 + 3 * k] = 0;
    s2[3 + 3 * k] = reg[k];
    if (k < nc) {
      w[k][0] = ends[k][1][max((int)threadIdx.x - 1, 0)];
      w[k][PN + 1] = ends[k][0][min((int)threadIdx.x + 1, TH - 1)];
#pragma unroll
      for (int j = 0; j < PN + 2; ++j) w[k][j] += -s1[1 + k];
#pragma unroll
      for (int j = 0; j < PN; ++j)
        if (i0 + j < n) {
          const double m = xs_mass_row(w[k][j], w[k][j + 1], w[k][j + 2], i0 + j, n, l00, l01, l11);
          s2[1 + 3 * k] += w[k][j + 1] * m;
          s2[2 + 3 * k] += r[j + 1] * m;
        }
    }
  }
  xs_sums<1 + 3 * NC, TH>(s2, red2);
  if (threadIdx.x == 0) {
    const double vr = sqrt(s2[0]);
    const double dr = fabs(vr - 0.) < 1e-15 ? 1. : vr;
#pragma unroll
    for (int k = 0; k < NC; ++k)
      if (k < nc) {
        const double vt = sqrt(s2[1 + 3 * k]);
        const double dt = fabs(vt - 0.) < 1e-15 ? 1. : vt;
        part[((size_t)(pair * MAX_CAND + k) * 2 + 0) * n + line] = skip ? 0. : -(s2[2 + 3 * k] / (dt * dr));
        part[((size_t)(pair * MAX_CAND + k) * 2 + 1) * n + line] = s2[3 + 3 * k];
      }
  }
}

// ================================================================================================
// Variation: DE_x = (row derivative of the NCC energy) / n + lambda (K_xx + y K_yy) phi_x, DE_y = 0.
// Row derivative (VariationOfNormalizedCrossCorrelationEnergy / CrossCorrelationForce on the row):
// w = (rn + E tn) / var_t, and at each quad point whose shifted position stays on the row
// -w(x_q) T'(x_q + phi(x_q)), integrated against the two basis functions; an element's two quad points
// once for its two nodes. K_xx = M_y K_x and K_yy = M_x K_y with the 1-D matrices K = [1 -1; -1 1] and
// M = [2 1; 1 2] / 6. Dynamic LDS: n doubles. Two FP64 pairs of
// 1024^2: 66 us with the stencil's entries assembled at every node, 37 us so.
// ================================================================================================
template <typename S, int TH, int PN>
__global__ void __launch_bounds__(TH)
k_grad_xshift(const S *__restrict__ R, const S *__restrict__ T, const S *__restrict__ phi, S *__restrict__ DE, int n,
              double h, double yreg, const PairState *st, double lambda_default, int npairs) {
  const int pair = blockIdx.x / n, line = blockIdx.x - pair * n;
  if (st && !participates(st[pair])) return;  // uniform across the workgroup
  const double lambda = st ? st[pair].lambda : lambda_default;
  extern __shared__ double xs_lds[];
  double *tl = xs_lds;
  __shared__ double ends[2][TH];
  __shared__ double red1[TH / 64 * 2], red2[TH / 64 * 3];
  const size_t nn = (size_t)n * n, row = (size_t)line * n;
  const S *Rr = R + pair * nn + row, *Tr = T + pair * nn + row;
  const S *px = phi + pair * 2 * nn;
  S *o = DE + pair * 2 * nn;
  const bool skip = (Rr[0] != Rr[0]) || (Tr[0] != Tr[0]);
  const Div hd = make_div(h);
  double l00, l01, l11;
  xs_mass_local(h, l00, l01, l11);
  const int i0 = (int)threadIdx.x * PN;

  // phi on the rows above, here and below, from the node before this thread's run to the one after it
  // (clamped: what lies outside the grid gets weight 0), and R's
  double y[3][PN + 2], r[PN + 2];
#pragma unroll
  for (int q = 0; q < 3; ++q)
#pragma unroll
    for (int j = 0; j < PN + 2; ++j)
      y[q][j] = (double)px[(size_t)min(max(line + q - 1, 0), n - 1) * n + min(max(i0 + j - 1, 0), n - 1)];
#pragma unroll
  for (int j = 0; j < PN + 2; ++j) r[j] = (double)Rr[min(max(i0 + j - 1, 0), n - 1)];
  double out[PN];
#pragma unroll
  for (int j = 0; j < PN; ++j) out[j] = 0;

  if (!skip) {  // uniform
#pragma unroll
    for (int j = 0; j < PN; ++j)
      if (i0 + j < n) tl[i0 + j] = (double)Tr[i0 + j];
    __syncthreads();
    double w[PN + 2] = {}, s1[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < PN; ++j) {
      const int i = i0 + j;
      if (i < n) {
        double ds = i + y[1][j + 1] / hd;
        ds = ds < 0 ? 0 : (ds > (double)(n - 1) ? (double)(n - 1) : ds);
        w[j + 1] = xs_interp(tl, n, ds);
        const double cs = xs_mass_row(1.0, 1.0, 1.0, i, n, l00, l01, l11);
        s1[0] += cs * r[j + 1];
        s1[1] += cs * w[j + 1];
      }
    }
    ends[0][threadIdx.x] = w[1];
    ends[1][threadIdx.x] = w[PN];
    xs_sums<2, TH>(s1, red1);  // its barrier also completes the runs' ends
    w[0] = ends[1][max((int)threadIdx.x - 1, 0)];
    w[PN + 1] = ends[0][min((int)threadIdx.x + 1, TH - 1)];
    double s2[3] = {0, 0, 0};
#pragma unroll
    for (int j = 0; j < PN + 2; ++j) {
      r[j] += -s1[0];
      w[j] += -s1[1];
    }
#pragma unroll
    for (int j = 0; j < PN; ++j)
      if (i0 + j < n) {
        const double m = xs_mass_row(w[j], w[j + 1], w[j + 2], i0 + j, n, l00, l01, l11);
        s2[0] += r[j + 1] * xs_mass_row(r[j], r[j + 1], r[j + 2], i0 + j, n, l00, l01, l11);
        s2[1] += w[j + 1] * m;
        s2[2] += r[j + 1] * m;
      }
    xs_sums<3, TH>(s2, red2);
    const double vr = sqrt(s2[0]), vt = sqrt(s2[1]);
    const Div dr = make_div(fabs(vr - 0.) < 1e-15 ? 1. : vr), dt = make_div(fabs(vt - 0.) < 1e-15 ? 1. : vt);
    const double e = -(s2[2] / (dt.d * dr.d));
#pragma unroll
    for (int j = 0; j < PN + 2; ++j) {
      double v = r[j] / dr;
      v += e * (w[j] / dt);
      w[j] = v / dt;
    }
    // element el = i0 - 1 + j: its dof 0 is node j - 1 of the run, its dof 1 node j
#pragma unroll
    for (int j = 0; j <= PN; ++j) {
      const int el = i0 + j - 1;
      if (el < 0 || el > n - 2) continue;
      double a[2] = {0, 0};
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const double xi = q ? MSG_QP1 : MSG_QP0;
        const double offq = (1 - xi) * y[1][j] + xi * y[1][j + 1];
        const double tc = (double)el + xi + offq / hd;
        int tel = (short)tc;
        const double tloc = tc - tel;
        if (tel == n - 1 && tloc == 0) tel = n - 2;
        double nl = 0;
        if (!(tc < 0. || tel < 0 || tel >= n - 1)) {
          const double g = (tl[tel + 1] - tl[tel]) / hd;
          nl = g * -((1 - xi) * w[j] + xi * w[j + 1]);
        }
        a[0] += (1 - xi) * 0.5 * nl;
        a[1] += xi * 0.5 * nl;
      }
      if (j > 0) out[j - 1] += h * a[0];
      if (j < PN) out[j] += h * a[1];
    }
  }
  // (K_xx + y K_yy) phi_x
  const double my[3] = {line > 0 ? 1.0 / 6 : 0., ((line > 0 ? 1 : 0) + (line < n - 1 ? 1 : 0)) * (2.0 / 6),
                        line < n - 1 ? 1.0 / 6 : 0.};
  double ky[PN + 2];  // K_y phi_x per column
#pragma unroll
  for (int j = 0; j < PN + 2; ++j)
    ky[j] = (line > 0 ? y[1][j] - y[0][j] : 0.) + (line < n - 1 ? y[1][j] - y[2][j] : 0.);
#pragma unroll
  for (int j = 0; j < PN; ++j) {
    const int i = i0 + j;
    if (i >= n) continue;
    double s = 0;
#pragma unroll
    for (int q = 0; q < 3; ++q)
      s += my[q] * ((i > 0 ? y[q][j + 1] - y[q][j] : 0.) + (i < n - 1 ? y[q][j + 1] - y[q][j + 2] : 0.));
    double m = ((i > 0 ? 1 : 0) + (i < n - 1 ? 1 : 0)) * (2.0 / 6) * ky[j + 1];
    if (i > 0) m += (1.0 / 6) * ky[j];
    if (i < n - 1) m += (1.0 / 6) * ky[j + 2];
    const double v = out[j] / n + lambda * (s + yreg * m);
    o[row + i] = (S)v;
    o[nn + row + i] = (S)0;
  }
}

}  // namespace msg
