// Deformation composition with harmonic extension: ConcatAndSmoothlyExtendDeformations
// (quoc/deformations.h:499-520) and SmoothlyExtendImage (L364-404). The extension solves the
// Q1 Laplace problem with Dirichlet data on the defined nodes by diagonally preconditioned CG
// (PCGInverse, aol/solver.h:264-359; absolute stop on |g|^2 < 1e-16, at most 1000 steps), both
// components in the same launches. All scalar work stays on the device; every kernel of an
// iteration reads the component's `done` flag, so iterations launched past convergence change
// nothing and the host only polls the flags every few iterations.
#pragma once

#include "ms_device.h"

namespace msg {

// r_c = phi1_c(x + phi2(x)) + phi2_c(x) (NaN where x + phi2(x) leaves the grid), the defined mask,
// and the Dirichlet data bc_c = defined ? r_c : 0.
template <typename S>
__global__ void k_compose_init(const S *__restrict__ phi1, const S *__restrict__ phi2, double *__restrict__ bc,
                               unsigned char *__restrict__ defined, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int nn = n * n;
  if (i >= nn) return;
  const int x = i % n, y = i / n;
  const Div h = make_div(1.0 / (double)(n - 1));
  const double dx = x + ld(phi2, i) / h, dy = y + ld(phi2, nn + i) / h;
  const double hi = (double)(n - 1);
  const bool inside = !(dx < 0.0 || dx > hi) && !(dy < 0.0 || dy > hi);
  double r0 = __builtin_nan(""), r1 = __builtin_nan("");
  if (inside) {
    r0 = interp(phi1, n, dx, dy);
    r1 = interp(phi1 + nn, n, dx, dy);
  }
  r0 += ld(phi2, i);
  r1 += ld(phi2, nn + i);
  const bool def = !isnan(r0);
  defined[i] = def ? 1 : 0;
  bc[i] = def ? r0 : 0.;
  bc[nn + i] = def ? r1 : 0.;
}

// The values a stiffness row reads: the 3 x 3 nodes around (x, y), loaded together (indices clamped into
// the grid; stiff_sum leaves out what lies outside), so a row costs one memory round trip.
template <typename Get, typename T>
__device__ __forceinline__ void load_3x3(const Get &get, int x, int y, int n, T (&v)[9]) {
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const int cx = min(max(x + k % 3 - 1, 0), n - 1), cy = min(max(y + k / 3 - 1, 0), n - 1);
    v[k] = get(cx + cy * n);
  }
}

// Assembled Q1 stiffness row of node (x, y) (element contributions in element order, K_loc of the unit
// element) applied to the 3 x 3 values v around it; nodes whose skip flag is set are left out (Dirichlet
// columns removed).
__device__ __forceinline__ double stiff_sum(const double (&v)[9], const unsigned char (&skip)[9], int x, int y, int n) {
  const double kl[4][4] = {{4. / 6, -1. / 6, -1. / 6, -2. / 6},
                           {-1. / 6, 4. / 6, -2. / 6, -1. / 6},
                           {-1. / 6, -2. / 6, 4. / 6, -1. / 6},
                           {-2. / 6, -1. / 6, -1. / 6, 4. / 6}};
  double s = 0;
#pragma unroll
  for (int dy = -1; dy <= 0; ++dy)
#pragma unroll
    for (int dx = -1; dx <= 0; ++dx) {
      const int ex = x + dx, ey = y + dy;
      const bool in = ex >= 0 && ey >= 0 && ex < n - 1 && ey < n - 1;
      const int bi = -dx - 2 * dy;
#pragma unroll
      for (int bj = 0; bj < 4; ++bj) {
        const int k = (dx + 1 + (bj & 1)) + 3 * (dy + 1 + (bj >> 1));
        const double t = s + kl[bi][bj] * v[k];
        s = in && !skip[k] ? t : s;
      }
    }
  return s;
}

// 1 / the diagonal of the assembled row (the elements around the node, 1, 2 or 4, times 4/6)
__device__ __forceinline__ double stiff_inv_diag(int x, int y, int n) {
  const int ne = (x == 0 || x == n - 1 ? 1 : 2) * (y == 0 || y == n - 1 ? 1 : 2);
  return ne == 4 ? 1.0 / (4 * (4.0 / 6.0)) : ne == 2 ? 1.0 / (2 * (4.0 / 6.0)) : 1.0 / (1 * (4.0 / 6.0));
}

// ------------------------------------------------------------------------------------------------
// PCG on the undefined nodes only. The Dirichlet matrix is block diagonal: identity rows on the
// defined nodes D, the masked stiffness K_UU on the undefined nodes U, and the preconditioner is
// the identity on D. On D every CG vector is therefore a scalar multiple of the start residual
// g0 = x0 - bc: g = gam g0, P g = eta g0, d = del g0, x = x0 + xi g0, and its share of every inner
// product is that product of scalars times G0 = |g0|^2. The kernels run over U (a compacted index
// list) and carry the D block as these scalars, so an iteration costs O(|U|) instead of O(n^2).
// The recurrences are the reference's (the oracle's pcgDirichlet) term by term; only the rounding
// of the D block differs (one scaling instead of per-node updates).
//
// Two kernels per iteration k: A forms d_k = beta d_{k-1} - P g (beta from B's partials, every
// workgroup reducing them the same way) and h = K_UU d_k; B takes alpha = <g, P g> / <d, h> and
// updates x, g and P g. d alternates between two buffers (A reads the previous one at stencil
// neighbours while it writes the new one). Workgroup 0 of each component records the scalars for
// the next kernel; a component that meets the stopping rule sets its done flag.
// ------------------------------------------------------------------------------------------------
struct CgState {
  double an;   // <g, P g> of the current iteration
  double spn;  // |g|^2
  double G0;   // |g0|^2 over D
  double gam, eta, del, xi;
  int it;
  int pad;
};

// Sum of cnt partials (every thread of the workgroup gets it; fixed order). Each thread loads a
// contiguous run of 8 before adding, so the loads of a sweep are in flight together.
__device__ __forceinline__ double wg_sum_partials(const double *__restrict__ p, int cnt, double *red) {
  double v = 0;
  for (int i0 = threadIdx.x * 8; i0 < cnt; i0 += 256 * 8) {
    double w[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) w[r] = (i0 + r < cnt) ? p[i0 + r] : 0.;
#pragma unroll
    for (int r = 0; r < 8; ++r) v += w[r];
  }
  __shared__ double out;
  const double s = block_sum<256>(v, red);
  if (threadIdx.x == 0) out = s;
  __syncthreads();
  return out;
}

// The same for two arrays at once, their loads together.
__device__ __forceinline__ void wg_sum_partials2(const double *__restrict__ p, const double *__restrict__ q, int cnt,
                                                 double *red, double (&out)[2]) {
  double v[2] = {0, 0};
  for (int i0 = threadIdx.x * 8; i0 < cnt; i0 += 256 * 8) {
    double w[2][8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int i = i0 + r < cnt ? i0 + r : cnt - 1;
      w[0][r] = p[i];
      w[1][r] = q[i];
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      v[0] += i0 + r < cnt ? w[0][r] : 0.;
      v[1] += i0 + r < cnt ? w[1][r] : 0.;
    }
  }
  __shared__ double both[2];
  block_sum_n<2>(v, red);
  if (threadIdx.x == 0) {
    both[0] = v[0];
    both[1] = v[1];
  }
  __syncthreads();
  out[0] = both[0];
  out[1] = both[1];
}

// Start, from the start value x0 (the result's previous content): on U x = x0, g = K_UU x - rhs with
// rhs = -K bc, P g, d = 0 - P g and the partials of <g,g>, <g,Pg>; on D the partial of |x0 - bc|^2. Grid
// (cdiv(n*n, 256), 2 components).
template <typename S>
__global__ void __launch_bounds__(256)
k_cg_start(const S *__restrict__ x0, const double *__restrict__ bc, const unsigned char *__restrict__ def,
           double *__restrict__ x, double *__restrict__ g, double *__restrict__ hb, double *__restrict__ d,
           double *__restrict__ part, int n, int nblk) {
  __shared__ double red[4 * 3];
  const int nn = n * n;
  const int c = blockIdx.y;
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  double acc[3] = {0, 0, 0};
  if (j < nn) {
    const int k = c * nn + j;
    const double xv = (double)x0[k];
    if (def[j]) {
      const double v = xv - bc[k];
      acc[2] = v * v;
    } else {
      const S *xc = x0 + c * nn;
      const double *bcc = bc + c * nn;
      double xs[9], bs[9];
      unsigned char ds[9], none[9];
      load_3x3([&](int m) { return (double)xc[m]; }, j % n, j / n, n, xs);
      load_3x3([&](int m) { return bcc[m]; }, j % n, j / n, n, bs);
      load_3x3([&](int m) { return def[m]; }, j % n, j / n, n, ds);
#pragma unroll
      for (int q = 0; q < 9; ++q) none[q] = 0;
      const double rhs = -stiff_sum(bs, none, j % n, j / n, n);
      const double gv = stiff_sum(xs, ds, j % n, j / n, n) - rhs;
      const double pv = stiff_inv_diag(j % n, j / n, n) * gv;
      x[k] = xv;
      g[k] = gv;
      hb[k] = pv;
      d[k] = 0.0 - pv;
      acc[0] = gv * gv;
      acc[1] = gv * pv;
    }
  }
  block_sum_n<3>(acc, red);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int t = 0; t < 3; ++t) part[(3 * c + t) * nblk + blockIdx.x] = acc[t];
  }
}

// Scalars of the start, one workgroup per component.
__global__ void k_cg_init(const double *__restrict__ part, int nblk, CgState *__restrict__ sb, int *__restrict__ done) {
  __shared__ double red[4];
  const int c = blockIdx.x;
  const double gg = wg_sum_partials(part + (3 * c + 0) * nblk, nblk, red);
  const double gh = wg_sum_partials(part + (3 * c + 1) * nblk, nblk, red);
  const double G0 = wg_sum_partials(part + (3 * c + 2) * nblk, nblk, red);
  if (threadIdx.x == 0) {
    CgState s;
    s.G0 = G0;
    s.gam = 1.0;   // g = g0 on D
    s.eta = 1.0;   // P g = g0
    s.del = -1.0;  // d = -P g
    s.xi = 0.0;
    s.spn = gg + G0;
    s.an = gh + G0;
    s.it = 0;
    s.pad = 0;
    sb[c] = s;
    done[c] = ((s.spn < 1e-16) || isnan(s.spn)) ? 1 : 0;
  }
}

// Iteration k, part A. Grid (nblkU, 2). Latency-bound: a few dozen workgroups, and every load waits on the
// other XCDs' writes of the kernel before. Two round trips: the flags, scalars, partial sums and the node's
// index, then the 3 x 3 fields around it (before it is known whether the iteration runs). 1024^2 with
// borders of up to 3 pixels undefined: parts A and B 8.0 + 3.7 us with a load after another through the
// row's 16 element nodes, 5.2 + 3.3 us so; a whole composition 771 -> 544 us.
__global__ void __launch_bounds__(256)
k_cg_a(int k, const int *__restrict__ U, int nu, const unsigned char *__restrict__ def,
       const double *__restrict__ dprev, double *__restrict__ dcur, const double *__restrict__ hb,
       double *__restrict__ h2, const double *__restrict__ partb, double *__restrict__ parta, int nblk,
       const CgState *__restrict__ sb, CgState *__restrict__ sa, int *__restrict__ done, int n) {
  __shared__ double red[4 * 2];
  const int c = blockIdx.y;
  const int nn = n * n;
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = nu > 0 ? U[u < nu ? u : 0] : 0;  // lanes past the list load an entry of it
  const int finished = done[c];
  CgState s = sb[c];
  const int x = j % n, y = j / n;
  const double *dp = dprev + c * nn, *hp = hb + c * nn;
  double dv9[9], hv9[9];
  unsigned char ds[9];
  load_3x3([&](int m) { return dp[m]; }, x, y, n, dv9);
  load_3x3([&](int m) { return hp[m]; }, x, y, n, hv9);
  load_3x3([&](int m) { return def[m]; }, x, y, n, ds);
  if (finished) return;
  double beta = 0;
  if (k > 0) {
    // end of iteration k-1: <g, P g>, |g|^2, the stopping rule, then beta and the new direction
    double t[2];
    wg_sum_partials2(partb + (2 * c + 0) * nblk, partb + (2 * c + 1) * nblk, nblk, red, t);
    const double bn = t[0] + (s.gam * s.eta) * s.G0;
    const double spn = t[1] + (s.gam * s.gam) * s.G0;
    beta = bn / s.an;
    s.an = bn;
    s.spn = spn;
    s.del = s.del * beta - s.eta;
  }
  s.it = k;
  if ((s.spn < 1e-16) || (k >= 1000) || isnan(s.spn)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      sa[c] = s;
      done[c] = 1;
    }
    return;
  }
  double dh = 0;
  if (u < nu) {
#pragma unroll
    for (int q = 0; q < 9; ++q) dv9[q] = k > 0 ? dv9[q] * beta - hv9[q] : dv9[q];
    if (k > 0) dcur[c * nn + j] = dv9[4];
    const double hv = stiff_sum(dv9, ds, x, y, n);
    h2[c * nn + j] = hv;
    dh = dv9[4] * hv;
  }
  const double v = block_sum<256>(dh, red);
  if (threadIdx.x == 0) parta[c * nblk + blockIdx.x] = v;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    s.eta = s.del;  // h = A d is d on D
    sa[c] = s;
  }
}

// Iteration k, part B. Grid (nblkU, 2). Its loads as in part A.
__global__ void __launch_bounds__(256)
k_cg_b(const int *__restrict__ U, int nu, double *__restrict__ x, const double *__restrict__ dcur,
       double *__restrict__ g, double *__restrict__ hb, const double *__restrict__ h2,
       const double *__restrict__ parta, double *__restrict__ partb, int nblk, const CgState *__restrict__ sa,
       CgState *__restrict__ sb, const int *__restrict__ done, int n) {
  __shared__ double red[4 * 2];
  const int c = blockIdx.y;
  const int nn = n * n;
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = nu > 0 ? U[u < nu ? u : 0] : 0, k = c * nn + j;
  const int finished = done[c];
  CgState s = sa[c];
  const double xv = x[k], dv = dcur[k], g0 = g[k], hv = h2[k];
  if (finished) return;
  const double ad = wg_sum_partials(parta + c * nblk, nblk, red) + (s.del * s.eta) * s.G0;
  const double alpha = s.an / ad;
  double acc[2] = {0, 0};
  if (u < nu) {
    x[k] = xv + alpha * dv;
    const double gv = g0 + alpha * hv;
    g[k] = gv;
    const double pv = stiff_inv_diag(j % n, j / n, n) * gv;
    hb[k] = pv;
    acc[0] = gv * pv;
    acc[1] = gv * gv;
  }
  block_sum_n<2>(acc, red);
  if (threadIdx.x == 0) {
    partb[(2 * c + 0) * nblk + blockIdx.x] = acc[0];
    partb[(2 * c + 1) * nblk + blockIdx.x] = acc[1];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    s.xi += alpha * s.del;
    s.gam += alpha * s.eta;
    s.eta = s.gam;  // P g on D
    sb[c] = s;
  }
}

// The result in the field type: x on U; on D x0 + xi g0 with g0 = x0 - bc, x0 its previous content.
template <typename D>
__global__ void k_cg_finish(const double *__restrict__ x, const double *__restrict__ bc,
                            const unsigned char *__restrict__ def, const CgState *__restrict__ sb, D *__restrict__ out,
                            int n) {
  const int nn = n * n;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 2 * nn) return;
  const int c = i >= nn ? 1 : 0, j = i - c * nn;
  double v;
  if (def[j]) {
    const double x0 = (double)out[i];
    v = x0 + sb[c].xi * (x0 - bc[i]);
  } else {
    v = x[i];
  }
  out[i] = static_cast<D>(v);
}

// stable list of the undefined nodes (for hipcub::DeviceSelect::If over node indices)
struct UndefinedNode {
  const unsigned char *def;
  __host__ __device__ bool operator()(int j) const { return def[j] == 0; }
};

}  // namespace msg
