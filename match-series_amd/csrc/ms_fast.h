// FP32-arithmetic kernels for FP32 fields: the SSD energy pass, the SSD variation and the V-cycle
// of the H1 metric. Same launch geometry, partial-sum layout and pair-state protocol as the FP64
// kernels in ms_kernels.h, which FP64 fields keep (they reproduce the reference's arithmetic).
//
// Numerics: the warp and the stencils run in FP32 with fused multiply-adds; energy sums, slopes and
// the step decisions stay FP64 (per-element values enter FP64 accumulators). A deformed quad point
// is computed in grid units relative to its element, e + u with u = quad offset + displacement / h,
// so the local coordinate keeps FP32 precision of the displacement (about 1e-6 px at 10 px) rather
// than of the absolute position (about 6e-5 px at 1023). Division by h becomes a multiplication by
// n - 1 and the Jacobi division by the diagonal a multiplication by its reciprocal.
#pragma once

#include "ms_kernels.h"

namespace msg {

__device__ __forceinline__ float qpxf(int q) { return (q >> 1) ? (float)MSG_QP1 : (float)MSG_QP0; }
__device__ __forceinline__ float qpyf(int q) { return (q & 1) ? (float)MSG_QP1 : (float)MSG_QP0; }
// basis value of dof b at quad point q (compile-time constants once the loops are unrolled)
__device__ __forceinline__ float bqf(int b, int q) { return (float)bq(b, q); }

// One axis of a deformed quad point: the position e + u in grid units (lo = -e, hi = n-1-e relative to the
// element e) clipped to [0, n-1] as transformAndClipCoord does: `fl` is the element hit relative to e and
// `loc` the position in it; `in` is false on a clipped axis. The element hit stays in [0, n-2] for every input
// (med3 takes a NaN to lo); at the upper bound it is the last one, with loc = 1 exactly.
__device__ __forceinline__ void clip_rel(float u, float lo, float hi, float &fl, float &loc, bool &in) {
  in = (u >= lo) && (u < hi);
  const float uc = __builtin_amdgcn_fmed3f(u, lo, hi);
  fl = fminf(floorf(uc), hi - 1.f);
  loc = uc - fl;
}

// Values of the Q1 interpolant of the element's nodal values p at the 4 quad points (q = 2 qx + qy),
// interpolating along x, then y.
__device__ __forceinline__ void quad_values(const float p[4], float v[4]) {
#pragma clang fp contract(fast)
  const float q0 = (float)MSG_QP0, q1 = (float)MSG_QP1;
  const float dx0 = p[1] - p[0], dx1 = p[3] - p[2];
  const float a0 = q0 * dx0 + p[0], a1 = q1 * dx0 + p[0];  // row y = 0 at qx = QP0, QP1
  const float b0 = q0 * dx1 + p[2], b1 = q1 * dx1 + p[2];  // row y = 1
  v[0] = q0 * (b0 - a0) + a0;
  v[1] = q1 * (b0 - a0) + a0;
  v[2] = q0 * (b1 - a1) + a1;
  v[3] = q1 * (b1 - a1) + a1;
}

// Gathers go through a buffer resource over one image: 32-bit offsets (no 64-bit address arithmetic
// per load), neighbouring nodes merged into one two-dword load, and reads past the image return 0.
// Resource word 3 is the gfx9-family raw-buffer format (32-bit data, no swizzle).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t image_rsrc(const float *p, int count) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), (short)0, count * 4, 0x00020000);
}

// a^T K_loc b of the Q1 stiffness matrix in the difference form of stiff_form, as its edge and
// diagonal sums e and d in FP32; the caller applies their weights 1/6 and 2/6 in FP64 (FP32's 1/6 is
// 3e-8 too large, a bias that every element would share)
__device__ __forceinline__ void stiff_parts_f(const float a[4], const float b[4], float &e, float &d) {
#pragma clang fp contract(fast)
  const float ea0 = a[0] - a[1], ea1 = a[0] - a[2], ea2 = a[1] - a[3], ea3 = a[2] - a[3];
  const float da0 = a[0] - a[3], da1 = a[1] - a[2];
  const float eb0 = b[0] - b[1], eb1 = b[0] - b[2], eb2 = b[1] - b[3], eb3 = b[2] - b[3];
  const float db0 = b[0] - b[3], db1 = b[1] - b[2];
  e = ea0 * eb0 + ea1 * eb1 + ea2 * eb2 + ea3 * eb3;
  d = da0 * db0 + da1 * db1;
}

// One axis of a deformed quad point for the energy's value: the position e + u clamped to the grid,
// [0, n-1] in grid units (lo = -e, hi = n-1-e), as element offset `off` from e and local coordinate
// `loc`. At the upper bound the element is the last node's (offset hi, loc 0) and the bilinear form
// returns that node's value exactly -- the interpolant's value there, which the reference's clip to
// width - eps reaches to rounding; the variation keeps clip_rel, which also reports a clipped axis.
// NaN clamps to the lower bound, so the node index stays in [0, n-1].
__device__ __forceinline__ void clamp_rel(float u, float lo, float hi, int &off, float &loc) {
  const float uc = fminf(fmaxf(u, lo), hi);
  const float fl = floorf(uc);
  off = (int)fl;
  loc = uc - fl;
}

// The 4 nodal values of T around byte offset vo (reads past the image return 0); the upper row's loads take
// the row pitch as their scalar offset.
__device__ __forceinline__ void gather4(__amdgpu_buffer_rsrc_t T, unsigned vo, int n, float t[4]) {
  const unsigned pitch = (unsigned)n * 4u;
  auto ld = [&](unsigned extra, unsigned so) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(T, vo + extra, so, 0));
  };
  t[0] = ld(0u, 0u);
  t[1] = ld(4u, 0u);
  t[2] = ld(0u, pitch);
  t[3] = ld(4u, pitch);
}
__device__ __forceinline__ float bilin(const float t[4], float lx, float ly) {
#pragma clang fp contract(fast)
  const float a = lx * (t[1] - t[0]) + t[0];
  const float b = lx * (t[3] - t[2]) + t[2];
  return ly * (b - a) + a;
}
// bilinear value of T at byte offset vo + (lx, ly) (a value read past the image meets a weight of 0)
__device__ __forceinline__ float bilin_at(__amdgpu_buffer_rsrc_t T, unsigned vo, int n, float lx, float ly) {
  float t[4];
  gather4(T, vo, n, t);
  return bilin(t, lx, ly);
}

// ================================================================================================
// SSD energy pass for up to PLAN_CAND step sizes (k_energy in FP32 arithmetic). Tiles of 64 x 4 RUN
// elements; each thread takes a vertical run of RUN elements, reusing the upper node row of one
// element as the lower row of the next.
// ================================================================================================
// FIDX: byte offsets of the gathers formed in FP32 arithmetic, exact while n^2 <= 2^24 (n <= 4096):
// two fused multiply-adds and one conversion instead of two conversions and integer arithmetic.
template <bool FIDX, int RUN>
__global__ void __launch_bounds__(256)
k_energy_f32(const float *__restrict__ R, const float *__restrict__ T, const float *__restrict__ phi,
             const float *__restrict__ z, const float *__restrict__ dold, int n, double vol,
             const PairState *st, double *__restrict__ part, int ntx, int nty, int npairs) {
#pragma clang fp contract(fast)
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * npairs);
  const int pair = wg / tiles, tile = wg - pair * tiles;
  const int nc = st[pair].ncand;
  if (nc == 0 || st[pair].exact) return;  // uniform across the workgroup (k_energy_exact_f32 takes exact pairs)
  const int dm = st[pair].dirmode;
  // Passes evaluate at most PLAN_CAND step sizes (armijo_plan; 2 for an FP64 re-evaluation, 1 for a
  // plain energy): candidate slots beyond it are never filled.
  constexpr int NC = PLAN_CAND;
  constexpr int NACC = NC + 3;  // E_SSD per candidate; sums of f'Kf, f'Kd, d'Kd
  __shared__ double red[4 * NACC];

  const size_t nn = (size_t)n * n;
  const float *Rp = R + pair * nn, *Tp = T + pair * nn;
  const __amdgpu_buffer_rsrc_t Trs = image_rsrc(Tp, (int)nn);
  const float *px = phi + pair * 2 * nn, *py = px + nn;
  const float *zx = z + pair * 2 * nn, *zy = zx + nn, *ox_ = dold + pair * 2 * nn, *oy_ = ox_ + nn;
  const bool cg = (dm == DIR_CG), use_old = st[pair].cg_old != 0;
  const double beta = st[pair].beta;
  const bool use_dir = (dm != DIR_NONE);
  const float nm1 = (float)(n - 1);
  float tau[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) tau[k] = (k < nc) ? (float)st[pair].cand[k] : 0.f;  // powers of two: exact

  const int ex = (tile % ntx) * EN_TX + (threadIdx.x % EN_TX);
  const int ey0 = (tile / ntx) * (4 * RUN) + (threadIdx.x / EN_TX) * RUN;

  double acc[NACC];
#pragma unroll
  for (int k = 0; k < NACC; ++k) acc[k] = 0.0;

  if (ex < n - 1) {
    // A run's sums in FP32 (a few terms each), converted once: per step size the SSD sum, and the
    // e and d parts of f'Kf, f'Kd, d'Kd
    float ssd[NC], se[3] = {0.f, 0.f, 0.f}, sd[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < NC; ++k) ssd[k] = 0.f;
    // node values of the element, b = x + 2 y: slots 0, 1 the lower row, 2, 3 the upper row
    float f0[4], f1[4], d0[4], d1[4], rn[4];
    auto load_row = [&](int y, int slot) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int g = ex + c + y * n;
        f0[slot + c] = px[g];
        f1[slot + c] = py[g];
        d0[slot + c] = use_dir ? search_dir<float>(zx, ox_, g, cg, use_old, beta) : 0.f;
        d1[slot + c] = use_dir ? search_dir<float>(zy, oy_, g, cg, use_old, beta) : 0.f;
        rn[slot + c] = Rp[g];
      }
    };
    if (ey0 < n - 1) load_row(ey0, 0);
#pragma unroll
    for (int j = 0; j < RUN; ++j) {
      const int ey = ey0 + j;
      if (ey >= n - 1) break;  // uniform across a wave (a wave is one row of 64 elements)
      if (j > 0) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          f0[c] = f0[2 + c];
          f1[c] = f1[2 + c];
          d0[c] = d0[2 + c];
          d1[c] = d1[2 + c];
          rn[c] = rn[2 + c];
        }
      }
      load_row(ey + 1, 2);
      // Positions are linear in the step size: the quad points of phi + tau d sit at u_f + tau u_d
      // (grid units relative to the element), and psi^T K psi of phi + tau d is a quadratic in tau. One
      // interpolation of phi and d per element serves every candidate; positions differ from those of
      // the stored phi + tau d (rounded per node) by that rounding, about 3e-7 px at 10 px.
      float rq[4], ufx[4], ufy[4], udx[4], udy[4];
      quad_values(rn, rq);
      quad_values(f0, ufx);
      quad_values(f1, ufy);
      quad_values(d0, udx);
      quad_values(d1, udy);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        ufx[q] = ufx[q] * nm1 + qpxf(q);
        ufy[q] = ufy[q] * nm1 + qpyf(q);
        udx[q] *= nm1;
        udy[q] *= nm1;
      }
      {
        float e, d;
        stiff_parts_f(f0, f0, e, d);
        se[0] += e;
        sd[0] += d;
        stiff_parts_f(f1, f1, e, d);
        se[0] += e;
        sd[0] += d;
        stiff_parts_f(f0, d0, e, d);
        se[1] += e;
        sd[1] += d;
        stiff_parts_f(f1, d1, e, d);
        se[1] += e;
        sd[1] += d;
        stiff_parts_f(d0, d0, e, d);
        se[2] += e;
        sd[2] += d;
        stiff_parts_f(d1, d1, e, d);
        se[2] += e;
        sd[2] += d;
      }
      // the quad point clamped to [0, n-1] in grid units: lo = -e, hi = n-1-e relative to the element
      const float lox = -(float)ex, hix = (float)(n - 1 - ex), loy = -(float)ey, hiy = (float)(n - 1 - ey);
      const int gbase = ex + ey * n;
      const float base4 = 4.f * (float)gbase, pitch4 = 4.f * (float)n;
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        if (k < nc) {
          float a = 0.f;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float lx, ly;
            unsigned vo;
            if constexpr (FIDX) {
              // med3 clamps; a NaN position gives offset 0 (the conversion's NaN result), in bounds
              const float cx = __builtin_amdgcn_fmed3f(tau[k] * udx[q] + ufx[q], lox, hix);
              const float cy = __builtin_amdgcn_fmed3f(tau[k] * udy[q] + ufy[q], loy, hiy);
              const float fx = floorf(cx), fy = floorf(cy);
              lx = cx - fx;
              ly = cy - fy;
              // 4 (gbase + fx + fy n): integers below 2^26 that are multiples of 4, exact in FP32
              vo = (unsigned)(fy * pitch4 + (fx * 4.f + base4));
            } else {
              int ox, oy;
              clamp_rel(tau[k] * udx[q] + ufx[q], lox, hix, ox, lx);
              clamp_rel(tau[k] * udy[q] + ufy[q], loy, hiy, oy, ly);
              vo = (unsigned)(gbase + ox + oy * n) * 4u;
            }
            const float t = bilin_at(Trs, vo, n, lx, ly) - rq[q];
            a += t * t;
          }
          ssd[k] += a;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < NC; ++k) acc[k] = (double)ssd[k] * (0.125 * vol);  // 1/2 t^2 * quad weight 1/4 * vol
#pragma unroll
    for (int m = 0; m < 3; ++m) acc[NC + m] = (double)se[m] * (1.0 / 6.0) + (double)sd[m] * (2.0 / 6.0);
  }
  const int nblk = tiles;
  block_sum_n<NACC>(acc, red);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NC; ++k)
      if (k < nc) {
        const double taud = st[pair].cand[k];
        part[((size_t)(pair * MAX_CAND + k) * 2 + 0) * nblk + tile] = acc[k];
        part[((size_t)(pair * MAX_CAND + k) * 2 + 1) * nblk + tile] =
            0.5 * (acc[NC] + taud * (2.0 * acc[NC + 1] + taud * acc[NC + 2]));
      }
  }
}

// The same pass in FP64 arithmetic at the stored positions (energy_elem<float>, the pass of FP64 data
// terms on FP32 fields) for the pairs whose control flagged a near-tie step decision (`exact`), on the
// tiles and partial layout of k_energy_f32. Its own kernel so that the FP32 pass keeps its register
// budget; a grid-stride loop over the tiles of the flagged pairs, so that a pass without any costs one
// check per pair.
__global__ void __launch_bounds__(256)
k_energy_exact_f32(const float *__restrict__ R, const float *__restrict__ T, const float *__restrict__ phi,
                   const float *__restrict__ z, const float *__restrict__ dold, int n, double h, int width,
                   const PairState *st, double *__restrict__ part, int ntx, int nty, int npairs) {
  const int tiles = ntx * nty;
  constexpr int NC = 2;  // plan_exact: the step, and 0 for the current position
  // usually no pair is flagged: 64 flags a look, their loads in flight together
  bool any = false;
  for (int p0 = 0; p0 < npairs; p0 += 64) {
    const int q = p0 + (int)(threadIdx.x & 63);
    any |= __any(q < npairs && st[min(q, npairs - 1)].exact && st[min(q, npairs - 1)].ncand);
  }
  if (!any) return;
  const size_t nn = (size_t)n * n;
  const int run = en32_run(n);
  const Div hd = make_div(h);
  for (int pair = 0; pair < npairs; ++pair) {
    if (!st[pair].exact || st[pair].ncand == 0) continue;  // uniform across the workgroup
    const float *Rp = R + pair * nn, *Tp = T + pair * nn;
    const float *px = phi + pair * 2 * nn, *py = px + nn;
    const float *zx = z + pair * 2 * nn, *zy = zx + nn, *ox_ = dold + pair * 2 * nn, *oy_ = ox_ + nn;
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
      const int ex = (tile % ntx) * EN_TX + (threadIdx.x % EN_TX);
      const int ey0 = (tile / ntx) * (4 * run) + (threadIdx.x / EN_TX) * run;
      double acc[2 * NC];
#pragma unroll
      for (int k = 0; k < 2 * NC; ++k) acc[k] = 0.0;
      if (ex < n - 1)
        for (int j = 0; j < run; ++j)
          if (ey0 + j < n - 1)
            energy_elem<float, NC>(Rp, Tp, px, py, zx, zy, ox_, oy_, n, hd, width, st[pair], ex, ey0 + j, acc);
      energy_write_partials<NC>(acc, st[pair].ncand, part, pair, tile, tiles);
    }
  }
}

// ================================================================================================
// SSD variation DE = F_SSD + lambda K phi (k_grad<S, DT_SSD> in FP32 arithmetic).
// ================================================================================================
// Contributions of one element to its 4 nodes (b = x + 2 y), from its nodal positions f0, f1 and reference
// values rn: the force cf and 6 K phi, ck, per dof and component.
template <bool FIDX>
__device__ __forceinline__ void grad_elem_f(__amdgpu_buffer_rsrc_t Trs, int ex, int ey, int n, float nm1, float wv,
                                            const float f0[4], const float f1[4], const float rn[4],
                                            float cf[4][2], float ck[4][2]) {
#pragma clang fp contract(fast)
  float nl[4][2], ox4[4], oy4[4], r4[4];
  quad_values(f0, ox4);
  quad_values(f1, oy4);
  quad_values(rn, r4);
  const float lox = -(float)ex, hix = (float)(n - 1 - ex), loy = -(float)ey, hiy = (float)(n - 1 - ey);
  const int gbase = ex + ey * n;
  const float base4 = 4.f * (float)gbase, pitch4 = 4.f * (float)n;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float fx, fy, lx, ly;
    bool inx, iny;
    clip_rel(ox4[q] * nm1 + qpxf(q), lox, hix, fx, lx, inx);
    clip_rel(oy4[q] * nm1 + qpyf(q), loy, hiy, fy, ly, iny);
    unsigned vo;
    if constexpr (FIDX)  // 4 (gbase + fx + fy n): integers below 2^26 that are multiples of 4, exact in FP32
      vo = (unsigned)(fy * pitch4 + (fx * 4.f + base4));
    else
      vo = (unsigned)(gbase + (int)fx + (int)fy * n) * 4u;
    float t4[4];
    gather4(Trs, vo, n, t4);
    const float diff = bilin(t4, lx, ly) - r4[q];
    // gradient of the bilinear T at the hit, in domain units
    const float ax = t4[1] - t4[0], bx = t4[3] - t4[2];
    const float ay = t4[2] - t4[0], by = t4[3] - t4[1];
    const float gx = (ly * (bx - ax) + ax) * nm1;
    const float gy = (lx * (by - ay) + ay) * nm1;
    nl[q][0] = inx ? gx * diff : 0.f;
    nl[q][1] = iny ? gy * diff : 0.f;
  }
#pragma unroll
  for (int dof = 0; dof < 4; ++dof) {
    float a0 = 0.f, a1 = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      a0 += bqf(dof, q) * nl[q][0];
      a1 += bqf(dof, q) * nl[q][1];
    }
    cf[dof][0] = wv * a0;
    cf[dof][1] = wv * a1;
  }
  // 6 K_loc = [4 -1 -1 -2; -1 4 -2 -1; -1 -2 4 -1; -2 -1 -1 4] applied to the element's dofs. Its
  // rows sum to zero, so row i is sum over j != i of K_ij (f_j - f_i): differences of close values
  // instead of a sum that cancels to the FP32 ulp of f for smooth fields. The integer weights are
  // exact; the factor lambda / 6 is applied in FP64 (FP32's 1/6 carries a 3e-8 bias).
  auto stiff = [&](const float f[4], int c) {
    const float d01 = f[1] - f[0], d02 = f[2] - f[0], d03 = f[3] - f[0];
    const float d12 = f[2] - f[1], d13 = f[3] - f[1], d23 = f[3] - f[2];
    ck[0][c] = -2.f * d03 + (-d02 - d01);
    ck[1][c] = -d13 + (-2.f * d12 + d01);
    ck[2][c] = -d23 + (2.f * d12 + d02);
    ck[3][c] = d23 + (d13 + 2.f * d03);
  };
  stiff(f0, 0);
  stiff(f1, 1);
}

__global__ void __launch_bounds__(256)
k_grad_f32(const float *__restrict__ R, const float *__restrict__ T, const float *__restrict__ phi,
           float *__restrict__ DE, int n, double vol_d, const PairState *st, double lambda_default, int ntx, int nty,
           int npairs) {
#pragma clang fp contract(fast)
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * npairs);
  const int pair = wg / tiles, tile = wg - pair * tiles;
  if (st && !participates(st[pair])) return;
  const double lambda6 = (st ? st[pair].lambda : lambda_default) * (1.0 / 6.0);

  // per dof, component and element (consecutive lanes, consecutive elements: no bank conflicts)
  __shared__ float cf[4][2][GR_NE];  // force contribution
  __shared__ float ck[4][2][GR_NE];  // stiffness contribution

  const size_t nn = (size_t)n * n;
  const float *Rp = R + pair * nn, *Tp = T + pair * nn;
  const __amdgpu_buffer_rsrc_t Trs = image_rsrc(Tp, (int)nn);
  const float *px = phi + pair * 2 * nn, *py = px + nn;
  const int x0 = (tile % ntx) * GR_TX, y0 = (tile / ntx) * GR_TY;
  const float nm1 = (float)(n - 1);
  const float wv = (float)(0.25 * vol_d);  // quad weight * vol

  for (int e = threadIdx.x; e < GR_EX * GR_EY; e += 256) {
    const int ex = x0 - 1 + (e % GR_EX), ey = y0 - 1 + (e / GR_EX);
    if (ex < 0 || ey < 0 || ex >= n - 1 || ey >= n - 1) continue;
    float f0[4], f1[4], rn[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int g = l2g(ex, ey, b, n);
      f0[b] = px[g];
      f1[b] = py[g];
      rn[b] = Rp[g];
    }
    float ef[4][2], ek[4][2];
    grad_elem_f<true>(Trs, ex, ey, n, nm1, wv, f0, f1, rn, ef, ek);
#pragma unroll
    for (int dof = 0; dof < 4; ++dof)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        cf[dof][c][e] = ef[dof][c];
        ck[dof][c][e] = ek[dof][c];
      }
  }
  __syncthreads();
  const int x = x0 + (threadIdx.x % GR_TX), y = y0 + (threadIdx.x / GR_TX);
  if (x >= n || y >= n) return;
  float F0 = 0.f, F1 = 0.f, K0 = 0.f, K1 = 0.f;
#pragma unroll
  for (int ey = y - 1; ey <= y; ++ey)
#pragma unroll
    for (int ex = x - 1; ex <= x; ++ex) {
      if (ex < 0 || ey < 0 || ex >= n - 1 || ey >= n - 1) continue;
      const int e = (ex - (x0 - 1)) + (ey - (y0 - 1)) * GR_EX;
      const int dof = (x - ex) + 2 * (y - ey);
      F0 += cf[dof][0][e];
      F1 += cf[dof][1][e];
      K0 += ck[dof][0][e];
      K1 += ck[dof][1][e];
    }
  float *o = DE + pair * 2 * nn;
  const int i = x + y * n;
  o[i] = (float)(lambda6 * (double)K0 + (double)F0);
  o[nn + i] = (float)(lambda6 * (double)K1 + (double)F1);
}

// The value of the lane to the left (0 in lane 0)
__device__ __forceinline__ float lane_left(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
// a + b, never fused with the product that b may be (as where the products pass through LDS)
__device__ __forceinline__ float add_rounded(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}

// The same variation for launches of GRAD_RUN_NODES nodes and more of grids from GRAD_RUN_GRID^2 on: a wave
// takes 64 element columns and the rows of RUN nodes from below to above; a node's contributions from the element
// column to its left come by a lane shift and those from the row below stay in registers, so there is no LDS and no
// barrier, node rows are loaded once per element row instead of twice, and of the elements only 1/64 (columns) and
// 1/RUN (rows) are worked on twice, where the 32 x 8 tiles take 5 passes of a wave for 4 waves of nodes. Same values
// as k_grad_f32's, bit for bit (a sum of zeros alone may differ in the zero's sign). Bound by vector arithmetic (312
// instructions per element, the tile kernel 417 before its clip and offsets took FP32 forms): 8 pairs of 1024^2,
// 106 us -> 102 us in tiles and 83 us here.
// A run of 7 beat 4 and 5 (87, 86 us: more rows done twice) and 8 (87 us; 16: 100 us, too few waves at the end).
// A wave's run is a chain of 8 elements at 1.6 us each, so small launches are faster in tiles: 512^2 6.9 us (runs
// 12.0), 1024^2 16.4 (18.5), 2 x 1024^2 27.7 (25.1), 4 x 1024^2 49.3 (42.9): runs from 2^21 nodes on. And a run's 63
// columns fit small grids badly (64^2: one node in the second column of waves), tiles of 32 x 8 well, whole calls of
// 2^22 nodes: 8^2 139 us (runs 261), 32^2 73 (128), 64^2 76 (112), 128^2 78 (82), 256^2 78 (81; of 2^23 nodes 130 and
// 126), 512^2 78.5 (77.0; 131 and 119): runs from 512^2 on. (So the tiles never see an image of more than 1024^2; FIDX
// holds to 4096^2.)
constexpr long GRAD_RUN_NODES = 1l << 21;
constexpr int GRAD_RUN_GRID = 512;
constexpr int GRR_TX = 63;  // nodes per wave and row (lane 0 only passes its element on)
constexpr int GRR_RUN = 7;
template <int RUN, bool FIDX>
__global__ void __launch_bounds__(256)
k_grad_run_f32(const float *__restrict__ R, const float *__restrict__ T, const float *__restrict__ phi,
               float *__restrict__ DE, int n, double vol_d, const PairState *st, double lambda_default, int ntx,
               int nty, int npairs) {
#pragma clang fp contract(fast)
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * npairs);
  const int pair = wg / tiles, tile = wg - pair * tiles;
  if (st && !participates(st[pair])) return;
  const double lambda6 = (st ? st[pair].lambda : lambda_default) * (1.0 / 6.0);

  const size_t nn = (size_t)n * n;
  const float *Rp = R + pair * nn, *Tp = T + pair * nn;
  const __amdgpu_buffer_rsrc_t Trs = image_rsrc(Tp, (int)nn);
  const float *px = phi + pair * 2 * nn, *py = px + nn;
  const int lane = threadIdx.x & 63;
  const int x = (tile % ntx) * GRR_TX - 1 + lane;  // element column, and the node stored by lanes 1 to 63
  const int y0 = __builtin_amdgcn_readfirstlane(((tile / ntx) * 4 + (threadIdx.x >> 6)) * RUN);
  if (y0 >= n) return;
  const float nm1 = (float)(n - 1);
  const float wv = (float)(0.25 * vol_d);  // quad weight * vol
  const bool ok = x >= 0 && x < n - 1;
  const int xa = min(max(x, 0), n - 1), xb = min(xa + 1, n - 1);
  float *o0 = DE + pair * 2 * nn, *o1 = o0 + nn;

  // slots 0, 1 the lower node row, 2, 3 the upper row, n* the row after it (loaded one element ahead)
  float f0[4], f1[4], rn[4], g0[2], g1[2], gr[2];
  auto load_row = [&](int y) {
    const int r = min(max(y, 0), n - 1) * n;
    g0[0] = px[r + xa];
    g0[1] = px[r + xb];
    g1[0] = py[r + xa];
    g1[1] = py[r + xb];
    gr[0] = Rp[r + xa];
    gr[1] = Rp[r + xb];
  };
  auto take_row = [&]() {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      f0[2 + c] = g0[c];
      f1[2 + c] = g1[c];
      rn[2 + c] = gr[c];
    }
  };
  load_row(y0 - 1);
  take_row();
  load_row(y0);
  float F[2] = {0.f, 0.f}, K[2] = {0.f, 0.f};  // node (x, ey): the sums of the elements below it
#pragma unroll 1
  for (int j = 0; j <= RUN; ++j) {
    const int ey = y0 - 1 + j;
    if (ey >= n) break;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      f0[c] = f0[2 + c];
      f1[c] = f1[2 + c];
      rn[c] = rn[2 + c];
    }
    take_row();
    load_row(ey + 2);
    float ef[4][2], ek[4][2];
    if (ey >= 0 && ey < n - 1 && ok) {
      grad_elem_f<FIDX>(Trs, x, ey, n, nm1, wv, f0, f1, rn, ef, ek);
    } else {
#pragma unroll
      for (int dof = 0; dof < 4; ++dof)
#pragma unroll
        for (int c = 0; c < 2; ++c) ef[dof][c] = ek[dof][c] = 0.f;
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      F[c] = add_rounded(add_rounded(F[c], lane_left(ef[1][c])), ef[0][c]);
      K[c] = add_rounded(add_rounded(K[c], lane_left(ek[1][c])), ek[0][c]);
    }
    if (j > 0 && lane > 0 && x < n) {
      const int i = x + ey * n;
      o0[i] = (float)(lambda6 * (double)K[0] + (double)F[0]);
      o1[i] = (float)(lambda6 * (double)K[1] + (double)F[1]);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      F[c] = add_rounded(lane_left(ef[3][c]), ef[2][c]);
      K[c] = add_rounded(lane_left(ek[3][c]), ek[2][c]);
    }
  }
}

// ================================================================================================
// V-cycle of the H1 metric in FP32 arithmetic (k_mg_down / k_mg_up / k_mg_coarse).
// ================================================================================================
__device__ __forceinline__ void level_consts_f(const PairState *st, int pair, double sigma_default, int n, float &hs,
                                               float &inv_diag) {
  const double sigma = st ? st[pair].sigma : sigma_default;
  const double tau = 0.5 * (sigma * sigma);
  const double s = (double)((n - 1) * (n - 1));
  hs = (float)(tau * s);
  inv_diag = (float)(1.0 / (1 + 4 * tau * s));
}

// A u of the FD heat operator (heat_apply) in FP32. The stencil 4u - (neighbours) is summed as
// differences u - u_nb: hs grows like n^2, and 4u - sum(u_nb) of a smooth field would cancel to a
// few FP32 ulps of u (a 1e-4 relative error of A u at n = 256), while each difference of close
// values is exact.
template <typename Get>
__device__ __forceinline__ float heat_apply_f(const Get &get, int x, int y, int n, float hs) {
#pragma clang fp contract(fast)
  if (n == 1) return get(0, 0);
  const float u = get(x, y);
  const int e = n - 1;
  // Neighbours outside the grid are mirrored inward, so on an edge the inward difference appears
  // twice (u - v) + (u - v) = 2 (u - v) exactly, and every node takes the same branch-free form:
  // interior ((u - r) + (u - l)) + ((u - t) + (u - b)); edge, e.g. y = 0, 2 (u - t) + ((u - r) + (u - l))
  // summed in the other order (FP addition commutes); corner 2 (u - r) + 2 (u - t) = 2 ((u - r) +
  // (u - t)) exactly. A wave covering a grid edge then runs one path instead of three.
  const int xl = x > 0 ? x - 1 : x + 1, xr = x < e ? x + 1 : x - 1;
  const int yb = y > 0 ? y - 1 : y + 1, yt = y < e ? y + 1 : y - 1;
  const float lap = ((u - get(xr, y)) + (u - get(xl, y))) + ((u - get(x, yt)) + (u - get(x, yb)));
  return hs * lap + u;
}

// One Jacobi sweep x + (rhs - A x) / diag on the tile + 1 (rows 1..18, columns 1..TX+2 of the halo tile), in
// heat_apply_f's order of operations.
template <int TX>
__device__ __forceinline__ void mg_sweep_tile1(const MgTile<TX> &t, const float (*sr)[TX + 4], const float (*sx)[TX + 4],
                                               float (*out)[TX + 4], float hs, float idg) {
#pragma clang fp contract(fast)
  auto cell = [&](int r, int lx, int xl, int xr) {
    const int gy = t.y0 + r - 2;
    const int yb = gy > 0 ? r - 1 : r + 1, yt = gy < t.n - 1 ? r + 1 : r - 1;
    const float u = sx[r][lx];
    const float lap = ((u - sx[r][xr]) + (u - sx[r][xl])) + ((u - sx[yt][lx]) + (u - sx[yb][lx]));
    const float au = hs * lap + u;
    out[r][lx] = (sr[r][lx] - au) * idg + u;
  };
#pragma unroll
  for (int k = 0; k < MgTile<TX>::SR; ++k) {
    const int r = 1 + t.g * MgTile<TX>::SR + k;
    if (r < MG_HY - 1 && t.row_in(r)) cell(r, t.tx + 2, t.xl, t.xr);
  }
  // the halo's inner columns: threads of the halo cells with column 1 or TX + 2
  const int c = threadIdx.x & 3;
  if ((c == 1 || c == 2) && t.hr >= 1 && t.hr < MG_HY - 1 && t.halo_in())
    cell(t.hr, t.hc, t.hx > 0 ? t.hc - 1 : t.hc + 1, t.hx < t.n - 1 ? t.hc + 1 : t.hc - 1);
}

// A u at a node of the tile (halo-tile row r)
template <int TX>
__device__ __forceinline__ float mg_heat_tile(const MgTile<TX> &t, const float (*sx)[TX + 4], int r, float hs) {
#pragma clang fp contract(fast)
  const int gy = t.y0 + r - 2, lx = t.tx + 2;
  const int yb = gy > 0 ? r - 1 : r + 1, yt = gy < t.n - 1 ? r + 1 : r - 1;
  const float u = sx[r][lx];
  const float lap = ((u - sx[r][t.xr]) + (u - sx[r][t.xl])) + ((u - sx[yt][lx]) + (u - sx[yb][lx]));
  return hs * lap + u;
}

template <int TX>
__global__ void __launch_bounds__(256)
k_mg_down_f32(const float *__restrict__ rhs, int negate, float *__restrict__ x2out, float *__restrict__ rhsc, int n,
              const PairState *st, double sigma_default, int ntx, int nty, int nfields) {
#pragma clang fp contract(fast)
  typedef MgTile<TX> Tile;
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * nfields);
  const int field = wg / tiles, tile = wg - field * tiles;
  const int pair = field >> 1;
  if (st && !participates(st[pair])) return;
  float hs, idg;
  level_consts_f(st, pair, sigma_default, n, hs, idg);

  __shared__ float sr[MG_HY][Tile::HX];  // rhs on tile+2
  __shared__ float s1[MG_HY][Tile::HX];  // x1 on tile+2
  __shared__ float s2[MG_HY][Tile::HX];  // x2 on tile+1
  __shared__ float sres[MG32_TY][TX];      // residual on tile
  const Tile t(tile, ntx, n);
  const float *rp = rhs + field * (size_t)n * n;
  const float sg = negate ? -1.f : 1.f;

  // every load issued before the first is used (clamped indices; cells outside the grid are not stored)
  float hv[Tile::LR];
#pragma unroll
  for (int k = 0; k < Tile::LR; ++k) hv[k] = rp[t.at(t.g * Tile::LR + k)];
  const float hh = rp[t.halo_at()];
#pragma unroll
  for (int k = 0; k < Tile::LR; ++k) {
    const int r = t.g * Tile::LR + k;
    if (r < MG_HY && t.row_in(r)) {
      const float v = sg * hv[k];
      sr[r][t.tx + 2] = v;
      s1[r][t.tx + 2] = v * idg;  // first Jacobi sweep from zero
    }
  }
  if (t.halo_in()) {
    const float v = sg * hh;
    sr[t.hr][t.hc] = v;
    s1[t.hr][t.hc] = v * idg;
  }
  __syncthreads();
  mg_sweep_tile1<TX>(t, sr, s1, s2, hs, idg);
  __syncthreads();
  float *xo = x2out + field * (size_t)n * n + (size_t)t.y0 * n + t.x0 + t.tx;
#pragma unroll
  for (int k = 0; k < MG32_TY / Tile::G; ++k) {
    const int r = t.g + Tile::G * k;
    sres[r][t.tx] = sr[r + 2][t.tx + 2] - mg_heat_tile<TX>(t, s2, r + 2, hs);
    xo[(size_t)r * n] = s2[r + 2][t.tx + 2];
  }
  __syncthreads();
  const int nc = n / 2;
  float *rc = rhsc + field * (size_t)nc * nc + (size_t)(t.y0 / 2) * nc + t.x0 / 2;
  for (int i = threadIdx.x; i < (TX / 2) * (MG32_TY / 2); i += 256) {
    const int cx = i % (TX / 2), cy = i / (TX / 2);
    rc[(size_t)cy * nc + cx] =
        0.25f * ((sres[2 * cy][2 * cx] + sres[2 * cy][2 * cx + 1]) + (sres[2 * cy + 1][2 * cx] + sres[2 * cy + 1][2 * cx + 1]));
  }
}

template <int TX>
__global__ void __launch_bounds__(256)
k_mg_up_f32(const float *__restrict__ x2in, const float *__restrict__ xc, const float *__restrict__ rhs, int negate,
            float *__restrict__ xout, int n, const PairState *st, double sigma_default, int ntx, int nty, int nfields,
            const float *__restrict__ dold, double *__restrict__ nrm_part) {
#pragma clang fp contract(fast)
  typedef MgTile<TX> Tile;
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * nfields);
  const int field = wg / tiles, tile = wg - field * tiles;
  const int pair = field >> 1;
  if (st && !participates(st[pair])) return;
  float hs, idg;
  level_consts_f(st, pair, sigma_default, n, hs, idg);

  __shared__ float sx[MG_HY][Tile::HX];  // x on tile+2
  __shared__ float sr[MG_HY][Tile::HX];  // rhs on tile+2
  __shared__ float s3[MG_HY][Tile::HX];  // x3 on tile+1
  __shared__ double red[4 * NORM_TERMS];
  const Tile t(tile, ntx, n);
  const size_t nn = (size_t)n * n;
  const int nc = n / 2;
  const float *x2p = x2in + field * nn, *rp = rhs + field * nn, *xcp = xc + field * (size_t)nc * nc;
  const float sg = negate ? -1.f : 1.f;
  const size_t o0 = field * nn + (size_t)t.y0 * n + t.x0 + t.tx;  // this thread's column of the tile
  constexpr int OUT = MG32_TY / Tile::G;                          // output rows per thread: g + G k

  // every load issued before the first is used (clamped indices; cells outside the grid are not stored);
  // the previous direction at the output nodes among them
  float dprev[OUT];
#pragma unroll
  for (int k = 0; k < OUT; ++k) dprev[k] = 0.f;
  if (nrm_part) {
#pragma unroll
    for (int k = 0; k < OUT; ++k) dprev[k] = dold[o0 + (size_t)(t.g + Tile::G * k) * n];
  }
  float hx2[Tile::LR], hxc[Tile::LR], hr[Tile::LR];
#pragma unroll
  for (int k = 0; k < Tile::LR; ++k) {
    const int r = t.g * Tile::LR + k, gi = t.at(r);
    hx2[k] = x2p[gi];
    hr[k] = rp[gi];
    hxc[k] = xcp[(min(max(t.y0 + r - 2, 0), n - 1) >> 1) * nc + ((t.x0 + t.tx) >> 1)];
  }
  const int gh = t.halo_at();
  const float hh2 = x2p[gh], hhr = rp[gh];
  const float hhc = xcp[(min(max(t.y0 + t.hr - 2, 0), n - 1) >> 1) * nc + (min(max(t.hx, 0), n - 1) >> 1)];
#pragma unroll
  for (int k = 0; k < Tile::LR; ++k) {
    const int r = t.g * Tile::LR + k;
    if (r < MG_HY && t.row_in(r)) {
      sx[r][t.tx + 2] = hx2[k] + hxc[k];
      sr[r][t.tx + 2] = sg * hr[k];
    }
  }
  if (t.halo_in()) {
    sx[t.hr][t.hc] = hh2 + hhc;
    sr[t.hr][t.hc] = sg * hhr;
  }
  __syncthreads();
  mg_sweep_tile1<TX>(t, sr, sx, s3, hs, idg);
  __syncthreads();
  double acc[NORM_TERMS] = {0., 0., 0., 0.};  // <z,z>, <DE,z>, <DE,d_old>, <DE,DE> (DE = the raw input)
#pragma unroll
  for (int k = 0; k < OUT; ++k) {
    const int r = t.g + Tile::G * k;
    const float rv = sr[r + 2][t.tx + 2];
    const float o = (rv - mg_heat_tile<TX>(t, s3, r + 2, hs)) * idg + s3[r + 2][t.tx + 2];
    xout[o0 + (size_t)r * n] = o;
    if (nrm_part) {
      const double od = (double)o, de = (double)(sg * rv);  // the raw input
      acc[0] += od * od;
      acc[1] += de * od;
      acc[2] += de * (double)dprev[k];
      acc[3] += de * de;
    }
  }
  if (nrm_part) {
    block_sum_n<NORM_TERMS>(acc, red);
    if (threadIdx.x == 0)
      for (int q = 0; q < NORM_TERMS; ++q) nrm_part[((size_t)field * NORM_TERMS + q) * tiles + tile] = acc[q];
  }
}

// Whole V-cycle below (and including) a level of at most 64x64 nodes in one workgroup of
// MGC_THREADS threads (k_mg_coarse, one level deeper: FP32 arrays of level 6 and below fit in LDS).
// The Jacobi sweeps write a second buffer instead of updating in place, the residual is restricted as
// it is formed and the prolongation is read on the fly by the first sweep of the up leg, so a level
// costs 3 barriers down and 2 up. Node coordinates come from shifts and masks (a division by the
// runtime level size would cost an integer-division sequence per node).
constexpr int MGC_MAXL_F32 = 6;

__global__ void __launch_bounds__(MGC_THREADS)
k_mg_coarse_f32(const float *__restrict__ rhs, int negate, float *__restrict__ xout, int L, const PairState *st,
                double sigma_default, int nfields, const float *__restrict__ dold, double *__restrict__ nrm_part) {
#pragma clang fp contract(fast)
  const int field = blockIdx.x;
  const int pair = field >> 1;
  if (st && !participates(st[pair])) return;
  const double sigma = st ? st[pair].sigma : sigma_default;
  const double tau = 0.5 * (sigma * sigma);
  __shared__ float X[MGC_OFF[MGC_MAXL_F32 + 1]], B[MGC_OFF[MGC_MAXL_F32 + 1]], Y[1 << (2 * MGC_MAXL_F32)];
  __shared__ double red[(MGC_THREADS / 64) * NORM_TERMS];
  // the levels' constants, formed once while the right-hand side loads (a division in FP64 on the chain
  // of every level and leg otherwise)
  __shared__ float lhs[MGC_MAXL_F32 + 1], lidg[MGC_MAXL_F32 + 1];
  if ((int)threadIdx.x <= L) {
    const int m = 1 << threadIdx.x;
    const double s = (double)((m - 1) * (m - 1));
    lhs[threadIdx.x] = (float)(tau * s);
    lidg[threadIdx.x] = (float)(1.0 / (1 + 4 * tau * s));
  }
  const int n = 1 << L;
  const size_t nn = (size_t)n * n;
  const float *rp = rhs + field * nn;
  const float sg = negate ? -1.f : 1.f;
  constexpr int PER = (1 << (2 * MGC_MAXL_F32)) / MGC_THREADS;  // nodes per thread at the largest level
  {
    float v[PER];  // every load issued before the first LDS store (indices clamped into the field)
#pragma unroll
    for (int k = 0; k < PER; ++k) v[k] = rp[min((int)threadIdx.x + MGC_THREADS * k, (int)nn - 1)];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int i = threadIdx.x + MGC_THREADS * k;
      if (i < (int)nn) B[MGC_OFF[L] + i] = sg * v[k];
    }
  }
  __syncthreads();

  auto consts = [&](int l, float &hs, float &idg) {
    hs = lhs[l];
    idg = lidg[l];
  };

  // Down leg of level l with nthr threads (thread tid): two Jacobi sweeps from zero, the second kept
  // in X for the up leg, then the residual restricted to level l - 1.
  auto down_level = [&](int l, int tid, int nthr, auto sync) {
    const int m = 1 << l, mm = m * m, mc = m / 2;
    float hs, idg;
    consts(l, hs, idg);
    float *x = X + MGC_OFF[l];
    const float *b = B + MGC_OFF[l];
    for (int i = tid; i < mm; i += nthr) Y[i] = b[i] * idg;  // first sweep from zero, into Y
    sync();
    auto gy = [&](int gx, int gyy) { return Y[gx + gyy * m]; };
    for (int i = tid; i < mm; i += nthr) x[i] = (b[i] - heat_apply_f(gy, i & (m - 1), i >> l, m, hs)) * idg + Y[i];
    sync();
    auto gx2 = [&](int px, int py) { return x[px + py * m]; };
    for (int i = tid; i < mc * mc; i += nthr) {  // residual at the 4 children of a coarse node, averaged
      const int cx = i & (mc - 1), cy = i >> (l - 1);
      float r[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int fx = 2 * cx + (c & 1), fy = 2 * cy + (c >> 1);
        r[c] = b[fx + fy * m] - heat_apply_f(gx2, fx, fy, m, hs);
      }
      B[MGC_OFF[l - 1] + i] = 0.25f * ((r[0] + r[1]) + (r[2] + r[3]));
    }
    sync();
  };
  // Up leg of level l: the injected coarse correction read on the fly by the first sweep, the
  // second sweep into X.
  auto up_level = [&](int l, int tid, int nthr, auto sync) {
    const int m = 1 << l, mm = m * m, mc = m / 2;
    float hs, idg;
    consts(l, hs, idg);
    float *x = X + MGC_OFF[l];
    const float *xc = X + MGC_OFF[l - 1];
    const float *b = B + MGC_OFF[l];
    auto gp = [&](int px, int py) { return x[px + py * m] + xc[(px >> 1) + (py >> 1) * mc]; };
    for (int i = tid; i < mm; i += nthr) {
      const int px = i & (m - 1), py = i >> l;
      Y[i] = (b[i] - heat_apply_f(gp, px, py, m, hs)) * idg + gp(px, py);
    }
    sync();
    auto gy = [&](int gx, int gyy) { return Y[gx + gyy * m]; };
    for (int i = tid; i < mm; i += nthr) x[i] = (b[i] - heat_apply_f(gy, i & (m - 1), i >> l, m, hs)) * idg + Y[i];
    sync();
  };
  auto block_sync = [] { __syncthreads(); };
  auto wave_sync = [] { mgc_wave_sync(); };
  constexpr int WAVE_LEVELS = MGC_WAVE_LEVELS;
  for (int l = L; l > WAVE_LEVELS; --l) down_level(l, (int)threadIdx.x, MGC_THREADS, block_sync);
  if (threadIdx.x < 64) {
    const int lw = L < WAVE_LEVELS ? L : WAVE_LEVELS;
    for (int l = lw; l >= 1; --l) down_level(l, (int)threadIdx.x, 64, wave_sync);
    if (threadIdx.x == 0) X[0] = B[0];  // 1x1 level: A = 1, the sweeps converge in one step
    wave_sync();
    for (int l = 1; l <= lw; ++l) up_level(l, (int)threadIdx.x, 64, wave_sync);
  }
  __syncthreads();
  for (int l = WAVE_LEVELS + 1; l <= L; ++l) up_level(l, (int)threadIdx.x, MGC_THREADS, block_sync);
  float *xo = xout + field * nn;
  double acc[NORM_TERMS] = {0., 0., 0., 0.};  // <z,z>, <DE,z>, <DE,d_old>, <DE,DE> (DE = the raw input)
  float rv[PER], ov[PER];
  if (nrm_part) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int i = min((int)threadIdx.x + MGC_THREADS * k, (int)nn - 1);
      rv[k] = rp[i];
      ov[k] = dold[field * nn + i];
    }
  }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = threadIdx.x + MGC_THREADS * k;
    if (i < (int)nn) {
      const float o = X[MGC_OFF[L] + i];
      xo[i] = o;
      if (nrm_part) {
        const double od = (double)o, de = (double)rv[k];
        acc[0] += od * od;
        acc[1] += de * od;
        acc[2] += de * (double)ov[k];
        acc[3] += de * de;
      }
    }
  }
  if (nrm_part) {
    block_sum_n<NORM_TERMS, MGC_THREADS>(acc, red);
    if (threadIdx.x == 0)
      for (int t = 0; t < NORM_TERMS; ++t) nrm_part[(size_t)field * NORM_TERMS + t] = acc[t];
  }
}

}  // namespace msg
