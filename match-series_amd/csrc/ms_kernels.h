// gfx950 kernels of the batched registration level solve. S is the storage type of the fields
// (float or double); arithmetic is double. A "pair" is one (reference, template) registration
// problem; pair p's images start at p*n*n and its fields at p*2*n*n.
#pragma once

#include "ms_device.h"
#include "ms_state.h"

namespace msg {

constexpr double TAU_MIN = 9.313225746154785e-10;  // 2^-30 (ArmijoSearch.h:64-73)
constexpr double TAU_MAX = 33554432.0;             // 2^25
constexpr double ARMIJO_SIGMA = 0.5;

// ================================================================================================
// Control: one workgroup per pair reduces the partial sums of the previous pass (fixed order) and
// advances the pair's state machine. Phases:
// ================================================================================================
// PH_NCC_REF0 / PH_NCC_REF1: the reference's mean, then its centred moments (NCC, once per level).
// An accepted step goes to the step slot of its iteration (iterations alternate between two slots);
// the update kernel of that iteration applies it and the next iteration's PH_ARMIJO_INIT clears the
// slot, so no phase of its own is needed after the update.
// PH_ARMIJO_INIT also forms the Fletcher-Reeves coefficient from the V-cycle's partial sums; the CG
// direction itself is never stored before the step: the energy passes and the update form it on
// the fly from z and the previous direction, and the update stores it for the next iteration.
enum CtrlPhase { PH_LEVEL_INIT = 0, PH_ARMIJO_INIT = 2, PH_ARMIJO_STEP = 3, PH_NCC_REF0 = 5, PH_NCC_REF1 = 6 };

constexpr int CTRL_THREADS = 256;  // threads of a control workgroup (a small workgroup finds a free slot sooner)
constexpr int CTRL_MAXT = 16;       // partial arrays one control sweep can reduce

// Sums of NT (<= 8) consecutive partial arrays base[t * len .. t * len + len) in the control
// workgroup, in a fixed order. The partials were just written by a kernel on other XCDs, so a load is
// a memory round trip: 256 threads issue all their loads (CTRL_RUN per array and sweep) before
// summing, from clamped indices with out-of-range values dropped by a select, so none waits for
// another. Each thread's sums go to LDS; 16 threads per array then sum 16 of them each, and one
// thread per array the 16 results -- plain LDS reads and adds (cross-lane shuffles of doubles by 16
// waves at once cost more than the loads). The sums land in out[0 .. NT) (shared memory), valid for
// every thread after the call; red / red2 are the caller's LDS blocks of RED_THREADS and 16 doubles
// per array.
constexpr int CTRL_RUN = 4;
constexpr int RED_THREADS = 256;
template <int NT>
__device__ __forceinline__ void reduce_arrays_n(const double *base, int len, double *out, double (*red)[RED_THREADS],
                                                double (*red2)[16]) {
  const int tid = threadIdx.x;
  if (tid < RED_THREADS) {
    double acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = 0.;
    for (int i0 = 0; i0 < len; i0 += RED_THREADS * CTRL_RUN) {
      double v[NT][CTRL_RUN];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < CTRL_RUN; ++r) {
          const int k = i0 + r * RED_THREADS + tid;
          v[t][r] = base[(size_t)t * len + (k < len ? k : len - 1)];
        }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < CTRL_RUN; ++r) {
          const int k = i0 + r * RED_THREADS + tid;
          acc[t] += (k < len) ? v[t][r] : 0.;
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) red[t][tid] = acc[t];
  }
  __syncthreads();
  if (tid < NT * 16) {
    const int t = tid >> 4, g = tid & 15;
    double a = 0.;
#pragma unroll
    for (int j = 0; j < 16; ++j) a += red[t][16 * g + j];
    red2[t][g] = a;
  }
  __syncthreads();
  if (tid < NT) {
    double a = 0.;
#pragma unroll
    for (int j = 0; j < 16; ++j) a += red2[tid][j];
    out[tid] = a;
  }
  __syncthreads();
}

// NT (<= CTRL_MAXT) arrays, in sweeps of at most 8
template <int NT>
__device__ __forceinline__ void reduce_arrays(const double *base, int len, double *out) {
  __shared__ double red[NT < 8 ? NT : 8][RED_THREADS];
  __shared__ double red2[NT < 8 ? NT : 8][16];
  static_assert(CTRL_THREADS >= RED_THREADS && NT <= CTRL_MAXT, "the reduction's threads are part of the control workgroup");
  if constexpr (NT <= 8) {
    reduce_arrays_n<NT>(base, len, out, red, red2);
  } else {
    reduce_arrays_n<8>(base, len, out, red, red2);
    reduce_arrays_n<NT - 8>(base + (size_t)8 * len, len, out + 8, red, red2);
  }
}

struct CtrlArgs {
  int nblk_energy;   // partial count per candidate and term
  int nblk_norm;     // partials per field and term of the V-cycle's last pass
  double lambda, stop_eps;
  int max_iter;
  int spec;          // candidates per energy pass (1..MAX_CAND)
  int trace_cap;
  int npairs;        // pairs of the batch (NCC: the reference statistics follow the candidates' partials)
  int sigma_fixed;   // 1: filter width fixed at sigma0 (H1GradientDescent, gradientDescent.h:639-650)
  double sigma0;
  int grad_stop;     // 1: USE_GRADIENT_BASED_STOPPING (gradientDescent.h:416)
  int slot;          // step slot of the current iteration (0 or 1)
  double exact_tol;  // > 0 (FP32 SSD passes): relative error bound of an evaluation; decisions whose
                     // margin lies within it are taken on FP64-arithmetic values (0: never)
};
// Partial sums of the V-cycle's last pass, per field and block: <z,z>, <DE,z>, <DE,d_old>, <DE,DE>.
constexpr int NORM_TERMS = 4;

// The search direction at element i: the smoothed gradient z, or the Fletcher-Reeves direction
// d = z + beta d_old (calcTaudAndDescentDir, gradientDescent.h:218-226) as the FP64 sum rounded to S,
// with d_old taken as zero after a fall-back to the gradient.
template <typename S>
__device__ __forceinline__ S search_dir(const S *__restrict__ z, const S *__restrict__ dold, size_t i, bool cg,
                                        bool use_old, double beta) {
  const S zv = z[i];
  if (!cg) return zv;
  const double od = use_old ? (double)dold[i] : 0.0;
  return static_cast<S>((double)zv + beta * od);
}
// The same from values already loaded (z_i, d_old_i); d_old_i is ignored unless use_old.
template <typename S>
__device__ __forceinline__ S search_dir_val(S zv, S ov, bool cg, bool use_old, double beta) {
  if (!cg) return zv;
  const double od = use_old ? (double)ov : 0.0;
  return static_cast<S>((double)zv + beta * od);
}
template <>
__device__ __forceinline__ float search_dir_val<float>(float zv, float ov, bool cg, bool use_old, double beta) {
  const float dv = __fmaf_rn((float)beta, ov, zv);
  return (cg && use_old) ? dv : zv;
}
// FP32 fields: one fused multiply-add in FP32 (the same expression in every kernel that forms d);
// both loads unconditional and the choice a select, so the loads of neighbouring nodes overlap.
template <>
__device__ __forceinline__ float search_dir<float>(const float *__restrict__ z, const float *__restrict__ dold,
                                                   size_t i, bool cg, bool use_old, double beta) {
  const float zv = z[i], ov = dold[i];
  const float dv = __fmaf_rn((float)beta, ov, zv);
  return (cg && use_old) ? dv : zv;
}

// Where the energy pass stores its partial sums. SSD: 2 terms per candidate (E_SSD, E_reg). NCC: 4
// per candidate (1'Mw, w'Mw, w'Mu, E_reg with w = t - c, u = r - m_r) and, after all candidates of
// all pairs, 2 per pair for the reference's statistics.
__device__ __host__ __forceinline__ size_t part_index(int data_term, int pair, int k, int term, int nblk) {
  return ((size_t)(pair * MAX_CAND + k) * (data_term == DT_NCC ? 4 : 2) + term) * nblk;
}
__device__ __host__ __forceinline__ size_t part_index_ref(int npairs, int pair, int term, int nblk) {
  return ((size_t)npairs * MAX_CAND * 4 + (size_t)pair * 2 + term) * nblk;
}
// NCC energy from the moments of one evaluation (NormalizedCrossCorrelationEnergy::computeEnergy,
// registration.h:1953-1964, with normalizeImageForNCC, L1934-1947, written in moments). The template
// t enters shifted, w = t - c, and the reference centred, u = r - m_r, so that no moment cancels:
// s1 = 1'Mw = m_t - c, s2 = w'Mw, s3 = w'Mu; then m_t = c + s1, v_t = sqrt(s2 - s1^2) (1'M1 = 1) and
// (t - m_t)'M(r - m_r) = s3 - s1 * rb with rb = 1'Mu. A deviation within 1e-15 of zero is not divided
// by (appeqAbsolute, aol.h:779-794).
__device__ __host__ __forceinline__ double ncc_value(double s1, double s2, double s3, double rb, double rv,
                                                    double *vt_out) {
  const double vt = sqrt(fmax(s2 - s1 * s1, 0.0));
  *vt_out = vt;
  const double dt = fabs(vt - 0.0) < 1e-15 ? 1.0 : vt;
  const double dr = fabs(rv - 0.0) < 1e-15 ? 1.0 : rv;
  return -((s3 - s1 * rb) / (dt * dr));
}

__device__ __forceinline__ double clampd(double v, double lo, double hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Plan the next energy pass of the Armijo machine: evaluations the sequential algorithm may ask for next
// (at most PLAN_CAND: the first step size with its double and half, or the next three doublings or
// halvings).
constexpr int PLAN_CAND = 3;
static_assert(PLAN_CAND <= MAX_CAND, "a plan fits the pair state's candidate slots");
__device__ __forceinline__ void armijo_plan(PairState &s, int spec) {
  double c[PLAN_CAND];
  int k = 0;
  const double t = s.a_tau;
  if (s.a_phase == AP_FIRST) {
    c[k++] = t;
    c[k++] = 2 * t;
    c[k++] = t > TAU_MIN ? 0.5 * t : t;
  } else if (s.a_phase == AP_GROW) {
    c[k++] = 2 * t;
    c[k++] = 4 * t;
    c[k++] = 8 * t;
  } else {
    double u = t > TAU_MIN ? 0.5 * t : t;
    for (int j = 0; j < 3; ++j) {
      c[k++] = u;
      u = u > TAU_MIN ? 0.5 * u : u;
    }
  }
  if (k > spec) k = spec;
  for (int j = 0; j < k; ++j) s.cand[j] = c[j];
  s.ncand = k;
  s.searching = 1;
  s.passes++;
}

// One energy evaluation: total E, unweighted E_reg and (NCC) the data energy and the warped
// template's mean / deviation.
struct EvalRec {
  double E, R, D, M, V;
  int ex;  // from an FP64-arithmetic pass
};

__device__ __forceinline__ bool armijo_lookup(const PairState &s, double t, EvalRec &ev) {
  for (int j = 0; j < s.ncand; ++j)
    if (s.cand[j] == t) {
      ev = {s.cand_E[j], s.cand_R[j], s.cand_D[j], s.cand_M[j], s.cand_V[j], s.cand_ex};
      return true;
    }
  for (int j = 0; j < 2; ++j)
    if (s.last_tau[j] == t) {
      ev = {s.last_E[j], s.last_R[j], s.last_D[j], s.last_M[j], s.last_V[j], s.last_ex[j]};
      return true;
    }
  return false;
}

__device__ __forceinline__ void armijo_consume(PairState &s, double t, const EvalRec &ev) {
  s.last_tau[1] = s.last_tau[0];
  s.last_E[1] = s.last_E[0];
  s.last_R[1] = s.last_R[0];
  s.last_D[1] = s.last_D[0];
  s.last_M[1] = s.last_M[0];
  s.last_V[1] = s.last_V[0];
  s.last_ex[1] = s.last_ex[0];
  s.last_tau[0] = t;
  s.last_E[0] = ev.E;
  s.last_R[0] = ev.R;
  s.last_D[0] = ev.D;
  s.last_M[0] = ev.M;
  s.last_V[0] = ev.V;
  s.last_ex[0] = ev.ex;
  s.evals++;
}

// A step decision compares E = E(phi + t d) with f = E(phi): Armijo's G >= 1/2, i.e.
// E - f <= 1/2 Df t, and f >= E (ArmijoSearch.h:148-190). With FP32 energy passes (tol > 0) a margin
// within tol (|f| + |E|) of either test could go either way on rounding alone; then both values are
// evaluated again in FP64 arithmetic at the stored positions before deciding.
__device__ __forceinline__ bool needs_exact(const PairState &s, double f, double t, const EvalRec &ev, double tol) {
  if (tol <= 0 || (ev.ex && s.f_ex) || !isfinite(ev.E) || !isfinite(f)) return false;
  const double b = tol * (fabs(f) + fabs(ev.E));
  return fabs(f - ev.E) <= b || fabs((ev.E - f) - ARMIJO_SIGMA * s.a_Df * t) <= b;
}
// Next pass: FP64 arithmetic at step t and, unless f already comes from such a pass at the current
// position (f_ex: consecutive near ties late in a level solve), at 0 (the current position: f).
__device__ __forceinline__ void plan_exact(PairState &s, double t) {
  s.cand[0] = t;
  s.cand[1] = 0.0;
  s.ncand = s.f_ex ? 1 : 2;
  s.exact = 1;
  s.searching = 1;
  s.passes++;
}

__device__ __forceinline__ void armijo_start(PairState &s, int dirmode, double Df, double oldTau) {
  s.dirmode = dirmode;
  s.a_Df = Df;
  s.a_tau = clampd(oldTau, TAU_MIN, TAU_MAX);
  s.a_phase = AP_FIRST;
  s.ncand = 0;
  s.last_tau[0] = s.last_tau[1] = -1.0;
}

// End of an iteration (GradientDescentBase::applySingle L361-439).
__device__ __forceinline__ void finish_iteration(PairState &s, double t, IterTrace *trace, int trace_cap, int pair, int slot) {
  s.step_tau[slot] = t;
  s.step_dir[slot] = s.dirmode;
  double En = s.energy, Rn = s.ereg_new;
  if (t != 0) {
    EvalRec ev;
    if (armijo_lookup(s, t, ev)) {
      En = ev.E;
      s.f_ex = ev.ex;
      Rn = ev.R;
      s.ncc_d = ev.D;  // the NCC variation at the new position needs these
      s.ncc_m = ev.M;
      s.ncc_v = ev.V;
      if (ev.M == ev.M) s.ncc_c = ev.M;  // later moments about the current mean
    } else {
      En = __builtin_nan("");  // cannot happen: the accepted step is one of the last two evaluations
    }
  }
  const double energy = s.energy;
  s.energy_new = En;
  s.ereg_new = Rn;
  s.tau = t;
  const double sigma_used = s.sigma;
  // the norm is of DE at the position the iteration started from (gradientDescent.h:416)
  const double crit = s.grad_stop ? sqrt(s.dd) : energy - En;
  bool stopping = (crit > s.stop_eps) && (s.iter < s.max_iter);
  if (s.sigma_fixed && t == 0) stopping = false;  // L418-422
  if (!s.sigma_fixed && (0.5 * s.sigma > 0.0001) && ((energy - En) < 0.00001)) {
    s.sigma *= 0.5;
    s.tau = 1.;
    stopping = (s.sigma > 0.0001) && (s.iter < s.max_iter);
  }
  if (trace && s.iter - 1 < trace_cap) {
    IterTrace &tr = trace[(size_t)pair * trace_cap + (s.iter - 1)];
    tr.energy = En;
    tr.ereg = Rn;
    tr.tau = t;
    tr.tau_first = s.tau_first;
    tr.sigma = sigma_used;
    tr.evals = s.evals;
    tr.passes = s.passes;
    tr.beta = s.beta;
  }
  s.total_evals += s.evals;
  s.total_passes += s.passes;
  s.energy = En;
  s.active = stopping ? 1 : 0;
  s.searching = 0;
  s.ncand = 0;
}

// Replays getTimestepWidthWithArmijoLineSearch (ArmijoSearch.h:118-200) over the evaluations
// available, including the fall-back to the smoothed gradient (gradientDescent.h:231-235).
__device__ __forceinline__ void armijo_run(PairState &s, int spec, double tol, IterTrace *trace, int trace_cap, int pair, int slot) {
  const double f = s.energy;
  for (int guard = 0; guard < 256; ++guard) {
    double t = s.a_tau;
    EvalRec ev;
    double result = -1;  // >= 0 when the search ends
    if (s.a_phase == AP_FIRST) {
      if (s.a_Df >= 0 || !isfinite(f)) {
        s.evals++;  // the reference evaluates E(tau0) before these checks
        result = 0;
      } else {
        if (!armijo_lookup(s, t, ev)) {
          armijo_plan(s, spec);
          return;
        }
        if (needs_exact(s, f, t, ev, tol)) {
          plan_exact(s, t);
          return;
        }
        armijo_consume(s, t, ev);
        const double E = ev.E;
        const double G = (E - f) / (s.a_Df * t);
        s.a_phase = (G >= ARMIJO_SIGMA && f >= E) ? AP_GROW : AP_SHRINK;
        continue;
      }
    } else if (s.a_phase == AP_GROW) {
      const double tn = t * 2.;
      if (!armijo_lookup(s, tn, ev)) {
        armijo_plan(s, spec);
        return;
      }
      if (needs_exact(s, f, tn, ev, tol)) {
        plan_exact(s, tn);
        return;
      }
      armijo_consume(s, tn, ev);
      const double E = ev.E;
      s.a_tau = tn;
      const double G = (E - f) / (s.a_Df * tn);
      if (G >= ARMIJO_SIGMA && f >= E && tn <= TAU_MAX) continue;
      s.a_tau *= 0.5;
      result = s.a_tau > TAU_MIN ? s.a_tau : 0.;
    } else {  // AP_SHRINK
      const double tn = t > TAU_MIN ? t * 0.5 : t;
      if (!armijo_lookup(s, tn, ev)) {
        armijo_plan(s, spec);
        return;
      }
      if (needs_exact(s, f, tn, ev, tol)) {
        plan_exact(s, tn);
        return;
      }
      armijo_consume(s, tn, ev);
      const double E = ev.E;
      s.a_tau = tn;
      const double G = (E - f) / (s.a_Df * tn);
      if ((!isfinite(E) || (G < ARMIJO_SIGMA || f < E)) && (tn > TAU_MIN)) continue;
      result = tn > TAU_MIN ? tn : 0.;
    }
    // the search ended with `result`
    if (s.dirmode == DIR_CG) {
      s.tau_first = result;
      if (result == 0) {  // not a descent step along the CG direction: retry along the gradient
        s.olddir_zero = 1;
        armijo_start(s, DIR_GRAD, s.Dfz, 0.0);
        s.ncand = 0;
        continue;
      }
    }
    finish_iteration(s, result, trace, trace_cap, pair, slot);
    return;
  }
  finish_iteration(s, 0.0, trace, trace_cap, pair, slot);  // unreachable guard
}

// The first part of armijo_run, at the start of an iteration: no evaluation is known yet (no candidates,
// no last evaluations), so it either plans the first pass or ends without a step.
__device__ __forceinline__ void armijo_begin(PairState &s, int spec, IterTrace *trace, int trace_cap, int pair, int slot) {
  for (;;) {
    if (!(s.a_Df >= 0 || !isfinite(s.energy))) {
      armijo_plan(s, spec);
      return;
    }
    s.evals++;  // the reference evaluates E(tau0) before these checks
    if (s.dirmode != DIR_CG) break;
    s.tau_first = 0;
    s.olddir_zero = 1;
    armijo_start(s, DIR_GRAD, s.Dfz, 0.0);
  }
  finish_iteration(s, 0.0, trace, trace_cap, pair, slot);
}

// Runs one control phase for one pair with the whole workgroup (the reductions need every thread)
// on the workgroup's copy s of the pair state. A kernel per phase and data term: one kernel for all of
// them was 45 KB of code, whose fetches cost more than its arithmetic (5.0 us per phase of one pair at
// 512^2; so, with 4 to 10 KB: 3.7 us at the start of an iteration, 4.6 us per step).
template <int PH, int DT>
__device__ __forceinline__ void control_pair(int pair, PairState &s, const double *__restrict__ part_e,
                             const double *__restrict__ part_n, const CtrlArgs &a, int *__restrict__ flags,
                             IterTrace *__restrict__ trace) {
  __shared__ double sums[CTRL_MAXT];
  const bool participates = s.active && !s.searching;

  if constexpr (PH == PH_NCC_REF0 || PH == PH_NCC_REF1) {
    const int nb = a.nblk_energy;
    reduce_arrays<PH == PH_NCC_REF1 ? 2 : 1>(part_e + part_index_ref(a.npairs, pair, 0, nb), nb, sums);
    const double r1 = sums[0], r2 = PH == PH_NCC_REF1 ? sums[1] : 0;
    if (threadIdx.x == 0) {
      if constexpr (PH == PH_NCC_REF0) {
        s.ncc_rm = r1;  // 1'Mr
      } else {
        s.ncc_rb = r1;  // 1'M(r - m_r)
        s.ncc_rv = sqrt(fmax(r2, 0.0));
        s.ncc_c = s.ncc_rm;  // the first template moments are taken about the reference's mean
      }
    }
  } else if constexpr ((PH == PH_LEVEL_INIT || PH == PH_ARMIJO_STEP) && DT == DT_NCC) {
    const int nc = s.ncand;
    const int nb = a.nblk_energy;
    // candidate k, term t at 4k+t; slots beyond nc hold older values, which nothing reads
    if (nc > 0) reduce_arrays<4 * PLAN_CAND>(part_e + part_index(DT_NCC, pair, 0, 0, nb), nb, sums);
    if (threadIdx.x == 0) {
      for (int k = 0; k < nc; ++k) {
        double vt;
        const double D = ncc_value(sums[4 * k], sums[4 * k + 1], sums[4 * k + 2], s.ncc_rb, s.ncc_rv, &vt);
        double E = 0;
        E += D;
        E += s.lambda * sums[4 * k + 3];  // LinCombOp: (0 + E_NCC) + lambda E_reg
        s.cand_E[k] = E;
        s.cand_R[k] = sums[4 * k + 3];
        s.cand_D[k] = D;
        s.cand_M[k] = s.ncc_c + sums[4 * k];
        s.cand_V[k] = vt;
      }
    }
  } else if constexpr ((PH == PH_LEVEL_INIT || PH == PH_ARMIJO_STEP) && DT == DT_XSHIFT) {
    // rows' NCC energies summed, then divided by the number of rows (FELineShiftRegisEnergy::apply)
    const int nc = s.ncand;
    if (nc > 0) reduce_arrays<2 * PLAN_CAND>(part_e + part_index(DT_SSD, pair, 0, 0, a.nblk_energy), a.nblk_energy, sums);
    if (threadIdx.x == 0) {
      for (int k = 0; k < nc; ++k) {
        double D = sums[2 * k];
        D /= a.nblk_energy;
        double E = 0;
        E += D;
        E += s.lambda * sums[2 * k + 1];
        s.cand_E[k] = E;
        s.cand_R[k] = sums[2 * k + 1];
        s.cand_D[k] = D;
        s.cand_M[k] = s.cand_V[k] = 0;
      }
      s.cand_ex = 0;
    }
  } else if constexpr (PH == PH_LEVEL_INIT || PH == PH_ARMIJO_STEP) {
    const int nc = s.ncand;
    if (nc > 0) reduce_arrays<2 * PLAN_CAND>(part_e + part_index(DT_SSD, pair, 0, 0, a.nblk_energy), a.nblk_energy, sums);
    if (threadIdx.x == 0) {
      for (int k = 0; k < nc; ++k) {
        double E = 0;
        E += sums[2 * k];
        E += s.lambda * sums[2 * k + 1];  // LinCombOp: (0 + E_SSD) + lambda E_reg
        s.cand_E[k] = E;
        s.cand_R[k] = sums[2 * k + 1];
        s.cand_D[k] = s.cand_M[k] = s.cand_V[k] = 0;
      }
      s.cand_ex = s.exact;
      if (s.exact) {  // the value at 0 is the FP64-arithmetic energy of the current position
        for (int k = 0; k < nc; ++k)
          if (s.cand[k] == 0.0) s.energy = s.cand_E[k];
        s.f_ex = 1;
        s.exact = 0;
      }
    }
  }
  if constexpr (PH == PH_LEVEL_INIT || PH == PH_ARMIJO_STEP) {
    if (threadIdx.x == 0) {
      if constexpr (PH == PH_LEVEL_INIT) {
        s.ncc_d = s.cand_D[0];
        s.ncc_m = s.ncc_c = s.cand_M[0];
        s.ncc_v = s.cand_V[0];
        s.energy = s.energy_new = s.energy_start = s.cand_E[0];
        s.ereg_new = s.ereg_start = s.cand_R[0];
        s.tau = 1.0;
        s.sigma = a.sigma_fixed ? a.sigma0 : 1.0;
        s.sigma_fixed = a.sigma_fixed;
        s.grad_stop = a.grad_stop;
        s.dd = 0;
        s.iter = 0;
        s.max_iter = a.max_iter;
        s.stop_eps = a.stop_eps;
        s.active = a.max_iter > 0 ? 1 : 0;
        s.searching = 0;
        s.ncand = 0;
        s.olddir_zero = 1;
        s.zz_old = 0;
        s.total_evals = s.total_passes = 0;
        s.step_tau[0] = s.step_tau[1] = 0;
      } else if (s.searching) {
        armijo_run(s, a.spec, a.exact_tol, trace, a.trace_cap, pair, a.slot);
      }
    }
  } else if constexpr (PH == PH_ARMIJO_INIT) {
    // the previous iteration's update has run (stream order): free its slot
    if (threadIdx.x == 0) s.step_tau[a.slot ^ 1] = 0;
    if (!participates) return;
    // field f, term t at f * NORM_TERMS + t
    reduce_arrays<2 * NORM_TERMS>(part_n + (size_t)(2 * pair) * NORM_TERMS * a.nblk_norm, a.nblk_norm, sums);
    if (threadIdx.x == 0) {
      double zz = 0, Dfz = 0, Dfd = 0;
      zz += sums[0];
      zz += sums[NORM_TERMS];
      Dfz += sums[1];
      Dfz += sums[NORM_TERMS + 1];
      Dfd += sums[2];
      Dfd += sums[NORM_TERMS + 2];
      s.iter += 1;
      s.beta = ((s.iter - 1) % 10) ? (zz / s.zz_old) : 0.0;
      s.zz_old = zz;
      s.evals = 0;
      s.passes = 0;
      // <DE, d> of d = z + beta d_old, or of d = z when the old direction counts as zero
      s.cg_old = s.olddir_zero ? 0 : 1;
      const double Df = s.cg_old ? Dfz + s.beta * Dfd : Dfz;
      s.Df = Df;
      s.Dfz = Dfz;
      if (a.grad_stop) {
        double dd = 0;
        dd += sums[3];
        dd += sums[NORM_TERMS + 3];
        s.dd = dd;
      }
      s.olddir_zero = 0;  // the update stores this iteration's CG direction
      s.tau_first = 0;
      armijo_start(s, DIR_CG, Df, s.tau);
      s.searching = 1;
      armijo_begin(s, a.spec, trace, a.trace_cap, pair, a.slot);
    }
  }
  if (threadIdx.x == 0 && flags) flags[pair] = (s.searching ? 1 : 0) | (s.active ? 2 : 0);
}

template <int PH, int DT>
__global__ void __launch_bounds__(CTRL_THREADS)
k_control(PairState *__restrict__ st, const double *__restrict__ part_e, const double *__restrict__ part_n, CtrlArgs a,
          int *__restrict__ flags, IterTrace *__restrict__ trace) {
  // The state machine runs on an LDS copy of the pair state: one coalesced load and one store
  // instead of a chain of dependent global accesses by the thread that advances it.
  static_assert(sizeof(PairState) % 4 == 0, "pair state copied in 32-bit words");
  constexpr int NW = sizeof(PairState) / 4;
  __shared__ PairState ss;
  const int pair = blockIdx.x;
  unsigned *g = reinterpret_cast<unsigned *>(st + pair), *l = reinterpret_cast<unsigned *>(&ss);
  for (int i = threadIdx.x; i < NW; i += CTRL_THREADS) l[i] = g[i];
  __syncthreads();
  control_pair<PH, DT>(pair, ss, part_e, part_n, a, flags, trace);
  __syncthreads();
  for (int i = threadIdx.x; i < NW; i += CTRL_THREADS) g[i] = l[i];
}



// A pair takes part in a new iteration when it is still iterating and no step search is pending
// (device-driven iterations can leave one open across an iteration boundary); the update of its
// last step has run before (stream order).
__device__ __forceinline__ bool participates(const PairState &s) {
  return s.active && !s.searching;
}


// ================================================================================================
// Energy E(phi + tau d) for up to MAX_CAND step sizes per pair, element-centric.
// SSD part: SSDEnergy::evaluateIntegrand (registration.h:1607-1615) integrated as in
// FENonlinIntegrationVectorInterface::applyAdd (FEOpInterface.h:2586-2613).
// Regularisation part: DisplacementLengthEnergy (hyperelastic.h:178-183) = 1/2 sum_c psi_c^T K psi_c,
// assembled element by element. Output: per block partial sums (ssd, reg) per candidate.
// ================================================================================================
constexpr int EN_TX = 64, EN_TY = 4;  // elements per workgroup tile (one per thread)
// The FP32 SSD pass (k_energy_f32, and its FP64 re-evaluation) takes tiles of 64 x 4 * run elements,
// a vertical run of `run` elements per thread: the workgroup's reduction and partial sums are shared by
// the run, and a run reads run + 1 node rows instead of 2 run. Runs of 4 from 1024^2 up; runs of 2
// below, where a single pair would otherwise give too few workgroups to hide the gathers' latency
// (one pair at 512^2: 8.5 us per pass instead of 11.2 us; at 1024^2 runs of 4 are faster, 21.3 us
// against 22.6). The run depends on the grid size only, so a pair's partial sums do not depend on the
// batch it sits in.
constexpr int EN32_RUN_FROM_1024 = 4, EN32_RUN_BELOW = 2;
__host__ __device__ constexpr int en32_run(int n) { return n >= 1024 ? EN32_RUN_FROM_1024 : EN32_RUN_BELOW; }

// The terms of element (ex, ey) of one pair for each candidate step size, added to accS (SSD) and
// accR (regulariser): FP64 arithmetic at the stored positions (step_at). Used by the FP64 pass and by
// the FP64-arithmetic re-evaluation of the FP32 pass (S = float).
template <typename S, int NC>
__device__ __forceinline__ void energy_elem(const S *__restrict__ Rp, const S *__restrict__ Tp,
                                            const S *__restrict__ px, const S *__restrict__ py,
                                            const S *__restrict__ zx, const S *__restrict__ zy,
                                            const S *__restrict__ ox_, const S *__restrict__ oy_, int n, const Div &h,
                                            int width, const PairState &sp, int ex, int ey, double (&acc)[2 * NC]) {
  const int nc = sp.ncand;
  const int dm = sp.dirmode;
  const bool cg = (dm == DIR_CG), use_old = sp.cg_old != 0;
  const double beta = sp.beta;
  const bool use_dir = (dm != DIR_NONE);
  double f0[4], f1[4], d0[4], d1[4], rq[4];
  double rn[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int g = l2g(ex, ey, b, n);
    f0[b] = ld(px, g);
    f1[b] = ld(py, g);
    d0[b] = use_dir ? (double)search_dir<S>(zx, ox_, g, cg, use_old, beta) : 0.0;
    d1[b] = use_dir ? (double)search_dir<S>(zy, oy_, g, cg, use_old, beta) : 0.0;
    rn[b] = ld(Rp, g);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    double w = 0.;
    for (int b = 0; b < 4; ++b) w += rn[b] * bq(b, q);
    rq[q] = w;
  }
  const double vol = h.d * h.d;
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    if (k < nc) {
      const double tau = sp.cand[k];
      double p0[4], p1[4];
      for (int b = 0; b < 4; ++b) {
        p0[b] = use_dir ? (double)step_at<S>((S)f0[b], tau, (S)d0[b]) : f0[b];
        p1[b] = use_dir ? (double)step_at<S>((S)f1[b], tau, (S)d1[b]) : f1[b];
      }
      double a = 0.;
      for (int q = 0; q < 4; ++q) {
        double ox = 0., oy = 0.;
        for (int b = 0; b < 4; ++b) {
          ox += p0[b] * bq(b, q);
          oy += p1[b] * bq(b, q);
        }
        const Hit hp = deform_qp(ex, ey, q, ox, oy, n, h, width);
        double t4[4];
        const double t = eval_img(Tp, hp, n, t4) - rq[q];
        a += 0.5 * (t * t) * 0.25;
      }
      a *= vol;
      acc[2 * k] += a;
      acc[2 * k + 1] += 0.5 * (stiff_form(p0) + stiff_form(p1));
    }
  }
}

// Sums of acc (per candidate E_SSD, E_reg) over the workgroup written as the partials of block `tile`
// (nblk per candidate and term) of one pair, all in one reduction.
template <int NC>
__device__ __forceinline__ void energy_write_partials(double (&acc)[2 * NC], int nc, double *__restrict__ part,
                                                      int pair, int tile, int nblk) {
  __shared__ double red[4 * 2 * NC];
  block_sum_n<2 * NC>(acc, red);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NC; ++k)
      if (k < nc) {
        part[((size_t)(pair * MAX_CAND + k) * 2 + 0) * nblk + tile] = acc[2 * k];
        part[((size_t)(pair * MAX_CAND + k) * 2 + 1) * nblk + tile] = acc[2 * k + 1];
      }
  }
}

// One workgroup's tile of the FP64 pass for one pair: one element per thread.
template <typename S>
__device__ __forceinline__ void energy_tile(const S *__restrict__ R, const S *__restrict__ T,
                                            const S *__restrict__ phi, const S *__restrict__ z,
                                            const S *__restrict__ dold, int n, double h, int width,
                                            const PairState *st, double *__restrict__ part, int ntx, int nty,
                                            int pair, int tile) {
  const size_t nn = (size_t)n * n;
  const S *Rp = R + pair * nn, *Tp = T + pair * nn;
  const S *px = phi + pair * 2 * nn, *py = px + nn;
  const S *zx = z + pair * 2 * nn, *zy = zx + nn, *ox_ = dold + pair * 2 * nn, *oy_ = ox_ + nn;
  const int ex = (tile % ntx) * EN_TX + (threadIdx.x % EN_TX);
  const int ey = (tile / ntx) * EN_TY + (threadIdx.x / EN_TX);
  const Div hd = make_div(h);
  double acc[2 * PLAN_CAND];
#pragma unroll
  for (int k = 0; k < 2 * PLAN_CAND; ++k) acc[k] = 0.0;
  if ((ex < n - 1) && (ey < n - 1))
    energy_elem<S, PLAN_CAND>(Rp, Tp, px, py, zx, zy, ox_, oy_, n, hd, width, st[pair], ex, ey, acc);
  energy_write_partials<PLAN_CAND>(acc, st[pair].ncand, part, pair, tile, ntx * nty);
}

template <typename S>
__global__ void __launch_bounds__(256)
k_energy(const S *__restrict__ R, const S *__restrict__ T, const S *__restrict__ phi, const S *__restrict__ z,
         const S *__restrict__ dold, int n, double h, int width, const PairState *st,
         double *__restrict__ part, int ntx, int nty, int npairs) {
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * npairs);
  const int pair = wg / tiles, tile = wg - pair * tiles;
  if (st[pair].ncand == 0) return;  // uniform across the workgroup
  energy_tile<S>(R, T, phi, z, dold, n, h, width, st, part, ntx, nty, pair, tile);
}

// ================================================================================================
// Consistency energy pass of reduceDeformations (matchSeries.h:678-704): for up to MAX_CAND step
// sizes, the sum over the n deformations psi_i (2 fields each) of ConsistencyEnergyOp
// (AmbrosioTortorelli.h:687-735), 1/2 int |psi_i(x + phi(x)) + phi(x)|^2 at the clipped deformed quad
// point. Partials as the SSD pass (term 1, the regulariser, is absent: 0).
// ================================================================================================
template <typename S>
__global__ void __launch_bounds__(256)
k_energy_cons(const S *__restrict__ psi, int npsi, const S *__restrict__ phi, const S *__restrict__ z,
              const S *__restrict__ dold, int n, double h, int width, const PairState *st, double *__restrict__ part,
              int ntx, int nty, int npairs) {
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * npairs);
  const int pair = wg / tiles, tile = wg - pair * tiles;
  const int nc = st[pair].ncand;
  if (nc == 0) return;  // uniform across the workgroup
  const int dm = st[pair].dirmode;
  __shared__ double red[4];

  const size_t nn = (size_t)n * n;
  const S *px = phi + pair * 2 * nn, *py = px + nn;
  const S *zx = z + pair * 2 * nn, *zy = zx + nn, *ox_ = dold + pair * 2 * nn, *oy_ = ox_ + nn;
  const bool cg = (dm == DIR_CG), use_old = st[pair].cg_old != 0;
  const double beta = st[pair].beta;
  const bool use_dir = (dm != DIR_NONE);

  const int ex = (tile % ntx) * EN_TX + (threadIdx.x % EN_TX);
  const int ey = (tile / ntx) * EN_TY + (threadIdx.x / EN_TX);
  const bool valid = (ex < n - 1) && (ey < n - 1);
  const Div hd = make_div(h);

  double acc[MAX_CAND];
#pragma unroll
  for (int k = 0; k < MAX_CAND; ++k) acc[k] = 0.0;

  if (valid) {
    double f0[4], f1[4], d0[4], d1[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int g = l2g(ex, ey, b, n);
      f0[b] = ld(px, g);
      f1[b] = ld(py, g);
      d0[b] = use_dir ? (double)search_dir<S>(zx, ox_, g, cg, use_old, beta) : 0.0;
      d1[b] = use_dir ? (double)search_dir<S>(zy, oy_, g, cg, use_old, beta) : 0.0;
    }
    const double vol = h * h;
#pragma unroll
    for (int k = 0; k < MAX_CAND; ++k) {
      if (k < nc) {
        const double tau = st[pair].cand[k];
        double p0[4], p1[4];
        for (int b = 0; b < 4; ++b) {
          p0[b] = use_dir ? (double)step_at<S>((S)f0[b], tau, (S)d0[b]) : f0[b];
          p1[b] = use_dir ? (double)step_at<S>((S)f1[b], tau, (S)d1[b]) : f1[b];
        }
        double a = 0.;
        for (int q = 0; q < 4; ++q) {
          double ox = 0., oy = 0.;
          for (int b = 0; b < 4; ++b) {
            ox += p0[b] * bq(b, q);
            oy += p1[b] * bq(b, q);
          }
          const Hit hp = deform_qp(ex, ey, q, ox, oy, n, hd, width);
          double e = 0.;
          for (int i = 0; i < npsi; ++i) {
            const S *pi = psi + (size_t)i * 2 * nn;
            double u4[4];
            const double vx = eval_img(pi, hp, n, u4) + ox, vy = eval_img(pi + nn, hp, n, u4) + oy;
            e += vx * vx + vy * vy;
          }
          a += 0.5 * e * 0.25;
        }
        acc[k] = a * vol;
      }
    }
  }
  const int nblk = tiles;
#pragma unroll
  for (int k = 0; k < MAX_CAND; ++k) {
    if (k < nc) {
      const double s = block_sum<256>(acc[k], red);
      if (threadIdx.x == 0) {
        part[((size_t)(pair * MAX_CAND + k) * 2 + 0) * nblk + tile] = s;
        part[((size_t)(pair * MAX_CAND + k) * 2 + 1) * nblk + tile] = 0.0;
      }
    }
  }
}

// ================================================================================================
// NCC energy pass (deformationModel 0) for up to MAX_CAND step sizes per pair, element-centric.
// NormalizedCrossCorrelationEnergy::computeEnergy (registration.h:1953-1964) in moments of the
// assembled mass matrix: with t the nodal FastDeformImage of T at phi + tau d, w = t - c for a shift
// c near the M-mean of t (the last accepted one) and u = r - m_r the centred reference, every element
// adds its share of 1'Mw, w'Mw, w'Mu (the element matrix of the assembled M). Moments about a nearby
// shift keep the differences between the candidates of one pass resolvable in FP64. The control
// combines them (ncc_value).
// ================================================================================================
// Bound by FP64 arithmetic. The warp at a node (two divisions, an interpolation) serves the four elements
// around it, so the tile's 65 x 5 nodes are warped once into LDS with their positions, then every thread
// takes its element's nodes from there; the 4 moments of all candidates share one reduction. Three pairs
// of 512^2, 20 iterations with the variation's weights shared alike: 5.6 -> 4.3 ms.
constexpr int NC_NX = EN_TX + 1, NC_NY = EN_TY + 1;  // nodes of a tile

template <typename S>
__global__ void __launch_bounds__(256)
k_energy_ncc(const S *__restrict__ R, const S *__restrict__ T, const S *__restrict__ phi, const S *__restrict__ z,
             const S *__restrict__ dold, int n, double h, const PairState *st, double *__restrict__ part, int ntx,
             int nty, int npairs) {
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * npairs);
  const int pair = wg / tiles, tile = wg - pair * tiles;
  const int nc = st[pair].ncand;
  if (nc == 0) return;  // uniform across the workgroup
  const int dm = st[pair].dirmode;
  constexpr int NC = PLAN_CAND;
  __shared__ double red[4 * 4 * NC];
  __shared__ double sw[NC][NC_NX * NC_NY], s0[NC][NC_NX * NC_NY], s1[NC][NC_NX * NC_NY];

  const size_t nn = (size_t)n * n;
  const S *Rp = R + pair * nn, *Tp = T + pair * nn;
  const S *px = phi + pair * 2 * nn, *py = px + nn;
  const S *zx = z + pair * 2 * nn, *zy = zx + nn, *ox_ = dold + pair * 2 * nn, *oy_ = ox_ + nn;
  const bool cg = (dm == DIR_CG), use_old = st[pair].cg_old != 0;
  const double beta = st[pair].beta;
  const bool use_dir = (dm != DIR_NONE);
  const Div hd = make_div(h);
  const double rm = st[pair].ncc_rm, c = st[pair].ncc_c;

  const int x0 = (tile % ntx) * EN_TX, y0 = (tile / ntx) * EN_TY;
  for (int i = threadIdx.x; i < NC_NX * NC_NY; i += 256) {
    const int x = x0 + i % NC_NX, y = y0 + i / NC_NX;
    if (x < n && y < n) {
      const int g = x + y * n;
      const S f0 = px[g], f1 = py[g];
      const S d0 = use_dir ? search_dir<S>(zx, ox_, g, cg, use_old, beta) : (S)0;
      const S d1 = use_dir ? search_dir<S>(zy, oy_, g, cg, use_old, beta) : (S)0;
#pragma unroll
      for (int k = 0; k < NC; ++k)
        if (k < nc) {
          const double tau = st[pair].cand[k];
          const double p0 = use_dir ? (double)step_at<S>(f0, tau, d0) : (double)f0;
          const double p1 = use_dir ? (double)step_at<S>(f1, tau, d1) : (double)f1;
          s0[k][i] = p0;
          s1[k][i] = p1;
          sw[k][i] = fast_warp(Tp, n, hd, x, y, p0, p1) - c;
        }
    }
  }
  __syncthreads();

  const int tx = threadIdx.x % EN_TX, ty = threadIdx.x / EN_TX;
  const int ex = x0 + tx, ey = y0 + ty;
  double acc[4 * NC];
#pragma unroll
  for (int k = 0; k < 4 * NC; ++k) acc[k] = 0.0;
  if ((ex < n - 1) && (ey < n - 1)) {
    double u[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
      u[b] = ld(Rp, l2g(ex, ey, b, n)) + (-rm);  // the reference centred as normalizeImageForNCC does (addToAll)
    double ml[4][4];
    mass_local(h * h, ml);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      if (k < nc) {
        double p0[4], p1[4], w[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int i = (tx + (b & 1)) + (ty + ((b >> 1) & 1)) * NC_NX;
          p0[b] = s0[k][i];
          p1[b] = s1[k][i];
          w[b] = sw[k][i];
        }
        for (int i = 0; i < 4; ++i) {
          double m = 0.;
          for (int j = 0; j < 4; ++j) m += ml[i][j] * w[j];
          acc[4 * k + 0] += m;
          acc[4 * k + 1] += w[i] * m;
          acc[4 * k + 2] += u[i] * m;
        }
        acc[4 * k + 3] = 0.5 * (stiff_form(p0) + stiff_form(p1));
      }
    }
  }
  block_sum_n<4 * NC>(acc, red);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NC; ++k)  // static indices keep acc in registers; nc is uniform
      if (k < nc)
#pragma unroll
        for (int t = 0; t < 4; ++t) part[part_index(DT_NCC, pair, k, t, tiles) + tile] = acc[4 * k + t];
  }
}

// The reference's statistics for the NCC pass, once per level: pass 0 the M-mean 1'Mr, pass 1 (with
// the mean in the pair state) the centred moments 1'Mu and u'Mu of u = r - m_r (normalizeImageForNCC,
// registration.h:1934-1947). Partials in the reference slots of the energy layout.
template <typename S>
__global__ void __launch_bounds__(256)
k_ncc_ref(const S *__restrict__ R, int n, double h, const PairState *st, double *__restrict__ part, int ntx, int nty,
          int npairs, int centred) {
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * npairs);
  const int pair = wg / tiles, tile = wg - pair * tiles;
  __shared__ double red[4];
  const size_t nn = (size_t)n * n;
  const S *Rp = R + pair * nn;
  const int ex = (tile % ntx) * EN_TX + (threadIdx.x % EN_TX);
  const int ey = (tile / ntx) * EN_TY + (threadIdx.x / EN_TX);
  double a1 = 0., a2 = 0.;
  if ((ex < n - 1) && (ey < n - 1)) {
    const double rm = centred ? st[pair].ncc_rm : 0.0;
    double u[4];
    for (int b = 0; b < 4; ++b) u[b] = centred ? ld(Rp, l2g(ex, ey, b, n)) + (-rm) : ld(Rp, l2g(ex, ey, b, n));
    double ml[4][4];
    mass_local(h * h, ml);
    for (int i = 0; i < 4; ++i) {
      double m = 0.;
      for (int j = 0; j < 4; ++j) m += ml[i][j] * u[j];
      a1 += m;
      a2 += u[i] * m;
    }
  }
  const double s1 = block_sum<256>(a1, red);
  const double s2 = block_sum<256>(a2, red);
  if (threadIdx.x == 0) {
    part[part_index_ref(npairs, pair, 0, tiles) + tile] = s1;
    part[part_index_ref(npairs, pair, 1, tiles) + tile] = s2;
  }
}

// ================================================================================================
// Variation DE = F_SSD + lambda K phi, node-centric with the element contributions staged in LDS.
// F_SSD: SSDForce::getNonlinearity (registration.h:1646-1666) assembled as in
// FENonlinVectorOpInterface::applyAdd (FEOpInterface.h:1803-1853); every node sums the
// contributions of its (up to) four elements in the reference's element order.
// ================================================================================================
constexpr int GR_TX = 32, GR_TY = 8;  // nodes per workgroup tile
constexpr int GR_EX = GR_TX + 1, GR_EY = GR_TY + 1;
constexpr int GR_NE = GR_EX * GR_EY;                // elements that touch the tile's nodes
constexpr int GR_NX = GR_TX + 2, GR_NY = GR_TY + 2;  // their nodes

// Gradient of the bilinear T at the hit from its 4 nodal values, in domain units: sum over the nodes of
// (derivative of the basis function / h) * value, in node order. The basis functions' derivatives are
// +-(1 - c) and +-c, so two divisions per axis give all four.
__device__ __forceinline__ void eval_grad(const double t[4], const Hit &hp, const Div &h, double &g0, double &g1) {
  const double ax = (1.0 - hp.ly) / h, bx = hp.ly / h, ay = (1.0 - hp.lx) / h, by = hp.lx / h;
  g0 = ((-ax * t[0] + ax * t[1]) + -bx * t[2]) + bx * t[3];
  g1 = ((-ay * t[0] + -by * t[1]) + ay * t[2]) + by * t[3];
}

template <typename S, int DT>
__global__ void __launch_bounds__(256)
k_grad(const S *__restrict__ R, const S *__restrict__ T, const S *__restrict__ phi, S *__restrict__ DE, int n,
       double h, int width, const PairState *st, double lambda_default, int ntx, int nty, int npairs, int npsi) {
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * npairs);
  const int pair = wg / tiles, tile = wg - pair * tiles;
  if (st && !participates(st[pair])) return;
  const double lambda = st ? st[pair].lambda : lambda_default;

  __shared__ double cf[4][2][GR_NE];  // force contribution per dof, component, element
  __shared__ double ck[4][2][GR_NE];  // stiffness contribution
  __shared__ double wn[DT == DT_NCC ? GR_NX * GR_NY : 1];  // the NCC weight at the elements' nodes

  const size_t nn = (size_t)n * n;
  const S *Rp = R + pair * nn, *Tp = T + pair * nn;
  const S *px = phi + pair * 2 * nn, *py = px + nn;
  const int x0 = (tile % ntx) * GR_TX, y0 = (tile / ntx) * GR_TY;
  const double vol = h * h;
  const Div hd = make_div(h);

  if constexpr (DT == DT_NCC) {
    // NormalizedCrossCorrelationEnergy::applyDerivative (registration.h:1974-1984): nodal weight
    // w = (Rn + E Tn) / v_t with Rn, Tn the normalised reference and warped template, once per node
    const PairState &ps = st[pair];
    const bool divr = !(fabs(ps.ncc_rv - 0.0) < 1e-15), divt = !(fabs(ps.ncc_v - 0.0) < 1e-15);
    const Div rv = make_div(ps.ncc_rv), tv = make_div(ps.ncc_v);
    for (int i = threadIdx.x; i < GR_NX * GR_NY; i += 256) {
      const int x = x0 - 1 + i % GR_NX, y = y0 - 1 + i / GR_NX;
      if (x < 0 || y < 0 || x >= n || y >= n) continue;
      const int g = x + y * n;
      double rh = ld(Rp, g) + (-ps.ncc_rm);
      if (divr) rh = rh / rv;
      double th = fast_warp(Tp, n, hd, x, y, ld(px, g), ld(py, g)) + (-ps.ncc_m);
      if (divt) th = th / tv;
      double wb = rh;
      wb += ps.ncc_d * th;
      if (divt) wb = wb / tv;
      wn[i] = wb;
    }
    __syncthreads();
  }

  for (int e = threadIdx.x; e < GR_EX * GR_EY; e += 256) {
    const int ex = x0 - 1 + (e % GR_EX), ey = y0 - 1 + (e / GR_EX);
    if (ex < 0 || ey < 0 || ex >= n - 1 || ey >= n - 1) continue;
    double f0[4], f1[4], rn[4];
    for (int b = 0; b < 4; ++b) {
      const int g = l2g(ex, ey, b, n);
      f0[b] = ld(px, g);
      f1[b] = ld(py, g);
      rn[b] = ld(Rp, g);
    }
    double nl[4][2];
    if (DT == DT_CONS) {
      // reduceDeformations: sum over the n deformations psi_i (passed as T, 2 fields each) of
      // VariationOfConsistencyEnergyOp::getNonlinearity (AmbrosioTortorelli.h:755-799):
      // (Dpsi_i + I)^T (psi_i + offset) at the clipped deformed quad point, zero per clipped axis
      for (int q = 0; q < 4; ++q) {
        double ox = 0., oy = 0.;
        for (int b = 0; b < 4; ++b) {
          ox += f0[b] * bq(b, q);
          oy += f1[b] * bq(b, q);
        }
        const Hit hp = deform_qp(ex, ey, q, ox, oy, n, hd, width);
        double a0 = 0., a1 = 0.;
        for (int k = 0; k < npsi; ++k) {
          const S *pk = T + (size_t)k * 2 * nn;
          double u4[4], w4[4];
          double vx = eval_img(pk, hp, n, u4), vy = eval_img(pk + nn, hp, n, w4);
          double j00, j01, j10, j11;  // j[c][d] = d psi_c / d x_d
          eval_grad(u4, hp, hd, j00, j01);
          eval_grad(w4, hp, hd, j10, j11);
          vx += ox;
          vy += oy;
          j00 += 1.;
          j11 += 1.;
          a0 += j00 * vx + j10 * vy;
          a1 += j01 * vx + j11 * vy;
        }
        nl[q][0] = hp.inx ? a0 : 0;
        nl[q][1] = hp.iny ? a1 : 0;
      }
    } else if (DT == DT_NCC) {
      // CrossCorrelationForce (registration.h:1826-1862): -w(x_q) grad T at the unclipped deformed quad
      // point, zero where it leaves the grid
      double w[4];
      for (int b = 0; b < 4; ++b) w[b] = wn[(ex - x0 + 1 + (b & 1)) + (ey - y0 + 1 + ((b >> 1) & 1)) * GR_NX];
      for (int q = 0; q < 4; ++q) {
        double ox = 0., oy = 0.;
        for (int b = 0; b < 4; ++b) {
          ox += f0[b] * bq(b, q);
          oy += f1[b] * bq(b, q);
        }
        Hit hp;
        if (!transform_noclip(ex, ey, q, ox, oy, n, hd, hp)) {
          nl[q][0] = nl[q][1] = 0.;
          continue;
        }
        double t4[4];
        (void)eval_img(Tp, hp, n, t4);
        double g0, g1;
        eval_grad(t4, hp, hd, g0, g1);
        double wq = 0.;
        for (int b = 0; b < 4; ++b) wq += w[b] * bq(b, q);
        const double sc = -wq;
        nl[q][0] = g0 * sc;
        nl[q][1] = g1 * sc;
      }
    } else {
      for (int q = 0; q < 4; ++q) {
        double ox = 0., oy = 0., r = 0.;
        for (int b = 0; b < 4; ++b) {
          ox += f0[b] * bq(b, q);
          oy += f1[b] * bq(b, q);
        }
        for (int b = 0; b < 4; ++b) r += rn[b] * bq(b, q);
        const Hit hp = deform_qp(ex, ey, q, ox, oy, n, hd, width);
        double t4[4];
        const double td = eval_img(Tp, hp, n, t4);
        double g0, g1;
        eval_grad(t4, hp, hd, g0, g1);
        nl[q][0] = hp.inx ? g0 * (td - r) : 0;
        nl[q][1] = hp.iny ? g1 * (td - r) : 0;
      }
    }
    for (int dof = 0; dof < 4; ++dof) {
      double a0 = 0, a1 = 0;
      for (int q = 0; q < 4; ++q) {
        const double fct = bq(dof, q) * 0.25;
        a0 += fct * nl[q][0];
        a1 += fct * nl[q][1];
      }
      cf[dof][0][e] = vol * a0;
      cf[dof][1][e] = vol * a1;
    }
    // K_loc (1/6)[4 -1 -1 -2; -1 4 -2 -1; -1 -2 4 -1; -2 -1 -1 4] applied to the element's dofs
    const double kl[4][4] = {{4. / 6, -1. / 6, -1. / 6, -2. / 6},
                             {-1. / 6, 4. / 6, -2. / 6, -1. / 6},
                             {-1. / 6, -2. / 6, 4. / 6, -1. / 6},
                             {-2. / 6, -1. / 6, -1. / 6, 4. / 6}};
    for (int i = 0; i < 4; ++i) {
      double s0 = 0, s1 = 0;
      for (int j = 0; j < 4; ++j) {
        s0 += kl[i][j] * f0[j];
        s1 += kl[i][j] * f1[j];
      }
      ck[i][0][e] = s0;
      ck[i][1][e] = s1;
    }
  }
  __syncthreads();
  const int x = x0 + (threadIdx.x % GR_TX), y = y0 + (threadIdx.x / GR_TX);
  if (x >= n || y >= n) return;
  double F0 = 0, F1 = 0, K0 = 0, K1 = 0;
  for (int ey = y - 1; ey <= y; ++ey)
    for (int ex = x - 1; ex <= x; ++ex) {
      if (ex < 0 || ey < 0 || ex >= n - 1 || ey >= n - 1) continue;
      const int e = (ex - (x0 - 1)) + (ey - (y0 - 1)) * GR_EX;
      const int dof = (x - ex) + 2 * (y - ey);
      F0 += cf[dof][0][e];
      F1 += cf[dof][1][e];
      K0 += ck[dof][0][e];
      K1 += ck[dof][1][e];
    }
  S *o = DE + pair * 2 * nn;
  const int i = x + y * n;
  o[i] = static_cast<S>(F0 + lambda * K0);
  o[nn + i] = static_cast<S>(F1 + lambda * K1);
}

// ================================================================================================
// H1 metric: one V-cycle of the FD heat operator (LinearSmoothOp::apply, linearSmoothOp.cpp:591-612,
// MDMultigrid::solve L451-494, HeatMultigrid::jacobi L556-580) per field, 2 fields per pair.
// Down-leg kernel: x1 = rhs/diag (first Jacobi sweep from zero), x2 = x1 + (rhs - A x1)/diag,
// residual r = rhs - A x2, coarse rhs = 2x2 mean of r. Up-leg kernel: x = x2 + injected coarse
// correction, then two Jacobi sweeps. Tiles with a 2-node halo live in LDS.
// ================================================================================================
constexpr int MG_TX = 32, MG_TY = 16;
constexpr int MG_HY = MG_TY + 4;
// FP32 fields: tiles of 64 x 16 nodes (4 per thread) on levels of 1024^2 and above -- 512 workgroups
// per field at 1024^2, resident at once, and a halo of 1.33x the tile instead of 1.41x -- and of
// 32 x 16 below, where a workgroup's latency, not the level's traffic, sets the pass's time.
constexpr int MG32_TY = MG_TY;
constexpr int MG32_TX_WIDE = 64, MG32_WIDE_FROM = 1024;

__device__ __forceinline__ void level_consts(const PairState *st, int pair, double sigma_default, int n, double &hs,
                                             Div &diag) {
  const double sigma = st ? st[pair].sigma : sigma_default;
  const double tau = 0.5 * (sigma * sigma);  // LinearSmoothOp::setSigma (linearSmoothOp.h:50-52)
  const double s = (double)((n - 1) * (n - 1));
  hs = tau * s;
  diag = make_div(1 + 4 * tau * s);
}

// The fine passes' tiles of TX x 16 nodes with a 2-node halo in LDS (TX + 4 columns, 20 rows). A thread keeps
// one of the TX columns, so its global and LDS addresses, the mirrored neighbours of a border column and
// the bounds are worked out once and rows differ by constants; the 4 halo columns are a short extra step.
// (n is a multiple of TX and 16: only halo rows and columns lie outside the grid.) Indexing every cell modulo
// the halo's width took as many instructions as the sweeps: 8 pairs of 1024^2, the finest level down 59 -> 51 us
// and up 90 -> 84 us (their memory traffic alone: 29 and 54 us). FP64, 2 pairs of 1024^2, where the tiles away
// from the grid's border skip heat_apply's cases too, over a solve's launches: down 23.6 -> 18.5, up 29.6 -> 28.0 us.
template <int TX>
struct MgTile {
  static constexpr int HX = TX + 4, G = 256 / TX;        // halo row length; rows in flight
  static constexpr int LR = (MG_HY + G - 1) / G;       // rows per thread: of the halo tile
  static constexpr int SR = (MG_HY - 2 + G - 1) / G;   // of the tile + 1
  static constexpr int NHALO = 4 * MG_HY;              // cells of the halo columns
  int tx, g;           // column of the tile, row group
  int x0, y0, n;
  int xl, xr;          // LDS columns of the (mirrored) neighbours of column tx
  int hr, hc, hx;      // the halo cell of this thread (tid < NHALO): row, LDS column, grid column
  __device__ __forceinline__ MgTile(int tile, int ntx, int n_) : n(n_) {
    tx = threadIdx.x % TX;
    g = threadIdx.x / TX;
    x0 = (tile % ntx) * TX;
    y0 = (tile / ntx) * MG32_TY;
    const int gx = x0 + tx, lx = tx + 2;
    xl = gx > 0 ? lx - 1 : lx + 1;
    xr = gx < n - 1 ? lx + 1 : lx - 1;
    hr = threadIdx.x >> 2;
    const int c = threadIdx.x & 3;
    hc = c < 2 ? c : TX + c;
    hx = x0 + hc - 2;
  }
  // no halo cell outside the grid, nor on its border (uniform)
  __device__ __forceinline__ bool inner() const { return x0 > 0 && y0 > 0 && x0 + TX < n && y0 + MG_TY < n; }
  __device__ __forceinline__ bool row_in(int r) const { return (unsigned)(y0 + r - 2) < (unsigned)n; }
  __device__ __forceinline__ bool halo_in() const {
    return threadIdx.x < NHALO && (unsigned)hx < (unsigned)n && row_in(hr);
  }
  // clamped grid index of halo-tile row r, column of this thread / of its halo cell
  __device__ __forceinline__ int at(int r) const { return min(max(y0 + r - 2, 0), n - 1) * n + x0 + tx; }
  __device__ __forceinline__ int halo_at() const {
    return min(max(y0 + hr - 2, 0), n - 1) * n + min(max(hx, 0), n - 1);
  }
};

// A u at row r, LDS column lx of a halo tile of the FP64 passes: on tiles away from the grid's border
// (INNER, uniform) without heat_apply's cases.
template <bool INNER, int TX>
__device__ __forceinline__ double heat_at(const MgTile<TX> &t, const double (*u)[TX + 4], int r, int lx, double hs) {
  if constexpr (INNER) {
    const double c = u[r][lx];
    double b = 0.0;
    b -= u[r][lx + 1];
    b -= u[r][lx - 1];
    b -= u[r + 1][lx];
    b -= u[r - 1][lx];
    return c + hs * (c * 4 + b);
  } else {
    auto get = [&](int gx, int gy) { return u[gy - t.y0 + 2][gx - t.x0 + 2]; };
    return heat_apply(get, t.x0 + lx - 2, t.y0 + r - 2, t.n, hs);
  }
}
// One Jacobi sweep x + (rhs - A x) / diag on the tile + 1 (rows 1..18, columns 1..TX+2 of the halo tile).
template <bool INNER, int TX>
__device__ __forceinline__ void sweep_tile1(const MgTile<TX> &t, const double (*sr)[TX + 4], const double (*sx)[TX + 4],
                                            double (*out)[TX + 4], double hs, const Div &diag) {
  auto cell = [&](int r, int lx) {
    const double v = sr[r][lx] - heat_at<INNER>(t, sx, r, lx, hs);
    out[r][lx] = sx[r][lx] + 1.0 * v / diag;
  };
#pragma unroll
  for (int k = 0; k < MgTile<TX>::SR; ++k) {
    const int r = 1 + t.g * MgTile<TX>::SR + k;
    if (r < MG_HY - 1 && (INNER || t.row_in(r))) cell(r, t.tx + 2);
  }
  const int c = threadIdx.x & 3;
  if ((c == 1 || c == 2) && t.hr >= 1 && t.hr < MG_HY - 1 && (INNER || t.halo_in())) cell(t.hr, t.hc);
}

template <typename S>
__global__ void __launch_bounds__(256)
k_mg_down(const S *__restrict__ rhs, int negate, S *__restrict__ x2out, S *__restrict__ rhsc, int n,
          const PairState *st, double sigma_default, int ntx, int nty, int nfields) {
  typedef MgTile<MG_TX> Tile;
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * nfields);
  const int field = wg / tiles, tile = wg - field * tiles;
  const int pair = field >> 1;
  if (st && !participates(st[pair])) return;
  double hs;
  Div diag;
  level_consts(st, pair, sigma_default, n, hs, diag);

  __shared__ double sr[MG_HY][Tile::HX];  // rhs on tile+2
  __shared__ double s1[MG_HY][Tile::HX];  // x1 on tile+2, then the residual on the tile
  __shared__ double s2[MG_HY][Tile::HX];  // x2 on tile+1
  const Tile t(tile, ntx, n);
  const S *rp = rhs + field * (size_t)n * n;

  // every load issued before the first is used (clamped indices; cells outside the grid are not stored)
  double hv[Tile::LR];
#pragma unroll
  for (int k = 0; k < Tile::LR; ++k) hv[k] = ld(rp, t.at(t.g * Tile::LR + k));
  const double hh = ld(rp, t.halo_at());
#pragma unroll
  for (int k = 0; k < Tile::LR; ++k) {
    const int r = t.g * Tile::LR + k;
    if (r < MG_HY && t.row_in(r)) {
      const double v = negate ? -hv[k] : hv[k];
      sr[r][t.tx + 2] = v;
      s1[r][t.tx + 2] = v / diag;  // 0 + (1.0 * (rhs - A 0)) / diag
    }
  }
  if (t.halo_in()) {
    const double v = negate ? -hh : hh;
    sr[t.hr][t.hc] = v;
    s1[t.hr][t.hc] = v / diag;
  }
  __syncthreads();
  double res[MG_TY / Tile::G];
  auto sweeps = [&](auto inner) {
    constexpr bool INNER = decltype(inner)::value;
    sweep_tile1<INNER>(t, sr, s1, s2, hs, diag);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < MG_TY / Tile::G; ++k) {
      const int r = t.g + Tile::G * k + 2;
      res[k] = sr[r][t.tx + 2] - heat_at<INNER>(t, s2, r, t.tx + 2, hs);
    }
  };
  if (t.inner())
    sweeps(std::true_type());
  else
    sweeps(std::false_type());
  S *xo = x2out + field * (size_t)n * n + (size_t)t.y0 * n + t.x0 + t.tx;
#pragma unroll
  for (int k = 0; k < MG_TY / Tile::G; ++k) {
    const int r = t.g + Tile::G * k;
    s1[r][t.tx] = res[k];
    xo[(size_t)r * n] = static_cast<S>(s2[r + 2][t.tx + 2]);
  }
  __syncthreads();
  const int nc = n / 2;
  S *rc = rhsc + field * (size_t)nc * nc + (size_t)(t.y0 / 2) * nc + t.x0 / 2;
  for (int i = threadIdx.x; i < (MG_TX / 2) * (MG_TY / 2); i += 256) {
    const int cx = i % (MG_TX / 2), cy = i / (MG_TX / 2);
    double v = 0;
    v += s1[2 * cy][2 * cx];
    v += s1[2 * cy][2 * cx + 1];
    v += s1[2 * cy + 1][2 * cx];
    v += s1[2 * cy + 1][2 * cx + 1];
    rc[(size_t)cy * nc + cx] = static_cast<S>((1.0 / 4.0) * v);
  }
}

template <typename S>
__global__ void __launch_bounds__(256)
k_mg_up(const S *__restrict__ x2in, const S *__restrict__ xc, const S *__restrict__ rhs, int negate,
        S *__restrict__ xout, int n, const PairState *st, double sigma_default, int ntx, int nty,
        int nfields, const S *__restrict__ dold, double *__restrict__ nrm_part) {
  typedef MgTile<MG_TX> Tile;
  const int tiles = ntx * nty;
  const int wg = xcd_remap(blockIdx.x, tiles * nfields);
  const int field = wg / tiles, tile = wg - field * tiles;
  const int pair = field >> 1;
  if (st && !participates(st[pair])) return;
  double hs;
  Div diag;
  level_consts(st, pair, sigma_default, n, hs, diag);

  __shared__ double sx[MG_HY][Tile::HX];  // x on tile+2
  __shared__ double sr[MG_HY][Tile::HX];  // rhs on tile+2
  __shared__ double s3[MG_HY][Tile::HX];  // x3 on tile+1
  __shared__ double red[4 * NORM_TERMS];
  const Tile t(tile, ntx, n);
  const size_t nn = (size_t)n * n;
  const int nc = n / 2;
  const S *x2p = x2in + field * nn, *rp = rhs + field * nn, *xcp = xc + field * (size_t)nc * nc;
  const size_t o0 = field * nn + (size_t)t.y0 * n + t.x0 + t.tx;  // this thread's column of the tile
  constexpr int OUT = MG_TY / Tile::G;                            // output rows per thread: g + G k

  // every load issued before the first is used (clamped indices; cells outside the grid are not stored);
  // the previous direction at the output nodes among them
  double dprev[OUT];
  if (nrm_part) {
#pragma unroll
    for (int k = 0; k < OUT; ++k) dprev[k] = ld(dold, o0 + (size_t)(t.g + Tile::G * k) * n);
  }
  double hx2[Tile::LR], hxc[Tile::LR], hr[Tile::LR];
#pragma unroll
  for (int k = 0; k < Tile::LR; ++k) {
    const int r = t.g * Tile::LR + k, gi = t.at(r);
    hx2[k] = ld(x2p, gi);
    hr[k] = ld(rp, gi);
    hxc[k] = ld(xcp, (min(max(t.y0 + r - 2, 0), n - 1) >> 1) * nc + ((t.x0 + t.tx) >> 1));
  }
  const int gh = t.halo_at();
  const double hh2 = ld(x2p, gh), hhr = ld(rp, gh);
  const double hhc = ld(xcp, (min(max(t.y0 + t.hr - 2, 0), n - 1) >> 1) * nc + (min(max(t.hx, 0), n - 1) >> 1));
#pragma unroll
  for (int k = 0; k < Tile::LR; ++k) {
    const int r = t.g * Tile::LR + k;
    if (r < MG_HY && t.row_in(r)) {
      sx[r][t.tx + 2] = hx2[k] + hxc[k];
      sr[r][t.tx + 2] = negate ? -hr[k] : hr[k];
    }
  }
  if (t.halo_in()) {
    sx[t.hr][t.hc] = hh2 + hhc;
    sr[t.hr][t.hc] = negate ? -hhr : hhr;
  }
  __syncthreads();
  double acc[NORM_TERMS] = {0., 0., 0., 0.};  // <z,z>, <DE,z>, <DE,d_old>, <DE,DE> (DE = the raw input)
  auto sweeps = [&](auto inner) {
    constexpr bool INNER = decltype(inner)::value;
    sweep_tile1<INNER>(t, sr, sx, s3, hs, diag);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < OUT; ++k) {
      const int r = t.g + Tile::G * k;
      const double b = sr[r + 2][t.tx + 2];
      const double v = b - heat_at<INNER>(t, s3, r + 2, t.tx + 2, hs);
      const S o = static_cast<S>(s3[r + 2][t.tx + 2] + 1.0 * v / diag);
      xout[o0 + (size_t)r * n] = o;
      if (nrm_part) {
        const double od = static_cast<double>(o), de = negate ? -b : b;
        acc[0] += od * od;
        acc[1] += de * od;
        acc[2] += de * dprev[k];
        acc[3] += de * de;
      }
    }
  };
  if (t.inner())
    sweeps(std::true_type());
  else
    sweeps(std::false_type());
  if (nrm_part) {
    block_sum_n<NORM_TERMS>(acc, red);
    if (threadIdx.x == 0)
      for (int q = 0; q < NORM_TERMS; ++q) nrm_part[((size_t)field * NORM_TERMS + q) * tiles + tile] = acc[q];
  }
}

// Whole V-cycle below (and including) a level of at most 32x32 nodes in one workgroup, in LDS. With n
// equal to the registration level this is the complete metric; otherwise it is the coarse part of the cycle
// started by k_mg_down.
// A chain of barriers with few nodes per thread between them, so the fewer and shorter the links the
// better: the sweeps write a second buffer instead of updating in place, the residual is restricted as it is formed,
// the prolongation is read on the fly by the first sweep of the up leg (3 barriers a level down and 2 up, 65 in
// all before), a 32x32 level is one node per thread, and levels of at most 8x8 nodes run in wave 0 alone
// behind compiler barriers: 20 to 24 us -> 15.7 us for a level of 32x32, the same bits.
// MAXL bounds the level, TH is the workgroup: threads without a node hold a compute unit's slots and LDS idle, which
// is free while every field's workgroup is resident and not beyond (mg_coarse chooses, with the times).
constexpr int MGC_THREADS = 1024;
constexpr int MGC_WAVE_LEVELS = 3;  // 8x8 nodes and below
constexpr int MGC_MAXL = 5;
constexpr int MGC_OFF[8] = {0, 1, 5, 21, 85, 341, 1365, 5461};  // prefix sums of 4^l

// Wave 0's own levels: its instructions, LDS accesses included, execute in order for all lanes, so a
// wavefront fence (a compiler barrier) replaces the workgroup barrier.
__device__ __forceinline__ void mgc_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename S, int MAXL, int TH>
__global__ void __launch_bounds__(TH)
k_mg_coarse(const S *__restrict__ rhs, int negate, S *__restrict__ xout, int L, const PairState *st,
            double sigma_default, int nfields, const S *__restrict__ dold, double *__restrict__ nrm_part) {
  const int field = blockIdx.x;
  const int pair = field >> 1;
  if (st && !participates(st[pair])) return;
  const double sigma = st ? st[pair].sigma : sigma_default;
  const double tau = 0.5 * (sigma * sigma);
  constexpr int MAXN = 1 << (2 * MAXL);
  __shared__ double X[MGC_OFF[MAXL + 1]], B[MGC_OFF[MAXL + 1]], Y[MAXN];
  __shared__ double red[(TH / 64) * NORM_TERMS];
  __shared__ Div dg[MAXL + 1];  // the levels' Jacobi diagonals, divided once
  const int n = 1 << L;
  const int nn = n * n;
  const S *rp = rhs + (size_t)field * nn;
  const int tid = threadIdx.x;
  constexpr int NPT = MAXN / TH;  // nodes per thread
  double raw[NPT];
#pragma unroll
  for (int k = 0; k < NPT; ++k) raw[k] = ld(rp, min(tid + TH * k, nn - 1));
  // the scalar products are summed by 256 threads (all, where there are fewer); their operands load now, behind
  // the sweeps
  constexpr int NT = TH < 256 ? TH : 256, PER = MAXN / NT;
  double rv[PER], ov[PER];
  if (nrm_part && tid < NT) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int i = min(tid + NT * k, nn - 1);
      rv[k] = ld(rp, i);
      ov[k] = ld(dold + (size_t)field * nn, i);
    }
  }
  if (tid <= L) {
    const int m = 1 << tid;
    const double s = (double)((m - 1) * (m - 1));
    dg[tid] = make_div(1 + 4 * tau * s);
  }
#pragma unroll
  for (int k = 0; k < NPT; ++k) {
    const int i = tid + TH * k;
    if (i < nn) B[MGC_OFF[L] + i] = negate ? -raw[k] : raw[k];
  }
  __syncthreads();

  // x + (b - A x) / diag at a node, x read by get
  auto relaxed = [&](const auto &get, const double *b, int i, int l, double hs, const Div &diag) {
    const int m = 1 << l, px = i & (m - 1), py = i >> l;
    const double v = b[i] - heat_apply(get, px, py, m, hs);
    return get(px, py) + 1.0 * v / diag;
  };
  auto level_hs = [&](int l) {
    const int m = 1 << l;
    return tau * (double)((m - 1) * (m - 1));
  };
  // Two sweeps from zero, the second kept in X for the up leg, then the residual restricted to level l - 1.
  auto down_level = [&](int l, int nthr, auto sync) {
    const int m = 1 << l, mm = m * m, mc = m / 2;
    const double hs = level_hs(l);
    const Div diag = dg[l];
    double *x = X + MGC_OFF[l];
    const double *b = B + MGC_OFF[l];
    for (int i = tid; i < mm; i += nthr) Y[i] = 0.0 + b[i] / diag;
    sync();
    auto gy = [&](int px, int py) { return Y[px + py * m]; };
    for (int i = tid; i < mm; i += nthr) x[i] = relaxed(gy, b, i, l, hs, diag);
    sync();
    auto gx = [&](int px, int py) { return x[px + py * m]; };
    // the residual at the 4 children of a coarse node, one child per lane, added in order x, then y
    for (int i = tid; i < mm; i += nthr) {
      const int c = i & 3, ci = i >> 2;
      const int fx = 2 * (ci & (mc - 1)) + (c & 1), fy = 2 * (ci >> (l - 1)) + (c >> 1);
      const double r = b[fx + fy * m] - heat_apply(gx, fx, fy, m, hs);
      double v = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) v += __shfl(r, k, 4);
      if (c == 0) B[MGC_OFF[l - 1] + ci] = (1.0 / 4.0) * v;
    }
    sync();
  };
  // The injected coarse correction read on the fly by the first sweep, the second sweep into X.
  auto up_level = [&](int l, int nthr, auto sync) {
    const int m = 1 << l, mm = m * m, mc = m / 2;
    const double hs = level_hs(l);
    const Div diag = dg[l];
    double *x = X + MGC_OFF[l];
    const double *xc = X + MGC_OFF[l - 1];
    const double *b = B + MGC_OFF[l];
    auto gp = [&](int px, int py) { return x[px + py * m] + xc[(px >> 1) + (py >> 1) * mc]; };
    for (int i = tid; i < mm; i += nthr) Y[i] = relaxed(gp, b, i, l, hs, diag);
    sync();
    auto gy = [&](int px, int py) { return Y[px + py * m]; };
    for (int i = tid; i < mm; i += nthr) x[i] = relaxed(gy, b, i, l, hs, diag);
    sync();
  };
  auto block_sync = [] { __syncthreads(); };
  auto wave_sync = [] { mgc_wave_sync(); };
  for (int l = L; l > MGC_WAVE_LEVELS; --l) down_level(l, TH, block_sync);
  if (tid < 64) {
    const int lw = min(L, MGC_WAVE_LEVELS);
    for (int l = lw; l >= 1; --l) down_level(l, 64, wave_sync);
    if (tid == 0) {  // 1x1 level: of 100 sweeps of x += (rhs - x) / 1 the third and later change nothing
      const double b = B[0];
      double x = 0;
      x += b - x;
      x += b - x;
      X[0] = x;
    }
    wave_sync();
    for (int l = 1; l <= lw; ++l) up_level(l, 64, wave_sync);
  }
  __syncthreads();
  for (int l = MGC_WAVE_LEVELS + 1; l <= L; ++l) up_level(l, TH, block_sync);
  S *xo = xout + (size_t)field * nn;
  for (int i = tid; i < nn; i += TH) xo[i] = static_cast<S>(X[MGC_OFF[L] + i]);
  if (nrm_part) {
    double acc[NORM_TERMS] = {0., 0., 0., 0.};  // <z,z>, <DE,z>, <DE,d_old>, <DE,DE> (DE = the raw input)
    if (tid < NT) {
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int i = tid + NT * k;
        if (i < nn) {
          const double od = static_cast<double>(static_cast<S>(X[MGC_OFF[L] + i])), de = rv[k];
          acc[0] += od * od;
          acc[1] += de * od;
          acc[2] += de * ov[k];
          acc[3] += de * de;
        }
      }
    }
    block_sum_n<NORM_TERMS, TH>(acc, red);
    if (tid == 0)
      for (int t = 0; t < NORM_TERMS; ++t) nrm_part[(size_t)field * NORM_TERMS + t] = acc[t];
  }
}

// ================================================================================================
// Update phi += tau * dir for pairs whose search accepted a step (GradientDescentBase::applySingle
// L382-385). Along the CG direction the kernel forms d = z + beta d_old (search_dir) and stores it
// in place of d_old: it is the next iteration's old direction.
// ================================================================================================
constexpr int UPD_PER_THREAD = 4;

template <typename S>
__global__ void __launch_bounds__(256)
k_update(S *__restrict__ phi, S *__restrict__ d, const S *__restrict__ z, int n, const PairState *st, int nblk_pair,
         int npairs, int slot) {
  const int total = nblk_pair * npairs;
  const int wg = xcd_remap(blockIdx.x, total);
  const int pair = wg / nblk_pair, blk = wg - pair * nblk_pair;
  const double tau = st[pair].step_tau[slot];
  if (tau == 0) return;  // no step accepted in this iteration
  const bool cg = st[pair].step_dir[slot] == DIR_CG, use_old = st[pair].cg_old != 0;
  const double beta = st[pair].beta;
  const size_t off = pair * 2 * (size_t)n * n;
  S *p = phi + off, *dp = d + off;
  const S *zp = z + off;
  const int m = 2 * n * n;
  const int base = blk * 256 * UPD_PER_THREAD;
  // every load first (indices clamped into the field), then the stores: the loads of all
  // UPD_PER_THREAD nodes are in flight together instead of one node's at a time
  S zv[UPD_PER_THREAD], ov[UPD_PER_THREAD], pv[UPD_PER_THREAD];
#pragma unroll
  for (int k = 0; k < UPD_PER_THREAD; ++k) {
    const int i = min(base + k * 256 + (int)threadIdx.x, m - 1);
    zv[k] = zp[i];
    ov[k] = dp[i];
    pv[k] = p[i];
  }
#pragma unroll
  for (int k = 0; k < UPD_PER_THREAD; ++k) {
    const int i = base + k * 256 + threadIdx.x;
    if (i < m) {
      const S dv = search_dir_val<S>(zv[k], ov[k], cg, use_old, beta);
      if (cg) dp[i] = dv;
      p[i] = step_at<S>(pv[k], tau, dv);
    }
  }
}

// ================================================================================================
// Grid transfer and warps
// ================================================================================================

// CellCenteredRestrictOp::apply (cellCenteredGrid.h:165-180): 2x2 mean, one coarse node per thread.
template <typename S>
__global__ void k_restrict(const S *__restrict__ fine, S *__restrict__ coarse, int n, int nfields) {
  const int nc = n / 2;
  const size_t cnt = (size_t)nc * nc;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cnt * nfields) return;
  const int f = (int)(i / cnt);
  const int j = (int)(i - (size_t)f * cnt);
  const int cx = j % nc, cy = j / nc;
  const S *fp = fine + (size_t)f * n * n;
  double v = 0;
  v += ld(fp, 2 * cx + 2 * cy * n);
  v += ld(fp, 2 * cx + 1 + 2 * cy * n);
  v += ld(fp, 2 * cx + (2 * cy + 1) * n);
  v += ld(fp, 2 * cx + 1 + (2 * cy + 1) * n);
  coarse[i] = static_cast<S>((1.0 / 4.0) * v);
}

// CellCenteredProlongOp::apply (cellCenteredGrid.h:188-210): injection n -> 2n.
template <typename S>
__global__ void k_prolong(const S *__restrict__ coarse, S *__restrict__ fine, int nc, int nfields) {
  const int n = 2 * nc;
  const size_t cnt = (size_t)n * n;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cnt * nfields) return;
  const int f = (int)(i / cnt);
  const int j = (int)(i - (size_t)f * cnt);
  const int x = j % n, y = j / n;
  fine[i] = coarse[(size_t)f * nc * nc + (x >> 1) + (y >> 1) * nc];
}

// ScalarArray<QC_2D>::resampleFrom (scalarArray.h:308-331, 1052-1060); coord[k] = k * (nc-1)/(n-1)
// evaluated in long double on the host and rounded to double.
template <typename S>
__global__ void k_resample(const S *__restrict__ src, S *__restrict__ dst, int nc, int n,
                           const double *__restrict__ coord, int nfields) {
  const size_t cnt = (size_t)n * n;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cnt * nfields) return;
  const int f = (int)(i / cnt);
  const int j = (int)(i - (size_t)f * cnt);
  dst[i] = static_cast<S>(interp(src + (size_t)f * nc * nc, nc, coord[j % n], coord[j / n]));
}

// ScalarArray<QC_2D>::resampleFrom of a w x h source onto n x n nodes: node (x, y) takes the source
// interpolated at (cx[x], cy[y]).
template <typename S>
__global__ void k_resample_rect(const S *__restrict__ src, int w, int h, S *__restrict__ dst, int n,
                                const double *__restrict__ cx, const double *__restrict__ cy) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)n * n) return;
  const int x = (int)(i % n), y = (int)(i / n);
  dst[i] = static_cast<S>(interp_wh(src, w, h, cx[x], cy[y]));
}

// DeformImage (deformations.h:62-101; ExtendWithConstant, optional nearest-neighbour rounding),
// FastDeformImage (L140-162; clamp) and the NaN-extended variant of L226-256 (mode 2).
// img: nimg images; phi: one field per image (or one shared field if phi_shared). n is a power of two,
// logn its logarithm. Bound by HBM (phi, the image and the result once, 16 B per FP32 pixel). A workgroup
// takes tiles of 256 columns (or the whole width) and a thread RUN pixels one below another, step by step
// together, displacements, then the 4 neighbours each, so a wave waits for two memory round trips in RUN pixels
// and neighbouring rows meet in its cache lines. Pixels outside gather from clamped nodes and are replaced by a
// select (no branches). 31 frames of 1024^2 in FP32, whole calls: 200 us with one pixel per thread and 64-bit index
// divisions; 132 us so (the kernel 118 us, 4.4 TB/s), where the field is noisy (1.5 pixels) 205 and 137 us; FP64
// 226 and 197, noisy 261 and 229 us. RUN = 4 pixels in a row, 256 apart, instead: 135 us, but 205 us where noisy (FP64 206 and 378 us), four
// rows' neighbours at once being more than a compute unit's L1 holds. Few pixels have nothing to overlap:
// 128^2 20.7 us with RUN = 1, 21.7 with 4; from WARP_RUN_PIXELS (512 workgroups of 4) on the latter is no slower:
// 512^2 x 2 22.8 and 23.1 us, in FP64 up to 25.6 and 23.2. Positions rounded to nodes (NEAR) lie on one row, but on
// the grid's last, and read that one alone (4 x 2048^2 in FP64, half the positions outside: 150 us with both rows, 132 so).
constexpr int WARP_RUN = 4;
constexpr long WARP_RUN_PIXELS = 1l << 19;

// NEAR: positions rounded to nodes (mode 0 only).
template <typename S, int RUN, bool NEAR>
__global__ void __launch_bounds__(256)
k_warp(const S *__restrict__ img, const S *__restrict__ phi, S *__restrict__ out, int n, int logn, int nblk,
       int phi_shared, int mode, double ext) {
  const int f = blockIdx.x / nblk, tile = blockIdx.x - f * nblk;
  const int cnt = n * n;
  const int logw = logn < 8 ? logn : 8;  // a tile's columns; its 256 RUN >> logw rows
  const int x = ((tile & ((n >> logw) - 1)) << logw) + (threadIdx.x & ((1 << logw) - 1));
  const int y0 = (tile >> (logn - logw)) * ((256 * RUN) >> logw) + (threadIdx.x >> logw) * RUN;
  const double h = 1.0 / (double)(n - 1);
  const S *ph = phi + (phi_shared ? 0 : (size_t)f * 2 * cnt);
  const S *im = img + (size_t)f * cnt;
  S *o = out + (size_t)f * cnt;
  const double hi = (double)(n - 1);
  S p0[RUN], p1[RUN];
#pragma unroll
  for (int k = 0; k < RUN; ++k) {
    const int j = min(x + (y0 + k) * n, cnt - 1);
    p0[k] = ph[j];
    p1[k] = ph[(size_t)cnt + j];
  }
  double X[RUN], Y[RUN];
  S v[RUN][4];
  bool inside[RUN];
#pragma unroll
  for (int k = 0; k < RUN; ++k) {
    double dx = x + (double)p0[k] / h, dy = (y0 + k) + (double)p1[k] / h;
    inside[k] = true;
    if (mode == 1) {  // clamp
      dx = dx < 0 ? 0 : (dx > hi ? hi : dx);
      dy = dy < 0 ? 0 : (dy > hi ? hi : dy);
    } else {
      if (dx < 0.0 || dx > hi || (mode == 0 && isnan(dx))) inside[k] = false;
      if (dy < 0.0 || dy > hi || (mode == 0 && isnan(dy))) inside[k] = false;
      if (NEAR) {
        dx = floor(dx + 0.5);
        dy = floor(dy + 0.5);
      }
    }
    int xL, yL;  // ScalarArray<QC_2D>::interpolate as interp(), inside the image for every input
    interp_cell(dx, n, xL, X[k]);
    interp_cell(dy, n, yL, Y[k]);
    const S *c = im + xL + (size_t)yL * n;
    v[k][0] = c[0];
    v[k][1] = c[1];
    if (!NEAR || Y[k] != 0) {
      v[k][2] = c[n];
      v[k][3] = c[n + 1];
    } else {
      v[k][2] = v[k][3] = 0;
    }
  }
#pragma unroll
  for (int k = 0; k < RUN; ++k) {
    const double v0 = v[k][0], v1 = v[k][1], v2 = v[k][2], v3 = v[k][3];
    const double r0 = (1 - X[k]) * v0 + X[k] * v1;
    const double r1 = (1 - X[k]) * (1 - Y[k]) * v0 + X[k] * (1 - Y[k]) * v1 + (1 - X[k]) * Y[k] * v2 + X[k] * Y[k] * v3;
    const double r = inside[k] ? (Y[k] == 0 ? r0 : r1) : (mode == 2 ? __builtin_nan("") : ext);
    if (y0 + k < n) o[x + (y0 + k) * n] = static_cast<S>(r);
  }
}

}  // namespace msg
