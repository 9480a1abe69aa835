// gx_steps.hpp -- what the independent-orbit integrator's kernels share: their
// arguments, save times, and the step-size controller.
#pragma once

#include "gx_internal.hpp"
#include "gx_rk.hpp"

namespace gx {
namespace {

struct IArgs {
  double dt0, rtol, atol, safety, factormin, factormax, dtmin, dtmax;
  double c1, c2, c3;  // PID exponents (i+p+d)/k, -(p+2d)/k, d/k
  long long max_steps;
  int force_dtmin;
  int t_stride;
  int T;
  int ts_mode;
  int root8;  // c1 == 1/8 and c2 == c3 == 0: factor from three square roots
  const double* w0;
  const double* t0;
  const double* t1;
  const double* ts;
  long long n;
  const long long* order;
  double* out;
  int* status;
  long long* nsteps;
  long long* naccept;
  unsigned long long* counter;
  double* h0;  // first step per orbit, from the prepass (workspace)
  double* a0;  // start acceleration per orbit [n][3], from the prepass
  long long fixed_lanes;  // lanes that start on a fixed ticket
  long long head_lanes;  // the first of them, on the longest orbits
  int head_only_once;    // head lanes take no second ticket
  int chunk;             // tickets taken from the queue at a time
  double* rec;           // dense records [n][rec_cap][kDenseRec] (dense mode)
  long long rec_cap;
  long long* nrec;       // records written per orbit
  // which of two launches takes the batch is decided on the device (`choose`):
  // teams if its work (TeamLoad) is at most `most` times its longest orbit's and
  // it has at most one save to `step` units of it
  int choose;
  double most, step;
};

// What a batch asks of the integrators, summed up by the first-step prepass
// beside the workspace's counter (256 bytes).
struct TeamLoad {
  double sum, longest;
};
__device__ __forceinline__ TeamLoad* team_load(const IArgs& A) {
  return reinterpret_cast<TeamLoad*>(A.counter + 1);
}
__device__ __forceinline__ bool teams_take(const IArgs& A) {
  const TeamLoad& l = *team_load(A);
  return l.sum <= A.most * l.longest && (A.T == 1 || (double)A.n * A.T * A.step <= l.sum);
}

__device__ __forceinline__ double clip_to_end(double tprev, double tnext,
                                              double t1, bool keep) {
  return (tnext > t1 - 1e-10) ? (keep ? t1 : tprev + 0.5 * (t1 - tprev))
                              : tnext;
}

__device__ __forceinline__ double save_time(const IArgs& A, long long orb,
                                            int s, double t0, double t1) {
  switch (A.ts_mode) {
    case GX_TS_SHARED:
      return A.ts[s];
    case GX_TS_PER_ORBIT:
      return A.ts[orb * A.T + s];
    case GX_TS_LINSPACE:
      return (s == A.T - 1) ? t1 : t0 + s * ((t1 - t0) / (A.T - 1));
    default:
      return t1;
  }
}

__device__ __forceinline__ void orbit_span(const IArgs& A, long long orb, double& t0,
                                           double& t1) {
  t0 = A.t0[A.t_stride ? orb : 0];
  t1 = A.t1[A.t_stride ? orb : 0];
}

__device__ __forceinline__ void write_save(const IArgs& A, long long orb,
                                           int s, double dir,
                                           const double (&q)[3],
                                           const double (&p)[3]) {
  double* o = A.out + (orb * A.T + s) * 6;
  o[0] = q[0];
  o[1] = q[1];
  o[2] = q[2];
  o[3] = dir * p[0];
  o[4] = dir * p[1];
  o[5] = dir * p[2];
}

// NaN for the saves from s on.
__device__ __forceinline__ void write_rest(const IArgs& A, long long orb, int s) {
  const double nanv = __longlong_as_double(0x7ff8000000000000ULL);
  const double nq[3] = {nanv, nanv, nanv};
  for (; s < A.T; ++s) write_save(A, orb, s, 1.0, nq, nq);
}

__device__ __forceinline__ long long ticket_to_orbit(const IArgs& A,
                                                     long long idx) {
  if (idx >= A.n) return -1;
  if (!A.order) return idx;
  const long long o = A.order[idx];
  return (o >= 0 && o < A.n) ? o : -1;  // the host validates permutations
}

// The next step after an attempted one from (tau, q, p) to (tnext, q1, p1)
// with error estimate (eq, ep): whether it is accepted, and in next_t1 where
// the attempt after it would end.  diffrax's RMS norm of the scaled error is
// taken through its mean square ms (the norm is below 1 exactly when ms is);
// quotients and roots by the short primitives, within about an ulp of the
// correctly rounded operation.
template <bool PID>
__device__ __forceinline__ bool control_step(
    const IArgs& A, double tau, double tnext, const double (&q)[3],
    const double (&p)[3], const double (&q1)[3], const double (&p1)[3],
    const double (&eq)[3], const double (&ep)[3], double& prev_inv,
    double& prev_prev_inv, int& at_dtmin, int& st, double& next_t1) {
  if (!PID) {
    next_t1 = tnext + A.dt0;
    return true;
  }
  const double h = tnext - tau;
  double sq = 0.0;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const double uq =
        eq[m] * rcp(A.atol + fmax(fabs(q[m]), fabs(q1[m])) * A.rtol);
    const double up =
        ep[m] * rcp(A.atol + fmax(fabs(p[m]), fabs(p1[m])) * A.rtol);
    sq += uq * uq + up * up;
  }
  const double ms = div6(sq);
  bool keep = ms < 1.0;
  if (A.dtmin > 0.0) keep = keep || at_dtmin != 0;
  // inv = 1 / norm = ms^(-1/2); zero (and subnormal) ms gives +inf, infinite
  // ms 0, NaN stays NaN
  const bool normal = ms >= kMinNormal && ms <= kMaxFinite;
  const double special = (ms < kMinNormal)   ? __builtin_inf()
                         : (ms > kMaxFinite) ? 0.0
                                             : ms;
  const double a = rsqrt_fast(ms);
  const double inv = normal ? a : special;
  double f;
  if (A.root8) {
    // inv^(1/8) = 1 / rsqrt(rsqrt(rsqrt(inv)))
    f = normal ? rcp(rsqrt_fast(rsqrt_fast(rsqrt_fast(a)))) : special;
  } else {
    f = (A.c1 == 0.0) ? 1.0 : pow(inv, A.c1);
    if (A.c2 != 0.0) f *= pow(prev_inv, A.c2);
    if (A.c3 != 0.0) f *= pow(prev_prev_inv, A.c3);
  }
  const double fmin_ = keep ? 1.0 : A.factormin;
  const double factor = fmin(fmax(A.safety * f, fmin_), A.factormax);
  double dt = fmin(h * factor, A.dtmax);
  if (A.dtmin > 0.0) {
    if (!A.force_dtmin && dt < A.dtmin) st = GX_DT_MIN_REACHED;
    at_dtmin = dt <= A.dtmin ? 1 : 0;
    dt = fmax(dt, A.dtmin);
  }
  if (keep) {
    // a zero or infinite error does not steer later steps
    prev_prev_inv = prev_inv;
    prev_inv = (inv == 0.0 || isinf(inv)) ? 1.0 : inv;
  }
  next_t1 = (keep ? tnext : tau) + dt;
  return keep;
}

}  // namespace
}  // namespace gx
