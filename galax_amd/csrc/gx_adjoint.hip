// gx_adjoint.hip -- discrete adjoint of fixed-step orbit integration.
//
// Gradients of a loss through n independent fixed-step Dopri8/Dopri5 orbit
// integrations, with respect to each orbit's initial state and the
// potential's table parameters.  galax differentiates its solves with
// jax (ForwardMode adjoint, dynamics/_src/orbit/solver.py:133; the stream
// loss derivatives of tests/functional/test_mockstreamgenerator.py:24-116);
// here the derivative of the discrete map is formed exactly, in reverse.
//
// Per orbit (one lane of two waves): a forward sweep stores states, the
// reverse sweep walks the steps backwards, and for every step recomputes its
// stage positions and applies the adjoint of the step.  In Runge-Kutta-
// Nystrom form (stages Q_i, accelerations g_i = a(Q_i), weights b, A, (bA),
// (A A)) the adjoint of one step of size h with output cotangents (qb', pb')
// is
//   gb_j = h b_j pb' + h^2 (bA)_j qb'                 (all stages j)
//   qb = qb',  pb = pb' + h (sum b) qb'
//   for k = S-1 .. 0:
//     Qb_k = -H(Q_k) gb_k          (Hessian-vector product, a = -grad Phi)
//     thb += (da/dtheta (Q_k))^T gb_k
//     qb += Qb_k;  pb += h rs_k Qb_k
//     gb_j += h^2 (A A)_kj Qb_k     (j < k)
// which is the transpose of the forward recurrence in gx_integrate.hip.
// A save time inside a step is the step's dense output,
//   q_s = q + th h p + h^2 th sum_l Wq_l(th) g_l,  p_s = p + h th sum_l Wp_l(th) g_l
// over the stages and the end stage g_E = a(q1) (Dopri8), as the forward
// pass produced it; its cotangents (cq, cp) add
//   gb_l += h^2 th Wq_l cq + h th Wp_l cp,  qb += cq,  pb += th h cq + cp
// and the end stage is reversed first: Q1b = -H(q1) gb_E, thb += ...,
// qb += Q1b, pb += h (sum b) Q1b, gb_j += h^2 (bA)_j Q1b.
#include <cmath>
#include <utility>

#include "gx_internal.hpp"
#include "gx_rk.hpp"
#include "gx_tableau.hpp"

namespace gx {
namespace {

// Orbits of a workgroup: two waves of them, and two more waves for the same
// orbits (see k_adjoint).  One wave of each kind (64 orbits) was as fast
// while every workgroup had a CU of its own, but two workgroups on a CU put
// their second waves on the same SIMD (us a step at 20,000 orbits: 13.7
// against 9.9).
constexpr int kAdjOrbits = 128;
constexpr int kMaxTheta = 12;  // 3 table parameters x up to 4 components

// Every step's start state is kept (56 bytes a step and orbit) where the
// workspace holds them, which saves a third of the forward work; else every
// K-th, and a segment of K steps is integrated again before it is reversed.
// Callers that do not say how much they give keep up to this much: 4 GiB, a
// sixtieth of the device's memory, holds 25,000 orbits of 3,000 steps.
constexpr long long kAllStatesBytes = GX_ADJOINT_STATES_BYTES + 256;

struct AArgs {
  double dt0;
  const double* w0;
  const double* t0;
  const double* t1;
  int t_stride;
  int T;
  int ts_mode;
  int all;            // every step's state is kept: one segment
  long long K;        // steps of a segment
  long long limit;    // steps an orbit may take
  const double* ts;
  const double* cot;  // n x T x 6
  long long n;
  double* w0_bar;     // n x 6
  double* theta_bar;  // n x ntheta
  int ntheta;
  double* ckpt;  // [limit / K][7][n] segment starts (not `all`)
  double* seg;   // [K][7][n] step starts of a segment
  int* status;
};

__device__ __forceinline__ double save_time_a(const AArgs& A, long long i,
                                              int s, double t0, double t1) {
  switch (A.ts_mode) {
    case GX_TS_SHARED:
      return A.ts[s];
    case GX_TS_PER_ORBIT:
      return A.ts[i * A.T + s];
    case GX_TS_LINSPACE:
      return (s == A.T - 1) ? t1 : t0 + s * ((t1 - t0) / (A.T - 1));
    default:
      return t1;
  }
}

__device__ __forceinline__ double clip_end(double tprev, double tnext,
                                           double t1) {
  return (tnext > t1 - 1e-10) ? t1 : tnext;
}

// Forward step (no error estimate); optionally records the stage positions
// and the step's end in this lane's column of st.
template <class M, class E, bool REC>
__device__ __forceinline__ void step_fwd(const DPot& P, double* st, double h,
                                         double (&q)[3], double (&p)[3]) {
  constexpr int S = M::S;
  double g[S][3];
#pragma unroll
  for (int k = 0; k < S; ++k) {
    double Q[3];
    if (k == 0) {
      Q[0] = q[0];
      Q[1] = q[1];
      Q[2] = q[2];
    } else {
      double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
      for (int l = 0; l < k; ++l) {
        const double a = M::k.aa[k][l];
        if (a != 0.0) {
          s0 = fma(a, g[l][0], s0);
          s1 = fma(a, g[l][1], s1);
          s2 = fma(a, g[l][2], s2);
        }
      }
      const double rs = M::k.rs[k];
      Q[0] = fma(h, fma(rs, p[0], h * s0), q[0]);
      Q[1] = fma(h, fma(rs, p[1], h * s1), q[1]);
      Q[2] = fma(h, fma(rs, p[2], h * s2), q[2]);
    }
    if (REC) {
#pragma unroll
      for (int m = 0; m < 3; ++m) st[(k * 3 + m) * kAdjOrbits] = Q[m];
    }
    E::acc(P, Q[0], Q[1], Q[2], 0.0, g[k][0], g[k][1], g[k][2]);
  }
  double b0 = 0, b1 = 0, b2 = 0, c0 = 0, c1 = 0, c2 = 0;
#pragma unroll
  for (int l = 0; l < S; ++l) {
    if (M::k.b[l] != 0.0) {
      b0 = fma(M::k.b[l], g[l][0], b0);
      b1 = fma(M::k.b[l], g[l][1], b1);
      b2 = fma(M::k.b[l], g[l][2], b2);
    }
    if (M::k.ba[l] != 0.0) {
      c0 = fma(M::k.ba[l], g[l][0], c0);
      c1 = fma(M::k.ba[l], g[l][1], c1);
      c2 = fma(M::k.ba[l], g[l][2], c2);
    }
  }
  constexpr double sb = M::k.sb;
  const double q0 = fma(h, fma(sb, p[0], h * c0), q[0]);
  const double q1 = fma(h, fma(sb, p[1], h * c1), q[1]);
  const double q2 = fma(h, fma(sb, p[2], h * c2), q[2]);
  if (REC && M::SF > S) {
    st[(S * 3 + 0) * kAdjOrbits] = q0;
    st[(S * 3 + 1) * kAdjOrbits] = q1;
    st[(S * 3 + 2) * kAdjOrbits] = q2;
  }
  p[0] = fma(h, b0, p[0]);
  p[1] = fma(h, b1, p[1]);
  p[2] = fma(h, b2, p[2]);
  q[0] = q0;
  q[1] = q1;
  q[2] = q2;
}

// What a lane carries from step to step: in the first set of waves (see
// k_adjoint) a step's start state q, p and, in th[0], its time; in the second
// the cotangents of a state and of the parameters.  One set of registers
// serves both.
struct Carry {
  double q[3], p[3], th[kMaxTheta];
};

// State rows [7][n] in memory: q, p, tau of orbit i.
__device__ __forceinline__ void put_state(double* row, long long n, long long i, const Carry& s) {
  double* r = row + i;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    r[m * n] = s.q[m];
    r[(m + 3) * n] = s.p[m];
  }
  r[6 * n] = s.th[0];
}
__device__ __forceinline__ void get_state(const double* row, long long n, long long i, Carry& s) {
  const double* r = row + i;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    s.q[m] = r[m * n];
    s.p[m] = r[(m + 3) * n];
  }
  s.th[0] = r[6 * n];
}

__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return v;
}

__device__ __forceinline__ void add_save(const AArgs& A, long long i, int s, double dir, Carry& b) {
  const double* c = A.cot + (i * A.T + s) * 6;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    b.q[m] += c[m];
    b.p[m] += dir * c[m + 3];
  }
}

// Adjoint of one step of size h, whose stage positions are in this lane's
// column of st: b holds the cotangents of the step's end on entry and those
// of its start on return.  Save times inside the step (their index counts
// down in si) add to the stage and state cotangents; with none the end stage
// is skipped.
template <class M, class F>
__device__ __forceinline__ void step_adj(const DPot& P, const AArgs& A, const double* st,
                                         long long i, double dir, double t0v, double t1v,
                                         double tau, double tau1, int& si, Carry& b) {
  constexpr int S = M::S;
  constexpr int SF = M::SF;
  const double h = tau1 - tau, h2 = h * h;
  double gb[SF][3];
#pragma unroll
  for (int j = 0; j < SF; ++j)
#pragma unroll
    for (int m = 0; m < 3; ++m)
      gb[j][m] = j < S ? fma(h * M::k.b[j < S ? j : 0], b.p[m], h2 * M::k.ba[j < S ? j : 0] * b.q[m])
                       : 0.0;
  constexpr double sb = M::k.sb;
#pragma unroll
  for (int m = 0; m < 3; ++m) b.p[m] = fma(h * sb, b.q[m], b.p[m]);
  // saves inside: the step's dense output at th = (t_s - tau) / h
  bool any_save = false;
  while (si >= 0) {
    const double tsv = dir * save_time_a(A, i, si, t0v, t1v);
    if (!(tsv > tau && tsv < tau1)) break;
    const double* c = A.cot + (i * A.T + si) * 6;
    const double cq[3] = {c[0], c[1], c[2]}, cp[3] = {dir * c[3], dir * c[4], dir * c[5]};
    const double tht = (tsv - tau) / h;
    const double ht = h * tht, hht = h * ht;
    // one stage's weights at a time: all of them at once do not fit beside
    // the stage cotangents
    constexpr int D = sizeof(M::dn.wq[0]) / sizeof(double);
    ConstDouble* tq = table_here(&M::dn.wq[0][0]);
    ConstDouble* tp = table_here(&M::dn.wp[0][0]);
#pragma unroll
    for (int l = 0; l < SF; ++l) {
      if (M::dn.nq[l]) {
        const double w = hht * horner_here<D>(tq + D * l, tht);
#pragma unroll
        for (int m = 0; m < 3; ++m) gb[l][m] = fma(w, cq[m], gb[l][m]);
      }
      if (M::dn.np[l]) {
        const double w = ht * horner_here<D>(tp + D * l, tht);
#pragma unroll
        for (int m = 0; m < 3; ++m) gb[l][m] = fma(w, cp[m], gb[l][m]);
      }
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      b.q[m] += cq[m];
      b.p[m] = fma(ht, cq[m], b.p[m] + cp[m]);
    }
    any_save = true;
    --si;
  }
  auto stage = [&](int k, const double (&w)[3], double (&Hw)[3]) {
    double Q[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) Q[m] = st[(k * 3 + m) * kAdjOrbits];
    F::adjoint(P, Q, w, Hw, b.th);
  };
  if constexpr (SF > S) {
    if (any_save) {
      // the end stage g_E = a(q1), q1 = q + h (sb p + h sum (bA)_j g_j)
      double Hw[3];
      stage(S, gb[S], Hw);
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        b.q[m] -= Hw[m];
        b.p[m] = fma(-h * sb, Hw[m], b.p[m]);
      }
#pragma unroll
      for (int j = 0; j < S; ++j) {
        const double a = M::k.ba[j];
        if (a != 0.0) {
#pragma unroll
          for (int m = 0; m < 3; ++m) gb[j][m] = fma(-h2 * a, Hw[m], gb[j][m]);
        }
      }
    }
  }
#pragma unroll
  for (int k = S - 1; k >= 0; --k) {
    double Hw[3];
    stage(k, gb[k], Hw);
    // Qb_k = -H gb_k
    const double rs = M::k.rs[k];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      b.q[m] -= Hw[m];
      b.p[m] = fma(-h * rs, Hw[m], b.p[m]);
      Hw[m] *= -h2;
    }
#pragma unroll
    for (int j = 0; j < k; ++j) {
      const double a = M::k.aa[k][j];
      if (a != 0.0) {
#pragma unroll
        for (int m = 0; m < 3; ++m) gb[j][m] = fma(a, Hw[m], gb[j][m]);
      }
    }
  }
}

// Two sets of waves share a workgroup's orbits.  A step back needs its stage positions (13
// field evaluations from the step's start state, independent of the
// cotangents) and then 13 Hessian-vector products with the parameter
// partials, one after the other.  The first set recomputes the positions
// of one step into LDS while the second reverses the step after it, from the
// other of two buffers.  A stream fit's orbits fill a third of the device's
// SIMDs, so the second set costs nothing there.  Bound by instructions in
// flight of one wave per SIMD: a step takes 4.4 us forward and 5.5 us back
// up to 32,768 orbits (32.5 us in all with one set, IEEE divisions, 400
// spilled registers and the stage positions in HBM); 131,072 orbits, which
// fill the device, take 39 us a step (70).  20,000 orbits of up to 1,000
// steps: 39.0 ms before, 12.4 ms.
// The kernels' registers are checked in the tests: with spills the compiler
// has stored a spilled parameter cotangent before restoring the execution
// mask after a divergent loop, so that it was lost in some lanes.
template <class M, class F>
__global__ void __launch_bounds__(2 * kAdjOrbits)
    __attribute__((amdgpu_waves_per_eu(2))) k_adjoint(DPot P, AArgs A) {
  __shared__ double st[2][3 * M::SF + 1][kAdjOrbits];  // stage positions, tau
  __shared__ int steps[kAdjOrbits], stat[kAdjOrbits];
  const int lane = threadIdx.x & (kAdjOrbits - 1);  // the orbit in the workgroup
  const bool first = __builtin_amdgcn_readfirstlane(threadIdx.x) < kAdjOrbits;
  const long long i = (long long)blockIdx.x * kAdjOrbits + lane;
  const bool valid = i < A.n;
  const long long ic = valid ? i : 0;
  const double t0v = A.t0[A.t_stride ? ic : 0];
  const double t1v = A.t1[A.t_stride ? ic : 0];
  const double dir = (t0v < t1v) ? 1.0 : -1.0;
  const double tau1 = dir * t1v;
  // the end of step n from its start
  auto next_tau = [&](long long n, double tau) {
    return n == 0 ? fmin(tau + A.dt0, tau1) : clip_end(tau, tau + A.dt0, tau1);
  };

  Carry s;
#pragma unroll
  for (int m = 0; m < 3; ++m) s.q[m] = s.p[m] = 0.0;
#pragma unroll
  for (int k = 0; k < kMaxTheta; ++k) s.th[k] = 0.0;
  // ---- forward sweep, by the first set
  if (first) {
    long long N = 0;
    int status = GX_SUCCESS;
    const double* w = A.w0 + ic * 6;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      s.q[m] = w[m];
      s.p[m] = dir * w[3 + m];
    }
    double tau = dir * t0v;
    long long in_seg = 0;
    while (valid && t0v != t1v && tau < tau1) {
      if (N >= A.limit) {
        status = GX_MAX_STEPS_REACHED;
        break;
      }
      s.th[0] = tau;
      if (A.all)
        put_state(A.seg + N * 7 * A.n, A.n, i, s);
      else if (in_seg == 0)
        put_state(A.ckpt + N / A.K * 7 * A.n, A.n, i, s);
      in_seg = in_seg + 1 == A.K ? 0 : in_seg + 1;
      const double tn = next_tau(N, tau);
      step_fwd<M, F, false>(P, nullptr, tn - tau, s.q, s.p);
      ++N;
      tau = tn;
    }
    steps[lane] = status == GX_SUCCESS ? (int)N : 0;
    stat[lane] = status;
  }
  __syncthreads();
  const long long N = steps[lane];
  const int status = stat[lane];

  // ---- reverse sweep
  int si = A.T - 1;
  const long long nseg = (N + A.K - 1) / A.K;
  // trip counts that every wave agrees on: the longest orbit's
  const int other = steps[lane ^ 64];
  const int trips = wave_max((int)((max((int)N, other) + A.K - 1) / A.K));
  for (int it = 0; it < trips; ++it) {
    const long long c = nseg - 1 - it;
    const long long n0 = c * A.K;
    const int len = c < 0 ? 0 : (int)(N - n0 < A.K ? N - n0 : A.K);
    const long long oc = (other + A.K - 1) / A.K - 1 - it;
    const int olen = oc < 0 ? 0 : (int)(other - oc * A.K < A.K ? other - oc * A.K : A.K);
    const int longest = wave_max(max(len, olen));
    if (first && !A.all && len > 0) {
      // the segment's step starts again
      get_state(A.ckpt + c * 7 * A.n, A.n, i, s);
      for (int m = 0; m < len; ++m) {
        put_state(A.seg + (long long)m * 7 * A.n, A.n, i, s);
        if (m + 1 < len) {
          const double tn = next_tau(n0 + m, s.th[0]);
          step_fwd<M, F, false>(P, nullptr, tn - s.th[0], s.q, s.p);
          s.th[0] = tn;
        }
      }
    }
    if (first && len > 0) get_state(A.seg + (long long)(len - 1) * 7 * A.n, A.n, i, s);
    for (int k = 0; k <= longest; ++k) {
      if (first) {
        const int m = len - 1 - k;
        if (m >= 0) {
          Carry ahead = s;
          if (m > 0) get_state(A.seg + (long long)(m - 1) * 7 * A.n, A.n, i, ahead);
          double* col = &st[k & 1][0][lane];
          col[3 * M::SF * kAdjOrbits] = s.th[0];
          step_fwd<M, F, true>(P, col, next_tau(n0 + m, s.th[0]) - s.th[0], s.q, s.p);
#pragma unroll
          for (int j = 0; j < 3; ++j) {
            s.q[j] = ahead.q[j];
            s.p[j] = ahead.p[j];
          }
          s.th[0] = ahead.th[0];
        }
      } else {
        const int m = len - k;
        if (k > 0 && m >= 0) {
          const double* col = &st[(k - 1) & 1][0][lane];
          const double tau = col[3 * M::SF * kAdjOrbits];
          const double tau_e = next_tau(n0 + m, tau);
          // saves at the step end
          while (si >= 0 && dir * save_time_a(A, i, si, t0v, t1v) == tau_e) add_save(A, i, si--, dir, s);
          step_adj<M, F>(P, A, col, i, dir, t0v, t1v, tau, tau_e, si, s);
        }
      }
      __syncthreads();
    }
  }
  if (first || !valid) return;
  // saves at (or before) the start
  if (status == GX_SUCCESS)
    while (si >= 0) add_save(A, i, si--, dir, s);
  double* wb = A.w0_bar + i * 6;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    wb[m] = s.q[m];
    wb[3 + m] = dir * s.p[m];
  }
#pragma unroll
  for (int k = 0; k < kMaxTheta; ++k)
    if (k < A.ntheta) A.theta_bar[i * A.ntheta + k] = s.th[k];
  if (A.status) A.status[i] = status;
}

template <class M, class F>
int launch_adj(const gx_pot* pot, AArgs& A, hipStream_t s) {
  const long long blocks = (A.n + kAdjOrbits - 1) / kAdjOrbits;
  if (blocks > 0x7fffffffLL) return GX_EINVAL;
  hipLaunchKernelGGL((k_adjoint<M, F>), dim3((unsigned)blocks), dim3(2 * kAdjOrbits), 0, s,
                     pot->dev, A);
  return check(hipGetLastError());
}

template <class M>
int dispatch_adj(const gx_pot* pot, AArgs& A, hipStream_t s) {
  if (pot->sig == kSigMilkyWay) return launch_adj<M, AdjointMW>(pot, A, s);
  if (pot->ncomp == 1 && pot->basic) {
    switch (pot->kind0) {
      case GX_KEPLER:
        return launch_adj<M, AdjointFixed<GX_KEPLER>>(pot, A, s);
      case GX_HERNQUIST:
        return launch_adj<M, AdjointFixed<GX_HERNQUIST>>(pot, A, s);
      case GX_MIYAMOTO_NAGAI:
        return launch_adj<M, AdjointFixed<GX_MIYAMOTO_NAGAI>>(pot, A, s);
      case GX_NFW:
        return launch_adj<M, AdjointFixed<GX_NFW>>(pot, A, s);
      case GX_PLUMMER:
        return launch_adj<M, AdjointFixed<GX_PLUMMER>>(pot, A, s);
      default:
        break;
    }
  }
  return GX_EINVAL;
}

}  // namespace
}  // namespace gx

using namespace gx;

namespace {

// Steps an orbit may take: whole segments, at least max_steps.
int64_t step_limit(int64_t max_steps, int64_t K) { return (max_steps / K + 2) * K; }

// Workspaces: every step's state (56 bytes), or those of the segment starts
// and of one segment.
bool all_states(int64_t n, int64_t max_steps, int64_t K, int64_t bytes) {
  return n == 0 || (bytes >= 256 && step_limit(max_steps, K) <= (bytes - 256) / 56 / n);
}
int64_t all_bytes(int64_t n, int64_t max_steps, int64_t K) {
  return 56 * n * step_limit(max_steps, K) + 256;
}
int64_t checkpoint_bytes(int64_t n, int64_t max_steps, int64_t K) {
  return 56 * n * (max_steps / K + 2 + K) + 256;
}

}  // namespace

extern "C" {

int64_t gx_adjoint_workspace_within(int64_t n, int64_t max_steps, int32_t K, int64_t bytes) {
  if (n < 0 || max_steps < 0 || K < 1) return 0;
  return all_states(n, max_steps, K, bytes) ? all_bytes(n, max_steps, K)
                                            : checkpoint_bytes(n, max_steps, K);
}

int64_t gx_adjoint_workspace_bytes(int64_t n, int64_t max_steps, int32_t K) {
  if (n < 0 || max_steps < 0 || K < 1) return 0;
  if (all_states(n, max_steps, K, kAllStatesBytes)) return all_bytes(n, max_steps, K);
  // not less than any smaller batch or span takes, whose states may all be kept
  const int64_t checkpointed = checkpoint_bytes(n, max_steps, K);
  return checkpointed > kAllStatesBytes ? checkpointed : kAllStatesBytes;
}

int gx_adjoint(const gx_pot* pot, const gx_solver_cfg* cfg, const double* w0,
               const double* t0, const double* t1, int32_t t_stride,
               const double* ts, int32_t T, int32_t ts_mode, int64_t n,
               const double* cot, double* w0_bar, double* theta_bar,
               int32_t ntheta, int64_t max_steps, int32_t K, int32_t* status,
               void* workspace, void* stream) {
  return gx_adjoint_within(pot, cfg, w0, t0, t1, t_stride, ts, T, ts_mode, n, cot, w0_bar, theta_bar,
                           ntheta, max_steps, K, status, workspace,
                           gx_adjoint_workspace_bytes(n, max_steps, K), stream);
}

int gx_adjoint_within(const gx_pot* pot, const gx_solver_cfg* cfg, const double* w0,
                      const double* t0, const double* t1, int32_t t_stride,
                      const double* ts, int32_t T, int32_t ts_mode, int64_t n,
                      const double* cot, double* w0_bar, double* theta_bar,
                      int32_t ntheta, int64_t max_steps, int32_t K, int32_t* status,
                      void* workspace, int64_t workspace_bytes, void* stream) {
  if (!pot || !cfg || n < 0 || T < 1 || K < 1 || max_steps < 1) return GX_EINVAL;
  if (n == 0) return GX_OK;
  if (!w0 || !t0 || !t1 || !cot || !w0_bar || !workspace) return GX_EINVAL;
  if (ntheta < 0 || ntheta > kMaxTheta || (ntheta > 0 && !theta_bar)) return GX_EINVAL;
  if (cfg->controller != GX_CONSTANT || !(cfg->dt0 > 0.0)) return GX_EINVAL;
  if (cfg->method != GX_DOPRI8 && cfg->method != GX_DOPRI5) return GX_EINVAL;
  if (t_stride != 0 && t_stride != 1) return GX_EINVAL;
  if (ts_mode < GX_TS_SHARED || ts_mode > GX_TS_FINAL) return GX_EINVAL;
  if ((ts_mode == GX_TS_SHARED || ts_mode == GX_TS_PER_ORBIT) && !ts) return GX_EINVAL;
  if (ts_mode == GX_TS_FINAL && T != 1) return GX_EINVAL;
  const bool all = all_states(n, max_steps, K, workspace_bytes);
  if (!all && workspace_bytes < checkpoint_bytes(n, max_steps, K)) return GX_EINVAL;
  AArgs A{};
  A.dt0 = cfg->dt0;
  A.w0 = w0;
  A.t0 = t0;
  A.t1 = t1;
  A.t_stride = t_stride;
  A.T = T;
  A.ts_mode = ts_mode;
  A.limit = step_limit(max_steps, K);
  A.all = all ? 1 : 0;
  A.K = A.all ? A.limit : K;
  A.ts = ts;
  A.cot = cot;
  A.n = n;
  A.w0_bar = w0_bar;
  A.theta_bar = theta_bar;
  A.ntheta = ntheta;
  A.status = status;
  char* ws = static_cast<char*>(workspace);
  A.ckpt = reinterpret_cast<double*>(ws);
  A.seg = A.all ? A.ckpt : A.ckpt + 7 * (A.limit / K) * n;
  hipStream_t s = (hipStream_t)stream;
  if (cfg->method == GX_DOPRI8) return dispatch_adj<Dopri8>(pot, A, s);
  return dispatch_adj<Dopri5>(pot, A, s);
}

}  // extern "C"
