// gx_nbody.hip -- direct-summation N-body field and its integrator.
//
// galax's NBodyField (dynamics/_src/orbit/field_nbody.py:94-131):
//   a_j = sum_{i != j} G m_i (x_i - x_j) / (|x_i - x_j|^2 + eps^2)^(3/2)
//         - grad Phi_ext(x_j, t),
// integrated as ONE system by OrbitSolver (shared steps; the PID error norm
// is the RMS over all 6N state components, orbit/solver.py:121-141).
//
// One launch integrates the whole system (N <= 4096, the range in which the
// reference's (N, N, 3) pair arrays are practical), with no host round trip
// per step: k_nbody_grid divides the bodies among the workgroups of a
// cooperative launch.  Where that cannot be launched (a stream capture, a
// device partition too small), and for a few bodies, k_nbody integrates the
// system in one workgroup of 512 threads: the stage positions of all bodies sit in LDS,
// every thread sums the pull of all bodies on its own bodies (all lanes read
// the same LDS word: a broadcast), stage accelerations go to a workspace in
// HBM, and the error norm is a block reduction.
#include <hip/hip_runtime.h>

#include <cmath>

#include "gx_internal.hpp"
#include "gx_potential.hpp"
#include "gx_rk.hpp"
#include "gx_slots.hpp"
#include "gx_tableau.hpp"

namespace gx {
namespace {

constexpr int kNbThreads = 512;
constexpr int kNbMax = 4096;
// Bodies that one workgroup integrates, and fewest bodies of a workgroup when
// there are several.  A meeting takes about 4 us whatever its size; one
// workgroup takes that long for the pulls of 50 to 60 bodies (us a step, one
// against several workgroups: 37 bodies 67/72, 64 bodies 73/68, 96 bodies
// 112/69).  Workgroups of 4 bodies against 8: 1,024 bodies 103 us a step
// against 125, 128 bodies 71 against 73 (smaller ones change nothing).
constexpr int kNbOne = 48;
constexpr int kNbOwnMin = 4;

struct NArgs {
  double dt0, rtol, atol, safety, factormin, factormax, dtmin, dtmax;
  double c1, c2, c3;
  long long max_steps;
  int force_dtmin;
  int T;
  double eps2;
  double t0, t1;
  const double* gm;  // [n] G m
  const double* w0;  // [n][6]
  const double* ts;  // [T]
  long long n;
  double* out;       // [n][T][6]
  int* status;
  long long* nsteps;
  long long* naccept;
  double* q;         // workspace: state [n][3] (positions, solver-time velocities)
  double* p;
  double* q1;        // end of the current step [n][3]
  double* p1;
  double* G;         // stage accelerations [SF][n][3] (slot SF-1: the end stage)
};

struct NbShared {
  double x[kNbMax], y[kNbMax], z[kNbMax], gm[kNbMax];
  double red[kNbThreads / 64];
};

__device__ __forceinline__ double block_sum(NbShared& S, double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) S.red[w] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < kNbThreads / 64; ++i) s += S.red[i];
  return s;
}

// Acceleration of body j at (x, y, z) from the positions in LDS and the
// external field at physical time t.
__device__ __forceinline__ void nb_accel(const DPot& P, const NbShared& S, long long n,
                                         double eps2, long long j, double x, double y,
                                         double z, double t, double& ax, double& ay,
                                         double& az) {
  accel<true>(P, x, y, z, t, ax, ay, az);
  for (long long k = 0; k < n; ++k) {
    const double dx = S.x[k] - x, dy = S.y[k] - y, dz = S.z[k] - z;
    const double r2 = dx * dx + dy * dy + dz * dz + eps2;
    const double ir = rsqrt_fast(r2);
    const double w = (k == j) ? 0.0 : S.gm[k] * ir * ir * ir;
    ax = fma(w, dx, ax);
    ay = fma(w, dy, ay);
    az = fma(w, dz, az);
  }
}

// One method evaluation for the whole system from (q, p) at solver time tau
// with step h: writes q1, p1 and (ERR) returns the squared scaled error sum
// of this thread's bodies.
template <class M, bool ERR>
__device__ double nb_eval(const DPot& P, NbShared& S, const NArgs& A, double dir,
                          double tau, double h) {
  constexpr auto& K = M::k;
  const long long n = A.n;
  const int tid = threadIdx.x;
  for (int i = 0; i < M::S; ++i) {
    const double ti = dir * fma(K.c[i], h, tau);
    // stage positions of own bodies into LDS
    for (long long j = tid; j < n; j += kNbThreads) {
      double s[3] = {0.0, 0.0, 0.0};
      for (int l = 0; l < i; ++l) {
        const double a = K.aa[i][l];
        if (a != 0.0)
          for (int m = 0; m < 3; ++m) s[m] = fma(a, A.G[((long long)l * n + j) * 3 + m], s[m]);
      }
      const double rs = K.rs[i];
      S.x[j] = fma(h, fma(rs, A.p[3 * j], h * s[0]), A.q[3 * j]);
      S.y[j] = fma(h, fma(rs, A.p[3 * j + 1], h * s[1]), A.q[3 * j + 1]);
      S.z[j] = fma(h, fma(rs, A.p[3 * j + 2], h * s[2]), A.q[3 * j + 2]);
    }
    __syncthreads();
    for (long long j = tid; j < n; j += kNbThreads) {
      double ax, ay, az;
      nb_accel(P, S, n, A.eps2, j, S.x[j], S.y[j], S.z[j], ti, ax, ay, az);
      double* g = A.G + ((long long)i * n + j) * 3;
      g[0] = ax;
      g[1] = ay;
      g[2] = az;
    }
    __syncthreads();
  }
  double sq = 0.0;
  for (long long j = tid; j < n; j += kNbThreads) {
    double b[3] = {0.0, 0.0, 0.0}, ba[3] = {0.0, 0.0, 0.0};
    double e[3] = {0.0, 0.0, 0.0}, ea[3] = {0.0, 0.0, 0.0};
    for (int l = 0; l < M::S; ++l) {
      for (int m = 0; m < 3; ++m) {
        const double gl = A.G[((long long)l * n + j) * 3 + m];
        if (K.b[l] != 0.0) b[m] = fma(K.b[l], gl, b[m]);
        if (K.ba[l] != 0.0) ba[m] = fma(K.ba[l], gl, ba[m]);
        if (ERR && K.e[l] != 0.0) e[m] = fma(K.e[l], gl, e[m]);
        if (ERR && K.ea[l] != 0.0) ea[m] = fma(K.ea[l], gl, ea[m]);
      }
    }
    for (int m = 0; m < 3; ++m) {
      const double q0 = A.q[3 * j + m], p0 = A.p[3 * j + m];
      const double q1 = fma(h, fma(K.sb, p0, h * ba[m]), q0);
      const double p1 = fma(h, b[m], p0);
      A.q1[3 * j + m] = q1;
      A.p1[3 * j + m] = p1;
      if (ERR) {
        const double eq = h * fma(K.se, p0, h * ea[m]);
        const double ep = h * e[m];
        const double uq = eq / (A.atol + fmax(fabs(q0), fabs(q1)) * A.rtol);
        const double up = ep / (A.atol + fmax(fabs(p0), fabs(p1)) * A.rtol);
        sq += uq * uq + up * up;
      }
    }
  }
  return sq;
}

__device__ void nb_write(const NArgs& A, int s, double dir, const double* q, const double* p) {
  for (long long j = threadIdx.x; j < A.n; j += kNbThreads) {
    double* o = A.out + (j * A.T + s) * 6;
    for (int m = 0; m < 3; ++m) {
      o[m] = q[3 * j + m];
      o[3 + m] = dir * p[3 * j + m];
    }
  }
}

template <class M, bool PID>
__global__ void __launch_bounds__(kNbThreads) k_nbody(DPot P, NArgs A) {
  __shared__ NbShared S;
  const long long n = A.n;
  const int tid = threadIdx.x;
  const double dir = (A.t0 < A.t1) ? 1.0 : -1.0;
  for (long long j = tid; j < n; j += kNbThreads) {
    S.gm[j] = A.gm[j];
    for (int m = 0; m < 3; ++m) {
      A.q[3 * j + m] = A.w0[6 * j + m];
      A.p[3 * j + m] = dir * A.w0[6 * j + 3 + m];
    }
  }
  __syncthreads();
  double tau = dir * A.t0;
  const double tau1 = dir * A.t1;
  int si = 0;
  while (si < A.T && dir * A.ts[si] <= tau) nb_write(A, si++, dir, A.q, A.p);
  int status = GX_SUCCESS;
  long long nst = 0, nacc = 0;
  if (A.t0 != A.t1) {
    // first step: dt0; dtmin if the controller sets one (as the orbit
    // integrators); else diffrax's initial-step heuristic over the system
    double h0 = A.dt0 > 0.0 ? A.dt0 : (PID && A.dtmin > 0.0 ? A.dtmin : 0.0);
    if (!(h0 > 0.0)) {
      double s0 = 0.0, s1 = 0.0;
      for (long long j = tid; j < n; j += kNbThreads) {
        S.x[j] = A.q[3 * j];
        S.y[j] = A.q[3 * j + 1];
        S.z[j] = A.q[3 * j + 2];
      }
      __syncthreads();
      for (long long j = tid; j < n; j += kNbThreads) {
        double a[3];
        nb_accel(P, S, n, A.eps2, j, S.x[j], S.y[j], S.z[j], dir * tau, a[0], a[1], a[2]);
        for (int m = 0; m < 3; ++m) {
          const double sq = A.atol + fabs(A.q[3 * j + m]) * A.rtol;
          const double sp = A.atol + fabs(A.p[3 * j + m]) * A.rtol;
          s0 += (A.q[3 * j + m] / sq) * (A.q[3 * j + m] / sq) + (A.p[3 * j + m] / sp) * (A.p[3 * j + m] / sp);
          s1 += (A.p[3 * j + m] / sq) * (A.p[3 * j + m] / sq) + (a[m] / sp) * (a[m] / sp);
          A.G[3 * j + m] = a[m];  // f0's acceleration part, kept for d2
        }
      }
      const double nn = 6.0 * (double)n;
      const double d0 = sqrt(block_sum(S, s0) / nn);
      const double d1 = sqrt(block_sum(S, s1) / nn);
      const bool cond = (d0 < 1e-5) || (d1 < 1e-5);
      const double hh = cond ? 1e-6 : 0.01 * (d0 / (cond ? 1.0 : d1));
      __syncthreads();
      for (long long j = tid; j < n; j += kNbThreads) {
        S.x[j] = A.q[3 * j] + A.p[3 * j] * hh;
        S.y[j] = A.q[3 * j + 1] + A.p[3 * j + 1] * hh;
        S.z[j] = A.q[3 * j + 2] + A.p[3 * j + 2] * hh;
      }
      __syncthreads();
      double s2 = 0.0;
      for (long long j = tid; j < n; j += kNbThreads) {
        double a[3];
        nb_accel(P, S, n, A.eps2, j, S.x[j], S.y[j], S.z[j], dir * (tau + hh), a[0], a[1], a[2]);
        for (int m = 0; m < 3; ++m) {
          const double sq = A.atol + fabs(A.q[3 * j + m]) * A.rtol;
          const double sp = A.atol + fabs(A.p[3 * j + m]) * A.rtol;
          const double p1 = A.p[3 * j + m] + dir * A.G[3 * j + m] * dir * hh;
          const double u = (p1 - A.p[3 * j + m]) / sq;
          const double v = dir * (a[m] - A.G[3 * j + m]) / sp;
          s2 += u * u + v * v;
        }
      }
      const double d2 = sqrt(block_sum(S, s2) / nn) / hh;
      const double maxd = fmax(d1, d2);
      const double h1 = (maxd <= 1e-15) ? fmax(1e-6, hh * 1e-3)
                                        : pow(0.01 / maxd, 1.0 / ((double)M::order + 1.0));
      h0 = fmin(100.0 * hh, h1);
    }
    bool at_dtmin = false;
    if (PID) {
      h0 = fmin(h0, A.dtmax);
      if (A.dtmin > 0.0) {
        at_dtmin = h0 <= A.dtmin;
        h0 = fmax(h0, A.dtmin);
      }
    }
    double tnext = fmin(tau + h0, tau1);
    double prev_inv = 1.0, prev_prev_inv = 1.0;
    while (tau < tau1) {
      if (nst >= A.max_steps) {
        status = GX_MAX_STEPS_REACHED;
        break;
      }
      const double h = tnext - tau;
      if (!(h >= 0.0)) {
        status = GX_NONFINITE;
        break;
      }
      const double sq = block_sum(S, nb_eval<M, PID>(P, S, A, dir, tau, h));
      ++nst;
      // a non-finite state anywhere stops the system
      double bad = 0.0;
      for (long long j = tid; j < n; j += kNbThreads)
        for (int m = 0; m < 3; ++m)
          if (!isfinite(A.q1[3 * j + m]) || !isfinite(A.p1[3 * j + m])) bad = 1.0;
      if (block_sum(S, bad) != 0.0) {
        status = GX_NONFINITE;
        break;
      }
      bool keep = true;
      double next_tau1;
      if (PID) {
        const double scaled = sqrt(sq / (6.0 * (double)n));
        keep = scaled < 1.0;
        if (A.dtmin > 0.0) keep = keep || at_dtmin;
        const double inv = 1.0 / scaled;
        double f = (A.c1 == 0.0) ? 1.0 : pow(inv, A.c1);
        if (A.c2 != 0.0) f *= pow(prev_inv, A.c2);
        if (A.c3 != 0.0) f *= pow(prev_prev_inv, A.c3);
        const double fmin_ = keep ? 1.0 : A.factormin;
        const double factor = fmin(fmax(A.safety * f, fmin_), A.factormax);
        double dt = fmin(h * factor, A.dtmax);
        if (A.dtmin > 0.0) {
          if (!A.force_dtmin && dt < A.dtmin) status = GX_DT_MIN_REACHED;
          at_dtmin = dt <= A.dtmin;
          dt = fmax(dt, A.dtmin);
        }
        if (keep) {
          prev_prev_inv = prev_inv;
          prev_inv = (inv == 0.0 || isinf(inv)) ? 1.0 : inv;
        }
        next_tau1 = (keep ? tnext : tau) + dt;
      } else {
        next_tau1 = tnext + A.dt0;
      }
      if (keep) {
        // saves in (tau, tnext]: the step end, or the step's dense output
        // (diffrax's interpolant), which reads the end stage a(q1, tnext)
        bool have_end = M::SF == M::S;  // Dopri5's last stage is at q1
        while (si < A.T && dir * A.ts[si] <= tnext) {
          const double ts_tau = dir * A.ts[si];
          if (ts_tau == tnext) {
            nb_write(A, si, dir, A.q1, A.p1);
          } else {
            if (!have_end) {
              for (long long j = tid; j < n; j += kNbThreads) {
                S.x[j] = A.q1[3 * j];
                S.y[j] = A.q1[3 * j + 1];
                S.z[j] = A.q1[3 * j + 2];
              }
              __syncthreads();
              for (long long j = tid; j < n; j += kNbThreads) {
                double* g = A.G + ((long long)(M::SF - 1) * n + j) * 3;
                nb_accel(P, S, n, A.eps2, j, S.x[j], S.y[j], S.z[j], dir * tnext, g[0], g[1], g[2]);
              }
              __syncthreads();
              have_end = true;
            }
            double wq[M::SF], wp[M::SF];
            const double th = (ts_tau - tau) / h;
            dense_weights<M>(th, wq, wp);
            const double ht = h * th, hht = h * ht;
            for (long long j = tid; j < n; j += kNbThreads) {
              double sq_[3] = {0.0, 0.0, 0.0}, sp_[3] = {0.0, 0.0, 0.0};
              for (int l = 0; l < M::SF; ++l)
                for (int m = 0; m < 3; ++m) {
                  const double gl = A.G[((long long)l * n + j) * 3 + m];
                  sq_[m] = fma(wq[l], gl, sq_[m]);
                  sp_[m] = fma(wp[l], gl, sp_[m]);
                }
              double* o = A.out + (j * A.T + si) * 6;
              for (int m = 0; m < 3; ++m) {
                const double q0 = A.q[3 * j + m], p0 = A.p[3 * j + m];
                o[m] = fma(hht, sq_[m], fma(ht, p0, q0));
                o[3 + m] = dir * fma(ht, sp_[m], p0);
              }
            }
          }
          ++si;
        }
        __syncthreads();
        for (long long j = tid; j < n; j += kNbThreads)
          for (int m = 0; m < 3; ++m) {
            A.q[3 * j + m] = A.q1[3 * j + m];
            A.p[3 * j + m] = A.p1[3 * j + m];
          }
        ++nacc;
      }
      __syncthreads();
      const double tprev = fmin(keep ? tnext : tau, tau1);
      tnext = (next_tau1 > tau1 - 1e-10) ? (keep ? tau1 : tprev + 0.5 * (tau1 - tprev)) : next_tau1;
      tau = tprev;
      if (status == GX_DT_MIN_REACHED) break;
    }
  }
  if (status != GX_SUCCESS) {
    const double nanv = __longlong_as_double(0x7ff8000000000000ULL);
    for (; si < A.T; ++si)
      for (long long j = tid; j < n; j += kNbThreads)
        for (int m = 0; m < 6; ++m) A.out[(j * A.T + si) * 6 + m] = nanv;
  }
  if (tid == 0) {
    if (A.status) *A.status = status;
    if (A.nsteps) *A.nsteps = nst;
    if (A.naccept) *A.naccept = nacc;
  }
}

// ---- the system over many workgroups -------------------------------------
// One workgroup's CU holds 1/256 of the device's FP64 rate: 1,024 bodies
// took 600 us a stage on it (60 Myr of a cluster, 23 steps: 180.8 ms; here
// 2.4 ms, of which the meetings take most; 128 bodies 12.3 ms, here 1.85;
// 16 bodies, one workgroup, 4.0 ms, here 1.4).  Here the bodies are divided among G resident
// workgroups (a cooperative launch): a workgroup owns `own` bodies, keeps
// their state and stage accelerations in LDS, and a stage is
//   1. the owner computes its bodies' stage positions and publishes them,
//   2. the workgroups meet (below),
//   3. every workgroup copies all positions to LDS, and its eight waves sum
//      the pull on the owned bodies, lanes over the sources (a wave for a
//      body; several waves for one when there are fewer than eight),
//   4. the owner adds the external field, which it evaluated while waiting.
// A meeting costs more than the sums of 1,024 bodies, so it is one store and
// one load through the level that all XCDs share, with no flag, no
// read-modify-write and no cache flush: every published value is its own
// flag (gx_slots.hpp).
// Three buffers take turns by meeting.  Having read meeting k - 1, an owner
// knows that every workgroup has come to it and so has read meeting k - 2,
// whose buffer is the one of meeting k + 1: it empties its own slots there,
// and waits for those stores (s_waitcnt vmcnt(0)) before it publishes for
// meeting k, without which nobody looks at meeting k + 1.
// Every workgroup runs the controller on the same sums in the same order
// and takes the same decisions.  The start of a step and the end of the
// accepted one before it are the same point, so its acceleration is kept
// (first same as last): 13 meetings a step.
// G = 1 is the same kernel with a workgroup barrier for a meeting and 16
// lanes a body, for systems whose sums take less time than a meeting.
constexpr int kNbWaves = kNbThreads / 64;
constexpr int kNbGroups = 256;  // most workgroups
constexpr int kNbOwnMax = kNbMax / kNbGroups;  // bodies of a workgroup of the largest system

struct NGrid {
  int G;         // workgroups
  int own;       // bodies of a workgroup
  Slot* pos;   // [3][3][n] published positions
  Slot* part;  // [3][2][G] published error sums and non-finite counts
};

__global__ void k_nb_empty(Slot* slots, long long m) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m) slots[i] = kSlotEmpty;
}

// Dynamic LDS of a workgroup (doubles): all positions and masses, then the
// owned bodies' [3][own] arrays.
struct NbOwn {
  double *x, *y, *z, *gm;       // [n]
  double *q, *p, *q1, *p1;      // [3][own]
  double *Q, *ext;              // stage position, external field
  double* aa;                   // [S][S] the tableau squared
  double *g;                    // [SF][3][own] stage accelerations
  double *part;                 // [3][max(own, waves)] partial pulls
};
__host__ __device__ inline size_t nb_lds_doubles(long long n, int own, int SF) {
  return (size_t)(4 * n + (long long)3 * own * (6 + SF) + 3 * (own > kNbWaves ? own : kNbWaves) +
                  (long long)SF * SF);
}

template <class M, bool PID, class E>
struct NbGridSolve {
  const DPot& P;
  const NArgs& A;
  const NGrid& X;
  NbOwn S;
  double2* red;  // [waves]
  int n, own, first, cnt, tid;
  double dir;
  int turn = 0;  // the buffer of the coming meeting

  // Sums over the workgroup, in a fixed order; every thread gets them.
  __device__ __forceinline__ void sum(double& a, double& b) const {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      a += __shfl_xor(a, o, 64);
      b += __shfl_xor(b, o, 64);
    }
    __syncthreads();
    if ((tid & 63) == 0) red[tid >> 6] = make_double2(a, b);
    __syncthreads();
    a = b = 0.0;
#pragma unroll
    for (int i = 0; i < kNbWaves; ++i) {
      a += red[i].x;
      b += red[i].y;
    }
  }

  // Position of owned body j, component m, for the coming meeting (wave 0
  // does all of a workgroup's publishing: own <= 16).
  __device__ __forceinline__ void publish(int m, int j, double v) {
    S.Q[m * own + j] = v;
    if (X.G == 1)
      (m == 0 ? S.x : m == 1 ? S.y : S.z)[j] = v;
    else
      put_slot(X.pos + ((size_t)turn * 3 + m) * n + first + j, v);
  }

  // The workgroup's two sums for the coming meeting.
  __device__ __forceinline__ void offer(double a, double b) {
    if (X.G == 1 || tid != 0) return;
    Slot* p = X.part + (size_t)turn * 2 * X.G + blockIdx.x;
    put_slot(p, a);
    put_slot(p + X.G, b);
  }

  // The meeting's sums over all workgroups.
  __device__ __forceinline__ void total(double& a, double& b) {
    if (X.G == 1) return;
    const Slot* p = X.part + (size_t)turn * 2 * X.G + tid;
    const bool in = tid < X.G;
    const Slot va = in ? get_slot(p) : 0, vb = in ? get_slot(p + X.G) : 0;
    a = await_slot(p, va);
    b = await_slot(p + X.G, vb);
    sum(a, b);
  }

  // Close the meeting: empty the buffer after next, which everyone has read.
  __device__ __forceinline__ void close() {
    if (X.G > 1 && tid < 64) {
      const int next = turn == 0 ? 2 : turn - 1;  // of the meeting after next
      if (tid < 3 * cnt)
        put_slot(X.pos + ((size_t)next * 3 + tid / cnt) * n + first + tid % cnt, kSlotEmpty);
      if (tid < 2) put_slot(X.part + ((size_t)next * 2 + tid) * X.G + blockIdx.x, kSlotEmpty);
    }
    turn = turn == 2 ? 0 : turn + 1;
  }
  // Before publishing: the emptied slots have reached the shared level.
  __device__ __forceinline__ void settle() {
    if (X.G > 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  // The external field at the owned bodies' published positions.
  __device__ __forceinline__ void external(double t) {
    for (int j = tid; j < cnt; j += kNbThreads) {
      double a[3];
      E::acc(P, S.Q[j], S.Q[own + j], S.Q[2 * own + j], t, a[0], a[1], a[2]);
      for (int m = 0; m < 3; ++m) S.ext[m * own + j] = a[m];
    }
  }

  // All positions of the meeting into LDS.
  __device__ __forceinline__ void fetch() {
    if (X.G > 1) {
      constexpr int R = 6;  // loads in flight
      const Slot* src = X.pos + (size_t)turn * 3 * n;
      for (int k0 = tid; k0 < 3 * n; k0 += R * kNbThreads) {
        Slot v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int k = k0 + r * kNbThreads;
          v[r] = k < 3 * n ? get_slot(src + k) : 0;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int k = k0 + r * kNbThreads;
          if (k < 3 * n) S.x[k] = await_slot(src + k, v[r]);
        }
      }
    }
    __syncthreads();
  }

  // Pull on body `self` at (x, y, z) of the sources k0, k0 + dk, ...
  __device__ __forceinline__ void pull(int self, double x, double y, double z, int k0, int dk,
                                       double& ax, double& ay, double& az) const {
    ax = ay = az = 0.0;
#pragma unroll 8
    for (int k = k0; k < n; k += dk) {
      const double dx = S.x[k] - x, dy = S.y[k] - y, dz = S.z[k] - z;
      const double r2 = dx * dx + dy * dy + dz * dz + A.eps2;
      const double ir = rsqrt_fast(r2);
      const double w = (k == self) ? 0.0 : S.gm[k] * ir * ir * ir;
      ax = fma(w, dx, ax);
      ay = fma(w, dy, ay);
      az = fma(w, dz, az);
    }
  }

  // Accelerations of the owned bodies at the positions in LDS, into g.
  __device__ __forceinline__ void accelerate(double* g) {
    const int lane = tid & 63, wave = tid >> 6;
    int parts = 1;
    if (X.G == 1) {
      // 16 lanes a body, 32 bodies a round
      for (int j0 = 0; j0 < own; j0 += kNbThreads / 16) {
        const int j = j0 + (tid >> 4), c = j < own ? j : own - 1;
        double ax, ay, az;
        pull(c, S.Q[c], S.Q[own + c], S.Q[2 * own + c], tid & 15, 16, ax, ay, az);
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) {
          ax += __shfl_xor(ax, o, 64);
          ay += __shfl_xor(ay, o, 64);
          az += __shfl_xor(az, o, 64);
        }
        if ((tid & 15) == 0 && j < own) {
          S.part[j] = ax;
          S.part[own + j] = ay;
          S.part[2 * own + j] = az;
        }
      }
    } else {
      // a wave for a body, or `parts` waves when that leaves waves idle
      while (2 * own * parts <= kNbWaves) parts *= 2;
      for (int u = wave; u < own * parts; u += kNbWaves) {
        const int j = u / parts, c = j < cnt ? j : 0;
        double ax, ay, az;
        pull(first + c, S.Q[c], S.Q[own + c], S.Q[2 * own + c], (u % parts) * 64 + lane, 64 * parts, ax, ay,
             az);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          ax += __shfl_xor(ax, o, 64);
          ay += __shfl_xor(ay, o, 64);
          az += __shfl_xor(az, o, 64);
        }
        if (lane == 0) {
          S.part[u] = ax;
          S.part[own * parts + u] = ay;
          S.part[2 * own * parts + u] = az;
        }
      }
    }
    __syncthreads();
    for (int i = tid; i < 3 * own; i += kNbThreads) {
      const int m = i / own, j = i - m * own;
      double a = S.ext[i];
      for (int k = 0; k < parts; ++k) a += S.part[(m * own + j) * parts + k];
      g[i] = a;
    }
    __syncthreads();
  }

  __device__ __forceinline__ void save(int s, const double* q, const double* p) const {
    for (int i = tid; i < 3 * own; i += kNbThreads) {
      const int m = i / own, j = i - m * own;
      if (j >= cnt) continue;
      double* o = A.out + ((size_t)(first + j) * A.T + s) * 6 + m;
      o[0] = q[i];
      o[3] = dir * p[i];
    }
  }

  // A save inside the step: the method's dense output at th of it.
  __device__ __forceinline__ void save_inside(int s, double th, double h) const {
    constexpr int SF = M::SF;
    double wq[SF], wp[SF];
    dense_weights<M>(th, wq, wp);
    const double ht = h * th, hht = h * ht;
    for (int k = tid; k < 3 * own; k += kNbThreads) {
      const int m = k / own, j = k - m * own;
      if (j >= cnt) continue;
      double a = 0.0, b = 0.0;
#pragma unroll
      for (int l = 0; l < SF; ++l) {
        const double gl = S.g[l * 3 * own + k];
        a = fma(wq[l], gl, a);
        b = fma(wp[l], gl, b);
      }
      double* o = A.out + ((size_t)(first + j) * A.T + s) * 6 + m;
      o[0] = fma(hht, a, fma(ht, S.p[k], S.q[k]));
      o[3] = dir * fma(ht, b, S.p[k]);
    }
  }

  __device__ __forceinline__ void run() {
    constexpr auto& K = M::k;
    constexpr int SF = M::SF;
    const int own3 = 3 * own;
    double* const gend = S.g + (SF - 1) * own3;
    dir = (A.t0 < A.t1) ? 1.0 : -1.0;
    for (int k = tid; k < n; k += kNbThreads) S.gm[k] = A.gm[k];
    for (int k = tid; k < M::S * M::S; k += kNbThreads) S.aa[k] = K.aa[k / M::S][k % M::S];
    for (int k = tid; k < SF * own3; k += kNbThreads) S.g[k] = 0.0;
    for (int i = tid; i < own3; i += kNbThreads) {
      const int m = i / own, j = i - m * own;
      const double* w = A.w0 + 6 * (size_t)(first + (j < cnt ? j : 0));
      S.q[i] = w[m];
      S.p[i] = dir * w[3 + m];
      S.ext[i] = 0.0;
      S.Q[i] = S.q[i];
    }
    __syncthreads();
    double tau = dir * A.t0;
    const double tau1 = dir * A.t1;
    int si = 0;
    while (si < A.T && dir * A.ts[si] <= tau) save(si++, S.q, S.p);
    int status = GX_SUCCESS;
    long long nst = 0, nacc = 0;
    const double nn = 6.0 * (double)n;
    // Each trip publishes one set of positions, meets, and evaluates the
    // field there: at the start, at the trial point of the first-step rule,
    // at a stage, or at a step's end (with the step's error).
    enum { kStart, kTrial, kStage, kEnd };
    int phase = kStart, stage = 0;
    double h = 0.0, hh = 0.0, d1 = 0.0, t_eval = dir * tau;
    double tnext = tau, prev_inv = 1.0, prev_prev_inv = 1.0;
    bool at_dtmin = false;
    while (A.t0 != A.t1) {
      double sq = 0.0, bad = 0.0;
      const bool last = phase == kEnd && SF == M::S;  // Dopri5's end stage is done
      settle();
      for (int k = tid; k < own3; k += kNbThreads) {
        const int m = k / own, j = k - m * own;
        if (j >= cnt) continue;
        double x = S.q[k];
        if (phase == kTrial) {
          x += S.p[k] * hh;
        } else if (phase == kStage) {
          // zero weights from `stage` on, where g holds the last step's
          const double* a = S.aa + stage * M::S;
          double s = 0.0;
#pragma unroll
          for (int l = 0; l < M::S - 1; ++l) s = fma(a[l], S.g[l * own3 + k], s);
          x = fma(h, fma(K.rs[stage], S.p[k], h * s), x);
        } else if (phase == kEnd) {
          double b = 0.0, ba = 0.0, e = 0.0, ea = 0.0;
#pragma unroll
          for (int l = 0; l < M::S; ++l) {
            const double gl = S.g[l * own3 + k];
            b = fma(K.b[l], gl, b);
            ba = fma(K.ba[l], gl, ba);
            if (PID) {
              e = fma(K.e[l], gl, e);
              ea = fma(K.ea[l], gl, ea);
            }
          }
          const double q0 = x, p0 = S.p[k];
          x = fma(h, fma(K.sb, p0, h * ba), q0);
          const double p1 = fma(h, b, p0);
          S.q1[k] = x;
          S.p1[k] = p1;
          if (!isfinite(x) || !isfinite(p1)) bad = 1.0;
          if (PID) {
            const double eq = h * fma(K.se, p0, h * ea);
            const double ep = h * e;
            const double uq = eq / (A.atol + fmax(fabs(q0), fabs(x)) * A.rtol);
            const double up = ep / (A.atol + fmax(fabs(p0), fabs(p1)) * A.rtol);
            sq += uq * uq + up * up;
          }
        }
        publish(m, j, x);
      }
      if (phase == kEnd) {
        sum(sq, bad);
        offer(sq, bad);
      }
      __syncthreads();
      if (!last) external(t_eval);
      bool keep = true;
      double next_tau1 = 0.0;
      if (phase == kEnd) {
        total(sq, bad);
        ++nst;
        if (bad != 0.0) {
          status = GX_NONFINITE;
          break;
        }
        if (PID) {
          const double scaled = sqrt(sq / nn);
          keep = scaled < 1.0;
          if (A.dtmin > 0.0) keep = keep || at_dtmin;
          const double inv = 1.0 / scaled;
          double f = (A.c1 == 0.0) ? 1.0 : pow(inv, A.c1);
          if (A.c2 != 0.0) f *= pow(prev_inv, A.c2);
          if (A.c3 != 0.0) f *= pow(prev_prev_inv, A.c3);
          const double fmin_ = keep ? 1.0 : A.factormin;
          const double factor = fmin(fmax(A.safety * f, fmin_), A.factormax);
          double dt = fmin(h * factor, A.dtmax);
          if (A.dtmin > 0.0) {
            if (!A.force_dtmin && dt < A.dtmin) status = GX_DT_MIN_REACHED;
            at_dtmin = dt <= A.dtmin;
            dt = fmax(dt, A.dtmin);
          }
          if (keep) {
            prev_prev_inv = prev_inv;
            prev_inv = (inv == 0.0 || isinf(inv)) ? 1.0 : inv;
          }
          next_tau1 = (keep ? tnext : tau) + dt;
        } else {
          next_tau1 = tnext + A.dt0;
        }
      }
      const bool field = keep && !last;
      if (field) fetch();
      close();
      if (field) accelerate(S.g + (phase == kStart ? 0 : phase == kStage ? stage : SF - 1) * own3);
      bool begin = false;  // the next trip begins a step
      if (phase == kStart || phase == kTrial) {
        // first step: dt0; dtmin if the controller sets one (as the orbit
        // integrators); else diffrax's initial-step heuristic over the system
        double h0 = A.dt0 > 0.0 ? A.dt0 : (PID && A.dtmin > 0.0 ? A.dtmin : 0.0);
        if (!(h0 > 0.0)) {
          double s0 = 0.0, s1 = 0.0;
          for (int k = tid; k < own3; k += kNbThreads) {
            if (k % own >= cnt) continue;
            const double q = S.q[k], p = S.p[k], a = S.g[k];
            const double wq = A.atol + fabs(q) * A.rtol, wp = A.atol + fabs(p) * A.rtol;
            if (phase == kStart) {
              s0 += (q / wq) * (q / wq) + (p / wp) * (p / wp);
              s1 += (p / wq) * (p / wq) + (a / wp) * (a / wp);
            } else {
              const double u = ((p + dir * a * dir * hh) - p) / wq;
              const double v = dir * (gend[k] - a) / wp;
              s0 += u * u + v * v;
            }
          }
          sum(s0, s1);
          settle();
          offer(s0, s1);
          total(s0, s1);
          close();
          if (phase == kStart) {
            const double d0 = sqrt(s0 / nn);
            d1 = sqrt(s1 / nn);
            const bool cond = (d0 < 1e-5) || (d1 < 1e-5);
            hh = cond ? 1e-6 : 0.01 * (d0 / (cond ? 1.0 : d1));
            phase = kTrial;
            t_eval = dir * (tau + hh);
            continue;
          }
          const double d2 = sqrt(s0 / nn) / hh;
          const double maxd = fmax(d1, d2);
          const double h1 = (maxd <= 1e-15) ? fmax(1e-6, hh * 1e-3)
                                            : pow(0.01 / maxd, 1.0 / ((double)M::order + 1.0));
          h0 = fmin(100.0 * hh, h1);
        }
        if (PID) {
          h0 = fmin(h0, A.dtmax);
          if (A.dtmin > 0.0) {
            at_dtmin = h0 <= A.dtmin;
            h0 = fmax(h0, A.dtmin);
          }
        }
        tnext = fmin(tau + h0, tau1);
        begin = true;
      } else if (phase == kStage) {
        if (++stage == M::S) {
          phase = kEnd;
          t_eval = dir * tnext;
        } else {
          t_eval = dir * fma(K.c[stage], h, tau);
        }
      } else {
        if (keep) {
          // saves in (tau, tnext]: the step end, or the step's dense output
          while (si < A.T && dir * A.ts[si] <= tnext) {
            const double ts_tau = dir * A.ts[si];
            if (ts_tau == tnext)
              save(si, S.q1, S.p1);
            else
              save_inside(si, (ts_tau - tau) / h, h);
            ++si;
          }
          __syncthreads();
          for (int k = tid; k < own3; k += kNbThreads) {
            S.q[k] = S.q1[k];
            S.p[k] = S.p1[k];
            S.g[k] = gend[k];
          }
          ++nacc;
        }
        __syncthreads();
        const double tprev = fmin(keep ? tnext : tau, tau1);
        tnext =
            (next_tau1 > tau1 - 1e-10) ? (keep ? tau1 : tprev + 0.5 * (tau1 - tprev)) : next_tau1;
        tau = tprev;
        if (status == GX_DT_MIN_REACHED) break;
        begin = true;
      }
      if (begin) {
        if (!(tau < tau1)) break;
        if (nst >= A.max_steps) {
          status = GX_MAX_STEPS_REACHED;
          break;
        }
        h = tnext - tau;
        if (!(h >= 0.0)) {
          status = GX_NONFINITE;
          break;
        }
        phase = kStage;
        stage = 1;
        t_eval = dir * fma(K.c[1], h, tau);
      }
    }
    if (status != GX_SUCCESS) {
      const double nanv = __longlong_as_double(0x7ff8000000000000ULL);
      for (; si < A.T; ++si)
        for (int j = tid; j < cnt; j += kNbThreads)
          for (int m = 0; m < 6; ++m) A.out[((size_t)(first + j) * A.T + si) * 6 + m] = nanv;
    }
    if (blockIdx.x == 0 && tid == 0) {
      if (A.status) *A.status = status;
      if (A.nsteps) *A.nsteps = nst;
      if (A.naccept) *A.naccept = nacc;
    }
  }
};

template <class M, bool PID, class E>
__global__ void __launch_bounds__(kNbThreads) k_nbody_grid(DPot P, NArgs A, NGrid X) {
  extern __shared__ double nb_lds[];
  __shared__ double2 red[kNbWaves];
  const int n = (int)A.n, own = X.own, o3 = 3 * X.own;
  NbGridSolve<M, PID, E> R{P, A, X};
  double* d = nb_lds;
  R.S.x = d;
  R.S.y = d + n;
  R.S.z = d + 2 * n;
  R.S.gm = d + 3 * n;
  d += 4 * n;
  R.S.q = d;
  R.S.p = d + o3;
  R.S.q1 = d + 2 * o3;
  R.S.p1 = d + 3 * o3;
  R.S.Q = d + 4 * o3;
  R.S.ext = d + 5 * o3;
  R.S.g = d + 6 * o3;
  R.S.part = d + (6 + M::SF) * o3;
  R.S.aa = R.S.part + 3 * (own > kNbWaves ? own : kNbWaves);
  R.red = red;
  R.n = n;
  R.own = own;
  R.tid = threadIdx.x;
  R.first = blockIdx.x * own;
  R.cnt = n - R.first < own ? n - R.first : own;
  R.run();
}

// The system over workgroups: GX_OK when launched, 1 when the device cannot
// hold them all at once (or the stream is being captured, which takes no
// cooperative launch).
template <class M, bool PID, class E>
int launch_grid(const gx_pot* ext, NArgs& A, void* workspace, hipStream_t s) {
  const auto kern = k_nbody_grid<M, PID, E>;
  NGrid X{};
  X.own = A.n <= kNbOne ? (int)A.n : (int)((A.n + kNbGroups - 1) / kNbGroups);
  if (A.n > kNbOne && X.own < kNbOwnMin) X.own = kNbOwnMin;
  X.G = (int)((A.n + X.own - 1) / X.own);
  // what G workgroups exchange (72 bytes a body, 48 a workgroup) fits where
  // the one-workgroup kernel keeps its state (432 bytes a body)
  X.pos = reinterpret_cast<Slot*>(static_cast<char*>(workspace) + 256);
  X.part = X.pos + 9 * A.n;
  const size_t lds = sizeof(double) * nb_lds_doubles(A.n, X.own, M::SF);
  // what the largest system takes, whatever this one does: the limit is the
  // function's, and another thread may be about to launch it
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                          hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)(sizeof(double) * nb_lds_doubles(kNbMax, kNbOwnMax, M::SF))) !=
      hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  if (X.G == 1) {
    hipLaunchKernelGGL(kern, dim3(1), dim3(kNbThreads), lds, s, ext->dev, A, X);
    return check(hipGetLastError());
  }
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  int coop = 0, occ = 0;
  if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone ||
      hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, ext->device) != hipSuccess ||
      !coop ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern, kNbThreads, lds) != hipSuccess ||
      (long long)occ * num_cus(ext->device) < X.G) {
    (void)hipGetLastError();
    return 1;
  }
  const long long slots = 9 * A.n + 6 * X.G;
  hipLaunchKernelGGL(k_nb_empty, dim3((unsigned)((slots + 255) / 256)), dim3(256), 0, s, X.pos, slots);
  DPot Pd = ext->dev;
  NArgs Ad = A;
  void* args[] = {&Pd, &Ad, &X};
  if (hipLaunchCooperativeKernel(reinterpret_cast<const void*>(kern), dim3(X.G), dim3(kNbThreads),
                                 args, (unsigned)lds, s) == hipSuccess)
    return GX_OK;
  (void)hipGetLastError();
  return 1;
}

template <class M, bool PID>
int launch_nbody(const gx_pot* ext, NArgs& A, void* workspace, hipStream_t s) {
  // A few bodies in another field than the Milky Way's stay with the plain
  // kernel: its step has fewer barriers, and their sums are nothing beside them
  // (ms of 50 fixed steps without a field, k_nbody / k_nbody_grid: Dopri8 2
  // bodies 1.9 / 2.8, 8 2.5 / 2.7, 12 more with k_nbody; Dopri5 4 bodies 1.16 /
  // 1.30, 6 as many; under PID 2 bodies 0.28 / 0.33, 5 as many).
  constexpr long long kFew = PID ? 4 : std::is_same_v<M, Dopri8> ? 8 : 5;
  int rc = 1;
  if (ext->sig == kSigMilkyWay)
    rc = launch_grid<M, PID, EvalMilkyWay>(ext, A, workspace, s);
  else if (A.n > kFew)
    rc = launch_grid<M, PID, EvalTable<true>>(ext, A, workspace, s);
  if (rc != 1) return rc;
  hipLaunchKernelGGL((k_nbody<M, PID>), dim3(1), dim3(kNbThreads), 0, s, ext->dev, A);
  return check(hipGetLastError());
}

// The field alone (NBodyField.__call__'s acceleration): one thread per body,
// positions staged through LDS in tiles.
__global__ void __launch_bounds__(256) k_nbody_accel(DPot P, const double* __restrict__ xyz,
                                                     const double* __restrict__ gm, double eps2,
                                                     double t, long long n,
                                                     double* __restrict__ acc) {
  __shared__ double tx[256], ty[256], tz[256], tg[256];
  const long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool own = j < n;
  const double x = own ? xyz[3 * j] : 0.0, y = own ? xyz[3 * j + 1] : 0.0,
               z = own ? xyz[3 * j + 2] : 0.0;
  double ax = 0.0, ay = 0.0, az = 0.0;
  if (own) accel<true>(P, x, y, z, t, ax, ay, az);
  for (long long k0 = 0; k0 < n; k0 += 256) {
    const long long k = k0 + threadIdx.x;
    __syncthreads();
    tx[threadIdx.x] = k < n ? xyz[3 * k] : 0.0;
    ty[threadIdx.x] = k < n ? xyz[3 * k + 1] : 0.0;
    tz[threadIdx.x] = k < n ? xyz[3 * k + 2] : 0.0;
    tg[threadIdx.x] = k < n ? gm[k] : 0.0;
    __syncthreads();
    const int m = (n - k0) < 256 ? (int)(n - k0) : 256;
    for (int i = 0; i < m; ++i) {
      const double dx = tx[i] - x, dy = ty[i] - y, dz = tz[i] - z;
      const double r2 = dx * dx + dy * dy + dz * dz + eps2;
      const double ir = rsqrt_fast(r2);
      const double w = (k0 + i == j) ? 0.0 : tg[i] * ir * ir * ir;
      ax = fma(w, dx, ax);
      ay = fma(w, dy, ay);
      az = fma(w, dz, az);
    }
  }
  if (own) {
    acc[3 * j] = ax;
    acc[3 * j + 1] = ay;
    acc[3 * j + 2] = az;
  }
}

}  // namespace
}  // namespace gx

using namespace gx;

extern "C" {

int64_t gx_nbody_workspace_bytes(int64_t n) {
  return n < 0 ? 0 : 256 + 8 * n * (12 + 3 * 14);
}

int gx_nbody_acceleration(const gx_pot* ext, const double* xyz, const double* gm,
                          double eps, double t, int64_t n, double* acc, void* stream) {
  if (!ext || !xyz || !gm || !acc || n < 0 || !(eps >= 0.0)) return GX_EINVAL;
  if (n == 0) return GX_OK;
  if ((n + 255) / 256 > 0x7fffffffLL) return GX_EINVAL;
  hipLaunchKernelGGL(k_nbody_accel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, ext->dev, xyz, gm, eps * eps, t, (long long)n, acc);
  return check(hipGetLastError());
}

int gx_nbody_integrate(const gx_pot* ext, const double* gm, double eps,
                       const gx_solver_cfg* cfg, const double* w0, double t0, double t1,
                       const double* ts, int32_t T, int64_t n, double* out, int32_t* status,
                       int64_t* nsteps, int64_t* naccept, void* workspace, void* stream) {
  if (!ext || !gm || !cfg || !w0 || !ts || !out || !workspace) return GX_EINVAL;
  if (n < 1 || n > kNbMax || T < 1 || !(eps >= 0.0)) return GX_EINVAL;
  if (!std::isfinite(t0) || !std::isfinite(t1)) return GX_EINVAL;
  if (cfg->method != GX_DOPRI8 && cfg->method != GX_DOPRI5) return GX_EINVAL;
  if (cfg->controller != GX_CONSTANT && cfg->controller != GX_PID) return GX_EINVAL;
  if (cfg->controller == GX_CONSTANT && !(cfg->dt0 > 0.0)) return GX_EINVAL;
  if (cfg->controller == GX_PID &&
      !(cfg->rtol >= 0.0 && cfg->atol >= 0.0 && cfg->rtol + cfg->atol > 0.0 &&
        cfg->safety > 0.0 && cfg->factormin > 0.0 && cfg->factormax >= 1.0))
    return GX_EINVAL;
  NArgs A{};
  A.dt0 = cfg->dt0;
  A.rtol = cfg->rtol;
  A.atol = cfg->atol;
  A.safety = cfg->safety;
  A.factormin = cfg->factormin;
  A.factormax = cfg->factormax;
  A.dtmin = cfg->dtmin > 0.0 ? cfg->dtmin : 0.0;
  A.dtmax = cfg->dtmax > 0.0 ? cfg->dtmax : INFINITY;
  const double korder = cfg->method == GX_DOPRI8 ? 8.0 : 5.0;
  A.c1 = (cfg->icoeff + cfg->pcoeff + cfg->dcoeff) / korder;
  A.c2 = -(cfg->pcoeff + 2.0 * cfg->dcoeff) / korder;
  A.c3 = cfg->dcoeff / korder;
  A.max_steps = (cfg->max_steps > 0 && cfg->max_steps < 10000000) ? cfg->max_steps : 10000000;
  A.force_dtmin = cfg->force_dtmin;
  A.T = T;
  A.eps2 = eps * eps;
  A.t0 = t0;
  A.t1 = t1;
  A.gm = gm;
  A.w0 = w0;
  A.ts = ts;
  A.n = n;
  A.out = out;
  A.status = status;
  A.nsteps = reinterpret_cast<long long*>(nsteps);
  A.naccept = reinterpret_cast<long long*>(naccept);
  double* w = reinterpret_cast<double*>(static_cast<char*>(workspace) + 256);
  A.q = w;
  A.p = w + 3 * n;
  A.q1 = w + 6 * n;
  A.p1 = w + 9 * n;
  A.G = w + 12 * n;
  hipStream_t s = (hipStream_t)stream;
  const bool pid = cfg->controller == GX_PID;
  if (cfg->method == GX_DOPRI8)
    return pid ? launch_nbody<Dopri8, true>(ext, A, workspace, s)
               : launch_nbody<Dopri8, false>(ext, A, workspace, s);
  return pid ? launch_nbody<Dopri5, true>(ext, A, workspace, s)
             : launch_nbody<Dopri5, false>(ext, A, workspace, s);
}

}  // extern "C"
