// gx_team.hpp -- Dopri8 orbits integrated by teams of waves, for launches that
// are bound by the latency of single orbits' steps.
//
// A wave that carries an orbit by itself issues about 2,000 instructions a
// step, one after the other (4.4 us at a fixed step, 5.0 us with the
// controller), whether the device is full or nearly empty, and the longest
// orbit of a batch, or a batch that does not fill the device, takes its step
// count times that.  In Runge-Kutta-Nystrom form stage i needs the
// accelerations of stages 0 .. i-2 only (A squared has two zero diagonals),
// so two stages can be evaluated at a time, and nothing but the last
// accelerations is on the way from one pair of stages to the next.  A team of
// waves shares 64 orbits (lane = orbit) accordingly, on a SIMD each:
//   wave 0   evaluates the odd stages 1, 3, .. 11 and the end stage 13,
//   wave 1   the even stages 2, 4, .. 12,
//   wave 2   sums the tableau rows of the stages to come, and at a step's end
//            takes the decision and draws new orbits from the queue,
//   wave 3   saves: the dense output of the step before, two stages a level;
//            in fields on a staged track it looks up the track at the stage
//            times instead, and wave 2 saves between two steps.
// Stages 2m-1 and 2m are level m; the team meets at a workgroup barrier after
// each of the seven levels.  In level m waves 0 and 1 add to their rows the
// terms of level m-1 (their own acceleration from registers, the other's from
// LDS); wave 2 meanwhile adds those of level m-1 to the later rows.  Stage
// accelerations stay in LDS for the dense output.  The end stage is evaluated
// while wave 2 decides on the step, and used if it is accepted.
// All sums run over the stages in the order of rk_step, so that results are
// the same bits as the one-wave integrator's.
//
// A step takes 2.6 us.  A field wave's 120 instructions a level (about 5
// cycles each) are two thirds of it, the hand-over at the barriers (LDS write,
// barrier, LDS read, some 250 cycles a level) most of the rest.  1,024 orbits
// of 2,000 fixed steps: 8.8 -> 5.2 ms; 131,072 orbits of 0.1 to 5 Gyr: 47 ->
// 27 ms; the 100,000 particles of a 4 Gyr stream: 24.9 -> 15.4 ms.
//
// Lanes need not be in step in any other sense: each has its own step
// sequence, ends and restarts by itself.  After a step in which some lane
// ends (wave 2 knows before the last barrier) the team meets once more, while
// waves 2 and 3 see to those lanes.
#pragma once

#include "gx_rk.hpp"
#include "gx_steps.hpp"

namespace gx {
namespace {

constexpr int kTeamOrbits = 64;

// A workgroup's LDS: one column a lane everywhere.
template <bool TRACK>
struct TeamShared {
  // stage accelerations; by the step's parity where wave 3 saves from them
  // during the next step
  double g[TRACK ? 1 : 2][Dopri8::SF][3][kTeamOrbits];
  double start[3][kTeamOrbits];    // the step's start acceleration, unless
  int from_end[kTeamOrbits];       // it is g[13] of the step before
  double x1[2][3][kTeamOrbits];    // level 1: q + rs h p of stages 1, 2
  double x[2][2][6][kTeamOrbits];  // levels 2.. by parity, two stages: the
                                   // same, and the row's sum so far
  double hh[kTeamOrbits];          // h^2
  double when[TRACK ? 4 : 1][kTeamOrbits];      // tau, h, tnext, dir
  double at[TRACK ? 2 : 1][TRACK ? 2 : 1][3][kTeamOrbits];  // track at a level's two
                                                // stages, by its parity
  // what wave 3 needs to save: tau, h, q, p; tnext, q1, p1; and the outcome
  double begin[TRACK ? 1 : 8][kTeamOrbits];
  double end[TRACK ? 1 : 7][kTeamOrbits];
  int kept[kTeamOrbits];           // record index + 1 of an accepted step
  int done[kTeamOrbits];           // the orbit has ended
  long long orb[kTeamOrbits];      // a new orbit, and its first
  int si[kTeamOrbits];             // save to come
  int serve;  // some lane ends (or saves, without wave 3) before the next step
  int alive;  // some lane has an orbit (read after `serve`)
};

// The row of stage i at level m = (i + 1) / 2: wave 2 sums the terms through
// stage 2m - 4, the wave that evaluates the stage adds the rest.
constexpr int team_summed(int i) { return 2 * ((i + 1) / 2) - 4; }

constexpr bool row_is_empty(int i) {
  for (int l = 0; l < i; ++l)
    if (Dopri8::kf.aa[i][l] != 0.0) return false;
  return true;
}
constexpr bool two_zero_diagonals() {
  for (int i = 1; i < Dopri8::SF; ++i)
    if (Dopri8::kf.aa[i][i - 1] != 0.0) return false;
  return row_is_empty(1);
}
static_assert(two_zero_diagonals(), "two stages are independent of each other");

// The start acceleration of the step in buffer b.
template <bool TRACK>
__device__ __forceinline__ void team_start(const TeamShared<TRACK>& S, int b, int lane,
                                           double (&g)[3]) {
  const auto& before = S.g[TRACK ? 0 : 1 - b][Dopri8::SF - 1];
  const bool end = S.from_end[lane] != 0;
#pragma unroll
  for (int m = 0; m < 3; ++m) g[m] = end ? before[m][lane] : S.start[m][lane];
}

// One field wave's stage I (position, acceleration, into LDS).  `own` is this
// wave's acceleration of the level before (stage I - 2), replaced by stage
// I's; for an even stage the other wave's is read from LDS.
template <int I, class E, bool TRACK>
__device__ __forceinline__ void team_stage(const DPot& P, TeamShared<TRACK>& S, int b,
                                           int lane, double hh, double (&own)[3]) {
  constexpr auto& aa = Dopri8::kf.aa;
  constexpr int level = (I + 1) / 2, which = (I + 1) % 2;
  double Q[3];
  if constexpr (level == 1) {
#pragma unroll
    for (int m = 0; m < 3; ++m) Q[m] = S.x1[which][m][lane];
    if constexpr (I == 2 && aa[2][0] != 0.0) {
      double g0[3];
      team_start(S, b, lane, g0);
#pragma unroll
      for (int m = 0; m < 3; ++m) Q[m] = fma(hh, fma(aa[2][0], g0[m], 0.0), Q[m]);
    }
  } else {
    double s[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      Q[m] = S.x[level & 1][which][m][lane];
      s[m] = S.x[level & 1][which][m + 3][lane];
    }
    if constexpr (I % 2 == 0 && aa[I][I - 3] != 0.0) {
#pragma unroll
      for (int m = 0; m < 3; ++m) s[m] = fma(aa[I][I - 3], S.g[b][I - 3][m][lane], s[m]);
    }
    if constexpr (aa[I][I - 2] != 0.0) {
#pragma unroll
      for (int m = 0; m < 3; ++m) s[m] = fma(aa[I][I - 2], own[m], s[m]);
    }
    if constexpr (!row_is_empty(I)) {
#pragma unroll
      for (int m = 0; m < 3; ++m) Q[m] = fma(hh, s[m], Q[m]);
    }
  }
  if constexpr (TRACK) {
    // the track's positions at level 1 are looked up during the host's field
    EvalMilkyWay::acc(P, Q[0], Q[1], Q[2], 0.0, own[0], own[1], own[2]);
    if constexpr (level == 1) __syncthreads();
    const auto& d = S.at[level & 1][which];
    E::template add_tracked<I != 1>(P, Q[0], Q[1], Q[2], d[0][lane], d[1][lane], d[2][lane],
                                    own[0], own[1], own[2]);
  } else {
    E::acc(P, Q[0], Q[1], Q[2], 0.0, own[0], own[1], own[2]);
  }
#pragma unroll
  for (int m = 0; m < 3; ++m) S.g[b][I][m][lane] = own[m];
}

// Odd (FIRST = 1) or even (FIRST = 2) stages from I on, a barrier after each.
template <int I, class E, bool TRACK>
__device__ __forceinline__ void team_stages(const DPot& P, TeamShared<TRACK>& S, int b,
                                            int lane, double hh, double (&own)[3]) {
  if constexpr (I < Dopri8::SF) team_stage<I, E, TRACK>(P, S, b, lane, hh, own);
  __syncthreads();
  if constexpr (I + 2 < Dopri8::SF + 1) team_stages<I + 2, E, TRACK>(P, S, b, lane, hh, own);
}

template <int FIRST, class E, bool TRACK>
__device__ void team_field(const DPot& P, TeamShared<TRACK>& S, int lane) {
  __syncthreads();
  if (!S.alive) return;
  double own[3] = {0.0, 0.0, 0.0};
  for (int b = 0;; b ^= TRACK ? 0 : 1) {
    team_stages<FIRST, E, TRACK>(P, S, b, lane, S.hh[lane], own);
    if (S.serve) {
      __syncthreads();
      if (!S.alive) return;
    }
  }
}

// The track at the stage times: level 1's at the start of the step, then
// those of level m + 1 during level m.
template <int LEVEL, class E, bool TRACK>
__device__ __forceinline__ void team_lookup(const DPot& P, TeamShared<TRACK>& S,
                                            int lane, double tau, double h,
                                            double tnext, double dir) {
  constexpr int i0 = 2 * LEVEL - 1;
  constexpr int N = i0 + 1 < Dopri8::SF ? 2 : 1;
  double t[N], d[N][3];
#pragma unroll
  for (int j = 0; j < N; ++j)
    t[j] = dir * (i0 + j == Dopri8::SF - 1 ? tnext : fma(Dopri8::kf.c[i0 + j], h, tau));
  E::template track_n<N>(P, t, d);
#pragma unroll
  for (int j = 0; j < N; ++j)
#pragma unroll
    for (int m = 0; m < 3; ++m) S.at[LEVEL & 1][j][m][lane] = d[j][m];
  __syncthreads();
  if constexpr (LEVEL < 7)
    team_lookup<LEVEL + 1, E, TRACK>(P, S, lane, tau, h, tnext, dir);
}

template <class E, bool TRACK>
__device__ void team_track(const DPot& P, TeamShared<TRACK>& S, int lane) {
  __syncthreads();
  if (!S.alive) return;
  for (;;) {
    team_lookup<1, E, TRACK>(P, S, lane, S.when[0][lane], S.when[1][lane],
                             S.when[2][lane], S.when[3][lane]);
    __syncthreads();  // level 7
    if (S.serve) {
      __syncthreads();
      if (!S.alive) return;
    }
  }
}

// Wave 2's sums over a step's stages: the rows of stages 3 .. 13 and the
// solution and error rows (13 .. 15 of `row_weight`).  Their weights lie in one
// table in the order of use, level by level, and are read by scalar loads
// where they are used (table_here): as compile-time constants they cost two
// moves or two lane reads a weight, and wave 2 then took longer than the
// fields (3.5 us a step).
constexpr int kTeamSums = Dopri8::SF + 3;
constexpr double team_weight(int i, int l) {
  constexpr auto& K = Dopri8::kf;
  if (i < Dopri8::SF) return i >= 3 && l <= team_summed(i) ? K.aa[i][l] : 0.0;
  return i == Dopri8::SF ? K.b[l] : i == Dopri8::SF + 1 ? K.e[l] : K.ea[l];
}
struct TeamTable {
  double w[Dopri8::S * kTeamSums];
  int at[Dopri8::S][kTeamSums];
  int first[Dopri8::S + 1];
};
constexpr TeamTable make_team_table() {
  TeamTable t{};
  int n = 0;
  for (int l = 0; l < Dopri8::S; ++l) {
    t.first[l] = n;
    for (int i = 0; i < kTeamSums; ++i) {
      t.at[l][i] = -1;
      if (team_weight(i, l) != 0.0) {
        t.at[l][i] = n;
        t.w[n++] = team_weight(i, l);
      }
    }
  }
  t.first[Dopri8::S] = n;
  return t;
}
struct TeamWeights {
  static constexpr TeamTable t = make_team_table();
};

struct TeamSums {
  double row[kTeamSums][3];

  // the terms of stage L; `w` is the table from stage L0 on
  template <int L, int L0, bool PID>
  __device__ __forceinline__ void add(ConstDouble* w, const double (&g)[3]) {
    static_for<3, PID ? kTeamSums : Dopri8::SF + 1>([&](auto row_) {
      constexpr int i = decltype(row_)::value;
      constexpr int at = TeamWeights::t.at[L][i];
      if constexpr (at >= 0) {
        const double a = w[at - TeamWeights::t.first[L0]];
#pragma unroll
        for (int m = 0; m < 3; ++m) row[i][m] = fma(a, g[m], row[i][m]);
      }
    });
  }
};

// What the field and track waves need at the start of a step.
template <bool TRACK>
__device__ __forceinline__ void team_publish(TeamShared<TRACK>& S, int lane, double tau,
                                             double tnext, double dir, const double (&q)[3],
                                             const double (&p)[3]) {
  constexpr auto& K = Dopri8::kf;
  const double h = tnext - tau;
  S.hh[lane] = h * h;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const double hp = h * p[m];
    S.x1[0][m][lane] = fma(K.rs[1], hp, q[m]);
    S.x1[1][m][lane] = fma(K.rs[2], hp, q[m]);
  }
  if constexpr (TRACK) {
    S.when[0][lane] = tau;
    S.when[1][lane] = h;
    S.when[2][lane] = tnext;
    S.when[3][lane] = dir;
  }
}

// What the saving wave needs at its end (kept: the record's index + 1).
__device__ __forceinline__ int record_slot(long long nacc, long long cap) {
  return (int)(nacc <= cap ? nacc : cap + 1);
}
__device__ __forceinline__ void team_outcome(TeamShared<false>& S, int lane, bool keep, int kept,
                                             bool done, double tend, const double (&q1)[3],
                                             const double (&p1)[3]) {
  S.kept[lane] = keep ? kept : 0;
  S.done[lane] = done ? 1 : 0;
  S.end[0][lane] = tend;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    S.end[1 + m][lane] = q1[m];
    S.end[4 + m][lane] = p1[m];
  }
}

template <bool TRACK>
__device__ __forceinline__ void team_stage_acc(const TeamShared<TRACK>& S, int b, int l, int lane,
                                               double (&g)[3]) {
#pragma unroll
  for (int m = 0; m < 3; ++m) g[m] = S.g[b][l][m][lane];
}

// Wave 2's sums from a step's start through its stage 12 (levels 1 to 6, a
// barrier after each): the end state and the error estimate; false if the end
// state is not finite.
template <bool PID, bool TRACK>
__device__ __forceinline__ bool team_rows(TeamShared<TRACK>& S, int b, int lane, double tau,
                                          double h, const double (&q)[3], const double (&p)[3],
                                          double (&q1)[3], double (&p1)[3], double (&eq)[3],
                                          double (&ep)[3]) {
  using M = Dopri8;
  constexpr int SF = M::SF;
  constexpr auto& K = M::kf;
  const double hh = h * h;
  const double hp[3] = {h * p[0], h * p[1], h * p[2]};
  auto load = [&](int l, double (&g)[3]) { team_stage_acc(S, b, l, lane, g); };
  TeamSums s;
#pragma unroll
  for (int i = 0; i < kTeamSums; ++i) s.row[i][0] = s.row[i][1] = s.row[i][2] = 0.0;
  // the next level's rows, for its two stages
  auto hand_over = [&](auto level) {
    constexpr int lv = decltype(level)::value;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      constexpr int i0 = 2 * lv - 1;
      if (i0 + w < SF) {
#pragma unroll
        for (int m = 0; m < 3; ++m) {
          S.x[lv & 1][w][m][lane] = fma(M::kf.rs[i0 + w < SF ? i0 + w : 0], hp[m], q[m]);
          S.x[lv & 1][w][m + 3][lane] = s.row[i0 + w < SF ? i0 + w : 0][m];
        }
      }
    }
  };
  auto add_two = [&](auto first, const double (&g1)[3], const double (&g2)[3]) {
    constexpr int L = decltype(first)::value;
    ConstDouble* w = table_here(TeamWeights::t.w + TeamWeights::t.first[L]);
    s.add<L, L, PID>(w, g1);
    s.add<L + 1, L, PID>(w, g2);
  };
  double ga[3], gb[3];
  // level 1: the start acceleration
  if (TRACK) __syncthreads();
  team_start(S, b, lane, ga);
#pragma unroll
  for (int m = 0; m < 3; ++m) S.start[m][lane] = S.g[b][0][m][lane] = ga[m];
  s.add<0, 0, PID>(table_here(TeamWeights::t.w), ga);
  hand_over(std::integral_constant<int, 2>{});
  __syncthreads();
  // levels 2 .. 6: the stages of the level before
  if constexpr (!TRACK) {
    S.begin[0][lane] = tau;
    S.begin[1][lane] = h;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      S.begin[2 + m][lane] = q[m];
      S.begin[5 + m][lane] = p[m];
    }
  }
  load(1, ga);
  load(2, gb);
  add_two(std::integral_constant<int, 1>{}, ga, gb);
  hand_over(std::integral_constant<int, 3>{});
  __syncthreads();
  load(3, ga);
  load(4, gb);
  add_two(std::integral_constant<int, 3>{}, ga, gb);
  hand_over(std::integral_constant<int, 4>{});
  __syncthreads();
  load(5, ga);
  load(6, gb);
  add_two(std::integral_constant<int, 5>{}, ga, gb);
  hand_over(std::integral_constant<int, 5>{});
  __syncthreads();
  load(7, ga);
  load(8, gb);
  add_two(std::integral_constant<int, 7>{}, ga, gb);
  hand_over(std::integral_constant<int, 6>{});
  __syncthreads();
  load(9, ga);
  load(10, gb);
  add_two(std::integral_constant<int, 9>{}, ga, gb);
  hand_over(std::integral_constant<int, 7>{});
  __syncthreads();
  // level 7: the step's end, beside the end stage
  load(11, ga);
  load(12, gb);
  add_two(std::integral_constant<int, 11>{}, ga, gb);
  bool finite = true;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const double a = K.aa[13][11] != 0.0 ? fma(K.aa[13][11], ga[m], s.row[13][m]) : s.row[13][m];
    q1[m] = fma(hh, a, fma(K.rs[SF - 1], hp[m], q[m]));
    p1[m] = fma(h, s.row[SF][m], p[m]);
    ep[m] = h * s.row[SF + 1][m];
    eq[m] = fma(hh, s.row[SF + 2][m], K.se * hp[m]);
    finite = finite && isfinite(q1[m]) && isfinite(p1[m]);
  }
  return finite;
}

// Wave 2: everything but the field.
template <bool PID, class E, bool DENSE, bool TRACK>
__device__ void team_control(const DPot& P, const IArgs& A, TeamShared<TRACK>& S,
                             int lane) {
  using M = Dopri8;
  constexpr int SF = M::SF;
  const long long slot = (long long)blockIdx.x * kTeamOrbits + lane;
  // the first tickets of a cost-ordered queue: no second ticket for them in a
  // grid large enough for the rest to drain the queue
  const bool head = slot < A.head_lanes;
  long long qnext = 0, qend = 0;
  auto draw = [&]() -> long long {
    if (head && A.head_only_once) return -1;
    long long idx = qnext;
    if (idx >= qend) {
      idx = A.head_lanes + (long long)atomicAdd(A.counter, (unsigned long long)A.chunk);
      qend = idx + A.chunk;
    }
    qnext = idx + 1;
    return ticket_to_orbit(A, idx);
  };
  long long orb = head ? ticket_to_orbit(A, slot) : draw();
  double q[3] = {1.0, 0.0, 0.0}, p[3] = {0.0, 0.0, 0.0};
  double tau = 0.0, tnext = 0.0, tau1 = 0.0, dir = 1.0, t0v = 0.0, t1v = 0.0;
  double prev_inv = 1.0, prev_prev_inv = 1.0;
  double tsave = 0.0;  // TRACK: the next save time (solver time), while si < A.T
  long long nst = 0, nacc = 0;
  int si = 0, st = GX_SUCCESS, at_dtmin = 0;

  auto next_save = [&]() { tsave = si < A.T ? dir * save_time(A, orb, si, t0v, t1v) : 0.0; };
  // whether the orbit stops before its next attempt
  auto stops = [&]() {
    if (nst >= A.max_steps) {
      st = GX_MAX_STEPS_REACHED;
      return true;
    }
    if (!(tnext - tau >= 0.0)) {
      st = GX_NONFINITE;
      return true;
    }
    return false;
  };
  auto finish = [&](bool rest) {
    if (rest) write_rest(A, orb, si);
    if (A.status) A.status[orb] = st;
    if (A.nsteps) A.nsteps[orb] = nst;
    if (A.naccept) A.naccept[orb] = nacc;
    if constexpr (DENSE) A.nrec[orb] = nacc < A.rec_cap ? nacc : A.rec_cap;
    orb = draw();
  };
  // a lane without a running orbit takes the next one that has a step to do
  auto start = [&]() {
    while (orb >= 0) {
      t0v = A.t0[A.t_stride ? orb : 0];
      t1v = A.t1[A.t_stride ? orb : 0];
      const double* w = A.w0 + orb * 6;
      dir = (t0v < t1v) ? 1.0 : -1.0;
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        q[m] = w[m];
        p[m] = dir * w[m + 3];
      }
      tau = dir * t0v;
      tau1 = dir * t1v;
      prev_inv = prev_prev_inv = 1.0;
      nst = nacc = 0;
      st = GX_SUCCESS;
      si = 0;
      if (t0v == t1v) {
        for (; si < A.T; ++si) write_save(A, orb, si, dir, q, p);
      } else {
        const double h0 = A.h0[orb];
        at_dtmin = (PID && A.dtmin > 0.0 && h0 == A.dtmin) ? 1 : 0;
        tnext = fmin(tau + h0, tau1);
        for (next_save(); si < A.T && tsave <= tau; next_save()) {
          write_save(A, orb, si, dir, q, p);
          ++si;
        }
        if (!stops()) {
#pragma unroll
          for (int m = 0; m < 3; ++m) S.start[m][lane] = A.a0[3 * orb + m];
          S.from_end[lane] = 0;
          break;
        }
      }
      finish(true);
    }
    if constexpr (!TRACK) {
      S.orb[lane] = orb;
      S.si[lane] = si;
    }
  };
  auto publish = [&]() { team_publish(S, lane, tau, tnext, dir, q, p); };
  int b = 0;  // the step's buffer of stage accelerations

  S.from_end[lane] = 0;
#pragma unroll
  for (int m = 0; m < 3; ++m) S.start[m][lane] = 0.0;
  start();
  publish();
  {
    const bool any = __any(orb >= 0);
    if (lane == 0) S.alive = any;
  }
  __syncthreads();
  if (!__any(orb >= 0)) return;

  for (;; b ^= TRACK ? 0 : 1) {
    const double h = tnext - tau;
    double q1[3], p1[3], eq[3], ep[3];
    const bool finite = team_rows<PID, TRACK>(S, b, lane, tau, h, q, p, q1, p1, eq, ep);
    const double tau_s = tau, tend = tnext;
    const double qs[3] = {q[0], q[1], q[2]}, ps[3] = {p[0], p[1], p[2]};
    bool keep = false, done = false;
    if (orb >= 0) {
      nst += 1;
      if (!finite) {
        st = GX_NONFINITE;
        done = true;
      } else {
        double next_t1;
        keep = control_step<PID>(A, tau, tnext, q, p, q1, p1, eq, ep, prev_inv,
                                 prev_prev_inv, at_dtmin, st, next_t1);
        if (keep) {
          if constexpr (DENSE)
            if (nacc >= A.rec_cap) st = GX_MAX_STEPS_REACHED;  // out of record slots
#pragma unroll
          for (int m = 0; m < 3; ++m) {
            q[m] = q1[m];
            p[m] = p1[m];
          }
          tau = tnext;
          nacc += 1;
        }
        const double tprev = fmin(tau, tau1);
        tnext = clip_to_end(tprev, next_t1, tau1, keep);
        tau = tprev;
        done = st == GX_DT_MIN_REACHED || (DENSE && st == GX_MAX_STEPS_REACHED) || tau >= tau1;
        if (!done) done = stops();
      }
    }
    S.from_end[lane] = keep ? 1 : 0;
    if constexpr (!TRACK) {
      team_outcome(S, lane, keep, DENSE ? record_slot(nacc, A.rec_cap) : 1, done, tend, q1, p1);
    }
    const bool saves = TRACK && keep && si < A.T && !(tsave > tend);
    const bool serve = __any(done || saves);
    if (lane == 0) S.serve = serve ? 1 : 0;
    publish();
    __syncthreads();
    if (!serve) continue;

    // some lane ends (or saves): see to it while the field waits
    if (saves) {
      double g[SF][3];
#pragma unroll
      for (int l = 0; l < SF; ++l) team_stage_acc(S, b, l, lane, g[l]);
      while (si < A.T && !(tsave > tend)) {
        if (tsave == tend) {
          write_save(A, orb, si, dir, q1, p1);
        } else {
          double qo[3], po[3];
          dense_eval<M, true>(div(tsave - tau_s, h), h, qs, ps, g, qo, po);
          write_save(A, orb, si, dir, qo, po);
        }
        ++si;
        next_save();
      }
    }
    if (done) {
      finish(TRACK);
      start();
      publish();
    }
    const bool any = __any(orb >= 0);
    if (lane == 0) S.alive = any ? 1 : 0;
    __syncthreads();
    if (!any) return;
  }
}

// Wave 3 without a track: the saves (and dense records) of the step before,
// from its buffer of stage accelerations, while the others take the next one.
// A lane's first save in the step is summed two stages a level; further ones
// follow in the last level.  When some lane ends, all saves of the step come
// before the team goes on.
template <bool DENSE, class Args>
__device__ void team_saves(const Args& A, TeamShared<false>& S, int lane) {
  using M = Dopri8;
  constexpr int SF = M::SF;
  __syncthreads();
  if (!S.alive) return;
  long long orb = -1;
  int si = 0;
  double tsave = 0.0, dir = 1.0, t0v = 0.0, t1v = 0.0;
  double tau, h, tend, q[3], p[3], q1[3], p1[3];
  int kept = 0;
  auto next_save = [&]() { tsave = si < A.T ? dir * save_time(A, orb, si, t0v, t1v) : 0.0; };
  auto take = [&]() {
    orb = S.orb[lane];
    si = S.si[lane];
    if (orb >= 0) {
      orbit_span(A, orb, t0v, t1v);
      dir = (t0v < t1v) ? 1.0 : -1.0;
      next_save();
    }
  };
  auto fetch = [&]() {
    kept = orb >= 0 ? S.kept[lane] : 0;
    tau = S.begin[0][lane];
    h = S.begin[1][lane];
    tend = S.end[0][lane];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      q[m] = S.begin[2 + m][lane];
      p[m] = S.begin[5 + m][lane];
      q1[m] = S.end[1 + m][lane];
      p1[m] = S.end[4 + m][lane];
    }
  };
  auto due = [&]() { return kept != 0 && si < A.T && !(tsave > tend); };
  auto load = [&](int b, int l, double (&g)[3]) { team_stage_acc(S, b, l, lane, g); };
  auto write = [&](const double (&qo)[3], const double (&po)[3]) {
    if (tsave == tend)
      write_save(A, orb, si, dir, q1, p1);
    else
      write_save(A, orb, si, dir, qo, po);
    ++si;
    next_save();
  };
  // the remaining saves and the record of the step in buffer b
  auto all_saves = [&](int b) {
    while (due()) {
      double g[SF][3], qo[3], po[3];
#pragma unroll
      for (int l = 0; l < SF; ++l) load(b, l, g[l]);
      const double th = div(tsave - tau, h);
      dense_eval<M, true>(th, h, q, p, g, qo, po);
      write(qo, po);
    }
  };
  auto record = [&](int b) {
    if constexpr (DENSE) {
      if (kept != 0 && kept <= A.rec_cap) {
        double g[SF][3];
#pragma unroll
        for (int l = 0; l < SF; ++l) load(b, l, g[l]);
        write_record<M>(A.rec + (orb * A.rec_cap + kept - 1) * kDenseRec, dir, tau, h, q, p, g);
      }
    }
  };
  take();
  bool pending = false;
  for (int b = 0;; b ^= 1) {
    if (pending) fetch();
    if (pending && __any(due())) {
      const bool mine = due();
      const double th = div(tsave - tau, h);
      DenseSum sum;
      static_for<0, 7>([&](auto level) {
        constexpr int l = 2 * decltype(level)::value;
        ConstDouble* tq = table_here(&M::dn.wq[0][0]);
        ConstDouble* tp = table_here(&M::dn.wp[0][0]);
        double g[3];
        load(1 - b, l, g);
        sum.add<M, l>(tq, tp, th, g);
        load(1 - b, l + 1, g);
        sum.add<M, l + 1>(tq, tp, th, g);
        if constexpr (l < 12) __syncthreads();
      });
      if (mine) {
        double qo[3], po[3];
        sum.result(th, h, q, p, qo, po);
        write(qo, po);
        all_saves(1 - b);
      }
    } else {
      for (int l = 1; l < 7; ++l) __syncthreads();
    }
    if (pending) record(1 - b);
    __syncthreads();  // level 7
    pending = true;
    if (S.serve) {
      fetch();
      all_saves(b);
      record(b);
      const bool ended = S.done[lane] != 0 && orb >= 0;
      if (ended) write_rest(A, orb, si);
      __syncthreads();
      if (!S.alive) return;
      if (ended) take();
      pending = false;
    }
  }
}

template <bool PID, class E, bool DENSE>
__global__ void __launch_bounds__(256) k_team(DPot P, IArgs A) {
  constexpr bool TRACK = track_prefetch<E>::value;
  __shared__ TeamShared<TRACK> S;
  if (A.choose && !teams_take(A)) return;
  if constexpr (TRACK) {
    E::stage(P);
    __syncthreads();
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  if ((long long)blockIdx.x * kTeamOrbits < A.head_lanes) __builtin_amdgcn_s_setprio(3);
  if (wave == 0)
    team_field<1, E, TRACK>(P, S, lane);
  else if (wave == 1)
    team_field<2, E, TRACK>(P, S, lane);
  else if (wave == 2)
    team_control<PID, E, DENSE, TRACK>(P, A, S, lane);
  else if constexpr (TRACK)
    team_track<E, TRACK>(P, S, lane);
  else
    team_saves<DENSE>(A, S, lane);
}

}  // namespace
}  // namespace gx
