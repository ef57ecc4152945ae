// rodas5p_team.hpp -- the Rodas5P ensemble step of a sparse system shared out
// over a workgroup's wavefronts.
//
// Included after rodas5p.hpp when MDX_TEAM > 0, in a source
// whose sys namespace holds, beside neg_jac (reading y by slot) and the
// pattern's sparse_factor and sparse_solve:
//   rhs_rows(wave, y, t, p, out)  wavefront ``wave``'s rows of the right-hand
//                                 side, reading y by slot
//   sens_rhs_rows, sens_coupling_rows  the same rows of a sensitivity
//                                 direction's right-hand side and of the
//                                 coupling of its stage (MDX_NSENS > 0)
//   ROW_OF[(W - 1) * R]           the variable a slot holds, -1 for padding
//   SLOT_OF[N]                    the slot of a variable
// Macros: MDX_TEAM wavefronts, MDX_TEAM_ROWS slots of each but the first,
// MDX_BLOCK trajectories (the same in the same lanes of every wavefront).
//
// Wavefront 0 forms and factorises the iteration matrix and runs the stage
// solves, which are chains along the elimination tree; the others own the rows:
// their state, stage vectors and sums are registers, the stage argument and
// the right-hand side go through LDS. A stage is three barriers: argument
// written, right-hand side written, solution written. The owners form the
// next stage's sums, all but the newest term, while the solve runs. One lane a
// trajectory keeps one wavefront of the compute unit busy with all of it and
// every vector in LDS or scratch. Each element sees that step's operations in
// their order, and the error norm is summed in ascending order by wavefront 0,
// so the bits are the same. A step is bounded by latency: at 20 variables 8 us,
// of which eight solves are 3, the factorisation 1, the controller 1, the dense
// output 1 and three exchanges a stage most of the rest; one lane a trajectory
// takes 20. Kept out: the factors in LDS (the 64-variable ring 0.84 -> 2.2 ms:
// the solves then wait for each element) and a wavefront's reads ahead of its
// arithmetic (more registers, no faster).
//
// The joint [y, S] solve puts its blocks side by side in the lanes: lane
// b * MDX_BLOCK + l holds block b (0: the state, then the directions) of
// trajectory l, so the sums, which are alike for all blocks, cost what the
// plain solve's cost and no lane holds more than R rows of one block. The
// blocks' right-hand sides run one after the other under a mask, and a stage
// takes two solves against the same factors, the directions' once the state's
// solution is known (rodas5P.py:512-561). The 64-variable ring with one
// parameter direction, 1,000 trajectories: 12.0 ms with one lane a trajectory,
// 2.9 ms with a team.
//
// With MDX_ADJOINT=1 (rodas5p_adjoint_team.hpp, included next) the steps write
// no history, and every stage has a place of its own in LDS.
#pragma once

#if !MDX_DT_ZERO || !MDX_SPARSE || MDX_HOOK || MDX_REFINE || (MDX_ADJOINT && MDX_NSENS > 0)
#error "a team makes the plain or joint solve of a sparse system whose right-hand side does not read t"
#endif

namespace mdx {
namespace r5 {

constexpr int W = MDX_TEAM;
constexpr int R = MDX_TEAM_ROWS;
constexpr int T = MDX_BLOCK;
constexpr int SLOTS = (W - 1) * R;
constexpr int BLOCKS = 1 + NS;     // the state, and each direction
constexpr int LANES = T * BLOCKS;  // lanes at work

#if MDX_ADJOINT
// the adjoint keeps every stage's argument and solution for the sweep back
constexpr int STAGE = SLOTS * LANES;
__shared__ double lds_u[8 * STAGE];
__shared__ LUT lds_r[8 * STAGE];
#else
constexpr int STAGE = 0;  // each stage in the place of the one before
__shared__ double lds_u[SLOTS * LANES];  // stage argument, [slot][lane]; then the error terms
__shared__ LUT lds_r[SLOTS * LANES];     // a stage's right-hand side, then its solution
#endif
#if MDX_NSENS > 0
__shared__ double lds_b[SLOTS * LANES];  // the step's base point
#endif
__shared__ double lds_c[2 * T];  // the step's outcome: next step size, error norm
__shared__ i64 lds_claim[T];
#if MDX_TEAM_LDS_PARAMS
__shared__ double lds_p[MDX_NP * T];
struct TeamParams {
  const double* base;
  __device__ __forceinline__ TeamParams(int l) : base(&lds_p[l]) {}
  __device__ __forceinline__ double operator[](int m) const { return base[m * T]; }
  // wavefront w brings in every W-th parameter; the step's first barrier makes
  // them visible
  __device__ __forceinline__ void load(const SolveArgs& a, i64 i, int w, int l) {
    for (int m = w; m < MDX_NP; m += W) lds_p[m * T + l] = a.params[i * a.p_ts + (i64)m * a.p_vs];
  }
};
#else
struct TeamParams : RegParams<MDX_NP> {
  __device__ __forceinline__ TeamParams(int) : RegParams<MDX_NP>{} {}
  __device__ __forceinline__ void load(const SolveArgs& a, i64 i, int, int) {
    RegParams<MDX_NP>::load(a, i);
  }
};
#endif

struct Slots {
  const double* base;
  __device__ __forceinline__ double operator[](int s) const { return base[s * LANES]; }
};
#if MDX_NSENS > 0 || MDX_ADJOINT
struct Solution {
  const LUT* base;
  __device__ __forceinline__ double operator[](int s) const { return (double)base[s * LANES]; }
};
#endif

// The step control, the same values in every wavefront (err_prev and err_prev2
// only in wavefront 0, which forms the step size).
struct Control {
  double t, dt, tf, ts, err_prev, err_prev2;
  int save_idx, n_steps, accepted, rejected;
};

__device__ __forceinline__ void control_init(Control& s, const SolveArgs& a, i64 i) {
  const double* __restrict__ times = a.times;
  const double tf = times[a.n_save - 1];
  s.t = times[0];
  s.dt = a.dt0 > 0.0 ? a.dt0 : (tf - times[0]) * 1e-6;
#if MDX_TF_INDEX >= 0
  s.tf = a.params[i * a.p_ts + (i64)MDX_TF_INDEX * a.p_vs];
#else
  s.tf = tf;
#endif
  s.err_prev = 1.0;
  s.err_prev2 = 1.0;
  s.save_idx = 1;
  s.n_steps = 0;
  s.accepted = 0;
  s.rejected = 0;
  if (a.resume && !a.cost) {
    // where a cost pilot left the trajectory (layout as in rodas5p.hpp's init)
    const double* __restrict__ r = a.resume + i;
    const i64 st = a.n_traj;
    s.t = r[(NA + 0) * st];
    s.dt = r[(NA + 1) * st];
    s.err_prev = r[(NA + 2) * st];
    s.err_prev2 = r[(NA + 3) * st];
    s.save_idx = (int)r[(NA + 4) * st];
    s.n_steps = (int)r[(NA + 5) * st];
    s.accepted = (int)r[(NA + 6) * st];
    s.rejected = (int)r[(NA + 7) * st];
  }
  s.ts = next_save(a, s.save_idx);
}

__device__ __forceinline__ bool team_active(const Control& s, const SolveArgs& a) {
  return s.save_idx < a.n_save && s.t < s.tf && s.n_steps < a.max_steps;
}

// The step size this step takes (the one-lane step's first lines).
__device__ __forceinline__ double step_length(const Control& s) {
  double dt_use = s.dt;
  if (dt_use > s.tf - s.t) dt_use = s.tf - s.t;
  if (dt_use < 1e-30) dt_use = 1e-30;
  return dt_use;
}

// Whether the next save lies in the step that ends at t_new.
__device__ __forceinline__ bool save_due(const Control& s, const SolveArgs& a, double t_new) {
  const double at = absT(s.ts);
  return s.save_idx < a.n_save && s.ts <= t_new + 1e-12 * (1.0 > at ? 1.0 : at);
}

// Wavefront 0: the iteration matrix, its factors, the stage solves, the error
// norm and the step control.
struct Solver {
  static constexpr bool FIRST = true;
  __device__ __forceinline__ void init(const SolveArgs&, i64, int, int) {}

  // The factorisation at the state in lds_u and the stage solves.
  __device__ __forceinline__ void stages(double t, double dt_use, const TeamParams& p, int lane,
                                         LUT (&lu)[MDX_NLU], Pivots& ipiv) {
    const int l = lane % T;
    const bool state = lane < T;
    (void)state;
    const double dtgamma_inv = 1.0 / (dt_use * GAMMA);
#if MDX_NEEDS_CLEAR
#pragma unroll
    for (int q = 0; q < MDX_NLU; ++q) lu[q] = (LUT)0;
#endif
    __syncthreads();  // the state is in lds_u
    {
      double dT[N];
      sys::neg_jac(Slots{&lds_u[l]}, t, p, lu, dT);
    }
#pragma unroll
    for (int d = 0; d < N; ++d) lu[diag_slot(d)] = lu[diag_slot(d)] + (LUT)dtgamma_inv;
    factor(lu, ipiv);
#pragma unroll 1
    for (int S = 0; S < 8; ++S) {
      if (S > 0) __syncthreads();  // the owners wrote the stage argument
      // the state's blocks, then the directions'
#pragma unroll 1
      for (int pass = 0; pass < (NS > 0 ? 2 : 1); ++pass) {
        __syncthreads();  // the right-hand side is written
        if (NS == 0 || state == (pass == 0)) {
          LUT r[N];
#pragma unroll
          for (int v = 0; v < N; ++v) r[v] = lds_r[S * STAGE + sys::SLOT_OF[v] * LANES + lane];
          solve(lu, ipiv, r);
#pragma unroll
          for (int v = 0; v < N; ++v) lds_r[S * STAGE + sys::SLOT_OF[v] * LANES + lane] = r[v];
        }
        __syncthreads();
      }
    }
  }

  __device__ __forceinline__ void step(Control& s, const TeamParams& p, const SolveArgs& a, i64,
                                       int, int lane, bool act) {
    const int l = lane % T;
    const bool state = lane < T;
    const double dt_use = step_length(s);
    {
      LUT lu[MDX_NLU];
      Pivots ipiv;
      stages(s.t, dt_use, p, lane, lu, ipiv);
    }
    __syncthreads();  // the error terms are in lds_u
    double err = 0.0;
#pragma unroll MDX_SENS_UNROLL
    for (int b = 0; b < BLOCKS; ++b)
#pragma unroll
      for (int v = 0; v < N; ++v) {
        const double r = lds_u[sys::SLOT_OF[v] * LANES + b * T + l];
        err = fmaT(r, r, err);
      }
    const double err_norm = __builtin_sqrt(err / (double)MDX_N_ERROR);
    const bool accept = err_norm <= 1.0 && !__builtin_isnan(err_norm);
    double e1 = s.err_prev, e2 = s.err_prev2;
    const double factor_ = pid_factor(err_norm, accept, e1, e2, MDX_E1, MDX_E2, MDX_E3, 0.2, 6.0);
    const double dt_next = dt_use * factor_;
    if (state) {
      lds_c[l] = dt_next;
      lds_c[T + l] = err_norm;
    }
    __syncthreads();
    if (act) {
      s.err_prev = e1, s.err_prev2 = e2;
      s.dt = dt_next;
      if (accept) {
        const double t_new = s.t + dt_use;
        while (save_due(s, a, t_new)) {
          s.save_idx++;
          s.ts = next_save(a, s.save_idx);
        }
        s.t = t_new;
        s.accepted++;
      } else {
        s.rejected++;
      }
      s.n_steps++;
    }
  }

  __device__ __forceinline__ void finish(Control& s, const SolveArgs& a, i64 i, int, int lane) {
    if (lane >= T) return;
    if (a.cost) {
      // a cost pilot (see rodas5p.hpp's finish): the steps left, and the step state
      a.cost[i] = (s.save_idx < a.n_save && s.t < s.tf) ? (s.tf - s.t) / s.dt : 0.0;
      if (a.resume) {
        double* __restrict__ r = a.resume + i;
        const i64 st = a.n_traj;
        r[(NA + 0) * st] = s.t;
        r[(NA + 1) * st] = s.dt;
        r[(NA + 2) * st] = s.err_prev;
        r[(NA + 3) * st] = s.err_prev2;
        r[(NA + 4) * st] = (double)s.save_idx;
        r[(NA + 5) * st] = (double)s.n_steps;
        r[(NA + 6) * st] = (double)s.accepted;
        r[(NA + 7) * st] = (double)s.rejected;
      }
      return;
    }
    a.accepted[i] = s.accepted;
    a.rejected[i] = s.rejected;
    a.loop[i] = s.n_steps;
  }
};

// Wavefronts 1 .. W-1: the rows.
struct Owner {
  static constexpr bool FIRST = false;
  double y[R];

  __device__ __forceinline__ int row(int w, int j) const { return sys::ROW_OF[(w - 1) * R + j]; }
  __device__ __forceinline__ int at(int w, int j, int lane) const {
    return ((w - 1) * R + j) * LANES + lane;
  }
  // a row's place in the joint vector
  __device__ __forceinline__ i64 joint(int v, int lane) const {
    return NS > 0 ? (i64)(v + lane / T * N) : (i64)v;
  }

  __device__ __forceinline__ void init(const SolveArgs& a, i64 i, int w, int lane) {
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int v = row(w, j);
      y[j] = 0.0;
      if (v >= 0) {
        const i64 q = joint(v, lane);
        y[j] = a.y0[i * a.y0_ts + q * a.y0_vs];
#if !MDX_ADJOINT
        a.hist[i * a.h_ts + q * a.h_vs] = y[j];
#endif
        if (a.resume && !a.cost) y[j] = a.resume[i + q * a.n_traj];
      }
    }
  }

  // One stage: sa and sc are the sums of the earlier stage vectors in the stage
  // argument and the right-hand side, without the newest one's term.
  template <int S>
  __device__ __forceinline__ void stage(KT (&k)[8][R], double (&u)[R], double (&sa)[R],
                                        double (&sc)[R], const double (&dT)[R],
                                        const TeamParams& p, int w, int lane, double t,
                                        double dt_use, double inv_dt) {
#pragma unroll
    for (int j = 0; j < R; ++j) {
      if constexpr (S == 0) {
        u[j] = y[j];
      } else if constexpr (S < 6) {
        const double kn = (double)k[S - 1][j];
        const double acc = S == 1 ? AM[S - 1][S - 1] * kn : fmaT(AM[S - 1][S - 1], kn, sa[j]);
        u[j] = y[j] + acc;
      } else {
        u[j] = u[j] + (double)k[S - 1][j];
      }
      lds_u[S * STAGE + at(w, j, lane)] = u[j];
#if MDX_NSENS > 0
      if constexpr (S == 0) lds_b[at(w, j, lane)] = u[j];
#endif
    }
    __syncthreads();
    const int l = lane % T;
    const bool state = lane < T;
    double work[R];
    const double ts = S == 0 ? t : S < 5 ? t + CT[S > 0 && S < 5 ? S - 1 : 0] * dt_use : t + dt_use;
#if MDX_NSENS > 0
    const OneHot pd{state ? -1 : PCOL[state ? 0 : lane / T - 1]};
    if (state)
      sys::rhs_rows(w, Slots{&lds_u[l]}, ts, p, work);
    else
      sys::sens_rhs_rows(w, Slots{&lds_u[l]}, ts, p, Slots{&lds_u[lane]}, pd, work);
#else
    (void)l;
    sys::rhs_rows(w, Slots{&lds_u[S * STAGE + lane]}, ts, p, work);
#endif
#pragma unroll
    for (int j = 0; j < R; ++j) {
      double v;
      if constexpr (S == 0) {
        v = fmaT(dt_use * DV[0], dT[j], work[j]);
      } else {
        const double kn = (double)k[S - 1][j];
        const double acc = S == 1 ? CM[S][S - 1] * kn : fmaT(CM[S][S - 1], kn, sc[j]);
        if constexpr (S < 5)
          v = fmaT(acc, inv_dt, fmaT(dt_use * DV[S], dT[j], work[j]));
        else
          v = fmaT(acc, inv_dt, work[j]);
      }
      work[j] = v;
      if (NS == 0 || state) lds_r[S * STAGE + at(w, j, lane)] = (LUT)v;
    }
    __syncthreads();
    // while wavefront 0 solves: the next stage's sums up to the vector before
    // this one
    if constexpr (S >= 1 && S < 7) {
#pragma unroll
      for (int j = 0; j < R; ++j) {
        sc[j] = CM[S + 1][0] * (double)k[0][j];
#pragma unroll
        for (int q = 1; q < S; ++q) sc[j] = fmaT(CM[S + 1][q], (double)k[q][j], sc[j]);
        if constexpr (S < 5) {
          sa[j] = AM[S][0] * (double)k[0][j];
#pragma unroll
          for (int q = 1; q < S; ++q) sa[j] = fmaT(AM[S][q], (double)k[q][j], sa[j]);
        }
      }
    }
    __syncthreads();
#if MDX_NSENS > 0
    // the directions' right-hand sides, corrected by the coupling to the
    // state's solution at the step's base point
    if (!state) {
      double c[R];
      sys::sens_coupling_rows(w, Slots{&lds_b[l]}, t, p, Slots{&lds_b[lane]}, pd,
                              Solution{&lds_r[l]}, c);
#pragma unroll
      for (int j = 0; j < R; ++j) lds_r[at(w, j, lane)] = (LUT)(work[j] + c[j]);
    }
    __syncthreads();
    __syncthreads();
#endif
#pragma unroll
    for (int j = 0; j < R; ++j) k[S][j] = lds_r[S * STAGE + at(w, j, lane)];
  }

  // The eight stage vectors k, and the last stage's argument u.
  __device__ __forceinline__ void stages(KT (&k)[8][R], double (&u)[R], const TeamParams& p, int w,
                                         int lane, double t, double dt_use) {
    const double inv_dt = 1.0 / dt_use;
    double sa[R], sc[R], dT[R];
#pragma unroll
    for (int j = 0; j < R; ++j) sa[j] = sc[j] = dT[j] = 0.0;
    stage<0>(k, u, sa, sc, dT, p, w, lane, t, dt_use, inv_dt);
    stage<1>(k, u, sa, sc, dT, p, w, lane, t, dt_use, inv_dt);
    stage<2>(k, u, sa, sc, dT, p, w, lane, t, dt_use, inv_dt);
    stage<3>(k, u, sa, sc, dT, p, w, lane, t, dt_use, inv_dt);
    stage<4>(k, u, sa, sc, dT, p, w, lane, t, dt_use, inv_dt);
    stage<5>(k, u, sa, sc, dT, p, w, lane, t, dt_use, inv_dt);
    stage<6>(k, u, sa, sc, dT, p, w, lane, t, dt_use, inv_dt);
    stage<7>(k, u, sa, sc, dT, p, w, lane, t, dt_use, inv_dt);
  }

  __device__ __forceinline__ void step(Control& s, const TeamParams& p, const SolveArgs& a, i64 i,
                                       int w, int lane, bool act) {
    const double dt_use = step_length(s);
    const double t = s.t;
    KT k[8][R];
    double u[R];
    stages(k, u, p, w, lane, t, dt_use);
    // the error terms (rodas5P.py:903-911)
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int v = row(w, j);
      const double k7 = (double)k[7][j];
      const double y_new = u[j] + k7;
      const double ya = absT(y[j]), yb = absT(y_new);
      const double scale = fmaT(a.rtol, ya > yb ? ya : yb, a.atol);
      lds_u[at(w, j, lane)] = weight(a, i, v < 0 ? 0 : (int)joint(v, lane)) * k7 / scale;
    }
    __syncthreads();
    __syncthreads();
    const double err_norm = lds_c[T + lane % T];
    const bool accept = err_norm <= 1.0 && !__builtin_isnan(err_norm);
    if (act) {
      s.dt = lds_c[lane % T];
      if (accept) {
        const double t_new = t + dt_use;
        while (save_due(s, a, t_new)) {
          const double ts = s.ts;
          (void)ts;
          s.ts = next_save(a, s.save_idx + 1);
#if !MDX_ADJOINT
          const double theta = (ts - t) / dt_use;
          const double theta1 = 1.0 - theta;
          double* __restrict__ out = a.hist + i * a.h_ts + (i64)s.save_idx * a.h_ss;
#pragma unroll
          for (int j = 0; j < R; ++j) {
            const int v = row(w, j);
            const double k0 = (double)k[0][j];
            double h1 = H1[0] * k0;
            double h2 = H2[0] * k0;
            double h3 = H3[0] * k0;
#pragma unroll
            for (int q = 1; q < 8; ++q) {
              const double kv = (double)k[q][j];
              h1 = fmaT(H1[q], kv, h1);
              h2 = fmaT(H2[q], kv, h2);
              h3 = fmaT(H3[q], kv, h3);
            }
            const double y_new = u[j] + (double)k[7][j];
            double x = fmaT(theta, h3, h2);
            x = fmaT(theta, x, h1);
            x = fmaT(theta1, x, y_new);
            if (v >= 0) out[joint(v, lane) * a.h_vs] = fmaT(theta, x, theta1 * y[j]);
          }
#endif
          s.save_idx++;
        }
#pragma unroll
        for (int j = 0; j < R; ++j) y[j] = u[j] + (double)k[7][j];
        s.t = t_new;
        s.accepted++;
      } else {
        s.rejected++;
      }
      s.n_steps++;
    }
  }

  __device__ __forceinline__ void finish(Control& s, const SolveArgs& a, i64 i, int w, int lane) {
    if (a.cost) {
      if (a.resume) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const int v = row(w, j);
          if (v >= 0) a.resume[i + joint(v, lane) * a.n_traj] = y[j];
        }
      }
      return;
    }
    while (s.save_idx < a.n_save) {
      double* __restrict__ out = a.hist + i * a.h_ts + (i64)s.save_idx * a.h_ss;
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int v = row(w, j);
        if (v >= 0) out[joint(v, lane) * a.h_vs] = y[j];
      }
      s.save_idx++;
    }
  }
};

// Every wavefront of a workgroup holds the same trajectories in the same lanes
// and the same step control, so loops and branches around the barriers are
// decided alike in all of them; each role has a loop of its own, with matching
// barriers.
template <class Role>
__device__ __forceinline__ void solve_block(const SolveArgs& a, int w, int lane) {
  const i64 i = (i64)blockIdx.x * T + lane % T;
  if (lane >= LANES || i >= a.n_traj) return;
  TeamParams p(lane % T);
  p.load(a, i, w, lane % T);
  Control s;
  Role role;
  control_init(s, a, i);
  role.init(a, i, w, lane);
  settle();
  for (;;) {
    const bool act = team_active(s, a);
    if (!__any(act)) break;
    role.step(s, p, a, i, w, lane, act);
  }
  role.finish(s, a, i, w, lane);
}

template <class Role>
__device__ __forceinline__ void solve_claimed(const SolveArgs& a, int w, int lane) {
  if (lane >= LANES) return;
  const int l = lane % T;
  TeamParams p(l);
  Control s = {};
  Role role = {};
  i64 i = -1;
  bool exhausted = false;
  for (;;) {
    const bool want = (i < 0) && !exhausted;
    if (__any(want)) {
      // wavefront 0 claims for all of them
      if (Role::FIRST) {
        const i64 claim = wave_claim(a.queue, want && lane < T);
        if (lane < T) lds_claim[l] = claim;
      }
      __syncthreads();
      const i64 got = lds_claim[l];
      __syncthreads();
      if (want) {
        if (got < a.n_traj) {
          const i64 j = a.order ? a.order[got] : got;
          if (j >= 0 && j < a.n_traj) {
            i = j;
            p.load(a, i, w, l);
            control_init(s, a, i);
            role.init(a, i, w, lane);
            settle();
          }
        } else {
          exhausted = true;
        }
      }
    }
    if (!__any(i >= 0)) break;
    const bool act = i >= 0 && team_active(s, a);
    if (__any(act)) role.step(s, p, a, i < 0 ? 0 : i, w, lane, act);
    if (i >= 0 && !team_active(s, a)) {
      role.finish(s, a, i, w, lane);
      i = -1;
    }
  }
}

}  // namespace r5
}  // namespace mdx

#if !MDX_ADJOINT
extern "C" __global__ __launch_bounds__(64 * MDX_TEAM) void mdx_rodas5p(mdx::SolveArgs a) {
  using namespace mdx::r5;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int lane = (int)threadIdx.x % 64;
  if (w == 0)
    solve_block<Solver>(a, w, lane);
  else
    solve_block<Owner>(a, w, lane);
}

extern "C" __global__ __launch_bounds__(64 * MDX_TEAM) void mdx_rodas5p_refill(mdx::SolveArgs a) {
  using namespace mdx::r5;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int lane = (int)threadIdx.x % 64;
  if (w == 0)
    solve_claimed<Solver>(a, w, lane);
  else
    solve_claimed<Owner>(a, w, lane);
}
#endif  // !MDX_ADJOINT
