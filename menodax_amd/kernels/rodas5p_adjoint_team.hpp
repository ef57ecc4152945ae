// rodas5p_adjoint_team.hpp -- the discrete adjoint of the Rodas5P ensemble solve
// of a sparse system, shared out over a workgroup's wavefronts.
//
// Included after rodas5p_team.hpp (whose roles, slots and macros it uses) in a
// source generated with MDX_ADJOINT=1, whose sys namespace also holds, reading
// every vector by slot,
//   f_vjp_rows, jac_vjp_rows      a wavefront's rows of the state's part of
//                                 rodas5p_adjoint.hpp's f_vjp and jac_vjp
//   f_vjp_params, jac_vjp_params  their parameters' part
// and sparse_solve_t. The arithmetic, element by element, is
// rodas5p_adjoint.hpp's, so the bits are the same; its comment has the reverse
// of a step. The forward pass is the team's step, recording each accepted step
// (state, time, step size, saves it produced), so the workspace is that of
// max_ckpt = 1 with room for every step in ckpt_every records.
//
// Going back, a step is first taken again (the stage arguments and solutions
// stay in LDS, one place a stage), then the stages are reversed last to first.
// The owners keep their rows' k_bar, u_bar and y_bar in registers; wavefront 0
// keeps the factors and runs the transposed solves, then sums the parameters'
// gradient while the owners form their rows' products. Two barriers a stage:
// k_bar written, r_bar written; r_bar has two places in turn, since owners still
// read one stage's when the next one's k_bar comes. What bounds it is the
// latency of one step after the other, as in the team's forward step; one lane
// a trajectory runs the same chain with a single wavefront a compute unit
// issuing all of it. Gradients of the 20-variable chain (FP64, some 1,400 steps),
// 8,192 trajectories on an MI355X with the solve before them: 155 ms with one
// lane a trajectory, 49 ms with a team.
#pragma once

#if !MDX_ADJOINT || !MDX_TEAM
#error "the team's adjoint goes with the team placement"
#endif

namespace mdx {
namespace r5 {

constexpr int RC = N + 4;   // step record words: y, t, h, first and last save
constexpr int CK = N + 8;   // a checkpoint's words, left unused ahead of the records
constexpr int NPB = MDX_NP > 0 ? MDX_NP : 1;

__shared__ double lds_x[2 * SLOTS * LANES];  // k_bar of a stage, then its r_bar

__device__ __forceinline__ double& record(const AdjointArgs& g, i64 i, int r, int word) {
  return workspace_at<N>(g, i, (i64)g.max_ckpt * CK + (i64)r * RC + word);
}

__device__ __forceinline__ double gbar_at(const AdjointArgs& g, i64 i, int sv, int v) {
  return g.gbar[i * g.g_ts + (i64)sv * g.g_ss + (i64)v * g.g_vs];
}

__device__ __forceinline__ double stage_time(int S, double t, double h) {
  return S == 0 ? t : S < 5 ? t + CT[S > 0 && S < 5 ? S - 1 : 0] * h : t + h;
}

// A step as the forward pass left it, the rows an owner's: plain words, since a
// conversion where they are loaded would wait for them there. The step before
// is loaded while one is reversed (50.2 -> 49.3 ms; loading a save's cotangent
// ahead as well gains nothing).
struct Record {
  double t, h, save_lo, save_hi, y[R];
};
template <class Role>
__device__ __forceinline__ void load_record(Role& role, Record& x, const AdjointArgs& g, i64 i,
                                            int r, int w) {
  x.t = record(g, i, r, N + 0);
  x.h = record(g, i, r, N + 1);
  x.save_lo = record(g, i, r, N + 2);
  x.save_hi = record(g, i, r, N + 3);
  role.load(x, g, i, r, w);
}

struct SolverBack : Solver {
  double pbar[NPB];

  __device__ __forceinline__ void record_step(const AdjointArgs& g, i64 i, int r, const Control& s,
                                              int, int) {
    record(g, i, r, N + 0) = s.t;
    record(g, i, r, N + 1) = step_length(s);
    record(g, i, r, N + 2) = (double)s.save_idx;
  }

  __device__ __forceinline__ void begin(const AdjointArgs&, i64, int, int) {
#pragma unroll
    for (int m = 0; m < NPB; ++m) pbar[m] = 0.0;
  }

  __device__ __forceinline__ void load(Record&, const AdjointArgs&, i64, int, int) {}

  __device__ __forceinline__ void reverse(const AdjointArgs& g, i64 i, Record& rec, int before,
                                          const TeamParams& p, int w, int lane, bool act) {
    LUT lu[MDX_NLU];
    Pivots ipiv;
    const double t = rec.t, h = rec.h;
    load_record(*this, rec, g, i, before, w);
    stages(t, h, p, lane, lu, ipiv);
    double lud[MDX_NLU];
#pragma unroll
    for (int q = 0; q < MDX_NLU; ++q) lud[q] = (double)lu[q];
    double pb[NPB];
#pragma unroll
    for (int m = 0; m < NPB; ++m) pb[m] = pbar[m];
#pragma unroll 1
    for (int S = 7; S >= 0; --S) {
      double* const x = &lds_x[(S & 1) * SLOTS * LANES];
      __syncthreads();  // k_bar of the stage is written
      double r[N];
#pragma unroll
      for (int v = 0; v < N; ++v) r[v] = x[sys::SLOT_OF[v] * LANES + lane];
      solve_t(lud, ipiv, r);
#pragma unroll
      for (int v = 0; v < N; ++v) x[sys::SLOT_OF[v] * LANES + lane] = r[v];
      __syncthreads();
      sys::jac_vjp_params(Slots{&lds_u[lane]}, t, p, Slots{&x[lane]},
                          Solution{&lds_r[S * STAGE + lane]}, pb);
      sys::f_vjp_params(Slots{&lds_u[S * STAGE + lane]}, stage_time(S, t, h), p, Slots{&x[lane]},
                        pb);
    }
    if (act) {
#pragma unroll
      for (int m = 0; m < NPB; ++m) pbar[m] = pb[m];
    }
    __syncthreads();  // the stages' places may be written again
  }

  __device__ __forceinline__ void output(const AdjointArgs& g, i64 i, int, int, int status) {
    const double bad = status != 0 ? __builtin_nan("") : 0.0;
    for (int m = 0; m < MDX_NP; ++m) g.grad_p[i * g.gp_ts + (i64)m * g.gp_vs] = pbar[m] + bad;
    g.status[i] = status;
  }
};

struct OwnerBack : Owner {
  double lam[R];  // dL/d(this wavefront's rows) after, then before the step

  __device__ __forceinline__ void record_step(const AdjointArgs& g, i64 i, int r, const Control&,
                                              int w, int) {
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int v = row(w, j);
      if (v >= 0) record(g, i, r, v) = y[j];
    }
  }

  // saves the solve never reached hold the final state
  __device__ __forceinline__ void begin(const AdjointArgs& g, i64 i, int w, int first) {
#pragma unroll
    for (int j = 0; j < R; ++j) lam[j] = 0.0;
    for (int sv = first; sv < g.s.n_save; ++sv)
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int v = row(w, j);
        if (v >= 0) lam[j] += gbar_at(g, i, sv, v);
      }
  }

  template <int S>
  __device__ __forceinline__ void reverse_stage(double (&kb)[8][R], double (&yb)[R],
                                                double (&uc)[R], const TeamParams& p, int w,
                                                int lane, double t, double h, double inv_dt) {
    double* const x = &lds_x[(S & 1) * SLOTS * LANES];
#pragma unroll
    for (int j = 0; j < R; ++j) x[at(w, j, lane)] = kb[S][j];
    __syncthreads();
    __syncthreads();  // r_bar is written
    sys::jac_vjp_rows(w, Slots{&lds_u[lane]}, t, p, Slots{&x[lane]},
                      Solution{&lds_r[S * STAGE + lane]}, yb);
#pragma unroll
    for (int q = 0; q < S; ++q) {
      const double c = CM[S][q] * inv_dt;
#pragma unroll
      for (int j = 0; j < R; ++j) kb[q][j] += c * x[at(w, j, lane)];
    }
    double ub[R];
#pragma unroll
    for (int j = 0; j < R; ++j) ub[j] = 0.0;
    sys::f_vjp_rows(w, Slots{&lds_u[S * STAGE + lane]}, stage_time(S, t, h), p, Slots{&x[lane]},
                    ub);
    if constexpr (S >= 5) {
#pragma unroll
      for (int j = 0; j < R; ++j) ub[j] += uc[j];
    }
    if constexpr (S >= 6) {
      // u_S = u_{S-1} + k_{S-1}
#pragma unroll
      for (int j = 0; j < R; ++j) uc[j] = ub[j], kb[S - 1][j] += ub[j];
    } else {
      // u_S = y + sum_q A_{S,q} k_q
#pragma unroll
      for (int j = 0; j < R; ++j) yb[j] += ub[j];
#pragma unroll
      for (int q = 0; q < S; ++q)
#pragma unroll
        for (int j = 0; j < R; ++j) kb[q][j] += AM[S > 0 ? S - 1 : 0][q] * ub[j];
    }
  }

  __device__ __forceinline__ void load(Record& x, const AdjointArgs& g, i64 i, int r, int w) {
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int v = row(w, j);
      x.y[j] = v >= 0 ? record(g, i, r, v) : 0.0;
    }
  }

  __device__ __forceinline__ void reverse(const AdjointArgs& g, i64 i, Record& rec, int before,
                                          const TeamParams& p, int w, int lane, bool act) {
    const double t = rec.t, h = rec.h;
    const int save_lo = act ? (int)rec.save_lo : 0, save_hi = act ? (int)rec.save_hi : 0;
    const double inv_dt = 1.0 / h;
#pragma unroll
    for (int j = 0; j < R; ++j) y[j] = rec.y[j];
    {
      KT k[8][R];
      double u[R];
      stages(k, u, p, w, lane, t, h);
    }
    double kb[8][R], yb[R], uc[R];
#pragma unroll
    for (int q = 0; q < 8; ++q)
#pragma unroll
      for (int j = 0; j < R; ++j) kb[q][j] = 0.0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      yb[j] = 0.0;
      uc[j] = lam[j];  // y_{n+1} = u7 + k7
      kb[7][j] = lam[j];
    }
    for (int sv = save_lo; sv < save_hi; ++sv) {
      const double theta = (g.s.times[sv] - t) / h;
      const double theta1 = 1.0 - theta;
      const double c1 = theta * theta1, c2 = c1 * theta, c3 = c2 * theta;
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int v = row(w, j);
        if (v < 0) continue;
        const double gj = gbar_at(g, i, sv, v);
        yb[j] += theta1 * gj;
        uc[j] += theta * gj;
        kb[7][j] += theta * gj;
#pragma unroll
        for (int q = 0; q < 8; ++q) kb[q][j] += (H1[q] * c1 + H2[q] * c2 + H3[q] * c3) * gj;
      }
    }
    // after the saves, which would wait for these loads too
    load_record(*this, rec, g, i, before, w);
    reverse_stage<7>(kb, yb, uc, p, w, lane, t, h, inv_dt);
    reverse_stage<6>(kb, yb, uc, p, w, lane, t, h, inv_dt);
    reverse_stage<5>(kb, yb, uc, p, w, lane, t, h, inv_dt);
    reverse_stage<4>(kb, yb, uc, p, w, lane, t, h, inv_dt);
    reverse_stage<3>(kb, yb, uc, p, w, lane, t, h, inv_dt);
    reverse_stage<2>(kb, yb, uc, p, w, lane, t, h, inv_dt);
    reverse_stage<1>(kb, yb, uc, p, w, lane, t, h, inv_dt);
    reverse_stage<0>(kb, yb, uc, p, w, lane, t, h, inv_dt);
    if (act) {
#pragma unroll
      for (int j = 0; j < R; ++j) lam[j] = yb[j];
    }
    __syncthreads();  // the stages' places may be written again
  }

  __device__ __forceinline__ void output(const AdjointArgs& g, i64 i, int w, int, int status) {
    const double bad = status != 0 ? __builtin_nan("") : 0.0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int v = row(w, j);
      // hist[0] is y0 itself
      if (v >= 0) g.grad_y0[i * g.gy_ts + (i64)v * g.gy_vs] = lam[j] + gbar_at(g, i, 0, v) + bad;
    }
  }
};

// As in the forward solve, every wavefront holds the same trajectories and step
// control in the same lanes and takes the same number of steps.
template <class Role>
__device__ __forceinline__ void adjoint_block(const AdjointArgs& g, int w, int lane) {
  const SolveArgs& a = g.s;
  const i64 i = (i64)blockIdx.x * T + lane;
  if (lane >= T || i >= a.n_traj) return;
  TeamParams p(lane);
  p.load(a, i, w, lane);
  Control s;
  Role role;
  control_init(s, a, i);
  role.init(a, i, w, lane);
  settle();
  const int room = g.ckpt_every;
  for (;;) {
    const bool act = team_active(s, a);
    if (!__any(act)) break;
    const int r = s.accepted;
    if (act && r < room) role.record_step(g, i, r, s, w, lane);
    role.step(s, p, a, i, w, lane, act);
    if (Role::FIRST && act && s.accepted > r && r < room)
      record(g, i, r, N + 3) = (double)s.save_idx;
  }
  // not enough room: report, leave the gradients NaN
  const int status = s.accepted > room ? 1 : 0;
  __syncthreads();  // wavefront 0's words of the records are written
  role.begin(g, i, w, s.save_idx);
  int r = status ? -1 : s.accepted - 1;
  Record rec;
  load_record(role, rec, g, i, r > 0 ? r : 0, w);
  for (;; --r) {
    const bool act = r >= 0;
    if (!__any(act)) break;
    // a trajectory already back at its start goes through the motions
    role.reverse(g, i, rec, r > 1 ? r - 1 : 0, p, w, lane, act);
  }
  role.output(g, i, w, lane, status);
}

}  // namespace r5
}  // namespace mdx

extern "C" __global__ __launch_bounds__(64 * MDX_TEAM) void mdx_rodas5p_adjoint(
    mdx::AdjointArgs g) {
  using namespace mdx::r5;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int lane = (int)threadIdx.x % 64;
  if (w == 0)
    adjoint_block<SolverBack>(g, w, lane);
  else
    adjoint_block<OwnerBack>(g, w, lane);
}
