// tsit5_team.hpp -- the Tsit5 ensemble step shared out over a workgroup's
// wavefronts, for systems too large for one wavefront's registers.
//
// Included after tsit5.hpp when MDX_TEAM > 0, in a source whose
// sys namespace holds, beside rhs:
//   rhs_rows(wave, y, t, p, out)  wavefront ``wave``'s rows of the right-hand
//                                 side, reading y by slot
//   ROW_OF[W * R]                 the variable a slot holds, -1 for padding
//   SLOT_OF[N]                    the slot of a variable
// Macros: MDX_TEAM wavefronts, MDX_TEAM_ROWS slots each, MDX_BLOCK
// trajectories (lanes 0 .. MDX_BLOCK-1 of every wavefront carry the same ones).
//
// One lane per trajectory leaves such a system's nine vectors in LDS or
// scratch, one wavefront a compute unit and three SIMDs idle, and every lane
// walks all N rows. Here wavefront w owns R rows of every one of the
// workgroup's trajectories: their state, seven stage vectors and sums are
// registers, and what a right-hand side needs of the other rows -- the stage
// argument -- is exchanged through LDS, double buffered, so a stage costs one
// barrier (about 10 cycles here; a write, barrier and read about 160). Each
// element still sees the operations of the one-lane step in their order, and
// the error norm is summed over the variables in ascending order by one
// wavefront, so the bits are the same.
#pragma once

namespace mdx {
namespace t5 {

constexpr int W = MDX_TEAM;
constexpr int R = MDX_TEAM_ROWS;
constexpr int T = MDX_BLOCK;
constexpr int SLOTS = W * R;

__shared__ double lds_u[2][SLOTS * T];  // stage argument, [slot][lane]; buffer 1 then holds the error terms
__shared__ double lds_c[2 * T];         // the step's outcome: next step size, error norm
__shared__ i64 lds_claim[T];
#if MDX_TEAM_LDS_PARAMS
__shared__ double lds_p[MDX_NP * T];
struct TeamParams {
  const double* base;
  __device__ __forceinline__ TeamParams(int lane) : base(&lds_p[lane]) {}
  __device__ __forceinline__ double operator[](int m) const { return base[m * T]; }
  // wavefront w brings in every W-th parameter; the step's first barrier makes
  // them visible
  __device__ __forceinline__ void load(const SolveArgs& a, i64 i, int w, int lane) {
    for (int m = w; m < MDX_NP; m += W) lds_p[m * T + lane] = a.params[i * a.p_ts + (i64)m * a.p_vs];
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

// What every wavefront knows of each trajectory (the same values in all of
// them; err_prev and err_prev2 only in wavefront 0, which forms the step size).
struct TeamState {
  double y[R], k[7][R];  // row 6 of k is the first-same-as-last carry
  double t, dt, tf, ts, err_prev, err_prev2;
  int save_idx, n_steps, accepted, rejected;
  bool has_fsal;
};

struct Slots {
  const double* base;
  __device__ __forceinline__ double operator[](int s) const { return base[s * T]; }
};

__device__ __forceinline__ void team_init(TeamState& s, const SolveArgs& a, i64 i, int w) {
  const double* __restrict__ times = a.times;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int v = sys::ROW_OF[w * R + j];
    s.y[j] = 0.0;
    s.k[6][j] = 0.0;
    if (v >= 0) {
      s.y[j] = a.y0[i * a.y0_ts + (i64)v * a.y0_vs];
      a.hist[i * a.h_ts + (i64)v * a.h_vs] = s.y[j];
    }
  }
  s.t = times[0];
  s.tf = times[a.n_save - 1];
  s.dt = a.dt0 > 0.0 ? a.dt0 : (s.tf - s.t) * 1e-6;
  s.err_prev = 1.0;
  s.err_prev2 = 1.0;
  s.save_idx = 1;
  s.n_steps = 0;
  s.accepted = 0;
  s.rejected = 0;
  s.has_fsal = false;
  if (a.resume && !a.cost) {
    // where a cost pilot left the trajectory (layout as in tsit5.hpp's init)
    const double* __restrict__ r = a.resume + i;
    const i64 st = a.n_traj;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int v = sys::ROW_OF[w * R + j];
      if (v >= 0) {
        s.y[j] = r[v * st];
        s.k[6][j] = r[(N + v) * st];
      }
    }
    s.t = r[(2 * N + 0) * st];
    s.dt = r[(2 * N + 1) * st];
    s.err_prev = r[(2 * N + 2) * st];
    s.err_prev2 = r[(2 * N + 3) * st];
    s.save_idx = (int)r[(2 * N + 4) * st];
    s.n_steps = (int)r[(2 * N + 5) * st];
    s.accepted = (int)r[(2 * N + 6) * st];
    s.rejected = (int)r[(2 * N + 7) * st];
    s.has_fsal = r[(2 * N + 8) * st] != 0.0;
  }
  s.ts = next_save(a, s.save_idx);
}

__device__ __forceinline__ bool team_active(const TeamState& s, const SolveArgs& a) {
  return s.save_idx < a.n_save && s.t < s.tf && s.n_steps < a.max_steps;
}

// One attempted step of every lane's trajectory; a lane whose ``act`` is false
// computes along and keeps its state. All wavefronts call it together.
__device__ __forceinline__ void team_step(TeamState& s, const TeamParams& p, const SolveArgs& a,
                                          i64 i, int w, int lane, bool act) {
  double dt_use = s.dt;
  if (dt_use > s.tf - s.t) dt_use = s.tf - s.t;
  if (dt_use < 1e-30) dt_use = 1e-30;
  const double t = s.t;
  double u[R];
  if (__any(act && !s.has_fsal)) {
    double out[R];
#pragma unroll
    for (int j = 0; j < R; ++j) lds_u[0][(w * R + j) * T + lane] = s.y[j];
    __syncthreads();
    sys::rhs_rows(w, Slots{&lds_u[0][lane]}, t, p, out);
#pragma unroll
    for (int j = 0; j < R; ++j) s.k[0][j] = s.has_fsal ? s.k[6][j] : out[j];
  } else {
#pragma unroll
    for (int j = 0; j < R; ++j) s.k[0][j] = s.k[6][j];
  }
  // unrolled: a wavefront's rows are a few hundred instructions a stage, and a
  // taken branch costs a lone wavefront about as much as six of them
#pragma unroll
  for (int S = 1; S < 7; ++S) {
    double q[R], out[R];
#pragma unroll
    for (int j = 0; j < R; ++j) q[j] = AT[S][0] * s.k[0][j];
#pragma unroll
    for (int r = 1; r < S; ++r)
#pragma unroll
      for (int j = 0; j < R; ++j) q[j] = fmaT(AT[S][r], s.k[r][j], q[j]);
    double* __restrict__ buf = lds_u[S & 1];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      u[j] = fmaT(dt_use, q[j], s.y[j]);
      buf[(w * R + j) * T + lane] = u[j];
    }
    __syncthreads();
    sys::rhs_rows(w, Slots{&buf[lane]}, t + CS[S] * dt_use, p, out);
    // k7 is state: a lane that has finished keeps its own
#pragma unroll
    for (int j = 0; j < R; ++j) s.k[S][j] = S < 6 || act ? out[j] : s.k[S][j];
  }

  // the embedded error's terms, each by its row's owner
  constexpr double EW[7] = {E1, E2, E3, E4, E5, E6, E7};
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int v = sys::ROW_OF[w * R + j];
    double e = EW[0] * s.k[0][j];
#pragma unroll
    for (int r = 1; r < 7; ++r) e = fmaT(EW[r], s.k[r][j], e);
    const double err_est = dt_use * e;
    const double ya = absT(s.y[j]), yb = absT(u[j]);
    const double scale = fmaT(a.rtol, ya > yb ? ya : yb, a.atol);
    lds_u[1][(w * R + j) * T + lane] = weight(a, i, v < 0 ? 0 : v) * err_est / scale;
  }
  __syncthreads();
  if (w == 0) {
    double err = 0.0;
#pragma unroll
    for (int v = 0; v < N; ++v) {
      const double r = lds_u[1][sys::SLOT_OF[v] * T + lane];
      err = fmaT(r, r, err);
    }
    const double err_norm = __builtin_sqrt(err / (double)MDX_N_ERROR);
    const bool accept = err_norm <= 1.0 && !__builtin_isnan(err_norm);
    double e1 = s.err_prev, e2 = s.err_prev2;
    const double factor_ = pid_factor(err_norm, accept, e1, e2, MDX_E1, MDX_E2, MDX_E3, 0.2, 10.0);
    if (act) s.err_prev = e1, s.err_prev2 = e2;
    lds_c[lane] = dt_use * factor_;
    lds_c[T + lane] = err_norm;
  }
  __syncthreads();
  const double err_norm = lds_c[T + lane];
  const bool accept = err_norm <= 1.0 && !__builtin_isnan(err_norm);
  if (act) {
    s.dt = lds_c[lane];
    if (accept) {
      const double t_new = t + dt_use;
      while (s.save_idx < a.n_save) {
        const double ts = s.ts;
        const double at = absT(ts);
        if (!(ts <= t_new + 1e-12 * (1.0 > at ? 1.0 : at))) break;
        const double ts_next = next_save(a, s.save_idx + 1);
        double b[7];
        dense_weights((ts - t) / dt_use, b);
        double* __restrict__ row = a.hist + i * a.h_ts + (i64)s.save_idx * a.h_ss;
#pragma unroll
        for (int j = 0; j < R; ++j) {
          const int v = sys::ROW_OF[w * R + j];
          if (v >= 0) {
            double q = b[0] * s.k[0][j];
#pragma unroll
            for (int r = 1; r < 7; ++r) q = fmaT(b[r], s.k[r][j], q);
            row[(i64)v * a.h_vs] = fmaT(dt_use, q, s.y[j]);
          }
        }
        s.save_idx++;
        s.ts = ts_next;
      }
#pragma unroll
      for (int j = 0; j < R; ++j) s.y[j] = u[j];
      s.accepted++;
      s.has_fsal = true;
      s.t = t_new;
    } else {
      s.rejected++;
#pragma unroll
      for (int j = 0; j < R; ++j) s.k[6][j] = 0.0;
      s.has_fsal = false;
    }
    s.n_steps++;
  }
}

__device__ __forceinline__ void team_finish(TeamState& s, const SolveArgs& a, i64 i, int w) {
  if (a.cost) {
    // a cost pilot (see tsit5.hpp's finish): the steps left, and the step state
    if (w == 0) a.cost[i] = (s.save_idx < a.n_save && s.t < s.tf) ? (s.tf - s.t) / s.dt : 0.0;
    if (a.resume) {
      double* __restrict__ r = a.resume + i;
      const i64 st = a.n_traj;
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const int v = sys::ROW_OF[w * R + j];
        if (v >= 0) {
          r[v * st] = s.y[j];
          r[(N + v) * st] = s.k[6][j];
        }
      }
      if (w == 0) {
        r[(2 * N + 0) * st] = s.t;
        r[(2 * N + 1) * st] = s.dt;
        r[(2 * N + 2) * st] = s.err_prev;
        r[(2 * N + 3) * st] = s.err_prev2;
        r[(2 * N + 4) * st] = (double)s.save_idx;
        r[(2 * N + 5) * st] = (double)s.n_steps;
        r[(2 * N + 6) * st] = (double)s.accepted;
        r[(2 * N + 7) * st] = (double)s.rejected;
        r[(2 * N + 8) * st] = s.has_fsal ? 1.0 : 0.0;
      }
    }
    return;
  }
  const double nan = __builtin_nan("");
  while (s.save_idx < a.n_save) {
    double* __restrict__ row = a.hist + i * a.h_ts + (i64)s.save_idx * a.h_ss;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int v = sys::ROW_OF[w * R + j];
      if (v >= 0) row[(i64)v * a.h_vs] = nan;
    }
    s.save_idx++;
  }
  if (w == 0) {
    a.accepted[i] = s.accepted;
    a.rejected[i] = s.rejected;
    a.loop[i] = s.n_steps;
  }
}

}  // namespace t5
}  // namespace mdx

// Every wavefront of a workgroup holds the same trajectories in the same lanes
// and the same step control, so loops and branches around the barriers are
// decided alike in all of them.
extern "C" __global__ __launch_bounds__(64 * MDX_TEAM) void mdx_tsit5(mdx::SolveArgs a) {
  using namespace mdx::t5;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int lane = (int)threadIdx.x % 64;
  const mdx::i64 i = (mdx::i64)blockIdx.x * T + lane;
  if (lane >= T || i >= a.n_traj) return;
  TeamParams p(lane);
  p.load(a, i, w, lane);
  TeamState s;
  team_init(s, a, i, w);
  mdx::settle();
  for (;;) {
    const bool act = team_active(s, a);
    if (!__any(act)) break;
    team_step(s, p, a, i, w, lane, act);
  }
  team_finish(s, a, i, w);
}

extern "C" __global__ __launch_bounds__(64 * MDX_TEAM) void mdx_tsit5_refill(mdx::SolveArgs a) {
  using namespace mdx::t5;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int lane = (int)threadIdx.x % 64;
  if (lane >= T) return;
  TeamParams p(lane);
  TeamState s = {};
  mdx::i64 i = -1;
  bool exhausted = false;
  for (;;) {
    const bool want = (i < 0) && !exhausted;
    if (__any(want)) {
      // wavefront 0 claims for all of them
      if (w == 0) lds_claim[lane] = mdx::wave_claim(a.queue, want);
      __syncthreads();
      const mdx::i64 got = lds_claim[lane];
      __syncthreads();
      if (want) {
        if (got < a.n_traj) {
          const mdx::i64 j = a.order ? a.order[got] : got;
          if (j >= 0 && j < a.n_traj) {
            i = j;
            p.load(a, i, w, lane);
            team_init(s, a, i, w);
            mdx::settle();
          }
        } else {
          exhausted = true;
        }
      }
    }
    if (!__any(i >= 0)) break;
    const bool act = i >= 0 && team_active(s, a);
    if (__any(act)) team_step(s, p, a, i < 0 ? 0 : i, w, lane, act);
    if (i >= 0 && !team_active(s, a)) {
      team_finish(s, a, i, w);
      i = -1;
    }
  }
}
