// rodas5p_rows.hpp -- the plain Rodas5P solve of a dense system in the wave
// placement: one trajectory a wavefront, lane r holding row r.
//
// Included after rodas5p.hpp for MDX_COOP (MDX_ROWS > 0) without sensitivity
// directions. Lane r keeps row r of the iteration matrix in registers together
// with its component of the state, of the stage vectors and of every sum, so a
// vector operation is one instruction for all rows. The factorisation leaves
// the rows where they are: a pivot search moves positions, not rows, and the
// pivot row's elements reach the other lanes by readlane. The forward
// substitution takes a column a step in every lane; the back substitution of
// row i is the chain of its N - 1 - i terms in ascending column order (the
// order the sequential solve sums them in), run in the lane that holds row i.
// The right-hand side and the Jacobian need every component: they are evaluated
// once, by lane 0, from and into LDS.
//
// Each element sees the operations of the sequential factorisation and solves
// in the same order, hence the same bits. What bounds it is the back
// substitutions' dependent chains, N^2 / 2 multiply-adds and N quotients a
// stage (through the pivot's reciprocal, which its lane keeps); the
// LDS-resident form this replaces also waited on LDS and a six-step butterfly
// through it at every pivot.
#pragma once

namespace mdx {
namespace r5 {

constexpr int WAVES = MDX_ROWS;

__shared__ double rows_v[WAVES][N];         // a vector every row reads
__shared__ double rows_f[WAVES][N];         // the right-hand side
__shared__ LUT rows_m[WAVES][N * MDX_LD];   // the matrix as it is formed

struct RowVec {
  const double* base;
  __device__ __forceinline__ double operator[](int j) const { return base[j]; }
};
struct RowMat {
  typedef LUT value_type;
  LUT* base;
  __device__ __forceinline__ LUT& operator[](int e) const {
    return base[(e / N) * MDX_LD + e % N];
  }
};

// Orders one wavefront's LDS accesses: its lanes run together, so a wait for
// what is outstanding is all it takes.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// The largest of v over the wavefront, in every lane (no NaN among them).
template <int CTRL>
__device__ __forceinline__ float dpp_max(float v) {
  const int o = __builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, 0xf, 0xf,
                                            false);
  return __builtin_fmaxf(v, __int_as_float(o));
}
template <int CTRL>
__device__ __forceinline__ double dpp_max(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_fmax(v, __longlong_as_double(((long long)hi << 32) | (unsigned)lo));
}
template <class V>
__device__ __forceinline__ V wave_max(V v) {
  v = dpp_max<0x111>(v);  // row_shr:1, 2, 4, 8: the largest of 16 lanes in their last
  v = dpp_max<0x112>(v);
  v = dpp_max<0x114>(v);
  v = dpp_max<0x118>(v);
  v = dpp_max<0x142>(v);  // row_bcast:15 and :31: of all 64 in the last
  v = dpp_max<0x143>(v);
  return lane_value(v, 63);
}

// Pivot i: the lane holding the first maximum of |c| over the rows at positions
// >= i, as the sequential scan finds it (a NaN below the diagonal never wins, a
// NaN diagonal keeps its row); the positions are swapped. c is the rows'
// column-i element.
__device__ __forceinline__ int choose_pivot(LUT c, int i, int lane, int& pos) {
  typedef LUT V;
  const int at_i = __builtin_ctzll(__ballot(pos == i));
  const V dii = absT(lane_value(c, at_i));
  int best = at_i;
  if (dii == dii) {
    V v = absT(c);
    if (!(v == v) || pos < i || lane >= N) v = (V)-1;
    const V top = wave_max(v);
    u64 mask = __ballot(v == top);
    best = __builtin_ctzll(mask);
    mask &= mask - 1;
    if (mask) {  // equal magnitudes: the smallest position
      int p = __builtin_amdgcn_readlane(pos, best);
      while (mask) {
        const int l = __builtin_ctzll(mask);
        mask &= mask - 1;
        const int q = __builtin_amdgcn_readlane(pos, l);
        if (q < p) p = q, best = l;
      }
    }
  }
  if (best != at_i) {
    const int p = __builtin_amdgcn_readlane(pos, best);
    pos = lane == at_i ? p : lane == best ? i : pos;
  }
  return best;
}

// The factorisation, in place: on return a[j] is the lane's row of L and U in
// factorised form, ``pos`` the row's position, and lane i's ``perm`` the lane
// of the row at position i. Up to MDX_ROWS_UNROLL rows the elimination is
// unrolled (updates of exactly the trailing columns, the element indices
// constants); above, that would leave the instruction cache, so it is a loop
// over the columns in which every row shifts left by one element a step and
// the finished column goes to LDS, its width cut three times on the way.
#ifndef MDX_ROWS_UNROLL
#define MDX_ROWS_UNROLL 32
#endif
struct Own {   // the pivot that the lane's row became, and its double reciprocal
  LUT pivot;
  double inv;
};
__device__ __forceinline__ void eliminate(int i, int lane, int& pos, int& perm, LUT col, double& f,
                                          bool& below, bool& regular, int& piv, Own& own) {
  piv = choose_pivot(col, i, lane, pos);
  perm = lane == i ? piv : perm;
  const LUT pv = lane_value(col, piv);
  const double inv = 1.0 / (double)pv;
  own.pivot = lane == piv ? pv : own.pivot;
  own.inv = lane == piv ? inv : own.inv;
  regular = pv != (LUT)0;
  below = pos > i;
  f = (double)col * inv;
}

template <int FROM, int TO>
__device__ __forceinline__ void eliminate_columns(LUT (&a)[N], int lane, int& pos, int& perm,
                                                  LUT* __restrict__ m, Own& own) {
  constexpr int WIDTH = N - FROM;
#pragma unroll 1
  for (int i = FROM; i < TO; ++i) {
    double f;
    bool below, regular;
    int piv;
    const LUT col = a[0];
    eliminate(i, lane, pos, perm, col, f, below, regular, piv, own);
    below = below && regular;
    if (lane < N) m[lane * MDX_LD + i] = below ? (LUT)f : col;
#pragma unroll
    for (int j = 1; j < WIDTH; ++j) {
      const LUT u = lane_value(a[j], piv);
      const LUT x = (LUT)fmaT(-f, (double)u, (double)a[j]);
      a[j - 1] = below ? x : a[j];
    }
  }
}

__device__ __forceinline__ void factor_rows(LUT (&a)[N], int lane, int& pos, int& perm,
                                            LUT* __restrict__ m, Own& own) {
  pos = lane < N ? lane : N + lane;
  perm = 0;
  own = Own{(LUT)1, 1.0};
  if constexpr (N <= MDX_ROWS_UNROLL) {
    (void)m;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      double f;
      bool below, regular;
      int piv;
      eliminate(i, lane, pos, perm, a[i], f, below, regular, piv, own);
      if (regular) {
        LUT u[N];
#pragma unroll
        for (int j = i + 1; j < N; ++j) u[j] = lane_value(a[j], piv);
        if (below) {
          a[i] = (LUT)f;
#pragma unroll
          for (int j = i + 1; j < N; ++j) a[j] = (LUT)fmaT(-f, (double)u[j], (double)a[j]);
        }
      }
    }
  } else {
    constexpr int Q = N / 4;
    eliminate_columns<0, Q>(a, lane, pos, perm, m, own);
    eliminate_columns<Q, 2 * Q>(a, lane, pos, perm, m, own);
    eliminate_columns<2 * Q, 3 * Q>(a, lane, pos, perm, m, own);
    eliminate_columns<3 * Q, N>(a, lane, pos, perm, m, own);
    wave_sync();
#pragma unroll
    for (int j = 0; j < N; ++j) a[j] = m[(lane < N ? lane : 0) * MDX_LD + j];
  }
}

// A value that is the same in every lane, kept in a vector register: the
// solution's components would fill the scalar ones and spill.
__device__ __forceinline__ float in_vgpr(float x) {
  asm("" : "+v"(x));
  return x;
}
__device__ __forceinline__ double in_vgpr(double x) {
  asm("" : "+v"(x));
  return x;
}

// s over the lane's pivot through its reciprocal, as the division rounds it
// (see Pivots and divide_by); ``out`` takes what tells whether that held.
__device__ __forceinline__ double own_quotient(double s, const Own& own, double& out) {
  out = s;
  return divide_by(s, own.pivot, own.inv);
}
__device__ __forceinline__ float own_quotient(float s, const Own& own, double& out) {
  out = (double)s * own.inv;
  return (float)out;
}
__device__ __forceinline__ bool quotient_held(const Own& own, double out) {
  const int e = __builtin_amdgcn_frexp_exp(out);
  if constexpr (sizeof(LUT) == 4) return e > -126;
  const int b = __builtin_amdgcn_frexp_exp((double)own.pivot);
  return in_divide_range(e, e, b, b);
}

// Solve with the factors: lane r's r in, its component of the solution out.
__device__ __forceinline__ LUT solve_rows(const LUT (&a)[N], int lane, int pos, int perm,
                                          const Own& own, LUT r) {
  // read afresh at every solve: the masks and lanes formed from them below
  // would otherwise be kept across the stage loop, several times the scalar
  // registers there are
  asm volatile("" : "+v"(lane), "+v"(pos), "+v"(perm));
  LUT acc = r;
#pragma unroll
  for (int j = 0; j < N - 1; ++j) {
    const LUT x = lane_value(acc, __builtin_amdgcn_readlane(perm, j));
    const LUT y = fmaT(-a[j], x, acc);
    acc = pos > j ? y : acc;
  }
  LUT x[N];
  LUT mine = (LUT)0;
  double told = 1.0;
#pragma unroll
  for (int i = N - 1; i >= 0; --i) {
    LUT s = acc;
#pragma unroll
    for (int j = i + 1; j < N; ++j) s = fmaT(-a[j], x[j], s);
    double out;
    s = own_quotient(s, own, out);
    told = pos == i ? out : told;
    x[i] = in_vgpr(lane_value(s, __builtin_amdgcn_readlane(perm, i)));
    mine = lane == i ? x[i] : mine;
  }
  if (__any(!quotient_held(own, told))) {
    // out of range in some row: once more with divisions
#pragma unroll
    for (int i = N - 1; i >= 0; --i) {
      LUT s = acc;
#pragma unroll
      for (int j = i + 1; j < N; ++j) s = fmaT(-a[j], x[j], s);
      LUT d = own.pivot;
      asm volatile("; out of range" : "+v"(d));  // keeps the divisions here
      s = s / d;
      x[i] = in_vgpr(lane_value(s, __builtin_amdgcn_readlane(perm, i)));
      mine = lane == i ? x[i] : mine;
    }
  }
  return mine;
}

struct RowState {
  double y;  // this lane's component; everything else is the same in every lane
  double t, dt, tf, ts, err_prev, err_prev2;
  int save_idx, n_steps, accepted, rejected;
};

__device__ __forceinline__ void rows_step(RowState& s, const PA& p, const SolveArgs& a, i64 i,
                                          int w, int lane) {
  double dt_use = s.dt;
  if (dt_use > s.tf - s.t) dt_use = s.tf - s.t;
  if (dt_use < 1e-30) dt_use = 1e-30;
  const double inv_dt = 1.0 / dt_use;
  const double t = s.t;
  const double t_end = t + dt_use;
  const double dtgamma_inv = 1.0 / (dt_use * GAMMA);
  const bool row = lane < N;
  const int r = row ? lane : 0;
  double* __restrict__ v = rows_v[w];
  double* __restrict__ f = rows_f[w];
  LUT* __restrict__ m = rows_m[w];

  // M = I/(h gamma) - J: every slot -0.0, the Jacobian's nonzeros by lane 0,
  // the diagonal a row a lane
  if (row) {
    v[lane] = s.y;
#pragma unroll
    for (int j = 0; j < N; ++j) m[j * MDX_LD + lane] = (LUT)-0.0;
  }
  wave_sync();
  double dTr = 0.0;
  if (lane == 0) {
    double dT[N];
    sys::neg_jac(RowVec{v}, t, p, RowMat{m}, dT);
#if !MDX_DT_ZERO
#pragma unroll
    for (int j = 0; j < N; ++j) f[j] = dT[j];
#endif
  }
  wave_sync();
#if !MDX_DT_ZERO
  dTr = f[r];
#endif
  LUT lu[N];
  if (row) m[lane * MDX_LD + lane] = m[lane * MDX_LD + lane] + (LUT)dtgamma_inv;
  wave_sync();
#pragma unroll
  for (int j = 0; j < N; ++j) lu[j] = m[r * MDX_LD + j];
  wave_sync();
  int pos, perm;
  Own own;
  factor_rows(lu, lane, pos, perm, m, own);

  LUT k[8];
  double u = s.y;
  // the stages stay a loop, one copy of the right-hand side and the solve in
  // the instruction cache; the stage vectors are registers, reached through
  // uniform branches
#pragma unroll 1
  for (int S = 0; S < 8; ++S) {
    const double* __restrict__ am = AM[S < 6 ? (S > 0 ? S - 1 : 0) : 0];
    const double* __restrict__ cm = CM[S];
    double ts = t;
    if (S > 0 && S < 6) {
      double acc = am[0] * (double)k[0];
#pragma unroll
      for (int q = 1; q < 5; ++q)
        if (q < S) acc = fmaT(am[q], (double)k[q], acc);
      u = s.y + acc;
      ts = S < 5 ? t + CT[S - 1] * dt_use : t_end;
    } else if (S >= 6) {
      u = u + (double)(S == 6 ? k[5] : k[6]);
      ts = t_end;
    }
    if (row) v[lane] = u;
    wave_sync();
    if (lane == 0) {
      double work[N];
      sys::rhs(RowVec{v}, ts, p, work);
#pragma unroll
      for (int j = 0; j < N; ++j) f[j] = work[j];
    }
    wave_sync();
    const double work = f[r];
    double x;
    if (S == 0) {
      x = fmaT(dt_use * DV[0], dTr, work);
    } else {
      double acc = cm[0] * (double)k[0];
#pragma unroll
      for (int q = 1; q < 7; ++q)
        if (q < S) acc = fmaT(cm[q], (double)k[q], acc);
      x = S < 5 ? fmaT(acc, inv_dt, fmaT(dt_use * DV[S], dTr, work)) : fmaT(acc, inv_dt, work);
    }
    const LUT ks = solve_rows(lu, lane, pos, perm, own, (LUT)x);
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (q == S) k[q] = ks;
  }

  // the error norm (rodas5P.py:903-911), each lane its component's term, the
  // sum in ascending order
  const double k7 = (double)k[7];
  const double y_new = u + k7;
  const double ya = absT(s.y), yb = absT(y_new);
  const double scale = fmaT(a.rtol, ya > yb ? ya : yb, a.atol);
  const double term = weight(a, i, r) * k7 / scale;
  double err = 0.0;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const double e = lane_value(term, j);
    err = fmaT(e, e, err);
  }
  const double err_norm = __builtin_sqrt(err / (double)MDX_N_ERROR);
  const bool accept = err_norm <= 1.0 && !__builtin_isnan(err_norm);
  const double factor_ =
      pid_factor(err_norm, accept, s.err_prev, s.err_prev2, MDX_E1, MDX_E2, MDX_E3, 0.2, 6.0);
  s.dt = dt_use * factor_;
  if (accept) {
    while (s.save_idx < a.n_save) {
      const double ts = s.ts;
      const double at = absT(ts);
      if (!(ts <= t_end + 1e-12 * (1.0 > at ? 1.0 : at))) break;
      s.ts = next_save(a, s.save_idx + 1);
      const double theta = (ts - t) / dt_use;
      const double theta1 = 1.0 - theta;
      double h1 = H1[0] * (double)k[0];
      double h2 = H2[0] * (double)k[0];
      double h3 = H3[0] * (double)k[0];
#pragma unroll
      for (int q = 1; q < 8; ++q) {
        h1 = fmaT(H1[q], (double)k[q], h1);
        h2 = fmaT(H2[q], (double)k[q], h2);
        h3 = fmaT(H3[q], (double)k[q], h3);
      }
      double x = fmaT(theta, h3, h2);
      x = fmaT(theta, x, h1);
      x = fmaT(theta1, x, y_new);
      if (row)
        a.hist[i * a.h_ts + (i64)s.save_idx * a.h_ss + (i64)lane * a.h_vs] =
            fmaT(theta, x, theta1 * s.y);
      s.save_idx++;
    }
    s.y = y_new;
    s.t = t_end;
    s.accepted++;
  } else {
    s.rejected++;
  }
  s.n_steps++;
}

}  // namespace r5
}  // namespace mdx

extern "C" __global__ __launch_bounds__(64 * MDX_ROWS) MDX_REG_CAP void mdx_rodas5p(
    mdx::SolveArgs a) {
  using namespace mdx::r5;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int lane = (int)threadIdx.x % 64;
  // as many trajectories as the launch has wavefronts a workgroup: WAVES, or one
  // where the kernel was registered without them
  const mdx::i64 i = (mdx::i64)blockIdx.x * (blockDim.x / 64) + w;
  if (i >= a.n_traj) return;
  PA p;
  p.load(a, i);
  RowState s;
  const double* __restrict__ times = a.times;
  const double tf = times[a.n_save - 1];
  s.y = 0.0;
  if (lane < N) {
    s.y = a.y0[i * a.y0_ts + (mdx::i64)lane * a.y0_vs];
    a.hist[i * a.h_ts + (mdx::i64)lane * a.h_vs] = s.y;
  }
  s.t = times[0];
  s.dt = a.dt0 > 0.0 ? a.dt0 : (tf - times[0]) * 1e-6;
#if MDX_TF_INDEX >= 0
  s.tf = p[MDX_TF_INDEX];
#else
  s.tf = tf;
#endif
  s.err_prev = s.err_prev2 = 1.0;
  s.save_idx = 1;
  s.n_steps = s.accepted = s.rejected = 0;
  s.ts = mdx::next_save(a, 1);
  mdx::settle();
  while (s.save_idx < a.n_save && s.t < s.tf && s.n_steps < a.max_steps)
    rows_step(s, p, a, i, w, lane);
  if (a.cost) {
    if (lane == 0)
      a.cost[i] = (s.save_idx < a.n_save && s.t < s.tf) ? (s.tf - s.t) / s.dt : 0.0;
    return;
  }
  for (; s.save_idx < a.n_save; s.save_idx++)
    if (lane < N)
      a.hist[i * a.h_ts + (mdx::i64)s.save_idx * a.h_ss + (mdx::i64)lane * a.h_vs] = s.y;
  if (lane == 0) {
    a.accepted[i] = s.accepted;
    a.rejected[i] = s.rejected;
    a.loop[i] = s.n_steps;
  }
}
