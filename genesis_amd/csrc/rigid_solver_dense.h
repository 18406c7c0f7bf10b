// Newton solver of models whose dofs all belong to one entity (an arm, a legged robot), one wavefront per env.
//
// Same algorithm and operation order as the other solvers (func_init_solver / func_solve / func_linesearch / rank-1
// Cholesky updates of constraint_solver_decomp.py); the entity-block machinery of rigid_solver_wave.h has nothing to
// do here, since every row touches the one entity, the Hessian is one dense triangle and every row list is all rows.
// A quadruped solve is a few thousand dependent operations on 18 dofs and some twenty rows, so what bounds it is
// latency and the registers that limit how many envs a SIMD holds:
//   * lane d owns dof d (at most 64): vectors over dofs are registers, read by other lanes as scalars (v_readlane);
//   * lane r owns row r of the first 64 rows: weight, Jaref, force, activity and line-search terms are registers for
//     the whole solve; the rows lie densely in LDS (stride odd, so a row or a column is read without bank conflicts),
//     staged once; rows past 64 are staged 64 at a time on each pass and keep their scalars in the env's row arrays;
//   * M and the factor lie in LDS with the same stride, the factor's diagonal in registers.
// Sums over rows (J^T f, J^T D J) take the rows with a nonzero term in ascending order, one lane per dof or per
// entry: the per-row walk's terms in its order (skipped terms add +-0 to sums that start at +0), hence its bits.
// The stop test needs the gradient but not the Newton direction, so the factor's update and the substitutions of the
// last iteration, which nothing reads, are not done.
// Measured (MI355X, the solve of one step, entity-block solver -> this one): 64 arms 52 -> 20 us, 4,000 quadrupeds
// 377 -> 164 us, 32,768 quadrupeds 1,805 -> 543 us.
#pragma once
#include "rigid_env.h"
#include "rigid_solver_bodies.h"
#include "rigid_solver_wave.h"

namespace gsr {

constexpr int kDenseDofs = 64;

// one entity holds every dof and the triangle of its Hessian is within the model's LDS budget
__host__ __device__ inline bool dense_solver(const gsr_model& m) {
  return m.n_dofs > 0 && m.n_dofs <= kDenseDofs && m.max_entity_dofs == m.n_dofs &&
         m.n_dofs * (m.n_dofs + 1) / 2 <= m.wave_h_floats;
}
__host__ __device__ inline int dense_stride(int D) { return D | 1; }
__host__ __device__ inline size_t dense_lds_bytes(int D) {
  return sizeof(float) * (size_t)(2 * D + kWave) * (size_t)dense_stride(D);
}

struct DenseCtx {
  const Env& e;
  lds_f* H;     // [D][S] factor, lower triangle (its diagonal lives in the lanes)
  lds_f* M;     // [D][S] mass matrix
  lds_f* J;     // [64][S] staged rows
  int lane, D, S, n_con, ne, nef;
};

// scalars of this lane's row of the first 64
struct DenseRow {
  float Dc, ja, jv, f, q0, q1, q2, fl, rf;
  int act;  // bit 0: active, bit 1: active before the last update
};

// rows c0 .. c0 + 63 into J, zero where a row has no entry or does not exist
__device__ inline void dense_stage(const DenseCtx& w, int c0) {
  const Env& e = w.e;
  const int c = c0 + w.lane;
  lds_f* row = w.J + w.lane * w.S;
  __syncthreads();
  const int W = e.m.row_width;
  const int nnz = c < w.n_con ? e.EI(e.s.jac_nnz, c) : 0;
  RowStage r;
  if (W <= kStage) {
    const float* pv = &e.JV(c < w.n_con ? c : 0, 0);
    const int* pi = &e.JI(c < w.n_con ? c : 0, 0);
#pragma unroll
    for (int k = 0; k < kStage; k++) {
      r.v[k] = k < W ? pv[k] : 0.f;
      r.d[k] = k < W ? pi[k] : 0;
    }
  }
  for (int d = 0; d < w.D; d++) row[d] = 0.f;
  if (W <= kStage) {
#pragma unroll
    for (int k = 0; k < kStage; k++)
      if (k < nnz) row[r.d[k]] = r.v[k];
  } else {
    for (int k = 0; k < nnz; k++) row[e.JI(c, k)] = e.JV(c, k);
  }
  __syncthreads();
}

// acc + sum_d J[staged row of this lane][d] x[d], x held by the dof lanes
__device__ __forceinline__ float dense_row_dot(const DenseCtx& w, float acc, float x) {
  const lds_f* row = w.J + w.lane * w.S;
#pragma unroll 4
  for (int d = 0; d < w.D; d++) acc += row[d] * lane_value(x, d);
  return acc;
}

__device__ __forceinline__ float dense_mass_mul(const DenseCtx& w, float x) {
  const lds_f* row = w.M + (w.lane < w.D ? w.lane : 0) * w.S;
  float v = 0.f;
#pragma unroll 4
  for (int j = 0; j < w.D; j++) v += row[j] * lane_value(x, j);
  return v;
}

// activity, force and this row's cost terms from Jaref (func_update_constraint)
__device__ __forceinline__ void dense_row_state(const DenseCtx& w, int c, float ja, float Dc, float fl, float rf, int& act,
                                                float& force, double& ci) {
  int a = 1;
  float floss_force = 0.f;
  if (w.ne <= c && c < w.nef) {
    const bool ln = ja <= -rf, lp = ja >= rf;
    a = !(ln || lp);
    floss_force = (float)ln * fl + (float)lp * -fl;
    float fc = (float)ln * fl * (-0.5f * rf - ja);
    fc += (float)lp * fl * (-0.5f * rf + ja);
    ci += (double)fc;
  } else if (w.nef <= c) {
    a = ja < 0.f;
  }
  act = a | ((act & 1) << 1);
  force = floss_force + (-ja * Dc * (float)a);
  ci += (double)(0.5f * (ja * ja * Dc * (float)a));
}

// rows' activity and forces, J^T f (lane d: dof d) and the cost; the rows past 64 read and write the row arrays
__device__ inline void dense_update_constraint(const DenseCtx& w, DenseRow& r, float Ma, float qacc, float force,
                                               float acc_smooth, float& qfrc, double& cost, float& gauss) {
  const Env& e = w.e;
  const gsr_state& s = e.s;
  double ci = 0.0;
  float acc = 0.f;
  const lds_f* col = w.J + (w.lane < w.D ? w.lane : 0);
  for (int c0 = 0; c0 < w.n_con; c0 += kWave) {
    const int c = c0 + w.lane;
    float f = 0.f;
    if (c0 == 0) {
      if (c < w.n_con) dense_row_state(w, c, r.ja, r.Dc, r.fl, r.rf, r.act, r.f, ci);
      f = c < w.n_con ? r.f : 0.f;
    } else if (c < w.n_con) {
      int act = e.EI(s.efc_active, c);
      const bool is_fl = w.ne <= c && c < w.nef;
      const float fl = is_fl ? e.EF(s.efc_fl, c) : 0.f, rf = is_fl ? e.EF(s.efc_diag, c) * fl : 0.f;
      dense_row_state(w, c, e.EF(s.efc_Jaref, c), e.EF(s.efc_D, c), fl, rf, act, f, ci);
      e.EI(s.efc_active, c) = act;
      e.EF(s.efc_force, c) = f;
    }
    if (w.n_con > kWave) dense_stage(w, c0);
    unsigned long long on = __ballot(f != 0.f);
    while (on) {
      const int k = __ffsll((long long)on) - 1;
      on &= on - 1;
      acc = acc + col[k * w.S] * lane_value(f, k);
    }
  }
  qfrc = acc;
  double gi = 0.0;
  if (w.lane < w.D) gi += (double)(0.5f * (Ma - force) * (qacc - acc_smooth));
  const double gd = wave_sum_d(gi);
  gauss = (float)gd;
  cost = wave_sum_d(ci) + gd;
}

// entry t of the packed lower triangle: row i, column j <= i
__device__ __forceinline__ void tri_entry(int t, int& i, int& j) {
  i = (int)((sqrtf(8.f * (float)t + 1.f) - 1.f) * 0.5f);
  while (i * (i + 1) / 2 > t) i--;
  while ((i + 1) * (i + 2) / 2 <= t) i++;
  j = t - i * (i + 1) / 2;
}

// H = M + J^T D J over the active rows (func_nt_hessian_direct), lanes over the entries of the lower triangle, four
// entries a lane at a time; then its Cholesky factor, row i on lane i, column by column (func_nt_chol_factor's sums,
// each serial over its index); dg: the factor's diagonal, entry d on lane d
__device__ inline void dense_hessian(const DenseCtx& w, const DenseRow& r, float& dg) {
  const Env& e = w.e;
  const gsr_state& s = e.s;
  const int D = w.D, S = w.S, ntri = D * (D + 1) / 2, lane = w.lane;
  const float eps = e.m.eps;
  for (int c0 = 0; c0 == 0 || c0 < w.n_con; c0 += kWave) {
    const int c = c0 + lane;
    float Dc = r.Dc;
    int act = c < w.n_con ? r.act & 1 : 0;
    if (c0 > 0) {
      Dc = c < w.n_con ? e.EF(s.efc_D, c) : 0.f;
      act = c < w.n_con ? e.EI(s.efc_active, c) & 1 : 0;
    }
    if (w.n_con > kWave) dense_stage(w, c0);
    const unsigned long long rows = __ballot(act != 0);
    const bool last = c0 + kWave >= w.n_con;
    for (int t0 = 0; t0 < ntri; t0 += 4 * kWave) {
      int i[4], j[4];
      float a[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int t = t0 + q * kWave + lane;
        tri_entry(t < ntri ? t : 0, i[q], j[q]);
        a[q] = c0 == 0 ? 0.f : w.H[i[q] * S + j[q]];
      }
      const int nq = min(4, (ntri - t0 + kWave - 1) / kWave);
      unsigned long long on = rows;
      while (on) {
        const int k = __ffsll((long long)on) - 1;
        on &= on - 1;
        const lds_f* row = w.J + k * S;
        const float Dk = lane_value(Dc, k);
#pragma unroll
        for (int q = 0; q < 4; q++) {
          if (q < nq) {
            // pair (the row's later dof i, earlier dof j), skipped when |J[i]| <= eps
            const float vi = row[i[q]];
            const float vm = fabsf(vi) > eps ? vi : 0.f;
            a[q] = a[q] + row[j[q]] * vm * Dk;
          }
        }
      }
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (t0 + q * kWave + lane < ntri) w.H[i[q] * S + j[q]] = last ? a[q] + w.M[i[q] * S + j[q]] : a[q];
    }
    __syncthreads();
  }
  // factor: lane i's running sum of column i is H(i, i) less the squares, every later lane's the products
  const lds_f* own = w.H + (lane < D ? lane : 0) * S;
  for (int i = 0; i < D; i++) {
    const lds_f* ri = w.H + i * S;
    const float hji = own[i];
    const bool diag = lane == i;
    float acc = diag ? hji : 0.f;
#pragma unroll 8
    for (int k = 0; k < i; k++) {
      const float p = own[k] * ri[k];
      acc += diag ? -p : p;
    }
    const float hii = sqrtf(fmaxf(lane_value(acc, i), eps));
    const float inv = 1.f / hii;
    if (diag) dg = hii;
    if (lane > i && lane < D) w.H[lane * S + i] = (hji - acc) * inv;
    __syncthreads();
  }
}

// H^-1 g, entry d on lane d (func_nt_chol_solve)
__device__ inline float dense_chol_solve(const DenseCtx& w, float dg, float a) {
  const int D = w.D, S = w.S, lane = w.lane;
  const lds_f* own = w.H + (lane < D ? lane : 0) * S;
#pragma unroll 4
  for (int j = 0; j < D; j++) {
    const float l = own[j];
    const float y = lane_value(a / dg, j);
    a = lane == j ? y : lane > j ? a - l * y : a;
  }
  const lds_f* col = w.H + (lane < D ? lane : 0);
#pragma unroll 4
  for (int i = D - 1; i >= 0; i--) {
    const float l = col[i * S];
    const float x = lane_value(a / dg, i);
    a = lane == i ? x : lane < i ? a - l * x : a;
  }
  return a;
}

// rank-1 update / downdate of the factor with the vector x (entry d on lane d); false on rank loss (the update is then
// incomplete and the factor is rebuilt)
__device__ inline bool dense_rank1(const DenseCtx& w, float& dg, float x, float sgn) {
  const float eps = w.e.m.eps;
  const int D = w.D, lane = w.lane;
  lds_f* own = w.H + (lane < D ? lane : 0) * w.S;
  bool ok = true;
  for (int k = 0; k < D; k++) {
    const float vk = lane_value(x, k);
    if (!(fabsf(vk) > eps)) continue;
    const float Lkk = lane_value(dg, k);
    float tmp = Lkk * Lkk + vk * vk * sgn;
    if (tmp < eps) {
      tmp = eps;
      ok = false;
    }
    const float r = sqrtf(tmp), cc = r / Lkk, cinv = 1.f / cc, sv = vk / Lkk;
    if (lane > k && lane < D) {
      const float hv = (own[k] + sv * x * sgn) * cinv;
      own[k] = hv;
      x = x * cc - sv * hv;
    }
    if (lane == k) dg = r;
  }
  __syncthreads();
  return ok;
}

__device__ __forceinline__ void dense_ls_row(const DenseCtx& w, int c, float ja, float jv, float q0, float q1, float q2,
                                             float fl, float rf, float alpha, double& t0, double& t1, double& t2) {
  const float x = ja + alpha * jv;
  bool act = true;
  if (w.ne <= c && c < w.nef) {
    const bool ln = x <= -rf, lp = x >= rf;
    if (ln || lp) {
      q0 = (float)ln * fl * (-0.5f * rf - ja) + (float)lp * fl * (-0.5f * rf + ja);
      q1 = (float)ln * (-fl * jv) + (float)lp * (fl * jv);
      q2 = 0.f;
    }
  } else if (w.nef <= c) {
    act = x < 0.f;
  }
  t0 += (double)(q0 * (float)act);
  t1 += (double)(q1 * (float)act);
  t2 += (double)(q2 * (float)act);
}

struct DenseLine {
  float qg0, qg1, qg2;
};

__device__ inline WLS dense_ls_point(const DenseCtx& w, const DenseRow& r, const DenseLine& g, float alpha, int& ls_it) {
  const Env& e = w.e;
  const gsr_state& s = e.s;
  double t0 = 0.0, t1 = 0.0, t2 = 0.0;
  if (w.lane < w.n_con) dense_ls_row(w, w.lane, r.ja, r.jv, r.q0, r.q1, r.q2, r.fl, r.rf, alpha, t0, t1, t2);
  for (int c = w.lane + kWave; c < w.n_con; c += kWave) {
    const bool is_fl = w.ne <= c && c < w.nef;
    const float fl = is_fl ? e.EF(s.efc_fl, c) : 0.f, rf = is_fl ? e.EF(s.efc_diag, c) * fl : 0.f;
    dense_ls_row(w, c, e.EF(s.efc_Jaref, c), e.EF(s.efc_jv, c), e.QD(c, 0), e.QD(c, 1), e.QD(c, 2), fl, rf, alpha, t0,
                 t1, t2);
  }
  return ls_point_from(e, g.qg0, g.qg1, g.qg2, wave_sum_d(t0), wave_sum_d(t1), wave_sum_d(t2), alpha, ls_it);
}

__device__ __forceinline__ void wave_solve_dense(const Env& e, char* lds) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const int lane = threadIdx.x, D = m.n_dofs, S = dense_stride(D);
  const int n_con = e.I(s.n_con, 0), ne = e.I(s.n_con, 1), nef = ne + e.I(s.n_con, 2);
  lds_f* base = reinterpret_cast<lds_f*>((lds_c*)lds);
  const DenseCtx w{e, base, base + D * S, base + 2 * D * S, lane, D, S, n_con, ne, nef};
  const bool dof = lane < D;
  const float acc_smooth = dof ? e.F(s.acc_smooth, lane) : 0.f;
  float qacc = acc_smooth, qfrc = 0.f;
  int iters = 0;
  if (n_con > 0) {
    if (e.I(s.is_warmstart, 0)) qacc = dof ? e.F(s.qacc_ws, lane) : 0.f;
    const float force = dof ? e.F(s.force, lane) : 0.f;
    // the entity's mass block: all of mass_blk, row-major
    for (int t = lane; t < D * D; t += kWave) w.M[(t / D) * S + t % D] = e.F(s.mass_blk, t);
    DenseRow r;
    r.Dc = r.ja = r.jv = r.f = r.q0 = r.q1 = r.q2 = r.fl = r.rf = 0.f;
    r.act = 0;
    if (lane < n_con) {
      r.Dc = e.EF(s.efc_D, lane);
      r.ja = -e.EF(s.efc_aref, lane);
      if (ne <= lane && lane < nef) {
        r.fl = e.EF(s.efc_fl, lane);
        r.rf = e.EF(s.efc_diag, lane) * r.fl;
      }
    }
    dense_stage(w, 0);
    float Ma = dense_mass_mul(w, qacc);
    r.ja = dense_row_dot(w, r.ja, qacc);
    for (int c0 = kWave; c0 < n_con; c0 += kWave) {
      dense_stage(w, c0);
      const int c = c0 + lane;
      const float ja = dense_row_dot(w, c < n_con ? -e.EF(s.efc_aref, c) : 0.f, qacc);
      if (c < n_con) e.EF(s.efc_Jaref, c) = ja;
    }
    double cost;
    float gauss;
    dense_update_constraint(w, r, Ma, qacc, force, acc_smooth, qfrc, cost, gauss);
    const float scale = e.meaninertia() * (float)(D > 1 ? D : 1);
    float dg = 1.f;
    bool build = true;
    for (;;) {
      if (build) dense_hessian(w, r, dg);
      const float dir = dense_chol_solve(w, dg, Ma - force - qfrc);
      const float search = dof ? -dir : 0.f;
      if (iters >= m.iterations) break;
      iters++;
      // func_linesearch
      const float snorm = sqrtf((float)wave_sum_d((double)(search * search)));
      const float gtol = m.tolerance * m.ls_tolerance * snorm * scale;
      float alpha = 0.f, mv = 0.f;
      if (!(snorm < m.eps)) {
        mv = dense_mass_mul(w, search);
        mv = dof ? mv : 0.f;
        for (int c0 = 0; c0 < n_con; c0 += kWave) {
          if (n_con > kWave) dense_stage(w, c0);
          const int c = c0 + lane;
          const float jv = dense_row_dot(w, 0.f, search);
          if (c0 == 0) {
            r.jv = jv;
            r.q0 = r.Dc * (0.5f * r.ja * r.ja);
            r.q1 = r.Dc * (jv * r.ja);
            r.q2 = r.Dc * (0.5f * jv * jv);
          } else if (c < n_con) {
            const float Dc = e.EF(s.efc_D, c), ja = e.EF(s.efc_Jaref, c);
            e.EF(s.efc_jv, c) = jv;
            e.QD(c, 0) = Dc * (0.5f * ja * ja);
            e.QD(c, 1) = Dc * (jv * ja);
            e.QD(c, 2) = Dc * (0.5f * jv * jv);
          }
        }
        double a1 = 0.0, a2 = 0.0;
        if (dof) {
          a1 += (double)(search * Ma - search * force);
          a2 += (double)(0.5f * search * mv);
        }
        const DenseLine g{gauss, (float)wave_sum_d(a1), (float)wave_sum_d(a2)};
        __syncthreads();
        alpha = linesearch_points(m, gtol, [&](float x, int& ls_it) { return dense_ls_point(w, r, g, x, ls_it); });
      }
      if (fabsf(alpha) < m.eps) break;
      qacc = qacc + search * alpha;
      Ma = Ma + mv * alpha;
      r.ja = r.ja + r.jv * alpha;
      for (int c = lane + kWave; c < n_con; c += kWave)
        e.EF(s.efc_Jaref, c) = e.EF(s.efc_Jaref, c) + e.EF(s.efc_jv, c) * alpha;
      const double prev_cost = cost;
      dense_update_constraint(w, r, Ma, qacc, force, acc_smooth, qfrc, cost, gauss);
      const float grad = dof ? Ma - force - qfrc : 0.f;
      const float tol_scaled = scale * m.tolerance;
      const double improvement = prev_cost - cost;
      const float gn = sqrtf((float)wave_sum_d((double)(grad * grad)));
      if (gn < tol_scaled || improvement < tol_scaled || iters >= m.iterations) break;
      // activity changes in row order: rank-1 updates or a rebuild of the factor
      const bool in0 = lane < n_con;
      int n_changed = __popcll(__ballot(in0 && ((r.act ^ (r.act >> 1)) & 1)));
      for (int c0 = kWave; c0 < n_con; c0 += kWave) {
        const int a = c0 + lane < n_con ? e.EI(s.efc_active, c0 + lane) : 0;
        n_changed += __popcll(__ballot((a ^ (a >> 1)) & 1));
      }
      build = n_changed > kMaxRank1PerIter;
      for (int c0 = 0; c0 < n_con && n_changed > 0 && !build; c0 += kWave) {
        const int a = c0 == 0 ? (in0 ? r.act : 0) : c0 + lane < n_con ? e.EI(s.efc_active, c0 + lane) : 0;
        unsigned long long chg = __ballot((a ^ (a >> 1)) & 1);
        if (chg && n_con > kWave) dense_stage(w, c0);
        const float Dc = c0 == 0 ? r.Dc : c0 + lane < n_con ? e.EF(s.efc_D, c0 + lane) : 0.f;
        while (chg && !build) {
          const int k = __ffsll((long long)chg) - 1;
          chg &= chg - 1;
          const float sgn = (lane_value(a, k) & 1) ? 1.f : -1.f;
          const float sq = sqrtf(lane_value(Dc, k));
          const float x = dof ? w.J[k * S + lane] * sq : 0.f;
          build = !dense_rank1(w, dg, x, sgn);
        }
      }
    }
    if (lane < n_con) e.EF(s.efc_force, lane) = r.f;
  }
  // epilogue (func_update_qacc, func_update_contact_force)
  int bad = 0;
  if (dof) {
    e.F(s.acc, lane) = qacc;
    e.F(s.force, lane) = e.F(s.qf_smooth, lane) + qfrc;
    e.F(s.qacc_ws, lane) = qacc;
    bad = isnan(qacc) ? 1 : 0;
  }
  const bool any_bad = __any(bad);
  if (lane == 0) {
    e.I(s.solver_iters, 0) = iters;
    e.I(s.is_warmstart, 0) = 1;
    if (any_bad) e.I((int32_t*)s.errno_env, 0) |= (int)GSR_ERR_NAN_QACC;
  }
  __syncthreads();
  contact_forces(e, lane, kWave);
}

// the Newton solve of one env on one wavefront
__device__ __forceinline__ void wave_solve(const Env& e, char* lds) {
  if (dense_solver(e.m)) wave_solve_dense(e, lds);
  else if (bodies_solver(e.m)) solve_bodies<1>(e, lds);
  else wave_solve_blocks(e, lds);
}
// dynamic LDS of wave_solve
__host__ __device__ inline size_t solve_lds_bytes(const gsr_model& m) {
  return dense_solver(m)    ? dense_lds_bytes(m.n_dofs)
         : bodies_solver(m) ? bodies_lds_bytes(m.n_dofs, m.wave_h_floats)
                            : wave_lds_bytes(m);
}

}  // namespace gsr
