// Kinematics and smooth dynamics of articulated environments on wavefronts: the stages of rigid_kin.h and dev_integrate
// with the same operations per value in the same order (so the same bits), spread over G lanes per env (64: one env a
// wavefront, 16: four envs a wavefront).
//
// One lane walking the tree through the state in global memory costs a round trip to L2 per dependent access: 172 us
// for the step_1 of 64 arms, 475 us for that of 4,000 quadrupeds, whatever the env count up to tens of thousands. Here
// a stage's inputs are loaded at once, values that lanes exchange live in LDS, and only the work that is serial by
// nature stays serial:
//   * link poses, velocities and bias accelerations go level by level down the tree, the links of a level on their
//     own lanes; the joints' own rotations (sin, cos in double) do not depend on the parent and come first;
//   * sums up the tree (composite inertias, link forces) run over the links that have a parent, last first, one lane
//     per component; a root's mass and COM sums run on the root's lane in link order;
//   * the mass matrix has a lane per entry, its LDL^T one step per eliminated dof with a lane per updated entry; the
//     substitutions multiply a column's entries on their own lanes and subtract them in ascending order.
// A tree of 9 to 18 dofs occupies 16 lanes about as well as 64, and four neighbouring envs read 16 bytes of each line of
// the env-minor state instead of 4; one env alone is faster on 64 lanes. tree_lanes() holds the line between the two.
//
// Measured (MI355X, us per launch, one lane per env -> 64 lanes -> 16 lanes per env), step_1: 64 arms 172 -> 23, 5,001
// arms 204 -> 81 -> 31, 4,000 quadrupeds 475 -> 114 -> 58, 32,768 quadrupeds 571 -> 846 -> 232; step_2: 64 arms 92 -> 36,
// 5,001 arms 122 -> 72 -> 44, 32,768 quadrupeds 190 -> 259 -> 145; kinematics of 20,000 quadrupeds 198 -> 261 -> 113.
#pragma once
#include "rigid_kin.h"
#include "rigid_solver.h"
#include "rigid_wave.h"

namespace gsr {

constexpr size_t kTreeMaxLds = 40 * 1024;  // four workgroups a CU

// LDS words: the tables of the model once per workgroup, then each env's values (step_1 and the kinematics use the
// space one after the other)
__host__ __device__ inline int tree_table_words(int L, int D, int mass) { return 4 * L + 3 * D + (mass + D) / 2; }
__host__ __device__ inline int tree_env_words(const gsr_model& m) {
  const int L = m.n_links, D = m.n_dofs, J = m.n_joints;
  const int a = 25 * L + 13 * D + m.mass_blk_size, b = 20 * L + 7 * D + 13 * J + m.n_qs;
  return (a > b ? a : b) | 1;
}
__host__ __device__ inline size_t tree_lds_bytes(const gsr_model& m, int G) {
  return sizeof(float) * (size_t)(tree_table_words(m.n_links, m.n_dofs, m.mass_blk_size) + kWave / G * tree_env_words(m));
}
// Models this path serves: one with an entity of more than six dofs whose values fit kTreeMaxLds. Free bodies and fixed links
// alone are better off with one lane per entity: nothing in them is serial but the entity itself. Arms of up to six joints
// are told apart from those by nothing here and take a lane too, which walks their chain through global memory (one arm of
// six joints, 1 to 2,048 envs: step_1 72 to 79 us, step_2 64 to 68).
__host__ __device__ inline bool tree_dynamics(const gsr_model& m) {
  return m.max_entity_dofs > 6 && tree_lds_bytes(m, kWave) <= kTreeMaxLds;
}
// Lanes per env of a launch over n envs: 16 once there are more envs than SIMDs (1,024), unless four envs take more LDS
// than kTreeMaxLds. Measured around the line (us, 64 lanes, 16 lanes): quadrupeds step_1 1,024: 38, 45; 2,048: 42, 48; 3,072:
// 72, 48; step_2 1,024: 34, 28; 2,048: 32, 31; 3,072: 38, 30; arms step_1 1,024: 24, 27; 2,048: 26, 26; 3,072: 43, 28; step_2
// 1,024: 48, 36; 2,048: 44, 40; 3,072: 52, 41.
__host__ __device__ inline int tree_lanes(const gsr_model& m, int n) {
  return n > 1024 && tree_lds_bytes(m, 16) <= kTreeMaxLds ? 16 : kWave;
}

// tables of the model, built by the whole wavefront: parent, depth and root of each link, the links that have a parent
// (last first), link and entity range of each dof, and every lower-triangle entry of the entity blocks (row dof |
// column dof << 16), blocks one after the other, rows ascending
struct TreeTables {
  lds_i *par, *dep, *root, *up, *dlink, *dst, *den, *tri;
  int n_up, n_tri, levels;
};
template <bool kDofs>
__device__ inline TreeTables tree_tables(const gsr_model& m, char* lds) {
  const int lane = threadIdx.x, L = m.n_links, D = m.n_dofs;
  TreeTables t;
  t.par = reinterpret_cast<lds_i*>((lds_c*)lds);
  t.dep = t.par + L;
  t.root = t.dep + L;
  t.up = t.root + L;
  t.dlink = t.up + L;
  t.dst = t.dlink + D;
  t.den = t.dst + D;
  t.tri = t.den + D;
  t.n_up = t.n_tri = 0;
  int most = 0;
  for (int l0 = (L - 1) / kWave * kWave; l0 >= 0; l0 -= kWave) {
    const int l = l0 + lane;
    int pl = -1;
    if (l < L) {
      int n = 0;
      pl = m.link_parent[l];
      for (int q = pl; q != -1; q = m.link_parent[q]) n++;
      t.par[l] = pl;
      t.dep[l] = n;
      t.root[l] = m.link_root[l];
      most = max(most, n);
      if (kDofs)
        for (int d = m.link_dof_start[l]; d < m.link_dof_end[l]; d++) t.dlink[d] = l;
    }
    const unsigned long long has = __ballot(pl >= 0);
    if (pl >= 0) t.up[t.n_up + __popcll(lane < 63 ? has >> (lane + 1) : 0ull)] = l;
    t.n_up += __popcll(has);
  }
  t.levels = -wave_min_i(-most) + 1;
  if (kDofs) {
    for (int ie = 0; ie < m.n_entities; ie++) {
      const int st = m.ent_dof_start[ie], n = m.ent_dof_end[ie] - st;
      for (int k = lane; k < n * (n + 1) / 2; k += kWave) {
        int i = (int)((sqrtf(8.f * (float)k + 1.f) - 1.f) * 0.5f);
        while (i * (i + 1) / 2 > k) i--;
        while ((i + 1) * (i + 2) / 2 <= k) i++;
        t.tri[t.n_tri + k] = (st + i) | ((st + k - i * (i + 1) / 2) << 16);
      }
      for (int d = st + lane; d < st + n; d += kWave) {
        t.dst[d] = st;
        t.den[d] = st + n;
      }
      t.n_tri += n * (n + 1) / 2;
    }
  }
  __syncthreads();
  return t;
}

__device__ __forceinline__ f3 lds3(const lds_f* a, int i) { return f3{a[3 * i], a[3 * i + 1], a[3 * i + 2]}; }
__device__ __forceinline__ void set3(lds_f* a, int i, f3 v) {
  a[3 * i] = v.x;
  a[3 * i + 1] = v.y;
  a[3 * i + 2] = v.z;
}
__device__ __forceinline__ q4 lds4(const lds_f* a, int i) { return q4{a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3]}; }
__device__ __forceinline__ void set4(lds_f* a, int i, q4 v) {
  a[4 * i] = v.w;
  a[4 * i + 1] = v.x;
  a[4 * i + 2] = v.y;
  a[4 * i + 3] = v.z;
}

// ---- step_1 -------------------------------------------------------------------------------------------------------
// M^-1 f of one entity of D dofs from its LDL^T (func_solve_mass_batched): a row's products on their lanes, subtracted
// in ascending order. 64 lanes: dof d on lane d, read as scalars; 16 lanes: dofs r and r + 16 on lane r, read by row
// broadcasts, absent terms subtracted as +0.
__device__ inline void tree_solve_64(const Env& e, const lds_f* ML, const lds_f* vec, int D) {
  const int lane = threadIdx.x, d = lane < D ? lane : 0;
  float o = vec[d];
  for (int i = D - 2; i >= 0; i--) {
    const float pr = ML[d * D + i] * o;
    float r = lane_value(o, i);
    for (int j = i + 1; j < D; j++) r -= lane_value(pr, j);
    o = lane == i ? r : o;
  }
  o = o * e.F(e.s.mass_D_inv, d);
  for (int i = 1; i < D; i++) {
    const float pr = ML[i * D + d] * o;
    float r = lane_value(o, i);
    for (int j = 0; j < i; j++) r -= lane_value(pr, j);
    o = lane == i ? r : o;
  }
  if (lane < D) {
    e.F(e.s.acc_smooth, lane) = o;
    e.F(e.s.acc, lane) = o;
  }
}
template <int kJ>
__device__ __forceinline__ float sub_row16(float r, float p) {
  r -= dpp<0x150 + kJ>(p);
  if constexpr (kJ < 15) return sub_row16<kJ + 1>(r, p);
  else return r;
}
__device__ inline void tree_solve_16(const Env& e, const lds_f* ML, const lds_f* vec, int D) {
  const int r = threadIdx.x & 15;
  const bool has0 = r < D, has1 = r + 16 < D;
  const int d0 = has0 ? r : 0, d1 = has1 ? r + 16 : 0;
  float o0 = vec[d0], o1 = vec[d1];
  for (int i = D - 2; i >= 0; i--) {
    const float p0 = has0 && r > i ? ML[d0 * D + i] * o0 : 0.f, p1 = has1 && r + 16 > i ? ML[d1 * D + i] * o1 : 0.f;
    float x = i < 16 ? sub_row16<0>(o0, p0) : o1;
    if (D > 16) x = sub_row16<0>(x, p1);
    if (i < 16) o0 = r == i ? x : o0;
    else o1 = r + 16 == i ? x : o1;
  }
  if (has0) o0 = o0 * e.F(e.s.mass_D_inv, d0);
  if (has1) o1 = o1 * e.F(e.s.mass_D_inv, d1);
  for (int i = 1; i < D; i++) {
    const float p0 = has0 && r < i ? ML[i * D + d0] * o0 : 0.f, p1 = has1 && r + 16 < i ? ML[i * D + d1] * o1 : 0.f;
    float x = sub_row16<0>(i < 16 ? o0 : o1, p0);
    if (i > 16) x = sub_row16<0>(x, p1);
    if (i < 16) o0 = r == i ? x : o0;
    else o1 = r + 16 == i ? x : o1;
  }
  if (has0) e.F(e.s.acc_smooth, d0) = e.F(e.s.acc, d0) = o0;
  if (has1) e.F(e.s.acc_smooth, d1) = e.F(e.s.acc, d1) = o1;
}

// smooth dynamics of env e on the G lanes holding it; p: the env's LDS words
template <int G>
__device__ inline void tree_step1(const Env& e, const TreeTables& t, lds_f* p) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const int lane = threadIdx.x & (G - 1), L = m.n_links, D = m.n_dofs, E = m.n_entities;
  const float EPS = m.eps, dt = m.dt;
  lds_f* crb = p; p += 13 * L;   // component c of link l at c * L + l: inertia 0..8, position 9..11, mass 12
  lds_f* acc = p; p += 6 * L;    // bias accelerations, link l at 6 l: linear, angular
  lds_f* frc = p; p += 6 * L;    // link forces, component c of link l at c * L + l
  lds_f* cda = p; p += 3 * D;
  lds_f* cdv = p; p += 3 * D;
  lds_f* fa = p; p += 3 * D;     // cdofd * vel until the accelerations are done, then the composite forces
  lds_f* fv = p; p += 3 * D;
  lds_f* vec = p; p += D;
  lds_f* ML = p;
  const bool single = m.max_entity_dofs == D;  // one entity holds every dof: its block is the whole matrix

  // inputs
  for (int k = 0; k < 9; k++)
    for (int l = lane; l < L; l += G) crb[k * L + l] = e.F(s.cinr_inertial, 9 * l + k);
  for (int l = lane; l < L; l += G) {
    const f3 c = e.L3(s.cinr_pos, l);
    crb[9 * L + l] = c.x;
    crb[10 * L + l] = c.y;
    crb[11 * L + l] = c.z;
    crb[12 * L + l] = e.F(s.cinr_mass, l);
  }
  for (int d = lane; d < D; d += G) {
    const float v = e.F(s.vel, d);
    set3(cda, d, e.L3(s.cdof_ang, d));
    set3(cdv, d, e.L3(s.cdof_vel, d));
    set3(fa, d, e.L3(s.cdofd_ang, d) * v);
    set3(fv, d, e.L3(s.cdofd_vel, d) * v);
  }
  __syncthreads();

  // --- bias accelerations (rsd:6180-6281), level by level ---
  for (int lev = 0; lev < t.levels; lev++) {
    for (int l = lane; l < L; l += G) {
      if (t.dep[l] != lev) continue;
      const int pl = t.par[l];
      f3 cv, ca;
      if (pl == -1) {
        cv = -f3{m.gravity[0], m.gravity[1], m.gravity[2]};
        ca = zero3();
        for (int ie = 0; ie < E; ie++)
          if (l >= m.ent_link_start[ie] && l < m.ent_link_end[ie]) cv = cv * (1.f - m.ent_gravity_compensation[ie]);
      } else {
        cv = lds3(acc, 2 * pl);
        ca = lds3(acc, 2 * pl + 1);
      }
      for (int d = m.link_dof_start[l]; d < m.link_dof_end[l]; d++) {
        cv = cv + lds3(fv, d);
        ca = ca + lds3(fa, d);
      }
      set3(acc, 2 * l, cv);
      set3(acc, 2 * l + 1, ca);
    }
    __syncthreads();
  }
  // --- link forces (rsd:6284-6398) ---
  for (int l = lane; l < L; l += G) {
    float I[9];
    for (int k = 0; k < 9; k++) I[k] = crb[k * L + l];
    const f3 cp{crb[9 * L + l], crb[10 * L + l], crb[11 * L + l]};
    const float cm = crb[12 * L + l];
    f3 f1a, f1v, f2a, f2v, f3a, f3v;
    const f3 v = e.L3(s.cd_vel, l), a = e.L3(s.cd_ang, l);
    inertial_mul(cp, I, cm, lds3(acc, 2 * l), lds3(acc, 2 * l + 1), f1a, f1v);
    inertial_mul(cp, I, cm, v, a, f2a, f2v);
    motion_cross_force(a, v, f2a, f2v, f3a, f3v);
    // applied and coupling forces are zero on this path; their additions are kept for the same rounding
    const f3 fl = f1v + f3v + zero3() + zero3(), fg = f1a + f3a + zero3() + zero3();
    frc[l] = fl.x; frc[L + l] = fl.y; frc[2 * L + l] = fl.z;
    frc[3 * L + l] = fg.x; frc[4 * L + l] = fg.y; frc[5 * L + l] = fg.z;
  }
  __syncthreads();
  // --- composite inertias and forces up the tree, last link first, one component per lane ---
  for (int c = lane; c < 19; c += G) {
    lds_f* a = c < 13 ? crb + c * L : frc + (c - 13) * L;
    for (int k = 0; k < t.n_up; k++) {
      const int l = t.up[k], pl = t.par[l];
      a[pl] = a[pl] + a[l];
    }
  }
  __syncthreads();
  // --- composite forces per dof, bias force, actuation and total force ---
  for (int d = lane; d < D; d += G) {
    const int l = t.dlink[d];
    float I[9];
    for (int k = 0; k < 9; k++) I[k] = crb[k * L + l];
    f3 ga, gv;
    inertial_mul(f3{crb[9 * L + l], crb[10 * L + l], crb[11 * L + l]}, I, crb[12 * L + l], lds3(cdv, d), lds3(cda, d), ga, gv);
    set3(fa, d, ga);
    set3(fv, d, gv);
    // actuation and passive forces (rsd:5960-6177)
    const int dstart = m.link_dof_start[l], jt = m.joint_type[m.link_joint_start[l]];
    const int cm = e.I(s.ctrl_mode, d);
    const float kp = e.DP(m.dof_kp, d), kv = e.DP(m.dof_kv, d), vel = e.F(s.vel, d), pos = e.F(s.dofs_pos, d);
    const float damping = e.DP(m.dof_damping, d);
    float f = 0.f;
    if (jt == JOINT_FREE && d >= dstart + 3 && (e.I(s.ctrl_mode, dstart + 3) == CTRL_POSITION ||
                                                e.I(s.ctrl_mode, dstart + 4) == CTRL_POSITION ||
                                                e.I(s.ctrl_mode, dstart + 5) == CTRL_POSITION)) {
      const f3 xyz{e.F(s.dofs_pos, dstart + 3), e.F(s.dofs_pos, dstart + 4), e.F(s.dofs_pos, dstart + 5)};
      const f3 cxyz{e.F(s.ctrl_pos, dstart + 3), e.F(s.ctrl_pos, dstart + 4), e.F(s.ctrl_pos, dstart + 5)};
      const q4 qd = qrot_q(xyz_to_quat(cxyz), qinv(xyz_to_quat(xyz)));
      f = kp * comp(quat_to_rotvec(qd, EPS), d - dstart - 3) - kv * vel;
    } else if (cm == CTRL_FORCE) {
      f = e.F(s.ctrl_force, d);
    } else if (cm == CTRL_VELOCITY) {
      f = kv * (e.F(s.ctrl_vel, d) - vel);
    } else if (cm == CTRL_POSITION && !(jt == JOINT_FREE && d >= dstart + 3)) {
      f = kp * (e.F(s.ctrl_pos, d) - pos) + kv * (e.F(s.ctrl_vel, d) - vel);
    }
    const float applied = fminf(fmaxf(f, e.DP(m.dof_force_range, 2 * d)), e.DP(m.dof_force_range, 2 * d + 1));
    float passive = -damping * vel;
    if (jt != JOINT_FREE && jt != JOINT_FIXED) passive = passive + -pos * e.DP(m.dof_stiffness, d);
    // generalized bias force and total force (rsd:6425-6563)
    const f3 la{frc[3 * L + l], frc[4 * L + l], frc[5 * L + l]}, lv{frc[l], frc[L + l], frc[2 * L + l]};
    const float qb = dot(lds3(cda, d), la) + dot(lds3(cdv, d), lv);
    const float total = passive - qb + applied;
    e.F(s.qf_applied, d) = applied;
    e.F(s.qf_passive, d) = passive;
    e.F(s.qf_bias, d) = qb;
    e.F(s.force, d) = total;
    e.F(s.qf_smooth, d) = total;
    vec[d] = total;
  }
  __syncthreads();
  // --- mass matrix (rsd:3422-3678) with armature and the implicit damping of approximate_implicitfast ---
  for (int k = lane; k < t.n_tri; k += G) {
    const int i = t.tri[k] & 0xffff, j = t.tri[k] >> 16;
    const int st = single ? 0 : t.dst[i], n = single ? D : t.den[i] - st, off = single ? 0 : m.ent_mass_offset[m.dof_entity[i]];
    float v = (dot(lds3(fa, i), lds3(cda, j)) + dot(lds3(fv, i), lds3(cdv, j))) * m.mass_parent_mask[i * D + j];
    if (i == j) {
      v = v + e.DP(m.dof_armature, i);
      v = v + e.DP(m.dof_damping, i) * dt;
      const int cm = e.I(s.ctrl_mode, i);
      if (cm == CTRL_POSITION || cm == CTRL_VELOCITY) v = v + e.DP(m.dof_kv, i) * dt;
    }
    const int at = off + (i - st) * n + (j - st);
    ML[at] = v;
    e.F(s.mass_blk, at) = v;
    if (i != j) e.F(s.mass_blk, off + (j - st) * n + (i - st)) = v;
  }
  __syncthreads();
  // --- LDL^T (rsd:3697-3760): eliminating dof i updates the entries of the rows before it ---
  if (single) {
    for (int i = D - 1; i >= 0; i--) {
      lds_f* ri = ML + i * D;
      const float dinv = 1.f / ri[i];
#pragma unroll 2
      for (int k = lane; k < i * (i + 1) / 2; k += G) {
        const int j = t.tri[k] & 0xffff, c = t.tri[k] >> 16;
        const float a = ri[j] * dinv;
        ML[j * D + c] = ML[j * D + c] - a * ri[c];
      }
      __syncthreads();
      for (int d = lane; d <= i; d += G) {
        if (d == i) e.F(s.mass_D_inv, i) = dinv;
        ri[d] = d < i ? ri[d] * dinv : 1.f;
      }
      __syncthreads();
    }
  } else {
    // every entity's step k (its dof end - 1 - k) together
    for (int k = 0; k < m.max_entity_dofs; k++) {
      for (int q = lane; q < t.n_tri; q += G) {
        const int j = t.tri[q] & 0xffff, c = t.tri[q] >> 16;
        const int st = t.dst[j], en = t.den[j], i = en - 1 - k, n = en - st;
        if (j >= i) continue;
        const int off = m.ent_mass_offset[m.dof_entity[j]];
        const lds_f* ri = ML + off + (i - st) * n - st;
        const float a = ri[j] * (1.f / ri[i]);
        lds_f* o = ML + off + (j - st) * n + (c - st);
        *o = *o - a * ri[c];
      }
      __syncthreads();
      for (int d = lane; d < D; d += G) {
        const int st = t.dst[d], en = t.den[d], i = en - 1 - k, n = en - st;
        if (d > i || i < st) continue;
        lds_f* ri = ML + m.ent_mass_offset[m.dof_entity[d]] + (i - st) * n - st;
        const float dinv = 1.f / ri[i];
        if (d < i) ri[d] = ri[d] * dinv;
        else e.F(s.mass_D_inv, i) = dinv;
      }
      __syncthreads();
      for (int d = lane; d < D; d += G) {
        const int st = t.dst[d], en = t.den[d], n = en - st;
        if (d == en - 1 - k) ML[m.ent_mass_offset[m.dof_entity[d]] + (d - st) * n + (d - st)] = 1.f;
      }
    }
    __syncthreads();
  }
  for (int k = lane; k < t.n_tri; k += G) {
    const int i = t.tri[k] & 0xffff, j = t.tri[k] >> 16;
    const int st = single ? 0 : t.dst[i], n = single ? D : t.den[i] - st, off = single ? 0 : m.ent_mass_offset[m.dof_entity[i]];
    const int at = off + (i - st) * n + (j - st);
    e.F(s.mass_L_blk, at) = ML[at];
  }
  // --- M^-1 force (rsd:3932-4042) ---
  if (single && D <= (G == 64 ? 64 : 32)) {
    if constexpr (G == 64) tree_solve_64(e, ML, vec, D);
    else tree_solve_16(e, ML, vec, D);
    return;
  }
  for (int ie = lane; ie < E; ie += G) {
    const int st = m.ent_dof_start[ie], en = m.ent_dof_end[ie], n = en - st;
    const lds_f* B = ML + m.ent_mass_offset[ie];
    for (int i = n - 1; i >= 0; i--) {
      float o = vec[st + i];
      for (int j = i + 1; j < n; j++) o -= B[j * n + i] * vec[st + j];
      vec[st + i] = o;
    }
    for (int i = 0; i < n; i++) vec[st + i] = vec[st + i] * e.F(s.mass_D_inv, st + i);
    for (int i = 0; i < n; i++) {
      float o = vec[st + i];
      for (int j = 0; j < i; j++) o -= B[i * n + j] * vec[st + j];
      vec[st + i] = o;
    }
    for (int i = 0; i < n; i++) e.F(s.acc_smooth, st + i) = e.F(s.acc, st + i) = vec[st + i];
  }
}

// ---- kinematics ---------------------------------------------------------------------------------------------------
struct TreeLds {
  lds_f *pos, *quat, *com, *mass, *rcom, *cvel, *cda, *cdv, *vel, *jq, *jax, *q;
};
__device__ inline TreeLds tree_carve(const gsr_model& m, lds_f* p) {
  TreeLds t;
  const int L = m.n_links, D = m.n_dofs, J = m.n_joints;
  t.pos = p; p += 3 * L;
  t.quat = p; p += 4 * L;
  t.com = p; p += 3 * L;
  t.mass = p; p += L;
  t.rcom = p; p += 3 * L;
  t.cvel = p; p += 6 * L;
  t.cda = p; p += 3 * D;
  t.cdv = p; p += 3 * D;
  t.vel = p; p += D;
  t.jq = p; p += 7 * J;    // free: position and rotation; revolute and spherical: rotation; prismatic: displacement
  t.jax = p; p += 6 * J;   // joint anchors and axes in the world
  t.q = p;
  return t;
}

// link poses, COM and motion subspaces, geom poses and velocities from t.q and t.vel (dev_kinematics)
template <int G>
__device__ inline void tree_kinematics(const Env& e, const TreeTables& tt, const TreeLds& t) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const float EPS = m.eps;
  const int lane = threadIdx.x & (G - 1), L = m.n_links, levels = tt.levels;
  // --- the joints' own motion ---
  for (int j = lane; j < m.n_joints; j += G) {
    const int jt = m.joint_type[j], qs = m.joint_q_start[j], ds = m.joint_dof_start[j];
    lds_f* o = t.jq + 7 * j;
    if (jt == JOINT_FREE || jt == JOINT_SPHERICAL) {
      const int ro = jt == JOINT_FREE ? 3 : 0;
      const q4 q{t.q[qs + ro], t.q[qs + ro + 1], t.q[qs + ro + 2], t.q[qs + ro + 3]};
      const f3 xyz = quat_to_xyz(q, EPS);
      if (jt == JOINT_FREE)
        for (int k = 0; k < 3; k++) e.F(s.dofs_pos, ds + k) = t.q[qs + k];
      e.F(s.dofs_pos, ds + ro) = xyz.x;
      e.F(s.dofs_pos, ds + ro + 1) = xyz.y;
      e.F(s.dofs_pos, ds + ro + 2) = xyz.z;
      for (int k = 0; k < ro + 4; k++) o[k] = t.q[qs + k];
    } else if (jt == JOINT_REVOLUTE) {
      const float dp = t.q[qs] - m.qpos0[qs];
      e.F(s.dofs_pos, ds) = dp;
      const q4 q = rotvec_to_quat(T3(m.dof_motion_ang, ds) * dp, EPS);
      o[0] = q.w; o[1] = q.x; o[2] = q.y; o[3] = q.z;
    } else if (jt == JOINT_PRISMATIC) {
      const float dp = t.q[qs] - m.qpos0[qs];
      e.F(s.dofs_pos, ds) = dp;
      o[0] = dp;
    }
  }
  __syncthreads();
  // --- link poses, level by level; the constants of a lane's first link and of that link's first joint are loaded
  // before the loop ---
  const int l0 = lane < L ? lane : 0;
  const f3 lp0 = T3(m.link_pos, l0);
  const q4 lq0 = T4(m.link_quat, l0);
  const int j00 = m.link_joint_start[l0], j01 = m.link_joint_end[l0], fix0 = m.link_is_fixed[l0];
  const int jc = j00 < m.n_joints ? j00 : 0;
  const int jt0 = m.joint_type[jc], ds0 = m.joint_dof_start[jc];
  const f3 jp0 = T3(m.joint_pos, jc);
  f3 ax0{0.f, 0.f, 1.f};
  if (jt0 == JOINT_REVOLUTE) ax0 = T3(m.dof_motion_ang, ds0);
  else if (jt0 == JOINT_PRISMATIC) ax0 = T3(m.dof_motion_vel, ds0);
  for (int lev = 0; lev < levels; lev++) {
    for (int l = lane; l < L; l += G) {
      if (tt.dep[l] != lev) continue;
      const bool first = l == lane;
      const f3 lp = first ? lp0 : T3(m.link_pos, l);
      const q4 lq = first ? lq0 : T4(m.link_quat, l);
      const int ja = first ? j00 : m.link_joint_start[l], jb = first ? j01 : m.link_joint_end[l];
      f3 pos = lp;
      q4 quat = lq;
      const int par = tt.par[l];
      if (par != -1) {
        const q4 pq = lds4(t.quat, par);
        pos = lds3(t.pos, par) + qrot(lp, pq);
        quat = qrot_q(lq, pq);
      }
      for (int j = ja; j < jb; j++) {
        const bool pre = first && j == ja;
        const int jt = pre ? jt0 : m.joint_type[j], ds = pre ? ds0 : m.joint_dof_start[j];
        const lds_f* jq = t.jq + 7 * j;
        if (jt == JOINT_FREE) {
          pos = f3{jq[0], jq[1], jq[2]};
          quat = q4{jq[3], jq[4], jq[5], jq[6]};
          set3(t.jax, 2 * j, pos);
          set3(t.jax, 2 * j + 1, f3{0.f, 0.f, 1.f});
        } else if (jt != JOINT_FIXED) {
          const f3 jp = pre ? jp0 : T3(m.joint_pos, j);
          f3 axis{0.f, 0.f, 1.f};
          if (pre) axis = ax0;
          else if (jt == JOINT_REVOLUTE) axis = T3(m.dof_motion_ang, ds);
          else if (jt == JOINT_PRISMATIC) axis = T3(m.dof_motion_vel, ds);
          const f3 anchor = qrot(jp, quat) + pos, xaxis = qrot(axis, quat);
          set3(t.jax, 2 * j, anchor);
          set3(t.jax, 2 * j + 1, xaxis);
          if (jt == JOINT_PRISMATIC) {
            pos = pos + xaxis * jq[0];
          } else {
            quat = qrot_q(q4{jq[0], jq[1], jq[2], jq[3]}, quat);
            pos = anchor - qrot(jp, quat);
          }
        }
      }
      // fixed root links keep their build-time pose
      if (par == -1 && (first ? fix0 : m.link_is_fixed[l])) {
        pos = lp;
        quat = lq;
      }
      set3(t.pos, l, pos);
      set4(t.quat, l, quat);
    }
    __syncthreads();
  }
  for (int j = lane; j < m.n_joints; j += G)
    if (m.joint_type[j] != JOINT_FIXED) {
      e.S3(s.xanchor, j, lds3(t.jax, 2 * j));
      e.S3(s.xaxis, j, lds3(t.jax, 2 * j + 1));
    }
  // --- COM (func_COM_links): per link, then the roots' sums in link order ---
  for (int l = lane; l < L; l += G) {
    const f3 lp = lds3(t.pos, l);
    const q4 lq = lds4(t.quat, l);
    e.S3(s.links_pos, l, lp);
    e.S4(s.links_quat, l, lq);
    set3(t.com, l, lp + qrot(T3(m.link_inertial_pos, l) + e.L3(s.i_pos_shift, l), lq));
    t.mass[l] = e.LP(m.link_inertial_mass, l) + e.F(s.mass_shift, l);
  }
  __syncthreads();
  for (int l = lane; l < L; l += G) {
    if (tt.root[l] != l) continue;
    float mass = 0.f;
    f3 c = zero3();
    for (int k = 0; k < L; k++) {
      const float mk = t.mass[k];
      const f3 ck = mk * lds3(t.com, k);
      if (tt.root[k] == l) {
        mass = mass + mk;
        c = c + ck;
      }
    }
    set3(t.rcom, l, c / mass);
  }
  __syncthreads();
  for (int l = lane; l < L; l += G) {
    const f3 com = lds3(t.rcom, tt.root[l]);
    const q4 lq = lds4(t.quat, l);
    e.S3(s.root_com, l, com);
    const q4 iq = qrot_q(T4(m.link_inertial_quat, l), lq);
    e.S4(s.links_iquat, l, iq);
    const f3 r = lds3(t.com, l) - com;
    const float mass = t.mass[l];
    const float x = r.x, y = r.y, z = r.z;
    const float xx = x * x, xy = x * y, xz = x * z, yy = y * y, yz = y * z, zz = z * z;
    const float hhT[9] = {yy + zz, -xy, -xz, -xy, xx + zz, -yz, -xz, -yz, xx + yy};
    const m3 R = quat_to_R(iq, EPS);
    const float* I0 = m.link_inertial_i + 9 * l;
    float RI[9];
    for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) RI[3 * i + j] = R.a[3 * i] * I0[j] + R.a[3 * i + 1] * I0[3 + j] + R.a[3 * i + 2] * I0[6 + j];
    for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++) {
        const float v = RI[3 * i] * R.a[3 * j] + RI[3 * i + 1] * R.a[3 * j + 1] + RI[3 * i + 2] * R.a[3 * j + 2];
        e.F(s.cinr_inertial, 9 * l + 3 * i + j) = v + hhT[3 * i + j] * mass;
      }
    e.S3(s.cinr_pos, l, r * mass);
    e.F(s.cinr_mass, l) = mass;
    // motion subspaces of the link's joints
    if (m.link_dof_end[l] - m.link_dof_start[l] <= 0) continue;
    for (int j = m.link_joint_start[l]; j < m.link_joint_end[l]; j++) {
      const int jt = m.joint_type[j], ds = m.joint_dof_start[j];
      if (jt == JOINT_FIXED) continue;
      const f3 xaxis = lds3(t.jax, 2 * j + 1), off = com - lds3(t.jax, 2 * j);
      if (jt == JOINT_REVOLUTE) {
        set3(t.cda, ds, xaxis);
        set3(t.cdv, ds, cross(xaxis, off));
      } else if (jt == JOINT_PRISMATIC) {
        set3(t.cda, ds, zero3());
        set3(t.cdv, ds, xaxis);
      } else {
        const int ro = jt == JOINT_FREE ? 3 : 0;
        for (int i = 0; i < ro; i++) {
          set3(t.cda, ds + i, zero3());
          set3(t.cdv, ds + i, f3{i == 0 ? 1.f : 0.f, i == 1 ? 1.f : 0.f, i == 2 ? 1.f : 0.f});
        }
        const m3 Rl = quat_to_R(lq, EPS);
        for (int i = 0; i < 3; i++) {
          const f3 c = mcol(Rl, i);  // row i of R^T
          set3(t.cda, ds + ro + i, c);
          set3(t.cdv, ds + ro + i, cross(c, off));
        }
      }
    }
  }
  __syncthreads();
  for (int k = lane; k < 3 * m.n_dofs; k += G) {
    e.F(s.cdof_ang, k) = t.cda[k];
    e.F(s.cdof_vel, k) = t.cdv[k];
  }
  // --- geom poses ---
  for (int g = lane; g < m.n_geoms; g += G) {
    const int l = m.geom_link[g];
    const q4 lq = lds4(t.quat, l);
    e.S3(s.geoms_pos, g, lds3(t.pos, l) + qrot(T3(m.geom_pos, g), lq));
    e.S4(s.geoms_quat, g, qrot_q(T4(m.geom_quat, g), lq));
  }
  // --- velocities, level by level ---
  for (int lev = 0; lev < levels; lev++) {
    for (int l = lane; l < L; l += G) {
      if (tt.dep[l] != lev) continue;
      f3 cv = zero3(), ca = zero3();
      const int par = tt.par[l];
      if (par != -1) {
        cv = lds3(t.cvel, 2 * par);
        ca = lds3(t.cvel, 2 * par + 1);
      }
      for (int j = m.link_joint_start[l]; j < m.link_joint_end[l]; j++) {
        const int jt = m.joint_type[j], ds = m.joint_dof_start[j], de = m.joint_dof_end[j];
        int d0 = ds;
        if (jt == JOINT_FREE) {
          for (; d0 < ds + 3; d0++) {
            const float v = t.vel[d0];
            cv = cv + lds3(t.cdv, d0) * v;
            ca = ca + lds3(t.cda, d0) * v;
            e.S3(s.cdofd_ang, d0, zero3());
            e.S3(s.cdofd_vel, d0, zero3());
          }
        }
        const int d1 = jt == JOINT_FREE ? ds + 6 : de;
        for (int d = d0; d < d1; d++) {
          f3 oa, ov;
          motion_cross_motion(ca, cv, lds3(t.cda, d), lds3(t.cdv, d), oa, ov);
          e.S3(s.cdofd_ang, d, oa);
          e.S3(s.cdofd_vel, d, ov);
        }
        for (int d = d0; d < d1; d++) {
          const float v = t.vel[d];
          cv = cv + lds3(t.cdv, d) * v;
          ca = ca + lds3(t.cda, d) * v;
        }
      }
      set3(t.cvel, 2 * l, cv);
      set3(t.cvel, 2 * l + 1, ca);
    }
    __syncthreads();
  }
  for (int l = lane; l < L; l += G) {
    e.S3(s.cd_vel, l, lds3(t.cvel, 2 * l));
    e.S3(s.cd_ang, l, lds3(t.cvel, 2 * l + 1));
  }
}

// kinematics of the env's present positions and velocities
template <int G>
__device__ inline void tree_refresh(const Env& e, const TreeTables& tt, lds_f* p) {
  const TreeLds t = tree_carve(e.m, p);
  const int lane = threadIdx.x & (G - 1);
  for (int q = lane; q < e.m.n_qs; q += G) t.q[q] = e.F(e.s.qpos, q);
  for (int d = lane; d < e.m.n_dofs; d += G) t.vel[d] = e.F(e.s.vel, d);
  __syncthreads();
  tree_kinematics<G>(e, tt, t);
}

// step_2: integration with the NaN-guarded commit (dev_integrate), then the kinematics of the new pose
template <int G>
__device__ inline void tree_step2(const Env& e, const TreeTables& tt, lds_f* p) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const int lane = threadIdx.x & (G - 1);
  const float dt = m.dt;
  const TreeLds t = tree_carve(m, p);
  bool valid = true;
  for (int q = lane; q < m.n_qs; q += G) t.q[q] = e.F(s.qpos, q);
  for (int d = lane; d < m.n_dofs; d += G) {
    const float v = e.F(s.vel, d) + e.F(s.acc, d) * dt;
    t.vel[d] = v;
    valid &= !isnan(v);
  }
  __syncthreads();
  for (int l = lane; l < m.n_links; l += G) {
    const int ds = m.link_dof_start[l], qs = m.link_q_start[l], qe = m.link_q_end[l];
    if (m.link_dof_end[l] - ds <= 0) continue;
    const int jt = m.joint_type[m.link_joint_start[l]];
    if (jt == JOINT_SPHERICAL || jt == JOINT_FREE) {
      const int ro = jt == JOINT_FREE ? 3 : 0;
      for (int j = 0; j < ro; j++) t.q[qs + j] = t.q[qs + j] + t.vel[ds + j] * dt;
      const q4 rot0{t.q[qs + ro], t.q[qs + ro + 1], t.q[qs + ro + 2], t.q[qs + ro + 3]};
      const f3 ang = f3{t.vel[ds + ro], t.vel[ds + ro + 1], t.vel[ds + ro + 2]} * dt;
      const q4 rot = qrot_q(rotvec_to_quat(ang, m.eps), rot0);  // normalize(rot0 * qrot)
      t.q[qs + ro] = rot.w;
      t.q[qs + ro + 1] = rot.x;
      t.q[qs + ro + 2] = rot.y;
      t.q[qs + ro + 3] = rot.z;
    } else {
      for (int j = 0; j < qe - qs; j++) t.q[qs + j] = t.q[qs + j] + t.vel[ds + j] * dt;
    }
    for (int q = qs; q < qe; q++) valid &= !isnan(t.q[q]);
  }
  __syncthreads();
  // NaN anywhere in the env: a set bit among its G lanes
  const unsigned long long mine = (G == kWave ? ~0ull : ((1ull << (G & 63)) - 1ull)) << (threadIdx.x & ~(G - 1));
  if ((__ballot(!valid) & mine) == 0ull) {
    for (int q = lane; q < m.n_qs; q += G) e.F(s.qpos, q) = t.q[q];
    for (int d = lane; d < m.n_dofs; d += G) e.F(s.vel, d) = t.vel[d];
  } else {
    if (lane == 0) e.I((int32_t*)s.errno_env, 0) |= (int)GSR_ERR_NAN_STATE;
    for (int q = lane; q < m.n_qs; q += G) t.q[q] = e.F(s.qpos, q);
    for (int d = lane; d < m.n_dofs; d += G) t.vel[d] = e.F(s.vel, d);
  }
  __syncthreads();
  tree_kinematics<G>(e, tt, t);
}

// LDS words of the workgroup's env `sub`, after the tables
__device__ __forceinline__ lds_f* tree_words(const gsr_model& m, char* lds, int sub) {
  return reinterpret_cast<lds_f*>((lds_c*)lds) + tree_table_words(m.n_links, m.n_dofs, m.mass_blk_size) + sub * tree_env_words(m);
}
// the env of this lane's group among those of workgroup `blk`, and its LDS words; false past the last of n envs
template <int G>
__device__ __forceinline__ bool tree_env(const gsr_model& m, int blk, int n, char* lds, int& k, lds_f*& p) {
  const int sub = threadIdx.x / G;
  k = xcd_env(blk, (n + kWave / G - 1) / (kWave / G)) * (kWave / G) + sub;
  p = tree_words(m, lds, sub);
  return k < n;
}

}  // namespace gsr
