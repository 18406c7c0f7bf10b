// Newton solver of models whose entities have six dofs or none, kWaves wavefronts per env: free bodies, and arms of six
// joints, which are "bodies" below as well.
//
// Same algorithm as the other solvers (func_init_solver / func_solve / func_linesearch / rank-1 Cholesky updates of
// constraint_solver_decomp.py). A heap couples its bodies through contacts, so the Hessian is a sparse matrix of 6 x 6
// blocks; what bounds the solve is the latency of its dependent steps, and a heap of 64 boxes fills a quarter of a CU's
// LDS, so one wavefront per env left every SIMD with a single wave. Here
//   * an env has one, two or four wavefronts (bodies_waves); rows and dofs are dealt to all of them, the bodies of an
//     elimination level to its wavefronts; the elimination order, the substitutions and the rank-1 updates, chains of
//     short steps, run on the first without barriers;
//   * dof d belongs to body d / 6 and a row holds its bodies' six entries side by side, so no index is looked up: J^T f
//     and J^T D J read a row's entries at (row, first or second half + d mod 6); rows that hold fewer entries
//     (frictionloss, JOINT equalities, a part of an arm's chain) are first filled up with zeros;
//   * forces, weights, Jaref and the line search's terms of the first kBodyRows rows a thread stay in registers; the
//     forces (then the active rows' weights) lie in LDS for the lanes that walk a body's rows;
//   * blocks lie whole in LDS, so a row is read with three wide loads and a block with nine; a rank-1 update keeps a
//     body's columns in registers and passes the pivots between lanes as scalars;
//   * the elimination order (minimum degree), its levels and the layout are computed with one body a lane and ballots
//     instead of by one lane.
// No sum depends on the number of wavefronts: FP32 sums keep the order of the entity-block solver, sums in double are
// taken over 64 rows at a time into four classes (64-row block modulo 4) that are added in order. So the fused launch
// (one wavefront) and the plain step (several) give the same bits.
//
// Measured (MI355X, the solve of one step, entity-block solver -> this one, us): 100 envs of 7 boxes 217 -> 114, 1,500 of
// 20 boxes 1,231 -> 495, 96 of 64 boxes 6,059 -> 1,588, 4,096 of 64 boxes 22,890 -> 7,070.
#pragma once
#include "rigid_env.h"
#include "rigid_solver_wave.h"

namespace gsr {

constexpr int kBodyRows = 4;     // rows per thread whose scalars stay in registers
constexpr int kMaxBodies = 128;  // two 64-bit words per pattern row, two bodies per lane
constexpr int kBlk = 36;         // floats of a 6 x 6 block
constexpr int kDiaLds = 24, kDiaMem = 21;  // floats from one diagonal block's lower triangle to the next

// rows whose force and weight have a place in LDS: three a dof (a settled heap has 2.5 to 2.8)
__host__ __device__ inline int bodies_lds_rows(int D) { return (3 * D + 63) & ~63; }
__host__ __device__ inline size_t bodies_lds_bytes(int D, int H) {
  const int nb = D / 6;
  return sizeof(float) * (size_t)(6 * D + ((H + 3) & ~3) + bodies_lds_rows(D)) + 16 * (size_t)nb + 8 * 32 +
         sizeof(int) * (size_t)(12 * nb + 16 + 2 * (H / kBlk)) + 32;
}
// every entity has six dofs or none (sum of squares = 6 x sum), a row has room for all entries of its bodies, and the
// Hessian's budget leaves room for the rest (the entity-block solver needs less beside it)
__host__ __device__ inline bool bodies_solver(const gsr_model& m) {
  return m.n_dofs > 0 && m.max_entity_dofs == 6 && m.mass_blk_size == 6 * m.n_dofs && m.n_dofs <= 6 * kMaxBodies &&
         m.row_width == (m.n_dofs == 6 ? 6 : 12) && m.max_rows < (1 << 20) &&
         bodies_lds_bytes(m.n_dofs, m.wave_h_floats) <= kMaxSolveLds;
}

// Wavefronts per env of the plain step's solve: two up to 128 dofs, four above. Measured (us a pass of three steps at
// 1,500 envs of 20 boxes, four at 100 envs of 7, two at 4,096 envs of 64) with one, two, four: 20 boxes 3690, 3318, 3960;
// 7 boxes 1395, 1333, -; 64 boxes -, 27830, 25206.
__host__ __device__ inline int bodies_waves(int D) { return D <= 128 ? 2 : 4; }

struct BodyLds {
  lds_f *vec, *hl, *row, *qacc, *Ma, *search, *mv, *qfrc;
  lds_u64* pat;     // [nb][2] factor space: the bodies sharing a block with the one at each position, and itself
  GSR_LDS double* red;  // [2][4][4] sums of the four classes, two buffers
  lds_i *vof;           // position of each body
  lds_i *hb;            // blocks before each position's first
  lds_i *flv, *fst;     // positions by forward level, first of each level: position | neighbours before << 8 | hb << 16
  lds_i *rlv, *rst;     // the same by backward level, with the neighbours after and the first of them in cl
  lds_i *rl, *cl;       // blocks in LDS: earlier position of each; later neighbours of each position | their block << 8
  lds_i *ptr;           // [nb + 1] row list of each body
  lds_i *cnt;           // [4][nb] rows of each body in each wavefront's share
  lds_i *misc;          // levels forward, backward; 1 = blocks in LDS
};
__device__ inline BodyLds bodies_carve(char* lds, int D, int H) {
  BodyLds L;
  const int nb = D / 6;
  lds_f* f = reinterpret_cast<lds_f*>((lds_c*)lds);
  L.hl = f; f += (H + 3) & ~3;
  L.row = f; f += bodies_lds_rows(D);
  L.vec = f; f += D;
  L.qacc = f; f += D;
  L.Ma = f; f += D;
  L.search = f; f += D;
  L.mv = f; f += D;
  L.qfrc = f; f += D;
  L.red = reinterpret_cast<GSR_LDS double*>(f);  // 6 D floats and multiples of four before it: 8-byte aligned
  L.pat = reinterpret_cast<lds_u64*>(L.red + 32);
  L.vof = reinterpret_cast<lds_i*>(L.pat + 2 * nb);
  L.hb = L.vof + nb;
  L.flv = L.hb + nb;
  L.fst = L.flv + nb;
  L.rlv = L.fst + nb + 1;
  L.rst = L.rlv + nb;
  L.ptr = L.rst + nb + 1;
  L.cnt = L.ptr + nb + 1;
  L.misc = L.cnt + 4 * nb;
  L.rl = L.misc + 8;
  L.cl = L.rl + H / kBlk;
  return L;
}

template <int kWaves>
struct BodyCtx {
  static constexpr int kThreads = kWave * kWaves;
  const Env& e;
  const BodyLds& L;
  int tid, lane, wv, D, nb, n_con, ne, nef, n_lds;  // n_lds: rows with a place in LDS
  int& flip;
  __device__ __forceinline__ void sync() const { __syncthreads(); }
};

// N sums over the env of doubles that each thread holds per class it serves (class k of wavefront wv: wv + kWaves k),
// the classes' sums added in order; items: how many items were summed (classes past them are empty)
template <int kWaves, int N>
__device__ __forceinline__ void bodies_sum(const BodyCtx<kWaves>& w, int items, const double (&a)[N][4 / kWaves],
                                           double (&out)[N]) {
  constexpr int K = 4 / kWaves;
  if constexpr (kWaves == 1) {
    for (int n = 0; n < N; n++) {
      double s[4];
#pragma unroll
      for (int k = 0; k < 4; k++) s[k] = kWave * k < items ? wave_sum_d(a[n][k]) : 0.0;
      out[n] = (s[0] + s[1]) + (s[2] + s[3]);
    }
  } else {
    GSR_LDS double* r = w.L.red + 16 * w.flip;
    w.flip ^= 1;
#pragma unroll
    for (int n = 0; n < N; n++)
#pragma unroll
      for (int k = 0; k < K; k++) {
        const int c = w.wv + kWaves * k;
        const double s = kWave * c < items ? wave_sum_d(a[n][k]) : 0.0;
        if (w.lane == 0) r[4 * n + c] = s;
      }
    w.sync();
#pragma unroll
    for (int n = 0; n < N; n++) out[n] = (r[4 * n] + r[4 * n + 1]) + (r[4 * n + 2] + r[4 * n + 3]);
  }
}

// ---- rows -----------------------------------------------------------------------------------------------------------
// Bodies of row c (the second << 8). A row that does not store all six entries of its bodies (frictionloss, JOINT
// equalities, a part of an arm's chain) is rewritten with zeros in the places that lack, so that every row holds body a's entries first and, if it
// has two bodies, b's after them. A row without an entry (an equality between two fixed links) is counted to body 0, with
// six zeros.
__device__ inline int body_row(const Env& e, int c) {
  const int nnz = e.EI(e.s.jac_nnz, c);
  const int a = nnz > 0 ? e.JI(c, 0) / 6 : 0, b = nnz > 0 ? e.JI(c, nnz - 1) / 6 : 0;
  if (nnz != (a == b ? 6 : 12)) {
    float v[12];
#pragma unroll
    for (int k = 0; k < 12; k++) v[k] = 0.f;
    for (int q = 0; q < nnz; q++) {
      const int d = e.JI(c, q), at = d - 6 * a < 6 ? d - 6 * a : 6 + d - 6 * b;
      const float x = e.JV(c, q);
#pragma unroll
      for (int k = 0; k < 12; k++)
        if (at == k) v[k] = x;
    }
#pragma unroll
    for (int k = 0; k < 12; k++)
      if (k < (a == b ? 6 : 12)) {
        e.JV(c, k) = v[k];
        e.JI(c, k) = k < 6 ? 6 * a + k : 6 * b + k - 6;
      }
    e.EI(e.s.jac_nnz, c) = a == b ? 6 : 12;
  }
  return a | (b << 8);
}
// sum_k J[c, k] x[dof k] in entry order, from acc
__device__ __forceinline__ float body_row_dot(const Env& e, int c, int ent, float acc, const lds_f* x) {
  const int a = ent & 0xff, b = ent >> 8;
  const float* pv = &e.JV(c, 0);
  const lds_f* xa = x + 6 * a;
  const lds_f* xb = x + 6 * b;
  float v[12];
#pragma unroll
  for (int k = 0; k < 6; k++) v[k] = pv[k];
#pragma unroll
  for (int k = 6; k < 12; k++) v[k] = a != b ? pv[k] : 0.f;
#pragma unroll
  for (int k = 0; k < 6; k++) acc += v[k] * xa[k];
  if (a != b) {
#pragma unroll
    for (int k = 0; k < 6; k++) acc += v[6 + k] * xb[k];
  }
  return acc;
}

struct BodyRow {
  float Dc, ja, jv, q0, q1, q2;
  int act, ent;  // act: bit 0 active, bit 1 active before the last update
};

// M x of dof d (serial over the body's six)
__device__ __forceinline__ float body_mass_mul(const Env& e, int d, const lds_f* x) {
  const int b6 = d / 6 * 6;
  float v = 0.f;
#pragma unroll
  for (int j = 0; j < 6; j++) v += e.F(e.s.mass_blk, 6 * d + j) * x[b6 + j];
  return v;
}

typedef int i4 __attribute__((ext_vector_type(4)));

// ---- structure: elimination order, levels, block layout, row lists -------------------------------------------------
__device__ __forceinline__ unsigned long long low_mask(int n) { return n >= 64 ? ~0ull : n <= 0 ? 0ull : (1ull << n) - 1ull; }

// index of block (v, u), u < v a neighbour of v: the blocks of v before it
__device__ __forceinline__ int blk_index(const BodyLds& L, int v, int u) {
  const unsigned long long p0 = L.pat[2 * v], p1 = L.pat[2 * v + 1];
  return L.hb[v] + __popcll(p0 & low_mask(u)) + __popcll(p1 & low_mask(u - 64));
}

// one body per lane (and lane + 64) on the env's first wavefront; pat holds the contact graph in model numbering
__device__ inline void bodies_order(const BodyLds& L, int lane, int nb, int h_floats) {
  unsigned long long adj[2][2];
  bool has[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int b = lane + 64 * h;
    has[h] = b < nb;
    adj[h][0] = has[h] ? L.pat[2 * b] : 0ull;
    adj[h][1] = has[h] ? L.pat[2 * b + 1] : 0ull;
  }
  // minimum degree over the bodies left (ties: the lower index); eliminating one joins its neighbours
  unsigned long long al0 = __ballot(has[0]), al1 = __ballot(has[1]);
  if (nb <= 64) {  // one word, one body a lane
    for (int step = 0; step < nb; step++) {
      const int k = (al0 >> lane) & 1ull ? (__popcll(adj[0][0] & al0) << 8) | lane : 0x7fffffff;
      const int v = __builtin_amdgcn_readfirstlane(wave_min_i(k)) & 0xff;
      al0 &= ~(1ull << v);
      const unsigned long long n0 = lane_value(adj[0][0], v) & al0;
      if ((n0 >> lane) & 1ull) adj[0][0] |= n0 & ~(1ull << lane);
      if (lane == v) L.vof[lane] = step;
    }
  } else {
    for (int step = 0; step < nb; step++) {
      int k = 0x7fffffff;
      if ((al0 >> lane) & 1ull) k = ((__popcll(adj[0][0] & al0) + __popcll(adj[0][1] & al1)) << 8) | lane;
      if ((al1 >> lane) & 1ull) k = min(k, ((__popcll(adj[1][0] & al0) + __popcll(adj[1][1] & al1)) << 8) | (lane + 64));
      const int v = __builtin_amdgcn_readfirstlane(wave_min_i(k)) & 0xff, src = v & 63;
      unsigned long long n0 = lane_value(v < 64 ? adj[0][0] : adj[1][0], src);
      unsigned long long n1 = lane_value(v < 64 ? adj[0][1] : adj[1][1], src);
      if (v < 64) al0 &= ~(1ull << v); else al1 &= ~(1ull << (v - 64));
      n0 &= al0;
      n1 &= al1;
      if ((n0 >> lane) & 1ull) { adj[0][0] |= n0 & ~(1ull << lane); adj[0][1] |= n1; }
      if ((n1 >> lane) & 1ull) { adj[1][0] |= n0; adj[1][1] |= n1 & ~(1ull << lane); }
      if (lane == 0) {
        L.vof[v] = step;
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  // pattern rows in factor space
#pragma unroll
  for (int h = 0; h < 2; h++) {
    if (!has[h]) continue;
    const int vi = L.vof[lane + 64 * h];
    unsigned long long r0 = vi < 64 ? 1ull << vi : 0ull, r1 = vi < 64 ? 0ull : 1ull << (vi - 64);
#pragma unroll
    for (int word = 0; word < 2; word++) {
      unsigned long long t = adj[h][word];
      while (t) {
        const int vx = L.vof[word * 64 + __ffsll((long long)t) - 1];
        t &= t - 1;
        if (vx < 64) r0 |= 1ull << vx; else r1 |= 1ull << (vx - 64);
      }
    }
    L.pat[2 * vi] = r0;
    L.pat[2 * vi + 1] = r1;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  unsigned long long p[2][2];
  int np[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int v = lane + 64 * h;
    p[h][0] = has[h] ? L.pat[2 * v] : 0ull;
    p[h][1] = has[h] ? L.pat[2 * v + 1] : 0ull;
    np[h] = has[h] ? __popcll(p[h][0] & low_mask(v)) + __popcll(p[h][1] & low_mask(v - 64)) : 0;
  }
  // blocks before each position, and the same count by columns
  int total = 0, ctotal = 0, hb[2], cb[2], ns[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    ns[h] = has[h] ? __popcll(p[h][0]) + __popcll(p[h][1]) - 1 - np[h] : 0;
    int x = np[h] | (ns[h] << 16);
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    hb[h] = total + (x & 0xffff) - np[h];
    cb[h] = ctotal + (x >> 16) - ns[h];
    if (has[h]) L.hb[lane + 64 * h] = hb[h];
    const int all = lane_value(x, 63);
    total += all & 0xffff;
    ctotal += all >> 16;
  }
  const bool in_lds = total * kBlk + nb * kDiaLds <= h_floats;
  if (in_lds) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int h = 0; h < 2; h++) {
      if (!has[h]) continue;
      const int v = lane + 64 * h;
      int at = hb[h], to = cb[h];
#pragma unroll
      for (int word = 0; word < 2; word++) {
        unsigned long long t = p[h][word];
        while (t) {
          const int u = word * 64 + __ffsll((long long)t) - 1;
          t &= t - 1;
          if (u < v) L.rl[at++] = u;
          else if (u > v) L.cl[to++] = u | (blk_index(L, u, v) << 8);
        }
      }
    }
  }
  // levels: a position is ready once every earlier (later) position it shares a block with is done
  for (int back = 0; back < 2; back++) {
    lds_i* order = back ? L.rlv : L.flv;
    lds_i* first = back ? L.rst : L.fst;
    unsigned long long d0 = 0ull, d1 = 0ull;
    int n_done = 0, lev = 0;
    bool done[2] = {!has[0], !has[1]};
    while (n_done < nb) {
      bool ready[2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int v = lane + 64 * h;
        const unsigned long long m0 = back ? ~low_mask(v + 1) : low_mask(v), m1 = back ? ~low_mask(v + 1 - 64) : low_mask(v - 64);
        ready[h] = !done[h] && (p[h][0] & m0 & ~d0) == 0ull && (p[h][1] & m1 & ~d1) == 0ull;
      }
      const unsigned long long r0 = __ballot(ready[0]), r1 = __ballot(ready[1]);
      if (lane == 0) first[lev] = n_done;
      if (ready[0]) order[n_done + __popcll(r0 & low_mask(lane))] = lane | (back ? ns[0] << 8 | cb[0] << 16 : np[0] << 8 | hb[0] << 16);
      if (ready[1])
        order[n_done + __popcll(r0) + __popcll(r1 & low_mask(lane))] =
            (lane + 64) | (back ? ns[1] << 8 | cb[1] << 16 : np[1] << 8 | hb[1] << 16);
      done[0] |= ready[0];
      done[1] |= ready[1];
      d0 |= r0;
      d1 |= r1;
      n_done += __popcll(r0) + __popcll(r1);
      lev++;
    }
    if (lane == 0) {
      first[lev] = nb;
      L.misc[back] = lev;
    }
  }
  if (lane == 0) L.misc[2] = in_lds ? 1 : 0;
}

template <int kWaves>
__device__ inline void bodies_structure(const BodyCtx<kWaves>& w) {
  constexpr int NT = BodyCtx<kWaves>::kThreads;
  const Env& e = w.e;
  const BodyLds& L = w.L;
  const int nb = w.nb;
  int* rent = e.s.efc_ent + (size_t)e.b * e.m.max_rows;
  lds_i* rows = reinterpret_cast<lds_i*>(L.row);
  for (int i = w.tid; i < 2 * nb; i += NT) L.pat[i] = 0ull;
  w.sync();
  for (int c = w.tid; c < w.n_con; c += NT) {
    const int r = body_row(e, c), a = r & 0xff, b = r >> 8;
    rent[c] = r;
    if (c < w.n_lds) rows[c] = r;
    if (a != b) {
      atomicOr((unsigned long long*)&L.pat[2 * a + (b >> 6)], 1ull << (b & 63));
      atomicOr((unsigned long long*)&L.pat[2 * b + (a >> 6)], 1ull << (a & 63));
    }
  }
  w.sync();
  if (w.wv == 0) bodies_order(L, w.lane, nb, e.m.wave_h_floats);
  // row lists: each wavefront takes a share of the rows, each lane a body (and body + 64); the rows of a body in
  // ascending order, counted first
  const int share = ((w.n_con + kWaves - 1) / kWaves + 3) & ~3, r0 = min(w.wv * share, w.n_con), r1 = min(r0 + share, w.n_con);
  int* lst = e.s.ent_row_list + (size_t)e.b * 2 * e.m.max_rows;
  int n[2] = {0, 0};
  // f(row, its bodies) for the wavefront's rows in order, four read at a time from LDS
  auto each_row = [&](auto f) {
    const int in_lds = min(r1, w.n_lds);
    int c = r0;
    i4 next = c < in_lds ? *reinterpret_cast<const GSR_LDS i4*>(rows + c) : i4{0, 0, 0, 0};
    for (; c < in_lds; c += 4) {
      const i4 x = next;
      if (c + 4 < in_lds) next = *reinterpret_cast<const GSR_LDS i4*>(rows + c + 4);
      f(c, x.x);
      if (c + 1 < r1) f(c + 1, x.y);
      if (c + 2 < r1) f(c + 2, x.z);
      if (c + 3 < r1) f(c + 3, x.w);
    }
    for (; c < r1; c++) f(c, rent[c]);
  };
  each_row([&](int, int r) {
    const int a = r & 0xff, b = r >> 8;
    n[0] += (a == w.lane) | (b == w.lane);
    if (nb > 64) n[1] += (a == w.lane + 64) | (b == w.lane + 64);
  });
#pragma unroll
  for (int h = 0; h < 2; h++)
    if (w.lane + 64 * h < nb) L.cnt[w.wv * nb + w.lane + 64 * h] = n[h];
  w.sync();
  int at[2], base = 0;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int b = w.lane + 64 * h;
    int all = 0, before = 0;
    if (b < nb)
      for (int q = 0; q < kWaves; q++) {
        const int k = L.cnt[q * nb + b];
        if (q < w.wv) before += k;
        all += k;
      }
    int x = all;
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (w.lane >= o) x += y;
    }
    at[h] = base + x - all + before;
    if (w.wv == 0 && b < nb) L.ptr[b] = base + x - all;
    base += lane_value(x, 63);
  }
  if (w.tid == 0) L.ptr[nb] = base;
  // entry: row | 1 << 20 where the body's entries are the row's second six | the row's other body (or itself) << 21
  each_row([&](int c, int r) {
    const int a = r & 0xff, b = r >> 8;
    const int xa = c | b << 21, xb = c | 1 << 20 | a << 21;
    if ((a == w.lane) | (b == w.lane)) lst[at[0]++] = a == w.lane ? xa : xb;
    if (nb > 64 && ((a == w.lane + 64) | (b == w.lane + 64))) lst[at[1]++] = a == w.lane + 64 ? xa : xb;
  });
  w.sync();
}

// ---- constraint update ----------------------------------------------------------------------------------------------
__device__ __forceinline__ void body_row_state(const Env& e, int c, int ne, int nef, float ja, float Dc, int& act, float& force,
                                               double& ci) {
  const gsr_state& s = e.s;
  int a = 1;
  float floss_force = 0.f;
  if (ne <= c && c < nef) {
    const float f = e.EF(s.efc_fl, c), r = e.EF(s.efc_diag, c), rf = r * f;
    const bool ln = ja <= -rf, lp = ja >= rf;
    a = !(ln || lp);
    floss_force = (float)ln * f + (float)lp * -f;
    float fc = (float)ln * f * (-0.5f * rf - ja);
    fc += (float)lp * f * (-0.5f * rf + ja);
    ci += (double)fc;
  } else if (nef <= c) {
    a = ja < 0.f;
  }
  act = a | ((act & 1) << 1);
  force = floss_force + (-ja * Dc * (float)a);
  ci += (double)(0.5f * (ja * ja * Dc * (float)a));
}

template <int kWaves>
__device__ inline void bodies_update_constraint(const BodyCtx<kWaves>& w, BodyRow (&r)[kBodyRows], double& cost, float& gauss) {
  constexpr int NT = BodyCtx<kWaves>::kThreads, K = 4 / kWaves;
  const Env& e = w.e;
  const gsr_state& s = e.s;
  const BodyLds& L = w.L;
  double a[2][K];
#pragma unroll
  for (int k = 0; k < K; k++) a[0][k] = a[1][k] = 0.0;
#pragma unroll
  for (int q = 0; q < kBodyRows; q++) {
    const int c = w.tid + NT * q;
    if (c < w.n_con) {
      float f;
      double ci = 0.0;
      body_row_state(e, c, w.ne, w.nef, r[q].ja, r[q].Dc, r[q].act, f, ci);
      a[0][q % K] += ci;
      e.EF(s.efc_force, c) = f;
      if (c < w.n_lds) L.row[c] = f;
    }
  }
  for (int c = w.tid + NT * kBodyRows, q = kBodyRows; c < w.n_con; c += NT, q++) {
    float f;
    int act = e.EI(s.efc_active, c);
    double ci = 0.0;
    body_row_state(e, c, w.ne, w.nef, e.EF(s.efc_Jaref, c), e.EF(s.efc_D, c), act, f, ci);
#pragma unroll
    for (int k = 0; k < K; k++)
      if (q % K == k) a[0][k] += ci;
    e.EI(s.efc_active, c) = act;
    e.EF(s.efc_force, c) = f;
    if (c < w.n_lds) L.row[c] = f;
  }
  w.sync();
  // J^T f, one dof a lane: its body's rows in ascending order, four loaded at a time
  const int* lst = e.s.ent_row_list + (size_t)e.b * 2 * e.m.max_rows;
  const int W = e.m.row_width;
  const float* jv = &e.JV(0, 0);
  for (int d = w.tid, q = 0; d < w.D; d += NT, q++) {
    const int b = d / 6, dr = d - 6 * b, t1 = L.ptr[b + 1];
    float acc = 0.f;
    int x[4];
    int t = L.ptr[b];
#pragma unroll
    for (int k = 0; k < 4; k++) x[k] = t + k < t1 ? lst[t + k] : 0;
    for (; t < t1; t += 4) {
      float f[4], v[4];
      int y[4];
#pragma unroll
      for (int k = 0; k < 4; k++) y[k] = t + 4 + k < t1 ? lst[t + 4 + k] : 0;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int c = x[k] & 0xfffff;
        v[k] = jv[c * W + ((x[k] >> 20) & 1) * 6 + dr];
        f[k] = c < w.n_lds ? L.row[c] : e.EF(s.efc_force, c);
      }
#pragma unroll
      for (int k = 0; k < 4; k++) {
        if (t + k >= t1) continue;
        // a zero force adds +-0 to a sum that starts at +0 and so never holds -0: skipping a row changes no bit
        if (f[k] != 0.f) acc = acc + v[k] * f[k];
      }
#pragma unroll
      for (int k = 0; k < 4; k++) x[k] = y[k];
    }
    L.qfrc[d] = acc;
    const float g = 0.5f * (L.Ma[d] - e.F(s.force, d)) * (L.qacc[d] - e.F(s.acc_smooth, d));
#pragma unroll
    for (int k = 0; k < K; k++)
      if (q % K == k) a[1][k] += (double)g;
  }
  double out[2];
  bodies_sum<kWaves, 2>(w, max(w.n_con, w.D), a, out);
  gauss = (float)out[1];
  cost = out[0] + out[1];
}

// ---- Hessian blocks -------------------------------------------------------------------------------------------------
struct BlocksLds {
  typedef lds_f* ptr;
  static constexpr int kDia = kDiaLds;
  static constexpr bool kLists = true;  // L.rl and L.cl hold the blocks' bodies
  lds_f* p;
  int nb;
  __device__ __forceinline__ lds_f* dia(int v) const { return p + v * kDia; }
  __device__ __forceinline__ lds_f* blk(int i) const { return p + nb * kDia + i * kBlk; }
};
struct BlocksMem {
  typedef float* ptr;
  static constexpr int kDia = kDiaMem;
  static constexpr bool kLists = false;
  float* p;
  int nb;
  __device__ __forceinline__ float* dia(int v) const { return p + v * kDia; }
  __device__ __forceinline__ float* blk(int i) const { return p + nb * kDia + i * kBlk; }
};
// rows of blocks in LDS are 8-byte aligned, blocks 16-byte aligned; blocks in global memory are not
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void load6(const lds_f* p, float (&v)[6]) {
  const GSR_LDS f2* q = reinterpret_cast<const GSR_LDS f2*>(p);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const f2 x = q[k];
    v[2 * k] = x.x;
    v[2 * k + 1] = x.y;
  }
}
__device__ __forceinline__ void load6(const float* p, float (&v)[6]) {
#pragma unroll
  for (int k = 0; k < 6; k++) v[k] = p[k];
}
__device__ __forceinline__ void load36(const lds_f* p, float (&v)[kBlk]) {
  const GSR_LDS f4* q = reinterpret_cast<const GSR_LDS f4*>(p);
#pragma unroll
  for (int k = 0; k < 9; k++) {
    const f4 x = q[k];
    v[4 * k] = x.x;
    v[4 * k + 1] = x.y;
    v[4 * k + 2] = x.z;
    v[4 * k + 3] = x.w;
  }
}
__device__ __forceinline__ void load36(const float* p, float (&v)[kBlk]) {
#pragma unroll
  for (int k = 0; k < kBlk; k++) v[k] = p[k];
}

// H = M + J^T D J over the active rows (func_nt_hessian_direct): the lane of dof i (factor order) walks its body's rows
// in ascending order and adds row i's entries: the diagonal block's in registers, those of the block shared with the
// row's other body in registers too while that body stays the same
template <int kWaves, class HB>
__device__ inline void bodies_hessian(const BodyCtx<kWaves>& w, const HB& h, const BodyRow (&r)[kBodyRows]) {
  constexpr int NT = BodyCtx<kWaves>::kThreads;
  const Env& e = w.e;
  const gsr_state& s = e.s;
  const BodyLds& L = w.L;
  const float eps = e.m.eps;
  w.sync();
  // the active rows' weights in the rows' LDS places (their forces are not needed any more)
#pragma unroll
  for (int q = 0; q < kBodyRows; q++) {
    const int c = w.tid + NT * q;
    if (c < w.n_con) {
      if (c < w.n_lds) L.row[c] = (r[q].act & 1) ? r[q].Dc : 0.f;
      else e.EI(s.efc_active, c) = r[q].act;
    }
  }
  for (int c = w.tid + NT * kBodyRows; c < min(w.n_con, w.n_lds); c += NT)
    L.row[c] = (e.EI(s.efc_active, c) & 1) ? e.EF(s.efc_D, c) : 0.f;
  const int n_blk = L.hb[w.nb - 1] + __popcll(L.pat[2 * w.nb - 2] & low_mask(w.nb - 1)) + __popcll(L.pat[2 * w.nb - 1] & low_mask(w.nb - 65));
  for (int i = w.tid; i < n_blk * kBlk; i += NT) h.blk(0)[i] = 0.f;
  w.sync();
  const int* lst = s.ent_row_list + (size_t)e.b * 2 * e.m.max_rows;
  const int W = e.m.row_width;
  const float* jv = &e.JV(0, 0);
  // a row's entries: this body's, the other body's and this dof's
  auto load_row = [&](int x, int i, float (&va)[6], float (&vo)[6], float& vi) {
    const int c = x & 0xfffff, p0 = ((x >> 20) & 1) * 6;
    const float* row = jv + c * W;
    const float* oth = row + (W > 6 ? 6 - p0 : 0);
#pragma unroll
    for (int k = 0; k < 6; k++) va[k] = row[p0 + k];
#pragma unroll
    for (int k = 0; k < 6; k++) vo[k] = oth[k];
    vi = row[p0 + i];
  };
  for (int d = w.tid; d < w.D; d += NT) {
    const int b = d / 6, i = d - 6 * b, v = L.vof[b], t1 = L.ptr[b + 1];
    float own[6], off[6];
#pragma unroll
    for (int k = 0; k < 6; k++) own[k] = off[k] = 0.f;
    int cur = -1;  // other body of the entries in off (a neighbour eliminated before this one), -1: none
    typename HB::ptr q = h.dia(v);
    int t = L.ptr[b];
    // the next row's entries are loaded while a row is summed
    int x = t < t1 ? lst[t] : 0, x1 = t + 1 < t1 ? lst[t + 1] : 0;
    float va[6], vo[6], vi = 0.f;
#pragma unroll
    for (int k = 0; k < 6; k++) va[k] = vo[k] = 0.f;
    if (t < t1) load_row(x, i, va, vo, vi);
    for (; t < t1; t++) {
      const int x2 = t + 2 < t1 ? lst[t + 2] : 0;
      float na[6], no[6], ni;
      load_row(x1, i, na, no, ni);
      const int c = x & 0xfffff, o = x >> 21;
      float Dc;
      if (c < w.n_lds) Dc = L.row[c];
      else Dc = (e.EI(s.efc_active, c) & 1) ? e.EF(s.efc_D, c) : 0.f;
      // an inactive row adds +-0 to entries that start at +0 and so never hold -0: skipping it changes no bit
      if (Dc != 0.f) {
        // the pair (later entry, earlier entry) of a row counts when the later one's magnitude exceeds eps
        const bool on = fabsf(vi) > eps;
        if (on) {
#pragma unroll
          for (int k = 0; k < 6; k++)
            if (k <= i) own[k] = own[k] + va[k] * vi * Dc;
        }
        if (o != b && L.vof[o] < v) {
          if (o != cur) {
            if (cur >= 0) {
#pragma unroll
              for (int k = 0; k < 6; k++) q[k] = off[k];
            }
            cur = o;
            q = h.blk(blk_index(L, v, L.vof[o])) + 6 * i;
            load6(q, off);
          }
#pragma unroll
          for (int k = 0; k < 6; k++)
            if (o < b ? on : fabsf(vo[k]) > eps) off[k] = off[k] + vo[k] * vi * Dc;
        }
      }
      x = x1;
      x1 = x2;
      vi = ni;
#pragma unroll
      for (int k = 0; k < 6; k++) {
        va[k] = na[k];
        vo[k] = no[k];
      }
    }
    if (cur >= 0)
#pragma unroll
      for (int k = 0; k < 6; k++) q[k] = off[k];
    typename HB::ptr dd = h.dia(v) + i * (i + 1) / 2;
#pragma unroll
    for (int k = 0; k < 6; k++)
      if (k <= i) dd[k] = own[k] + e.F(s.mass_blk, 6 * d + k);
  }
  w.sync();
}

__device__ __forceinline__ constexpr int tri6(int r, int q) { return r * (r + 1) / 2 + q; }

// neighbours of v before position v (and) or after it, as two words
__device__ __forceinline__ void before_mask(const BodyLds& L, int v, unsigned long long& m0, unsigned long long& m1) {
  m0 = L.pat[2 * v] & low_mask(v);
  m1 = L.pat[2 * v + 1] & low_mask(v - 64);
}
__device__ __forceinline__ int pop_low(unsigned long long& m0, unsigned long long& m1) {
  if (m0) {
    const int x = __ffsll((long long)m0) - 1;
    m0 &= m0 - 1;
    return x;
  }
  const int x = 64 + __ffsll((long long)m1) - 1;
  m1 &= m1 - 1;
  return x;
}

// Cholesky of the block matrix (func_nt_chol_factor's entries), level by level. Of a body: the products of its diagonal
// block's rows over the earlier columns, terms dealt round-robin to G lanes and added by a butterfly (G as if the level's
// bodies shared one wavefront, so the sums do not depend on kWaves: with more wavefronts, subgroups of G lanes compute
// the same sums); the block's own factor, by every lane alike; then each row of the later bodies it shares a block with,
// one a lane of the body's kWaves G lanes.
template <int kWaves, class HB>
__device__ inline void bodies_factor(const BodyCtx<kWaves>& w, const HB& h) {
  const BodyLds& L = w.L;
  const float EPS = w.e.m.eps;
  const int nl = L.misc[0];
  for (int lv = 0; lv < nl; lv++) {
    const int i0 = L.fst[lv], i1 = L.fst[lv + 1];
    const int G = lane_group(i1 - i0, 0).G, Gw = min(kWave, G * kWaves);
    const int group = (w.lane / Gw) * kWaves + w.wv, n_groups = (kWave / Gw) * kWaves, r = w.lane & (Gw - 1);
    for (int k0 = i0 + group; k0 < i1; k0 += n_groups) {
      const int lw = L.flv[k0], v = lw & 0xff, hv = lw >> 16, n_terms = 6 * ((lw >> 8) & 0xff);
      const auto dia = h.dia(v);
      unsigned long long b0, b1;
      before_mask(L, v, b0, b1);
      float lc[21];
#pragma unroll
      for (int t = 0; t < 21; t++) lc[t] = 0.f;
      for (int t = r & (G - 1); t < n_terms; t += G) {
        const int j = t / 6;
        const auto p = h.blk(hv + j) + (t - 6 * j);
        float x[6];
#pragma unroll
        for (int i = 0; i < 6; i++) x[i] = p[6 * i];
#pragma unroll
        for (int i = 0; i < 6; i++)
#pragma unroll
          for (int q = 0; q <= i; q++) lc[tri6(i, q)] += x[i] * x[q];
      }
      if (n_terms > 0) {
#pragma unroll
        for (int t = 0; t < 21; t++) lc[t] = group_sum(lc[t], G);
      }
#pragma unroll
      for (int i = 0; i < 6; i++) {
#pragma unroll
        for (int q = 0; q <= i; q++) {
          float x = dia[tri6(i, q)] - lc[tri6(i, q)];
#pragma unroll
          for (int p = 0; p < q; p++) x -= lc[tri6(i, p)] * lc[tri6(q, p)];
          lc[tri6(i, q)] = q == i ? sqrtf(fmaxf(x, EPS)) : x / lc[tri6(q, q)];
        }
      }
      // rows of the later neighbours: row t of their concatenation, lane r takes t = r, r + Gw, ...
      unsigned long long a0 = L.pat[2 * v] & ~low_mask(v + 1), a1 = L.pat[2 * v + 1] & ~low_mask(v + 1 - 64);
      const int n_rows = 6 * (__popcll(a0) + __popcll(a1));
      int seen = 0, u = 0;
      for (int t = r; t < n_rows; t += Gw) {
        while (seen <= t) {
          u = pop_low(a0, a1);
          seen += 6;
        }
        const int j = t - (seen - 6);
        float acc[6];
#pragma unroll
        for (int q = 0; q < 6; q++) acc[q] = 0.f;
        const unsigned long long u0 = L.pat[2 * u], u1 = L.pat[2 * u + 1];
        unsigned long long c0 = b0 & u0, c1 = b1 & u1;
        const int hu = L.hb[u];
        while (c0 | c1) {
          const int x = pop_low(c0, c1);
          const unsigned long long l0 = low_mask(x), l1 = low_mask(x - 64);
          float bv[kBlk], y[6];
          load36(h.blk(hv + __popcll(b0 & l0) + __popcll(b1 & l1)), bv);
          load6(h.blk(hu + __popcll(u0 & l0) + __popcll(u1 & l1)) + 6 * j, y);
#pragma unroll
          for (int k = 0; k < 6; k++)
#pragma unroll
            for (int q = 0; q < 6; q++) acc[q] += y[k] * bv[6 * q + k];
        }
        const auto pj = h.blk(hu + __popcll(u0 & low_mask(v)) + __popcll(u1 & low_mask(v - 64))) + 6 * j;
        float y[6];
        load6(pj, y);
#pragma unroll
        for (int q = 0; q < 6; q++) {
          float x = y[q] - acc[q];
#pragma unroll
          for (int p = 0; p < q; p++) x -= y[p] * lc[tri6(q, p)];
          y[q] = x / lc[tri6(q, q)];
        }
#pragma unroll
        for (int q = 0; q < 6; q++) pj[q] = y[q];
      }
      if (r == 0) {
#pragma unroll
        for (int t = 0; t < 21; t++) dia[t] = lc[t];
      }
    }
    w.sync();
  }
}

// vec = H^-1 vec in factor space (func_nt_chol_solve) on the env's first wavefront: forward over the forward levels,
// backward over the backward ones, a group of G lanes per body of the level; the terms over the other bodies are dealt
// round-robin to the group for the body's six rows together and added by butterflies, the triangle of the diagonal block
// is solved by every lane alike
template <class HB>
__device__ inline void bodies_solve(const BodyLds& L, const HB& h, int lane) {
  for (int back = 0; back < 2; back++) {
    const int nl = L.misc[back];
    const lds_i* order = back ? L.rlv : L.flv;
    const lds_i* first = back ? L.rst : L.fst;
    for (int lv = 0; lv < nl; lv++) {
      const int i0 = first[lv], i1 = first[lv + 1];
      const LaneGroup g = lane_group(i1 - i0, lane);
      for (int k0 = i0 + g.q; k0 < i1; k0 += g.ng) {
        const int lw = order[k0], v = lw & 0xff, first_blk = lw >> 16, n_terms = 6 * ((lw >> 8) & 0xff);
        const auto dia = h.dia(v);
        float acc[6], lc[21], y[6];
#pragma unroll
        for (int t = 0; t < 21; t++) lc[t] = dia[t];
#pragma unroll
        for (int k = 0; k < 6; k++) {
          acc[k] = 0.f;
          y[k] = L.vec[6 * v + k];
        }
        if constexpr (HB::kLists) {
          if (back) {
#pragma unroll 4
            for (int t = g.r; t < n_terms; t += g.G) {
              const int idx = t / 6, j = t - 6 * idx, ent = L.cl[first_blk + idx];
              const float xj = L.vec[6 * (ent & 0xff) + j];
              float b[6];
              load6(h.blk(ent >> 8) + 6 * j, b);
#pragma unroll
              for (int k = 0; k < 6; k++) acc[k] += b[k] * xj;
            }
          } else {
#pragma unroll 4
            for (int t = g.r; t < n_terms; t += g.G) {
              const int idx = t / 6, j = t - 6 * idx;
              const float xj = L.vec[6 * L.rl[first_blk + idx] + j];
              const auto p = h.blk(first_blk + idx) + j;
#pragma unroll
              for (int k = 0; k < 6; k++) acc[k] += p[6 * k] * xj;
            }
          }
        } else {
          unsigned long long m0 = L.pat[2 * v], m1 = L.pat[2 * v + 1];
          m0 &= back ? ~low_mask(v + 1) : low_mask(v);
          m1 &= back ? ~low_mask(v + 1 - 64) : low_mask(v - 64);
          int seen = 0, u = 0;
          for (int t = g.r; t < n_terms; t += g.G) {
            while (seen <= t) {
              u = pop_low(m0, m1);
              seen += 6;
            }
            const int j = t - (seen - 6);
            const float xj = L.vec[6 * u + j];
            const auto p = back ? h.blk(blk_index(L, u, v)) + 6 * j : h.blk(first_blk + seen / 6 - 1) + j;
#pragma unroll
            for (int k = 0; k < 6; k++) acc[k] += p[back ? k : 6 * k] * xj;
          }
        }
#pragma unroll
        for (int k = 0; k < 6; k++) y[k] -= group_sum(acc[k], g.G);
        if (back) {
#pragma unroll
          for (int p = 5; p >= 0; p--) {
#pragma unroll
            for (int q = p + 1; q < 6; q++) y[p] -= lc[tri6(q, p)] * y[q];
            y[p] = y[p] / lc[tri6(p, p)];
          }
        } else {
#pragma unroll
          for (int p = 0; p < 6; p++) {
#pragma unroll
            for (int q = 0; q < p; q++) y[p] -= lc[tri6(p, q)] * y[q];
            y[p] = y[p] / lc[tri6(p, p)];
          }
        }
        if (g.r == 0) {
#pragma unroll
          for (int k = 0; k < 6; k++) L.vec[6 * v + k] = y[k];
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
}

// rank-1 update / downdate of the factor with row c (func_nt_hessian_incremental) on the first wavefront; false on rank
// loss (the caller then rebuilds the factor). The row's bodies, then every later body that shares a block with one whose
// entries were not all zero, in factor order; of each body the six rows of its diagonal block lie on lanes 0 to 5, the
// rows of the later blocks on the lanes after them (further ones are taken after the pivots are known).
template <class HB>
__device__ inline bool bodies_rank1(const Env& e, const BodyLds& L, const HB& h, int lane, int D, int c, int ent, float Dc,
                                    float sgn) {
  const float eps = e.m.eps;
  const float sq = sqrtf(Dc);
  for (int d = lane; d < D; d += kWave) L.vec[d] = 0.f;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  const int ea = ent & 0xff, eb = ent >> 8;
  if (lane < (ea == eb ? 6 : 12))
    L.vec[6 * L.vof[lane < 6 ? ea : eb] + (lane < 6 ? lane : lane - 6)] = e.JV(c, lane) * sq;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  bool ok = true;
  unsigned long long act0 = 0ull, act1 = 0ull;
  {
    const int va = __builtin_amdgcn_readfirstlane(L.vof[ea]), vb = __builtin_amdgcn_readfirstlane(L.vof[eb]);
    if (va < 64) act0 |= 1ull << va; else act1 |= 1ull << (va - 64);
    if (vb < 64) act0 |= 1ull << vb; else act1 |= 1ull << (vb - 64);
  }
  while (act0 | act1) {
    const int v = pop_low(act0, act1);
    const unsigned long long a0 = L.pat[2 * v] & ~low_mask(v + 1), a1 = L.pat[2 * v + 1] & ~low_mask(v + 1 - 64);
    const int n_rows = 6 + 6 * (__popcll(a0) + __popcll(a1));
    const auto dia = h.dia(v);
    float P[6], S[6], Q[6];  // of each pivot with a nonzero entry: r / L, its inverse, v / L; P = 0: none
    bool any = false;
    unsigned long long m0 = a0, m1 = a1;
    int seen = 6, u = 0;
    for (int t0 = 0; t0 < n_rows; t0 += kWave) {
      const int t = t0 + lane;
      // row t: a row of the diagonal block, or of block (u, v)
      typename HB::ptr p = dia;
      int xi = 6 * v;
      float l[6], x = 0.f;
#pragma unroll
      for (int k = 0; k < 6; k++) l[k] = 0.f;
      if (t < 6) {
        p = dia + t * (t + 1) / 2;
        xi = 6 * v + t;
#pragma unroll
        for (int k = 0; k < 6; k++) l[k] = k <= t ? p[k] : 0.f;
        x = L.vec[xi];
      } else if (t < n_rows) {
        while (seen <= t) {
          u = pop_low(m0, m1);
          seen += 6;
        }
        const int j = t - (seen - 6);
        p = h.blk(blk_index(L, u, v)) + 6 * j;
        xi = 6 * u + j;
        load6(p, l);
        x = L.vec[xi];
      }
#pragma unroll
      for (int k = 0; k < 6; k++) {
        if (t0 == 0) {
          const float vk = lane_value(x, k);
          P[k] = 0.f;
          if (fabsf(vk) > eps) {
            any = true;
            const float Lkk = lane_value(l[k], k);
            float tmp = Lkk * Lkk + vk * vk * sgn;
            if (tmp < eps) {
              tmp = eps;
              ok = false;
            }
            const float rr = sqrtf(tmp);
            P[k] = rr / Lkk;
            S[k] = 1.f / P[k];
            Q[k] = vk / Lkk;
            if (lane == k) l[k] = rr;
          }
        }
        if (P[k] != 0.f && t > k && t < n_rows) {
          const float hv = (l[k] + Q[k] * x * sgn) * S[k];
          l[k] = hv;
          x = x * P[k] - Q[k] * hv;
        }
      }
      if (any) {
        if (t < 6) {
#pragma unroll
          for (int k = 0; k < 6; k++)
            if (k <= t) p[k] = l[k];
        } else if (t < n_rows) {
#pragma unroll
          for (int k = 0; k < 6; k++) p[k] = l[k];
          L.vec[xi] = x;
        }
      }
      if (!any) break;
    }
    if (any) {
      act0 |= a0;
      act1 |= a1;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  }
  return ok;
}

// ---- line search ----------------------------------------------------------------------------------------------------
__device__ __forceinline__ void body_ls_row(const Env& e, int c, int ne, int nef, float ja, float jv, float q0, float q1,
                                            float q2, float alpha, double& t0, double& t1, double& t2) {
  const gsr_state& s = e.s;
  const float x = ja + alpha * jv;
  bool act = true;
  if (ne <= c && c < nef) {
    const float f = e.EF(s.efc_fl, c), r = e.EF(s.efc_diag, c), rf = r * f;
    const bool ln = x <= -rf, lp = x >= rf;
    if (ln || lp) {
      q0 = (float)ln * f * (-0.5f * rf - ja) + (float)lp * f * (-0.5f * rf + ja);
      q1 = (float)ln * (-f * jv) + (float)lp * (f * jv);
      q2 = 0.f;
    }
  } else if (nef <= c) {
    act = x < 0.f;
  }
  t0 += (double)(q0 * (float)act);
  t1 += (double)(q1 * (float)act);
  t2 += (double)(q2 * (float)act);
}

struct BodyLine {
  float qg0, qg1, qg2;
};
template <int kWaves>
__device__ inline WLS bodies_ls_point(const BodyCtx<kWaves>& w, const BodyRow (&r)[kBodyRows], const BodyLine& g, float alpha,
                                      int& ls_it) {
  constexpr int NT = BodyCtx<kWaves>::kThreads, K = 4 / kWaves;
  const Env& e = w.e;
  const gsr_state& s = e.s;
  double a[3][K];
#pragma unroll
  for (int k = 0; k < K; k++) a[0][k] = a[1][k] = a[2][k] = 0.0;
#pragma unroll
  for (int q = 0; q < kBodyRows; q++) {
    const int c = w.tid + NT * q;
    if (c < w.n_con)
      body_ls_row(e, c, w.ne, w.nef, r[q].ja, r[q].jv, r[q].q0, r[q].q1, r[q].q2, alpha, a[0][q % K], a[1][q % K], a[2][q % K]);
  }
  for (int c = w.tid + NT * kBodyRows, q = kBodyRows; c < w.n_con; c += NT, q++) {
    double t[3] = {0.0, 0.0, 0.0};
    body_ls_row(e, c, w.ne, w.nef, e.EF(s.efc_Jaref, c), e.EF(s.efc_jv, c), e.QD(c, 0), e.QD(c, 1), e.QD(c, 2), alpha, t[0],
                t[1], t[2]);
#pragma unroll
    for (int k = 0; k < K; k++)
      if (q % K == k) {
        a[0][k] += t[0];
        a[1][k] += t[1];
        a[2][k] += t[2];
      }
  }
  double out[3];
  bodies_sum<kWaves, 3>(w, w.n_con, a, out);
  return ls_point_from(e, g.qg0, g.qg1, g.qg2, out[0], out[1], out[2], alpha, ls_it);
}

template <int kWaves>
__device__ inline float bodies_linesearch(const BodyCtx<kWaves>& w, BodyRow (&r)[kBodyRows], float gauss, float scale) {
  constexpr int NT = BodyCtx<kWaves>::kThreads, K = 4 / kWaves;
  const Env& e = w.e;
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const BodyLds& L = w.L;
  double a[3][K], out[3];
#pragma unroll
  for (int k = 0; k < K; k++) a[0][k] = a[1][k] = a[2][k] = 0.0;
  for (int d = w.tid, q = 0; d < w.D; d += NT, q++) {
    const float mv = body_mass_mul(e, d, L.search), sd = L.search[d];
    L.mv[d] = mv;
    const double x0 = (double)(sd * sd), x1 = (double)(sd * L.Ma[d] - sd * e.F(s.force, d)), x2 = (double)(0.5f * sd * mv);
#pragma unroll
    for (int k = 0; k < K; k++)
      if (q % K == k) {
        a[0][k] += x0;
        a[1][k] += x1;
        a[2][k] += x2;
      }
  }
  bodies_sum<kWaves, 3>(w, w.D, a, out);
  const float snorm = sqrtf((float)out[0]);
  const float gtol = m.tolerance * m.ls_tolerance * snorm * scale;
  if (snorm < m.eps) return 0.f;
#pragma unroll
  for (int q = 0; q < kBodyRows; q++) {
    const int c = w.tid + NT * q;
    if (c < w.n_con) {
      const float jv = body_row_dot(e, c, r[q].ent, 0.f, L.search);
      r[q].jv = jv;
      r[q].q0 = r[q].Dc * (0.5f * r[q].ja * r[q].ja);
      r[q].q1 = r[q].Dc * (jv * r[q].ja);
      r[q].q2 = r[q].Dc * (0.5f * jv * jv);
    }
  }
  const int* rent = s.efc_ent + (size_t)e.b * m.max_rows;
  for (int c = w.tid + NT * kBodyRows; c < w.n_con; c += NT) {
    const float jv = body_row_dot(e, c, rent[c], 0.f, L.search);
    const float Dc = e.EF(s.efc_D, c), ja = e.EF(s.efc_Jaref, c);
    e.EF(s.efc_jv, c) = jv;
    e.QD(c, 0) = Dc * (0.5f * ja * ja);
    e.QD(c, 1) = Dc * (jv * ja);
    e.QD(c, 2) = Dc * (0.5f * jv * jv);
  }
  const BodyLine g{gauss, (float)out[1], (float)out[2]};
  return linesearch_points(m, gtol, [&](float x, int& ls_it) { return bodies_ls_point(w, r, g, x, ls_it); });
}

// ---- Newton iterations ----------------------------------------------------------------------------------------------
template <int kWaves, class HB>
__device__ inline int bodies_newton(const BodyCtx<kWaves>& w, const HB& h, BodyRow (&r)[kBodyRows], double cost, float gauss) {
  constexpr int NT = BodyCtx<kWaves>::kThreads, K = 4 / kWaves;
  const Env& e = w.e;
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const BodyLds& L = w.L;
  const float scale = e.meaninertia() * (float)(w.D > 1 ? w.D : 1), tol_scaled = scale * m.tolerance;
  int iters = 0;
  bool build = true;
  while (iters < m.iterations) {
    if (build) {
      bodies_hessian(w, h, r);
      bodies_factor(w, h);
    }
    for (int d = w.tid; d < w.D; d += NT) {
      const int b = d / 6;
      L.vec[6 * L.vof[b] + d - 6 * b] = L.Ma[d] - e.F(s.force, d) - L.qfrc[d];
    }
    w.sync();
    if (w.wv == 0) bodies_solve(L, h, w.lane);
    w.sync();
    for (int d = w.tid; d < w.D; d += NT) {
      const int b = d / 6;
      L.search[d] = -L.vec[6 * L.vof[b] + d - 6 * b];
    }
    w.sync();
    iters++;
    const float alpha = bodies_linesearch(w, r, gauss, scale);
    if (fabsf(alpha) < m.eps) break;
    for (int d = w.tid; d < w.D; d += NT) {
      L.qacc[d] = L.qacc[d] + L.search[d] * alpha;
      L.Ma[d] = L.Ma[d] + L.mv[d] * alpha;
    }
#pragma unroll
    for (int q = 0; q < kBodyRows; q++) r[q].ja = r[q].ja + r[q].jv * alpha;
    for (int c = w.tid + NT * kBodyRows; c < w.n_con; c += NT)
      e.EF(s.efc_Jaref, c) = e.EF(s.efc_Jaref, c) + e.EF(s.efc_jv, c) * alpha;
    const double prev_cost = cost;
    bodies_update_constraint(w, r, cost, gauss);
    const double improvement = prev_cost - cost;
    // |grad|^2 and the number of rows whose activity changed
    double a[2][K], out[2];
#pragma unroll
    for (int k = 0; k < K; k++) a[0][k] = a[1][k] = 0.0;
    for (int d = w.tid, q = 0; d < w.D; d += NT, q++) {
      const float g = L.Ma[d] - e.F(s.force, d) - L.qfrc[d];
#pragma unroll
      for (int k = 0; k < K; k++)
        if (q % K == k) a[0][k] += (double)(g * g);
    }
    int changed = 0;
#pragma unroll
    for (int q = 0; q < kBodyRows; q++)
      if (w.tid + NT * q < w.n_con) changed += (r[q].act ^ (r[q].act >> 1)) & 1;
    for (int c = w.tid + NT * kBodyRows; c < w.n_con; c += NT) {
      const int x = e.EI(s.efc_active, c);
      changed += (x ^ (x >> 1)) & 1;
    }
    a[1][0] = (double)changed;
    bodies_sum<kWaves, 2>(w, NT * 4, a, out);  // every class may hold a count
    const float gn = sqrtf((float)out[0]);
    if (gn < tol_scaled || improvement < tol_scaled) break;
    const int n_changed = (int)out[1];
    build = n_changed > kMaxRank1PerIter || (n_changed > 0 && w.n_con > 16 * w.n_lds);  // the bits below fit L.row
    if (n_changed > 0 && !build) {
      // the changed rows, in row order, as bits of the rows' LDS places: 64 rows a word
      lds_u64* bits = reinterpret_cast<lds_u64*>(L.row);
      const int words = (w.n_con + kWave - 1) / kWave;
      w.sync();  // the forces in L.row are read no more
      auto word = [&](int q, int x) {
        const unsigned long long on = __ballot((x ^ (x >> 1)) & 1);
        const int c0 = kWave * (w.wv + kWaves * q);
        if (w.lane == 0 && c0 < w.n_con) bits[2 * (c0 / kWave)] = on;
        const unsigned long long up = __ballot(((x ^ (x >> 1)) & 1) && (x & 1));
        if (w.lane == 0 && c0 < w.n_con) bits[2 * (c0 / kWave) + 1] = up;
      };
#pragma unroll
      for (int q = 0; q < kBodyRows; q++) word(q, w.tid + NT * q < w.n_con ? r[q].act : 0);
      for (int q = kBodyRows; NT * q < w.n_con; q++)
        word(q, w.tid + NT * q < w.n_con ? e.EI(s.efc_active, w.tid + NT * q) : 0);
      w.sync();
      if (w.wv == 0) {
        const int* rent = s.efc_ent + (size_t)e.b * m.max_rows;
        bool ok = true;
        for (int k = 0; k < words && ok; k++) {
          unsigned long long on = bits[2 * k];
          const unsigned long long up = bits[2 * k + 1];
          while (on && ok) {
            const int j = __ffsll((long long)on) - 1, c = kWave * k + j;
            on &= on - 1;
            ok = bodies_rank1(e, L, h, w.lane, w.D, c, rent[c], e.EF(s.efc_D, c), ((up >> j) & 1ull) ? 1.f : -1.f);
          }
        }
        if (w.lane == 0) L.misc[3] = ok ? 0 : 1;
      }
      w.sync();
      build = L.misc[3] != 0;
    }
  }
  return iters;
}

template <int kWaves>
__device__ __forceinline__ void solve_bodies(const Env& e, char* lds) {
  constexpr int NT = kWave * kWaves;
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const int tid = threadIdx.x, D = m.n_dofs;
  const BodyLds L = bodies_carve(lds, D, m.wave_h_floats);
  const int n_con = e.I(s.n_con, 0), ne = e.I(s.n_con, 1), nef = ne + e.I(s.n_con, 2);
  int flip = 0;
  const BodyCtx<kWaves> w{e, L, tid, tid & 63, tid >> 6, D, D / 6, n_con, ne, nef, bodies_lds_rows(D), flip};
  int iters = 0;
  if (n_con > 0) {
    const bool ws = e.I(s.is_warmstart, 0) != 0;
    for (int d = tid; d < D; d += NT) L.qacc[d] = ws ? e.F(s.qacc_ws, d) : e.F(s.acc_smooth, d);
    bodies_structure(w);
    for (int d = tid; d < D; d += NT) L.Ma[d] = body_mass_mul(e, d, L.qacc);
    BodyRow r[kBodyRows];
    const int* rent = s.efc_ent + (size_t)e.b * m.max_rows;
#pragma unroll
    for (int q = 0; q < kBodyRows; q++) {
      const int c = tid + NT * q;
      r[q] = BodyRow{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0, 0};
      if (c < n_con) {
        r[q].ent = rent[c];
        r[q].Dc = e.EF(s.efc_D, c);
        r[q].ja = body_row_dot(e, c, r[q].ent, -e.EF(s.efc_aref, c), L.qacc);
      }
    }
    for (int c = tid + NT * kBodyRows; c < n_con; c += NT)
      e.EF(s.efc_Jaref, c) = body_row_dot(e, c, rent[c], -e.EF(s.efc_aref, c), L.qacc);
    double cost;
    float gauss;
    bodies_update_constraint(w, r, cost, gauss);
    const int in_lds = L.misc[2];
    if (in_lds) iters = bodies_newton(w, BlocksLds{L.hl, w.nb}, r, cost, gauss);
    else iters = bodies_newton(w, BlocksMem{&e.H(0, 0), w.nb}, r, cost, gauss);
  } else {
    for (int d = tid; d < D; d += NT) {
      L.qacc[d] = e.F(s.acc_smooth, d);
      L.qfrc[d] = 0.f;
    }
  }
  w.sync();
  // epilogue (func_update_qacc, func_update_contact_force)
  int bad = 0;
  for (int d = tid; d < D; d += NT) {
    const float q = L.qacc[d];
    e.F(s.acc, d) = q;
    e.F(s.force, d) = e.F(s.qf_smooth, d) + L.qfrc[d];
    e.F(s.qacc_ws, d) = q;
    bad |= isnan(q) ? 1 : 0;
  }
  if (__any(bad) && w.lane == 0) atomicOr((unsigned*)&e.I((int32_t*)s.errno_env, 0), (unsigned)GSR_ERR_NAN_QACC);
  if (tid == 0) {
    e.I(s.solver_iters, 0) = iters;
    e.I(s.is_warmstart, 0) = 1;
  }
  contact_forces(e, tid, NT);
}

}  // namespace gsr
