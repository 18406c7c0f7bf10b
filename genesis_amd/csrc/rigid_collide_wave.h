// Collision detection and constraint rows of environments on wavefronts, W lanes per env (64: one env a wavefront, 16:
// four envs a wavefront; collide_lanes() says which).
//
// Same results as the one-lane-per-env path of rigid_collide.h / rigid_solver.h, spread over lanes:
//   * AABBs: one geom per lane (rigid_solver_decomp.py:5668-5689).
//   * Sweep-and-prune (collider_decomp.py:1331-1470): the reference warm-starts an insertion sort with strict `<`,
//     which is a stable sort of the previous order; here each lane ranks its entries (rank = #smaller + #equal
//     before it), which gives the same permutation. The sweep's active list at a min event holds the geoms whose
//     min event came earlier and whose max event comes later, in min-event order: event after event the earlier
//     geoms are tested on their own lanes, from AABBs in LDS, and a ballot places every pair where the serial sweep
//     puts it.
//   * Narrowphase: one broadphase pair per lane, contacts kept in the lane (LocalSink) and placed by a prefix sum,
//     convex pairs first and plane-box pairs second, both in broadphase order, as the reference appends them.
//   * Rows: equality rows on lane 0 (few), frictionloss and limit rows a link per lane, the 4 rows of each contact on its
//     own lane.
// What bounds it is dependent work on few lanes. Measured (us, whole stage; every event's set walked by one lane, every
// dof's tables by lane 0 and a general pow in each row -> events' sets across lanes, links across lanes, integer powers as
// products): 64 arms 45 -> 25, 100 7-box piles 62 -> 45, 1,500 20-box piles 250 -> 192, 96 64-box piles 641 -> 486,
// 4,096 of them 2063 -> 1713.
#pragma once
#include "rigid_collide.h"
#include "rigid_solver.h"

namespace gsr {

constexpr int kWaveMaxGeoms = 1024;

// exclusive prefix sum over the W lanes of an env, its total on every lane
template <int W>
__device__ __forceinline__ int wave_excl_scan(int v, int lane, int& total) {
  int x = v;
  for (int o = 1; o < W; o <<= 1) {
    int y = __shfl_up(x, o, W);
    if (lane >= o) x += y;
  }
  total = __shfl(x, W - 1, W);
  return x - v;
}
// the lanes of this lane's env for which v holds
template <int W>
__device__ __forceinline__ unsigned long long env_ballot(bool v) {
  const unsigned long long b = __ballot(v);
  if constexpr (W == 64) return b;
  else return (b >> (threadIdx.x & ~(W - 1))) & ((1ull << W) - 1ull);
}

// LDS words of one env: the sweep's arrays (16 a geom), then in their place the narrowphase's (32 a lane)
__host__ __device__ inline size_t wave_collide_words(int G, int W) {
  return (16 * (size_t)G > 32 * (size_t)W ? 16 * (size_t)G : 32 * (size_t)W) + 4;
}
__host__ __device__ inline size_t wave_collide_lds_bytes(int G, int W = 64) {
  return sizeof(float) * wave_collide_words(G, W) * (size_t)(64 / W) + 64;
}
// Models whose collision the wavefront form holds (its LDS, its contact buffer of a pair): all that any scene here has. The
// others take a lane per env.
__host__ __device__ inline bool collide_waves(const gsr_model& m) {
  return m.collide_variant == 1 ||
         (wave_collide_lds_bytes(m.n_geoms) <= 64 * 1024 && m.n_contacts_per_pair <= kMaxPairContacts);
}
// Models that may share a wavefront among four envs: with few entities a few pairs reach the narrowphase and a few contacts
// the rows, which leaves most of 64 lanes idle.
__host__ __device__ inline bool collide_packs(const gsr_model& m) { return m.n_entities <= 8 && m.n_geoms <= 32; }
// Lanes per env of a launch over n envs. Up to 2,048 envs there are SIMDs to spare and 64 lanes finish sooner; above, four
// envs a wavefront are faster where the model packs. Measured (us, collision and GJK/EPA pass; one lane per env, 64, 16
// lanes): quadrupeds 2,048: 576, 68, 68; 4,000: 585, 123, 80; 32,768: 824, 939, 374; arms 2,000: 707, 76, 89; 5,000: 726,
// 120, 98; 7-box piles 1,024: 465, 58, 55; 4,000: 488, 122, 105; 16,384: 569, 491, 342. Heaps do not pack: 20 boxes 300:
// 4213, 172, 354; 4,000: 4437, 403, 448; 64 boxes 1,024: 25968, 566, 1529 (heaps with a pair per lane throughout; wave_convex
// has taken 15 to 40 % off their 64-lane figures since).
__host__ __device__ inline int collide_lanes(const gsr_model& m, int n) { return n > 2048 && collide_packs(m) ? 16 : kWave; }
// Models of variant 0 with few entities over so many envs that a lane per env fills the chip too: its work per env is the
// least, and what the wavefront forms gain by spreading one env is lost. Where the line lies follows the geoms, since one lane
// walks them all. Measured (us, lane per env, 16 lanes where the model packs, else 64), below and at the line: one sphere
// 8,192: 32, 41; 16,384: 34, 71; one box 8,192: 54, 50; 16,384: 62, 85; two boxes 16,384: 205, 206; 32,768: 277, 411; three
// 16,384: 348, 281; 32,768: 500, 610; seven 32,768: 386, 397; a quadruped on a plane (28 geoms) 32,768: 276, 174; 65,536:
// 311, 344; an arm of 35 geoms 16,384: 380, 243; 32,768: 430, 479; of 121 geoms 16,384: 1265, 941; 32,768: 1419, 1942.
__host__ __device__ inline bool collide_by_lane(const gsr_model& m, int n) {
  const int line = m.n_geoms <= 2 ? 16384 : m.n_geoms <= 6 ? 32768 : m.n_geoms <= 32 ? 65536 : 32768;
  return m.collide_variant == 0 && m.n_entities <= 8 && n >= line;
}

template <int W>
__device__ inline void wave_broad_phase(const Env& e, char* lds, int lane) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const int G = m.n_geoms, G2 = 2 * G;
  const int MAXB = 1 << 30;
  float* sv = reinterpret_cast<float*>(lds);
  float* tv = sv + G2;
  int* sig = reinterpret_cast<int*>(tv + G2);
  int* tig = sig + G2;
  int* minpos = tig + G2;
  int* maxpos = minpos + G;
  const float* box = reinterpret_cast<const float*>(maxpos + G);
  const bool first = e.I(s.first_time, 0) != 0;
  for (int i = lane; i < G2; i += W) {
    int t;
    if (first) t = (i & 1) ? ((i >> 1) | MAXB) : (i >> 1);
    else t = e.I(s.sort_ig, i);
    int g = t & (MAXB - 1);
    sig[i] = t;
    sv[i] = box[6 * g + ((t & MAXB) ? 3 : 0)];
  }
  __syncthreads();
  if (first && lane == 0) e.I(s.first_time, 0) = 0;
  // stable rank sort
  for (int i = lane; i < G2; i += W) {
    float v = sv[i];
    int r = 0;
    for (int j = 0; j < G2; j++) {
      float u = sv[j];
      r += (u < v) || (u == v && j < i);
    }
    tv[r] = v;
    tig[r] = sig[i];
  }
  __syncthreads();
  for (int i = lane; i < G2; i += W) {
    float v = tv[i];
    int t = tig[i];
    sv[i] = v;
    sig[i] = t;
    e.F(s.sort_value, i) = v;
    e.I(s.sort_ig, i) = t;
    if (t & MAXB) maxpos[t & (MAXB - 1)] = i;
    else minpos[t] = i;
  }
  __syncthreads();
  // geoms in the order of their min events: order[k] (in tig's place, whose contents sig has now), the AABBs in LDS. The geoms a min event pairs with are
  // those before it in this order whose max event comes later; they are tested on their own lanes, W at a time, event
  // after event, and a ballot places the pairs in the serial sweep's order.
  int* order = tig;
  int n_min = 0;
  for (int i0 = 0; i0 < G2; i0 += W) {
    const int i = i0 + lane;
    const bool is_min = i < G2 && !(sig[i] & MAXB);
    const unsigned long long b = env_ballot<W>(is_min);
    const int t = is_min ? sig[i] : 0;
    __syncthreads();
    if (is_min) order[n_min + __popcll(b & ((1ull << lane) - 1ull))] = t;
    n_min += __popcll(b);
  }
  __syncthreads();
  int base = 0;
  bool overflow = false;
  const int g0 = lane < G ? order[lane] : 0, m0 = lane < G ? maxpos[g0] : -1;
  float b0[6];
  for (int q = 0; q < 6; q++) b0[q] = box[6 * g0 + q];
  for (int ev = 1; ev < G; ev++) {
    const int gi = order[ev], pos = minpos[gi];
    const int full = max(base, m.max_broad);  // the serial sweep leaves an event at the first pair that finds no room
    float bi[6];
    for (int q = 0; q < 6; q++) bi[q] = box[6 * gi + q];
    for (int k0 = 0; k0 < ev; k0 += W) {
      const int k = k0 + lane;
      int g = g0, mp = m0;
      float bx[6];
      for (int q = 0; q < 6; q++) bx[q] = b0[q];
      if (k0 > 0) {
        g = k < ev ? order[k] : 0;
        mp = k < ev ? maxpos[g] : -1;
        for (int q = 0; q < 6; q++) bx[q] = box[6 * g + q];
      }
      int pidx = -1;
      const int ga = min(g, gi), gb = max(g, gi);
      if (k < ev && mp > pos) pidx = m.pair_idx[(size_t)ga * G + gb];
      bool hit = false;
      if (pidx != -1) {
        // box: minimum then maximum of each geom
        const bool sep = bx[3] <= bi[0] || bx[4] <= bi[1] || bx[5] <= bi[2] || bx[0] >= bi[3] || bx[1] >= bi[4] || bx[2] >= bi[5];
        hit = !sep;
      }
      const unsigned long long b = env_ballot<W>(hit);
      const int at = base + __popcll(b & ((1ull << lane) - 1ull));
      if (pidx != -1 && !hit && at <= full) e.S3(s.cache_normal, pidx, zero3());
      if (hit) {
        if (at < m.max_broad) e.I(s.broad_pairs, at) = (ga << 16) | gb;
        else overflow = true;
      }
      base += __popcll(b);
    }
  }
  overflow = env_ballot<W>(overflow) != 0ull;
  if (lane == 0) {
    e.I(s.n_broad, 0) = min(base, m.max_broad);
    if (overflow) e.I((int32_t*)s.errno_env, 0) |= (int)GSR_ERR_BROAD_OVERFLOW;
  }
  __syncthreads();
}

// a contact of the env's list, or the overflow bit
__device__ __forceinline__ void put_contact(const Env& e, int k, int ga, int gb, f3 n, f3 p, float pen, uint32_t& err) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  if (k >= m.max_contacts) {
    err |= GSR_ERR_CONTACT_OVERFLOW;
    return;
  }
  e.I(s.contact_geoms, 2 * k) = ga;
  e.I(s.contact_geoms, 2 * k + 1) = gb;
  e.S3(s.contact_normal, k, n);
  e.S3(s.contact_pos, k, p);
  e.F(s.contact_pen, k) = pen;
  e.F(s.contact_friction, k) = fmaxf(fmaxf(m.geom_friction[ga] * e.F(s.friction_ratio, ga),
                                           m.geom_friction[gb] * e.F(s.friction_ratio, gb)), 1e-2f);
}
// records of the pairs that need GJK/EPA, with the index their contacts go to
template <int W>
__device__ __forceinline__ void defer_pairs(const Env& e, int lane, bool deferred, int pr, int k, int& n_def) {
  const unsigned long long def = env_ballot<W>(deferred);
  if (deferred) {
    const int slot = n_def + __popcll(def & ((1ull << lane) - 1ull));
    e.I(e.s.gjk_defer, 2 * slot) = pr;
    e.I(e.s.gjk_defer, 2 * slot + 1) = min(k, e.m.max_contacts);
  }
  n_def += __popcll(def);
}
// geoms of a pair in type order
__device__ __forceinline__ void pair_geoms(const gsr_model& m, int pr, int& ga, int& gb) {
  ga = pr >> 16;
  gb = pr & 0xffff;
  if (m.geom_type[ga] > m.geom_type[gb]) { int t = ga; ga = gb; gb = t; }
}

// Up to W pairs of one kind (q[lane], lane < cnt), a pair per lane, contacts appended at `base`.
// kGjk: pairs that need GJK/EPA are redone in place, one lane at a time (they share the env's workspace), instead of
// being deferred to the GJK/EPA pass
template <bool kGjk, int W>
__device__ inline int wave_pairs(const Env& e, int lane, const int* q, int cnt, bool plane_box, int base,
                                 uint32_t& err) {
  PairContacts pc;
  pc.cnt = 0;
  pc.err = 0;
  pc.deferred = false;
  int ga = 0, gb = 0;
  if (lane < cnt) {
    pair_geoms(e.m, q[lane], ga, gb);
    LocalSink<false> snk{pc};
    if (plane_box) dev_plane_box(e, ga, gb, snk);
    else if constexpr (kGjk) dev_convex_convex(e, ga, gb, snk);
  }
  if constexpr (kGjk) {
    unsigned long long redo = env_ballot<W>(pc.deferred);
    while (redo) {
      int j = __ffsll((long long)redo) - 1;
      redo &= redo - 1;
      if (lane == j) {
        pc.cnt = 0;
        pc.err = 0;
        pc.deferred = false;
        LocalSink<true> snk{pc};
        dev_convex_convex(e, ga, gb, snk);
      }
    }
  }
  int total;
  const int k = base + wave_excl_scan<W>(pc.cnt, lane, total);
  for (int c = 0; c < pc.cnt; c++) put_contact(e, k + c, ga, gb, pc.n[c], pc.p[c], pc.pen[c], err);
  err |= pc.err;
  return base + total;
}

// Up to W convex pairs (q[lane], lane < cnt): the first detection with a pair per lane, then the turned detections of the
// pairs that touch with a detection per lane, four lanes beside each other for a pair. They depend on the first alone,
// except that a contact near an earlier one of its pair is dropped, which the four lanes settle among themselves. lds: 30 W
// words; the turned contacts wait there too. What bounds it is the chain of support points of one detection: a pair's five in turn on its lane, with the
// lanes of other pairs idle, were most of a heap's collision. Measured (us, collision and GJK/EPA pass, a pair per lane ->
// this): 20-box piles 300: 172 -> 106, 1,500: 193 -> 145, 4,000: 403 -> 325; 1,024 64-box piles 566 -> 388.
template <int W>
__device__ inline int wave_convex(const Env& e, int lane, const int* q, int cnt, float* lds, int base, uint32_t& err,
                                  int& n_def) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  // of each touching pair: first contact, its normal and the two axes (12 words), then 7 words of each turned contact in
  // their place; the pair's geoms in the last word
  constexpr int kPair = 29;
  int* count = reinterpret_cast<int*>(lds + kPair * W);  // which turned contacts stay (4 bits, -1: deferred), first index << 4
  PairContacts none;
  LocalSink<false> snk{none};
  int ga = 0, gb = 0;
  Detection o;
  o.is_col = false;
  bool deferred = false, turn = false;
  f3 ax0 = zero3(), ax1 = zero3();
  if (lane < cnt) {
    pair_geoms(m, q[lane], ga, gb);
    const GPose A{e.L3(s.geoms_pos, ga), e.L4(s.geoms_quat, ga)}, Bp{e.L3(s.geoms_pos, gb), e.L4(s.geoms_quat, gb)};
    deferred = !dev_detect(e, ga, gb, A, Bp, true, e.L3(s.cache_normal, dev_pair_index(m, ga, gb)),
                           dev_tolerance(m, ga, gb, m.mc_tolerance), snk, o);
    turn = !deferred && o.is_col && dev_multi_contact(m, ga, gb);
    if (turn) dev_contact_orthogonals(e, ga, gb, o.normal, ax0, ax1);
  }
  const unsigned long long turned = env_ballot<W>(turn);
  const int n_turn = __popcll(turned), rank = __popcll(turned & ((1ull << lane) - 1ull));
  __syncthreads();
  if (turn) {
    const float v[12] = {o.pos.x, o.pos.y, o.pos.z, o.normal.x, o.normal.y, o.normal.z, ax0.x, ax0.y, ax0.z, ax1.x, ax1.y, ax1.z};
    for (int j = 0; j < 12; j++) lds[kPair * rank + j] = v[j];
    lds[kPair * rank + 28] = __int_as_float(q[lane]);
  }
  __syncthreads();
#pragma unroll 1
  for (int t0 = 0; t0 < 4 * n_turn; t0 += W) {
    const int t = t0 + lane, k = t >> 2, quad = t & 3;
    Detection d;
    d.is_col = false;
    d.pen = 0.f;
    d.pos = d.normal = zero3();
    bool def = false;
    float tol = 0.f;
    f3 p0 = zero3();
    float* v = lds + kPair * min(k, W - 1);
    if (k < n_turn) {
      p0 = f3{v[0], v[1], v[2]};
      const f3 n0{v[3], v[4], v[5]}, a0{v[6], v[7], v[8]}, a1{v[9], v[10], v[11]};
      int ta, tb;
      pair_geoms(m, __float_as_int(v[28]), ta, tb);
      tol = dev_tolerance(m, ta, tb, m.mc_tolerance);
      GPose A{e.L3(s.geoms_pos, ta), e.L4(s.geoms_quat, ta)}, Bp{e.L3(s.geoms_pos, tb), e.L4(s.geoms_quat, tb)};
      const q4 qr = dev_perturb(m, quad + 1, p0, a0, a1, A, Bp);
      def = !dev_detect(e, ta, tb, A, Bp, false, n0, tol, snk, d);
      if (!def && d.is_col) dev_unperturb(m, d, qr, p0, n0);
    }
    // which of the pair's four are contacts, in order, each against those before it
    const bool cand = !def && d.is_col && d.pen > -tol;
    f3 at[4];
    unsigned keep = 0, bad = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      at[j] = f3{__shfl(d.pos.x, j, 4), __shfl(d.pos.y, j, 4), __shfl(d.pos.z, j, 4)};
      bad |= __shfl((int)def, j, 4);
      bool c = __shfl((int)cand, j, 4) != 0 && !(norm(at[j] - p0) < tol);
#pragma unroll
      for (int i = 0; i < j; i++) c = c && !((keep >> i & 1u) && norm(at[j] - at[i]) < tol);
      keep |= (unsigned)c << j;
    }
    __syncthreads();
    if (k < n_turn) {
      if (quad == 0) count[k] = bad ? -1 : (int)keep;
      const float w[7] = {d.normal.x, d.normal.y, d.normal.z, d.pos.x, d.pos.y, d.pos.z, fmaxf(d.pen, 0.f)};
      for (int j = 0; j < 7; j++) v[7 * quad + j] = w[j];
    }
  }
  __syncthreads();
  int n = 0;
  if (lane < cnt && !deferred) {
    n = o.is_col ? 1 : 0;
    if (turn) {
      const int c = count[rank];
      deferred = c < 0;
      n = deferred ? 0 : n + __popc((unsigned)c);
    }
    if (!deferred) e.S3(s.cache_normal, dev_pair_index(m, ga, gb), o.is_col ? o.normal : zero3());
  }
  int total;
  const int k = base + wave_excl_scan<W>(n, lane, total);
  defer_pairs<W>(e, lane, deferred, (ga << 16) | gb, k, n_def);
  __syncthreads();
  if (turn) count[rank] = (k << 4) | (n > 0 ? count[rank] : 0);
  if (n > 0) put_contact(e, k, ga, gb, o.normal, o.pos, o.pen, err);
  __syncthreads();
  for (int t = lane; t < 4 * n_turn; t += W) {
    const int c = count[t >> 2], quad = t & 3;
    if (!(c >> quad & 1)) continue;
    const float* v = lds + kPair * (t >> 2);
    const float* w = v + 7 * quad;
    int ta, tb;
    pair_geoms(m, __float_as_int(v[28]), ta, tb);
    put_contact(e, (c >> 4) + 1 + __popc((unsigned)c & ((1u << quad) - 1u)), ta, tb, f3{w[0], w[1], w[2]}, f3{w[3], w[4], w[5]},
                w[6], err);
  }
  __syncthreads();
  return base + total;
}

// The broadphase pairs of one kind (convex pairs, or plane-box pairs), W at a time: they are gathered in a queue first,
// since the two kinds come mixed
template <bool kGjk, int W>
__device__ inline int wave_narrow_pass(const Env& e, int lane, float* lds, int nb, bool plane_box_pass, int base,
                                       uint32_t& err, int& n_def) {
  const gsr_model& m = e.m;
  int* q = reinterpret_cast<int*>(lds) + 30 * W;
  int n = 0;
  for (int p0 = 0; p0 < nb || n > 0; p0 += W) {
    const int ip = p0 + lane;
    int pr = 0;
    bool mine = false;
    if (ip < nb) {
      pr = e.I(e.s.broad_pairs, ip);
      int ga, gb;
      pair_geoms(m, pr, ga, gb);
      mine = (m.geom_type[ga] == GEOM_PLANE && m.geom_type[gb] == GEOM_BOX) == plane_box_pass;
    }
    const unsigned long long b = env_ballot<W>(mine);
    if (mine) q[n + __popcll(b & ((1ull << lane) - 1ull))] = pr;
    n += __popcll(b);
    __syncthreads();
    if (n < W && p0 + W < nb) continue;
    if (n == 0) break;
    const int cnt = min(n, W);
    if constexpr (kGjk) {
      base = wave_pairs<true, W>(e, lane, q, cnt, plane_box_pass, base, err);
    } else {
      if (plane_box_pass) base = wave_pairs<false, W>(e, lane, q, cnt, true, base, err);
      else base = wave_convex<W>(e, lane, q, cnt, lds, base, err, n_def);
    }
    n -= cnt;
    const int left = lane < n ? q[W + lane] : 0;
    __syncthreads();
    if (lane < n) q[lane] = left;
    __syncthreads();
  }
  return base;
}

template <bool kGjk, int W>
__device__ inline void wave_narrow_phase(const Env& e, char* lds, int lane) {
  const gsr_state& s = e.s;
  float* w = reinterpret_cast<float*>(lds);
  const int nb = e.I(s.n_broad, 0);
  uint32_t err = 0;
  int n_def = 0;
  int n = wave_narrow_pass<kGjk, W>(e, lane, w, nb, false, 0, err, n_def);
  n = wave_narrow_pass<kGjk, W>(e, lane, w, nb, true, n, err, n_def);
  for (int o = W / 2; o > 0; o >>= 1) err |= (uint32_t)__shfl_xor((int)err, o, W);
  if (lane == 0) {
    e.I(s.n_contacts, 0) = min(n, e.m.max_contacts);
    e.I(s.gjk_defer_n, 0) = n_def;
    if (err) e.I((int32_t*)s.errno_env, 0) |= (int)err;
  }
  __syncthreads();
}

// frictionloss and limit rows with a link per lane (counted, then placed by a prefix sum, so the rows come in link
// order), the 4 rows of each contact on its own lane. One lane walking every dof's tables took longer than the contacts.
template <int W = 64>
__device__ __forceinline__ void wave_rows(const Env& e) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const int lane = threadIdx.x & (W - 1);
  const int n_eq = e.I(s.n_con, 0);
  int n_con = n_eq;
  for (int l0 = 0; l0 < m.n_links; l0 += W) {
    const int l = l0 + lane;
    int cnt = 0, total = 0;
    if (l < m.n_links) each_frictionloss(e, l, [&](int, int) { cnt++; });
    if (env_ballot<W>(cnt != 0) == 0ull) continue;
    int c = n_con + wave_excl_scan<W>(cnt, lane, total);
    if (cnt) each_frictionloss(e, l, [&](int j, int d) { dev_frictionloss_row(e, j, d, c++); });
    n_con += total;
  }
  const int n_fl = n_con - n_eq;
  if (m.enable_collision) {
    int nc = e.I(s.n_contacts, 0);
    for (int ic = lane; ic < nc; ic += W) dev_contact_rows(e, ic, n_con + 4 * ic);
    n_con += 4 * nc;
  }
  for (int l0 = 0; m.enable_joint_limit && l0 < m.n_links; l0 += W) {
    const int l = l0 + lane;
    int cnt = 0, total = 0;
    if (l < m.n_links) each_limit(e, l, [&](int, int, float, float) { cnt++; });
    if (env_ballot<W>(cnt != 0) == 0ull) continue;
    int c = n_con + wave_excl_scan<W>(cnt, lane, total);
    if (cnt) each_limit(e, l, [&](int j, int d, float dmin, float dmax) { dev_limit_row(e, j, d, dmin, dmax, c++); });
    n_con += total;
  }
  if (lane == 0) {
    e.I(s.n_con, 0) = n_con;
    e.I(s.n_con, 2) = n_fl;
  }
  __syncthreads();
}

// equality rows, collision detection and inequality rows of one env (k_collide's work) on the W lanes holding it; lds: the
// env's words
template <bool kGjk = false, int W = 64>
__device__ __forceinline__ void wave_collide(const Env& e, char* lds) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const int lane = threadIdx.x & (W - 1);
  if (lane == 0) {
    dev_equality_rows(e);
    e.I(s.n_contacts, 0) = 0;
    e.I(s.n_broad, 0) = 0;
    e.I(s.gjk_defer_n, 0) = 0;
  }
  if (m.enable_collision) {
    dev_update_aabbs(e, lane, W, reinterpret_cast<float*>(lds) + 10 * m.n_geoms);
    __syncthreads();
    if (m.n_pairs > 0) {
      wave_broad_phase<W>(e, lds, lane);
      wave_narrow_phase<kGjk, W>(e, lds, lane);
    }
  }
  __syncthreads();
  // with deferred pairs the contact list is not final yet: the GJK/EPA pass builds the rows after inserting them
  if (e.I(s.gjk_defer_n, 0) > 0) return;
  wave_rows<W>(e);
}

// The GJK/EPA pass of one env on one wavefront: lane 0 recomputes the deferred pairs with GJK/EPA (they share the
// env's workspace), last first; the contacts above each pair's insertion index move up across the lanes (64 at a
// time from the top: every lane reads before any writes), and lane 0 writes the pair's contacts in the gap.
// Contacts pushed past max_contacts are dropped with the overflow bit, as the one-pass narrowphase drops them.
// Returns whether the env had deferred pairs (uniform).
__device__ inline bool wave_gjk_fixup(const Env& e) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const int lane = threadIdx.x;
  const int nd = e.I(s.gjk_defer_n, 0);
  if (nd == 0) return false;
  __syncthreads();
  for (int j = nd - 1; j >= 0; j--) {
    const int pr = e.I(s.gjk_defer, 2 * j), at = e.I(s.gjk_defer, 2 * j + 1);
    const int ga = pr >> 16, gb = pr & 0xffff;
    PairContacts pc;
    pc.cnt = 0;
    pc.err = 0;
    pc.deferred = false;
    if (lane == 0) {
      LocalSink<true> snk{pc};
      dev_convex_convex(e, ga, gb, snk);
      if (pc.err) e.I((int32_t*)s.errno_env, 0) |= (int)pc.err;
    }
    const int cnt = __shfl(pc.cnt, 0, 64);
    if (cnt == 0) continue;
    const int n = e.I(s.n_contacts, 0);
    const int kept = min(n + cnt, m.max_contacts);
    for (int top = n; top > at; top -= 64) {
      const int i = top - 1 - lane;
      const bool act = i >= at;
      int g0 = 0, g1 = 0;
      f3 cp = zero3(), cn = zero3();
      float pe = 0.f, fr = 0.f;
      if (act) {
        g0 = e.I(s.contact_geoms, 2 * i);
        g1 = e.I(s.contact_geoms, 2 * i + 1);
        cp = e.L3(s.contact_pos, i);
        cn = e.L3(s.contact_normal, i);
        pe = e.F(s.contact_pen, i);
        fr = e.F(s.contact_friction, i);
      }
      __syncthreads();
      const int t = i + cnt;
      if (act && t < kept) {
        e.I(s.contact_geoms, 2 * t) = g0;
        e.I(s.contact_geoms, 2 * t + 1) = g1;
        e.S3(s.contact_pos, t, cp);
        e.S3(s.contact_normal, t, cn);
        e.F(s.contact_pen, t) = pe;
        e.F(s.contact_friction, t) = fr;
      }
      __syncthreads();
    }
    if (lane == 0) {
      if (n + cnt > m.max_contacts) e.I((int32_t*)s.errno_env, 0) |= (int)GSR_ERR_CONTACT_OVERFLOW;
      const float fr = fmaxf(fmaxf(m.geom_friction[ga] * e.F(s.friction_ratio, ga),
                                   m.geom_friction[gb] * e.F(s.friction_ratio, gb)), 1e-2f);
      for (int c = 0; c < cnt; c++) {
        const int t = at + c;
        if (t >= kept) break;
        e.I(s.contact_geoms, 2 * t) = ga;
        e.I(s.contact_geoms, 2 * t + 1) = gb;
        e.S3(s.contact_pos, t, pc.p[c]);
        e.S3(s.contact_normal, t, pc.n[c]);
        e.F(s.contact_pen, t) = pc.pen[c];
        e.F(s.contact_friction, t) = fr;
      }
      e.I(s.n_contacts, 0) = kept;
    }
    __syncthreads();
  }
  if (lane == 0) e.I(s.gjk_defer_n, 0) = 0;
  __syncthreads();
  return true;
}

}  // namespace gsr
