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

// LDS words of one env
__host__ __device__ inline size_t wave_collide_words(int G) { return 16 * (size_t)G + 4; }
__host__ __device__ inline size_t wave_collide_lds_bytes(int G, int envs = 1) {
  return sizeof(float) * wave_collide_words(G) * (size_t)envs + 64;
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
// 4213, 172, 354; 4,000: 4437, 403, 448; 64 boxes 1,024: 25968, 566, 1529.
__host__ __device__ inline int collide_lanes(const gsr_model& m, int n) { return n > 2048 && collide_packs(m) ? 16 : kWave; }

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
  // geoms in the order of their min events: order[k] (tv's place), the AABBs in LDS. The geoms a min event pairs with are
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

// one pass over the broadphase pairs of one kind (convex pairs, then plane-box pairs), contacts appended at `base`
// kGjk: pairs that need GJK/EPA are redone in place, one lane at a time (they share the env's workspace), instead of
// being deferred to the GJK/EPA pass
template <bool kGjk, int W>
__device__ inline int wave_narrow_pass(const Env& e, int lane, int nb, bool plane_box_pass, int base,
                                       uint32_t& err, int& n_def) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  for (int p0 = 0; p0 < nb; p0 += W) {
    const int ip = p0 + lane;
    PairContacts pc;
    pc.cnt = 0;
    pc.err = 0;
    pc.deferred = false;
    int ga = 0, gb = 0;
    bool pb = false;
    if (ip < nb) {
      int pr = e.I(s.broad_pairs, ip);
      ga = pr >> 16;
      gb = pr & 0xffff;
      if (m.geom_type[ga] > m.geom_type[gb]) { int t = ga; ga = gb; gb = t; }
      pb = m.geom_type[ga] == GEOM_PLANE && m.geom_type[gb] == GEOM_BOX;
      if (pb == plane_box_pass) {
        LocalSink<false> snk{pc};
        if (pb) dev_plane_box(e, ga, gb, snk);
        else dev_convex_convex(e, ga, gb, snk);
      }
    }
    if (kGjk) {
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
    // a pair that needs GJK/EPA contributes no contact here; it is recorded with the index its contacts go to
    if (pc.deferred) {
      pc.cnt = 0;
      pc.err = 0;
    }
    const unsigned long long def = env_ballot<W>(pc.deferred);
    int total;
    int k = base + wave_excl_scan<W>(pc.cnt, lane, total);
    if (pc.deferred) {
      const int slot = n_def + __popcll(def & ((1ull << lane) - 1ull));
      e.I(s.gjk_defer, 2 * slot) = (ga << 16) | gb;
      e.I(s.gjk_defer, 2 * slot + 1) = min(k, m.max_contacts);
    }
    n_def += __popcll(def);
    float fr = fmaxf(fmaxf(m.geom_friction[ga] * e.F(s.friction_ratio, ga),
                           m.geom_friction[gb] * e.F(s.friction_ratio, gb)), 1e-2f);
    for (int c = 0; c < pc.cnt; c++, k++) {
      if (k < m.max_contacts) {
        e.I(s.contact_geoms, 2 * k) = ga;
        e.I(s.contact_geoms, 2 * k + 1) = gb;
        e.S3(s.contact_normal, k, pc.n[c]);
        e.S3(s.contact_pos, k, pc.p[c]);
        e.F(s.contact_pen, k) = pc.pen[c];
        e.F(s.contact_friction, k) = fr;
      } else {
        pc.err |= GSR_ERR_CONTACT_OVERFLOW;
      }
    }
    err |= pc.err;
    base += total;
  }
  return base;
}

template <bool kGjk, int W>
__device__ inline void wave_narrow_phase(const Env& e, int lane) {
  const gsr_model& m = e.m;
  const gsr_state& s = e.s;
  const int nb = e.I(s.n_broad, 0);
  uint32_t err = 0;
  int n_def = 0;
  int n = wave_narrow_pass<kGjk, W>(e, lane, nb, false, 0, err, n_def);
  n = wave_narrow_pass<kGjk, W>(e, lane, nb, true, n, err, n_def);
  for (int o = W / 2; o > 0; o >>= 1) err |= (uint32_t)__shfl_xor((int)err, o, W);
  if (lane == 0) {
    e.I(s.n_contacts, 0) = min(n, m.max_contacts);
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
      wave_narrow_phase<kGjk, W>(e, lane);
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
