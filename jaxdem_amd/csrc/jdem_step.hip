// jdem_step.hip -- (b) neighbour traversal with the pair laws and (c) the
// fused integration of one DEM time step on gfx950.
//
// The candidates of particle i are walked by a group of lanes or, in large
// systems, by one, a neighbour-list row always by one; F_i and T_i are summed
// in the reference's traversal order either way -- no atomics, so results are
// deterministic run to run.  The same kernel then applies
// ForceManager, step_after_force of step k, and domain.apply +
// step_before_force of step k+1 (system.py:60-82), writing positions and
// velocities to the other half of a ping-pong pair because neighbours of
// i still read the step-k values.
//
// Reference: colliders/naive.py:190-235, cell_list.py:188-261, 437-496,
// neighbor_list.py:594-669; forces/force_manager.py:341-425;
// integrators/velocity_verlet.py:57-94, direct_euler.py:62-65,
// velocity_verlet_spiral.py:83-180, spiral.py:60-144; domains/reflect.py:
// 102-297.
#include <hip/hip_runtime.h>

#include "jdem_internal.h"

namespace jdem {

template <class Real>
JD void to_arr_a(Vec<3, Real> v, Real* x) {
  to_arr(v, x);
}
template <class Real>
JD void to_arr_a(Ang1T<Real> v, Real* x) {
  x[0] = v.z;
}
template <class Real>
JD void from_arr_a(Vec<3, Real>& v, const Real* x) {
  from_arr(v, x);
}
template <class Real>
JD void from_arr_a(Ang1T<Real>& v, const Real* x) {
  v.z = x[0];
}

template <class Real>
JD bool is_bonded(const StepArgsT<Real>& a, int64_t i, int32_t j) {
  for (int w = 0; w < a.bond_w; ++w)
    if (a.bond_id[i * a.bond_w + w] == j) return true;
  return false;
}

template <int LAW, class Real>
JD int species_of(const LawPT<Real>& L, int64_t i) {
  if constexpr (LawTraits<LAW>::routed) return L.species ? L.species[i] : 0;
  return 0;
}

template <int D, int LAW, class Real>
JD void fill_partner(const StepArgsT<Real>& a, Side<D, Real>& b, int32_t j) {
  if (a.law.n_mat > 1) b.mat = a.mat_id[j];
  b.sp = species_of<LAW>(a.law, j);
  if constexpr (LawTraits<LAW>::kin) {
    b.v = ld<D>(a.vel_in, j);
    b.w = lda<D>(a.ang_in, j);
    b.m = a.mass[j];
  }
}

// The pair (i <- j) may touch: |rij| is within the law's reach (a margin over
// the law's own overlap test; past it delta of every law is exactly 0).
template <class Real>
JD bool in_reach(Real d_sq, Real R) {
  return !(d_sq > (R * R) * Real(1.0001));
}

// valid_interaction_mask: not the particle itself (its clump), not bonded
template <class Real>
JD bool may_interact(const StepArgsT<Real>& a, int64_t i, int32_t j) {
  if (a.clump ? a.clump[j] == a.clump[i] : j == (int32_t)i) return false;
  return a.isb || a.bond_w == 0 || !is_bonded(a, i, j);
}

// Evaluate the pair (i <- j) and accumulate.  Returns true if in contact.
template <int D, int LAW, bool PER, class Real>
JD bool visit(const StepArgsT<Real>& a, const Side<D, Real>& me, int64_t i, int32_t j, const Vec<D, Real>& xj,
              Real rj, Vec<D, Real>& F, Ang<D, Real>& T, const Vec<D, Real>& xi_old, Vec<D, Real>& xi_new) {
  const Vec<D, Real> rij = disp_<PER>(me.x, xj, a.dom);
  const Real d_sq = dot(rij, rij);
  if (!in_reach(d_sq, me.r + rj)) return false;
  if (!may_interact(a, i, j)) return false;
  Side<D, Real> b;
  b.x = xj;
  b.r = rj;
  b.mat = 0;
  fill_partner<D, LAW>(a, b, j);
  PairOut<D, Real> o = law_eval<D, LAW>(a.law, me, b, rij, d_sq, xi_old, a.dt);
  F = F + o.F;
  if constexpr (LawTraits<LAW>::torque) T = T + o.T;
  if constexpr (LawTraits<LAW>::hist) xi_new = o.xi;
  return o.contact;
}

// ---------------------------------------------------------------------------
// candidates of the cell list and of the naive collider
// ---------------------------------------------------------------------------
// A group of G lanes serves one particle.  For the cell list each lane loads
// the bounds of one stencil column, a scan over the group numbers the
// columns' candidates, and the group tests G of them at a time; the naive
// collider tests G consecutive particles at a time.  Candidates within reach
// are queued in LDS in candidate order, and `flush(n)` takes the first n of
// the queue: their pairs are evaluated one per lane and added up in queue
// order, so every sum is that of one lane walking all candidates in the
// reference's order (stencil order, ascending id within a cell).
//
// One lane per particle instead is a serial chain of dependent loads (27 cell
// bounds, then the candidates one by one), and below ~10^5 particles there
// are not even enough wavefronts to hide it.  Measured: the step kernel of
// 1000 spheres with the naive collider 145 -> 17 us (a step of 64 39 -> 23 us, of
// 30 k 5.1 -> 0.9 ms), of 16 k spheres with the cell list 61 -> 12 us, its energy
// kernel 58 -> 10 us.
//
// G: a 3D stencil holds about 40 candidates (27 cells of about 1.4), so 16
// lanes take it in three rounds; a 2D one holds about 13, two rounds of 8.
template <int D, int SRC>
constexpr int group_lanes() {
  return SRC == SRC_NAIVE ? 64 : (D == 3 ? 16 : 8);
}
template <int D, int SRC>
constexpr int queue_len() {
  return 2 * (group_lanes<D, SRC>() < 16 ? 16 : group_lanes<D, SRC>());
}

// The stencil of one cell as columns along the fastest axis, in the
// reference's 'ij' order (cell_list.py:425-427); a column is one run of the
// sorted particles, or two where a periodic axis wraps.
template <int D, bool PER>
struct ColumnWalk {
  int c0, c1, n1, ncol, r0a, r0b, r1a, r1b;
  template <class Real>
  JD void start(const GridPT<Real>& g, uint32_t key) {
    const int d0 = g.dims[0], d1 = g.dims[1], d2 = (D == 3) ? g.dims[2] : 1;
    int cf;
    if constexpr (D == 3) {
      cf = (int)(key % (uint32_t)d2);
      const uint32_t q = key / (uint32_t)d2;
      c1 = (int)(q % (uint32_t)d1);
      c0 = (int)(q / (uint32_t)d1);
    } else {
      cf = (int)(key % (uint32_t)d1);
      c0 = (int)(key / (uint32_t)d1);
      c1 = 0;
    }
    const int sr = g.sr;
    stencil_runs(PER, cf, sr, D == 3 ? d2 : d1, r0a, r0b, r1a, r1b);
    n1 = (D == 3) ? (PER ? min(sr, d1 - sr - 1) : sr) + sr + 1 : 1;
    ncol = ((PER ? min(sr, d0 - sr - 1) : sr) + sr + 1) * n1;
  }
  // first slots and lengths of column `col`'s two runs (0 off the grid)
  template <class Real>
  JD void bounds(const GridPT<Real>& g, const int32_t* __restrict__ starts, int col, int& s0, int& len0, int& s1,
                 int& len1) const {
    s0 = len0 = s1 = len1 = 0;
    if (col >= ncol) return;
    const int d0 = g.dims[0], d1 = g.dims[1];
    const int cx = stencil_cell(PER, c0, (D == 3 ? col / n1 : col) - g.sr, d0);
    const int cy = (D == 3) ? stencil_cell(PER, c1, col % n1 - g.sr, d1) : 0;
    if (cx < 0 || cy < 0) return;
    const int64_t base = (D == 3) ? ((int64_t)cx * d1 + cy) * g.dims[2] : (int64_t)cx * d1;
    s0 = starts[base + r0a];
    len0 = starts[base + r0b + 1] - s0;
    if (r1b >= r1a) {
      s1 = starts[base + r1a];
      len1 = starts[base + r1b + 1] - s1;
    }
  }
};

JD float4 cand_of(const float4* spos, int64_t k) { return spos[k]; }
JD Double4 cand_of(const Double4* spos, int64_t k) { return spos[k]; }

// position, radius and id of candidate k: a cell-sorted slot, or a particle
template <int D, int SRC, class Real>
JD void load_cand(const StepArgsT<Real>& a, int64_t k, Vec<D, Real>& x, Real& r) {
  if constexpr (SRC == SRC_CELLS) {
    const Real4<Real> p = cand_of(a.spos, k);
    if constexpr (D == 3)
      x = Vec<3, Real>{p.x, p.y, p.z};
    else
      x = Vec<2, Real>{p.x, p.y};
    r = p.w;
  } else {
    x = ld<D>(a.pos_in, k);
    r = a.rad[k];
  }
}
template <int SRC, class Real>
JD int32_t cand_id(const StepArgsT<Real>& a, int64_t k) {
  return SRC == SRC_CELLS ? a.perm[k] : (int32_t)k;
}

// FAR: an infinite squared distance counts as within reach (the energy and
// virial kernels, whose laws then return what they return there).  `queue`
// holds queue_len entries of this group; every lane of the group calls.
template <int D, int SRC, bool PER, bool FAR, class Real, class Flush>
JD void walk_candidates(const StepArgsT<Real>& a, int64_t idx, int64_t i, const Vec<D, Real>& x, Real r, int* queue,
                        Flush&& flush) {
  constexpr int G = group_lanes<D, SRC>();
  const int lane = threadIdx.x & 63, l = lane & (G - 1);
  const uint64_t below = (1ull << l) - 1ull;
  int nq = 0;
  ColumnWalk<D, PER> cols;
  if constexpr (SRC == SRC_CELLS) cols.start(a.grid, (uint32_t)a.skeys[idx]);
  int cb = -G, total = 0, b = 0;                // columns cb.. of the group, candidates b.. of their total
  int s0 = 0, len0 = 0, s1 = 0, len1 = 0, pre = 0;  // this lane's column
  int64_t k0 = 0;
  for (bool done = false; !done;) {
    bool in = false;
    int k = 0;
    if constexpr (SRC == SRC_NAIVE) {
      in = k0 + l < a.n;
      k = (int)(k0 + l);
      k0 += G;
      done = k0 >= a.n;
    } else if (b < total) {
      // candidate b + l lies in the last column whose prefix is not above it
      const int c = b + l;
      int q = 0;
#pragma unroll
      for (int st = G / 2; st > 0; st >>= 1) q += __shfl(pre, q + st, G) <= c ? st : 0;
      const int o = c - __shfl(pre, q, G), f0 = __shfl(s0, q, G), n_0 = __shfl(len0, q, G), f1 = __shfl(s1, q, G);
      in = c < total;
      k = o < n_0 ? f0 + o : f1 + (o - n_0);
      b += G;
      done = b >= total && cb + G >= cols.ncol;
    } else {
      cb += G;
      cols.bounds(a.grid, a.cstart, cb + l, s0, len0, s1, len1);
      int incl = len0 + len1;
#pragma unroll
      for (int d = 1; d < G; d <<= 1) {
        const int t = __shfl_up(incl, d, G);
        if (l >= d) incl += t;
      }
      pre = incl - (len0 + len1);
      total = __shfl(incl, G - 1, G);
      b = 0;
      done = total == 0 && cb + G >= cols.ncol;
    }
    bool hit = false;
    if (in) {
      Vec<D, Real> xj;
      Real rj;
      load_cand<D, SRC>(a, k, xj, rj);
      const Vec<D, Real> rij = disp_<PER>(x, xj, a.dom);
      const Real d_sq = dot(rij, rij);
      hit = in_reach(d_sq, r + rj) || (FAR && d_sq == Real(INFINITY));
      if (hit) hit = may_interact(a, i, cand_id<SRC>(a, k));
    }
    uint64_t m = __ballot(hit);
    if constexpr (G < 64) m = (m >> (lane & ~(G - 1))) & ((1ull << G) - 1ull);
    if (hit) queue[nq + __popcll(m & below)] = k;
    nq += __popcll(m);
    if (nq > queue_len<D, SRC>() - G || (done && nq > 0)) {
      wave_sync();
      flush(nq);
      wave_sync();
      nq = 0;
    }
  }
}

template <int G, class Real>
JD Vec<3, Real> group_get(Vec<3, Real> v, int src) {
  return {__shfl(v.x, src, G), __shfl(v.y, src, G), __shfl(v.z, src, G)};
}
template <int G, class Real>
JD Vec<2, Real> group_get(Vec<2, Real> v, int src) {
  return {__shfl(v.x, src, G), __shfl(v.y, src, G)};
}
template <int G, class Real>
JD Ang1T<Real> group_get(Ang1T<Real> v, int src) {
  return {__shfl(v.z, src, G)};
}

template <int D, int LAW, class Real>
JD void load_side(const StepArgsT<Real>& a, int64_t i, Side<D, Real>& me) {
  me.x = ld<D>(a.pos_in, i);
  me.r = a.rad[i];
  me.mat = (a.law.n_mat > 1) ? a.mat_id[i] : 0;
  me.sp = species_of<LAW>(a.law, i);
  me.v = ld<D>(a.vel_in, i);
  me.w = lda<D>(a.ang_in, i);
  me.m = a.mass[i];
}

// Calls use(o, rij, in) for the pairs of one flush, in groups of G: lane l
// holds the result of queue entry h0 + l (in: l < the entries left).
template <int D, int LAW, int SRC, bool PER, class Real, class Use>
JD void queued_pairs(const StepArgsT<Real>& a, const Side<D, Real>& me, const int* queue, int nq, Use&& use) {
  constexpr int G = group_lanes<D, SRC>();
  const int l = threadIdx.x & (G - 1);
  for (int h0 = 0; h0 < nq; h0 += G) {
    PairOut<D, Real> o;
    o.F = zero_vec<D, Real>();
    o.T = zero_ang<D, Real>();
    Vec<D, Real> rij = zero_vec<D, Real>();
    if (h0 + l < nq) {
      const int k = queue[h0 + l];
      Side<D, Real> b;
      load_cand<D, SRC>(a, k, b.x, b.r);
      b.mat = 0;
      fill_partner<D, LAW>(a, b, cand_id<SRC>(a, k));
      rij = disp_<PER>(me.x, b.x, a.dom);
      o = law_eval<D, LAW>(a.law, me, b, rij, dot(rij, rij), zero_vec<D, Real>(), a.dt);
    }
    use(o, rij, min(G, nq - h0));
  }
}

// Force and torque of the particle in sorted slot (or of id) idx; every lane
// of its group returns them.
template <int D, int LAW, int SRC, bool PER, class Real>
JD void group_force(const StepArgsT<Real>& a, int64_t idx, int64_t i, int* queue, Vec<D, Real>& F, Ang<D, Real>& T) {
  constexpr int G = group_lanes<D, SRC>();
  Side<D, Real> me;
  load_side<D, LAW>(a, i, me);
  F = zero_vec<D, Real>();
  T = zero_ang<D, Real>();
  walk_candidates<D, SRC, PER, false>(a, idx, i, me.x, me.r, queue, [&](int nq) {
    queued_pairs<D, LAW, SRC, PER>(a, me, queue, nq, [&](const PairOut<D, Real>& o, Vec<D, Real>, int cnt) {
      for (int q = 0; q < cnt; ++q) {
        F = F + group_get<G>(o.F, q);
        if constexpr (LawTraits<LAW>::torque) T = T + group_get<G>(o.T, q);
      }
    });
  });
}

// The same candidates with one lane per particle, for systems large enough
// to fill the chip that way: a lane walks its nine (2D: three) columns, four
// candidates at a time, and queues those within reach in LDS (kLaneQueue
// each); the wavefront's queued pairs are then numbered lane by lane and
// dealt out 64 at a time, one pair per lane, and each owner adds its results
// in queue order.  A candidate costs a third of the instructions of the
// lane-group walk (no search for its column, no half-empty rounds), which is
// what bounds the step once every SIMD has its wavefronts.
constexpr int kLaneQueue = 12;
template <int NR, class R>
struct LaneWalkLds {
  int queue[kLaneQueue][64];
  int pair[64];
  R res[NR][64];
};

// eval(o, k, out): the pair of owner lane o and candidate k (out: NR values);
// add(v): the owner takes the next pair's values.  Every lane of the wave
// calls; `on` is false for a lane without a particle.
template <int D, bool PER, bool FAR, int NR, class R, class Real, class Eval, class Add>
JD void lane_walk(const StepArgsT<Real>& a, bool on, int64_t idx, int64_t i, const Vec<D, Real>& x, Real r,
                  LaneWalkLds<NR, R>& lds, Eval&& eval, Add&& add) {
  const int lane = threadIdx.x & 63;
  ColumnWalk<D, PER> cols;
  cols.start(a.grid, on ? (uint32_t)a.skeys[idx] : 0u);
  int nq = 0;
  int s0, len0, s1, len1;
  cols.bounds(a.grid, a.cstart, on ? 0 : cols.ncol, s0, len0, s1, len1);
  for (int col = 0; col < cols.ncol; ++col) {  // uniform: the grid's column count
    int k = s0, ke = s0 + len0, k2 = s1, k2e = s1 + len1;
    // the next column's bounds are on their way while this one is walked
    cols.bounds(a.grid, a.cstart, on ? col + 1 : cols.ncol, s0, len0, s1, len1);
    for (bool more = true; more;) {
      if (k >= ke) {
        k = k2;
        ke = k2e;
        k2 = k2e = 0;
      }
      Vec<D, Real> xj[4];
      Real rj[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        xj[u] = zero_vec<D, Real>();
        rj[u] = Real(0);
        if (k + u < ke) load_cand<D, SRC_CELLS>(a, k + u, xj[u], rj[u]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (k + u >= ke) break;
        const Vec<D, Real> rij = disp_<PER>(x, xj[u], a.dom);
        const Real d_sq = dot(rij, rij);
        if (!in_reach(d_sq, r + rj[u]) && !(FAR && d_sq == Real(INFINITY))) continue;
        if (!may_interact(a, i, a.perm[k + u])) continue;
        lds.queue[nq][lane] = k + u;
        ++nq;
      }
      k += 4;
      more = __any(k < ke || k2 < k2e);
      if (__any(nq > kLaneQueue - 4) || (!more && col + 1 == cols.ncol)) {
        int incl = nq;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          const int t = __shfl_up(incl, d);
          if (lane >= d) incl += t;
        }
        const int off = incl - nq, total = __shfl(incl, 63);
        for (int c0 = 0; c0 < total; c0 += 64) {
          const int q0 = max(off, c0), q1 = min(off + nq, c0 + 64);
          for (int q = q0; q < q1; ++q) lds.pair[q - c0] = lane | (q - off) << 6;
          wave_sync();
          if (c0 + lane < total) {
            const int d = lds.pair[lane];
            R out[NR];
            eval(d & 63, lds.queue[d >> 6][d & 63], out);
#pragma unroll
            for (int c = 0; c < NR; ++c) lds.res[c][lane] = out[c];
          }
          wave_sync();
          for (int q = q0; q < q1; ++q) {
            R v[NR];
#pragma unroll
            for (int c = 0; c < NR; ++c) v[c] = lds.res[c][q - c0];
            add(v);
          }
          wave_sync();
        }
        nq = 0;
      }
    }
  }
}

// The pair of the particles in sorted slots s (owner) and k.
template <int D, int LAW, bool PER, class Real>
JD PairOut<D, Real> pair_of_slots(const StepArgsT<Real>& a, int64_t s, int64_t k, Vec<D, Real>& rij) {
  Side<D, Real> me, b;
  load_cand<D, SRC_CELLS>(a, s, me.x, me.r);
  load_cand<D, SRC_CELLS>(a, k, b.x, b.r);
  me.mat = 0;
  b.mat = 0;
  fill_partner<D, LAW>(a, me, a.perm[s]);
  fill_partner<D, LAW>(a, b, a.perm[k]);
  rij = disp_<PER>(me.x, b.x, a.dom);
  return law_eval<D, LAW>(a.law, me, b, rij, dot(rij, rij), zero_vec<D, Real>(), a.dt);
}

// Force of one particle from its row of the (N, M) neighbour list.
template <int D, int LAW, bool PER, class Real>
JD void row_force(const StepArgsT<Real>& a, int64_t i, const Side<D, Real>& me, Vec<D, Real>& F, Ang<D, Real>& T) {
  F = zero_vec<D, Real>();
  T = zero_ang<D, Real>();
  const int32_t* row = a.nl + i * a.M;
  for (int w = 0; w < a.W32; ++w) {
    uint32_t live_old = 0, live_new = 0;
    if constexpr (LawTraits<LAW>::hist) live_old = a.hist_live[i * a.W32 + w];
    const int s_end = min(a.M, (w + 1) * 32);
    bool done = false;
    for (int sl = w * 32; sl < s_end; ++sl) {
      const int32_t j = row[sl];
      if (j < 0) {
        done = true;
        break;
      }
      Vec<D, Real> xold = zero_vec<D, Real>();
      if constexpr (LawTraits<LAW>::hist) {
        if ((live_old >> (sl & 31)) & 1u) xold = ld<D>(a.hist_xi, i * a.M + sl);
      }
      Vec<D, Real> xnew;
      const bool c = visit<D, LAW, PER>(a, me, i, j, ld<D>(a.pos_in, j), a.rad[j], F, T, xold, xnew);
      if constexpr (LawTraits<LAW>::hist) {
        if (c) {
          st(a.hist_xi, i * a.M + sl, xnew);
          live_new |= 1u << (sl & 31);
        }
      }
    }
    if constexpr (LawTraits<LAW>::hist) a.hist_live[i * a.W32 + w] = live_new;
    if (done) {
      if constexpr (LawTraits<LAW>::hist)
        for (int w2 = w + 1; w2 < a.W32; ++w2) a.hist_live[i * a.W32 + w2] = 0u;
      break;
    }
  }
}

// The rest of a particle's step once its force F and torque T are known:
// phases of StepArgs (do_after runs ForceManager + step_after_force of step
// k; do_before runs domain.apply + step_before_force of step k+1 and the
// NeighborList displacement check).
template <int D, class Real>
JD void finish_particle(const StepArgsT<Real>& a, int64_t i, const Side<D, Real>& me, Vec<D, Real> F,
                        Ang<D, Real> T) {
  if (!a.write_kin) {  // Collider.compute_force only
    st(a.force, i, F);
    sta(a.torque, i, T);
    return;
  }
  Vec<D, Real> x = me.x, v = me.v;
  Ang<D, Real> w = me.w;
  QuatT<Real> q = ldq(a.q, i);
  const Ang<D, Real> I = lda<D>(a.inertia, i);
  const Real m = me.m;
  const bool fixed = a.fixed[i] != 0;
  const Real freef = fixed ? Real(0) : Real(1);
  if (a.do_after) {
    // ForceManager.apply for spheres (force_manager.py:358-424)
    if (a.has_fm) {
      Vec<D, Real> fp = a.ext_f ? ld<D>(a.ext_f, i) : zero_vec<D, Real>();
      Vec<D, Real> fc = a.ext_fc ? ld<D>(a.ext_fc, i) : zero_vec<D, Real>();
      Vec<D, Real> g;
      if constexpr (D == 3)
        g = Vec<3, Real>{a.g[0], a.g[1], a.g[2]};
      else
        g = Vec<2, Real>{a.g[0], a.g[1]};
      fc = fc + g * (m / Real(1));
      F = (F + fp) + fc;
      if (a.ext_t) T = T + lda<D>(a.ext_t, i);
    }
    // step_after_force
    if (a.lin == JDEM_LIN_VERLET) {
      const Real s = (a.dt * Real(0.5)) / m;
      v = v + (F * s) * freef;
    } else if (a.lin == JDEM_LIN_EULER) {
      const Real s = a.dt / m;
      v = v + (F * s) * freef;
      x = x + v * a.dt;
    }
    if (a.rot == JDEM_ROT_VERLET_SPIRAL)
      vvs_after<D>(q, w, T, I, a.dt, freef);
    else if (a.rot == JDEM_ROT_SPIRAL)
      spiral_after<D>(q, w, T, I, a.dt, freef);
  }
  if (a.do_before) {
    // domain.apply of step k+1 (reflect.py:102-297; free/periodic: no-op)
    if (a.dom.kind == JDEM_DOMAIN_REFLECT) reflect_apply<D>(a.dom, x, v, q, F, m, me.r, fixed, a.dt);
    // step_before_force of step k+1
    if (a.lin == JDEM_LIN_VERLET) {
      const Real s = (a.dt * Real(0.5)) / m;
      v = v + (F * s) * freef;
      x = x + v * a.dt;
    }
    if (a.rot == JDEM_ROT_VERLET_SPIRAL) vvs_before<D>(q, w, T, I, a.dt, freef);
  }
  st(a.pos_out, i, x);
  st(a.vel_out, i, v);
  sta(a.ang_out, i, w);
  stq(a.q, i, q);
  st(a.force, i, F);
  sta(a.torque, i, T);
  if (a.do_before && a.check_disp) {
    const Vec<D, Real> d = x - ld<D>(a.old_pos, i);
    if (dot(d, d) > a.trigger) *a.flag_wr = a.step_idx + 1;
  }
}

// The fused step kernel.  do_force computes F, T at the current positions
// (else they are read from force/torque).  A neighbour-list row is one lane's
// work, and so is a particle of SRC_CELLS_LANE (always do_force).  For
// SRC_CELLS and the naive collider a wavefront takes a.pw particles: its
// groups of lanes walk their candidates, 64 / G particles at a time, the sums
// go to LDS, and then each lane finishes one particle.
template <int D, int LAW, int SRC, bool PER, class Real>
__global__ void __launch_bounds__(kBlock) k_step(StepArgsT<Real> a) {
  if (a.flag_rd && *a.flag_rd) {  // a neighbour-list rebuild is pending
    if (a.flag_wr) *a.flag_wr = *a.flag_rd;
    return;
  }
  Vec<D, Real> F;
  Ang<D, Real> T;
  int64_t idx;
  if constexpr (SRC == SRC_NLIST) {
    idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= a.n) return;
  } else {
    constexpr int A = D == 3 ? 3 : 1;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t w0 = ((int64_t)xcd_tile(blockIdx.x, gridDim.x) * (kBlock / 64) + wv) * a.pw;
    if constexpr (SRC == SRC_CELLS_LANE) {
      __shared__ LaneWalkLds<D + A, Real> lds[kBlock / 64];
      const int64_t s = w0 + lane;
      const bool on = s < a.n;
      const int64_t i = a.perm[on ? s : 0];
      Side<D, Real> me;
      load_cand<D, SRC_CELLS>(a, on ? s : 0, me.x, me.r);
      F = zero_vec<D, Real>();
      T = zero_ang<D, Real>();
      lane_walk<D, PER, false>(
          a, on, s, i, me.x, me.r, lds[wv],
          [&](int o, int k, Real* out) {
            Vec<D, Real> rij;
            const PairOut<D, Real> r = pair_of_slots<D, LAW, PER>(a, w0 + o, k, rij);
            to_arr(r.F, out);
            to_arr_a(r.T, out + D);
          },
          [&](const Real* v) {
            Vec<D, Real> f;
            from_arr(f, v);
            F = F + f;
            if constexpr (LawTraits<LAW>::torque) {
              Ang<D, Real> t;
              from_arr_a(t, v + D);
              T = T + t;
            }
          });
    } else if (a.do_force && !a.force_zero) {
      constexpr int G = group_lanes<D, SRC>();
      __shared__ int queue[kBlock / G][queue_len<D, SRC>()];
      __shared__ Real sums[kBlock / 64][D + A][64];
      for (int p0 = 0; p0 < a.pw; p0 += 64 / G) {
        const int p = p0 + lane / G;
        const int64_t s = w0 + p;
        if (s < a.n) {
          const int64_t i = SRC == SRC_CELLS ? (int64_t)a.perm[s] : s;
          group_force<D, LAW, SRC, PER>(a, s, i, queue[threadIdx.x / G], F, T);
          if ((lane & (G - 1)) == 0) {
            Real f[D], t[A];
            to_arr(F, f);
            to_arr_a(T, t);
#pragma unroll
            for (int c = 0; c < D; ++c) sums[wv][c][p] = f[c];
#pragma unroll
            for (int c = 0; c < A; ++c) sums[wv][D + c][p] = t[c];
          }
        }
      }
      wave_sync();
      Real f[D], t[A];
#pragma unroll
      for (int c = 0; c < D; ++c) f[c] = sums[wv][c][lane];
#pragma unroll
      for (int c = 0; c < A; ++c) t[c] = sums[wv][D + c][lane];
      from_arr(F, f);
      from_arr_a(T, t);
    }
    idx = w0 + lane;
    if (lane >= a.pw || idx >= a.n) return;
  }
  const bool sorted = SRC == SRC_CELLS_LANE || (SRC == SRC_CELLS && a.do_force && !a.force_zero);
  const int64_t i = sorted ? (int64_t)a.perm[idx] : idx;
  Side<D, Real> me;
  load_side<D, LAW>(a, i, me);
  if (a.do_force && a.force_zero) {
    F = zero_vec<D, Real>();
    T = zero_ang<D, Real>();
  } else if (a.do_force) {
    if constexpr (SRC == SRC_NLIST) row_force<D, LAW, PER>(a, i, me, F, T);
    // clump member: the lever torque of its summed force (naive.py:231,
    // cell_list.py:462)
    if (a.ppr) T = T + cross_t(ld<D>(a.ppr, i), F);
  } else {
    F = ld<D>(a.force, i);
    T = lda<D>(a.torque, i);
  }
  finish_particle<D>(a, i, me, F, T);
}

// Potential energy: 1/2 sum of pair energies per particle, float64 sum.  Pairs
// out of reach have energy exactly 0.
template <int D, int LAW, int SRC, bool PER, class Real>
__global__ void __launch_bounds__(kBlock) k_energy(StepArgsT<Real> a) {
  if constexpr (SRC == SRC_NLIST) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    Side<D, Real> me;
    me.x = ld<D>(a.pos_in, i);
    me.r = a.rad[i];
    me.mat = (a.law.n_mat > 1) ? a.mat_id[i] : 0;
    me.sp = species_of<LAW>(a.law, i);
    double acc = 0.0;
    const int32_t* row = a.nl + i * a.M;
    for (int sl = 0; sl < a.M; ++sl) {
      const int32_t j = row[sl];
      if (j < 0) break;
      if (!may_interact(a, i, j)) continue;
      Side<D, Real> b;
      b.x = ld<D>(a.pos_in, j);
      b.r = a.rad[j];
      b.mat = (a.law.n_mat > 1) ? a.mat_id[j] : 0;
      b.sp = species_of<LAW>(a.law, j);
      const Vec<D, Real> rij = disp_<PER>(me.x, b.x, a.dom);
      acc += 0.5 * (double)law_energy<D, LAW>(a.law, me, b, dot(rij, rij));
    }
    a.e_out[i] = acc;
  } else if constexpr (SRC == SRC_CELLS_LANE) {
    __shared__ LaneWalkLds<1, double> lds[kBlock / 64];
    const int64_t w0 = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * kBlock + (threadIdx.x & ~63u);
    const int64_t s = w0 + (threadIdx.x & 63);
    const bool on = s < a.n;
    const int64_t i = a.perm[on ? s : 0];
    Side<D, Real> me;
    load_cand<D, SRC_CELLS>(a, on ? s : 0, me.x, me.r);
    double acc = 0.0;
    lane_walk<D, PER, true>(
        a, on, s, i, me.x, me.r, lds[threadIdx.x >> 6],
        [&](int o, int k, double* out) {
          Side<D, Real> mo, b;
          load_cand<D, SRC_CELLS>(a, w0 + o, mo.x, mo.r);
          load_cand<D, SRC_CELLS>(a, k, b.x, b.r);
          const int32_t io = a.perm[w0 + o], j = a.perm[k];
          mo.mat = (a.law.n_mat > 1) ? a.mat_id[io] : 0;
          mo.sp = species_of<LAW>(a.law, io);
          b.mat = (a.law.n_mat > 1) ? a.mat_id[j] : 0;
          b.sp = species_of<LAW>(a.law, j);
          const Vec<D, Real> rij = disp_<PER>(mo.x, b.x, a.dom);
          out[0] = 0.5 * (double)law_energy<D, LAW>(a.law, mo, b, dot(rij, rij));
        },
        [&](const double* v) { acc += v[0]; });
    if (on) a.e_out[i] = acc;
  } else {
    constexpr int G = group_lanes<D, SRC>();
    __shared__ int queues[kBlock / G][queue_len<D, SRC>()];
    int* queue = queues[threadIdx.x / G];
    const int l = threadIdx.x & (G - 1);
    const int64_t s = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * (kBlock / G) + threadIdx.x / G;
    if (s >= a.n) return;
    const int64_t i = SRC == SRC_CELLS ? (int64_t)a.perm[s] : s;
    Side<D, Real> me;
    me.x = ld<D>(a.pos_in, i);
    me.r = a.rad[i];
    me.mat = (a.law.n_mat > 1) ? a.mat_id[i] : 0;
    me.sp = species_of<LAW>(a.law, i);
    double acc = 0.0;
    walk_candidates<D, SRC, PER, true>(a, s, i, me.x, me.r, queue, [&](int nq) {
      for (int h0 = 0; h0 < nq; h0 += G) {
        double e = 0.0;
        if (h0 + l < nq) {
          const int k = queue[h0 + l];
          const int32_t j = cand_id<SRC>(a, k);
          Side<D, Real> b;
          load_cand<D, SRC>(a, k, b.x, b.r);
          b.mat = (a.law.n_mat > 1) ? a.mat_id[j] : 0;
          b.sp = species_of<LAW>(a.law, j);
          const Vec<D, Real> rij = disp_<PER>(me.x, b.x, a.dom);
          e = 0.5 * (double)law_energy<D, LAW>(a.law, me, b, dot(rij, rij));
        }
        const int cnt = min(G, nq - h0);
        for (int q = 0; q < cnt; ++q) acc += __shfl(e, q, G);
      }
    });
    if (l == 0) a.e_out[i] = acc;
  }
}

// Contact virial sum_{i<j} r_ij (x) F_ij (contacts.py:89-164): each i-side
// pair contributes 1/2 r_ij (x) F_ij, float64.
template <int D, int LAW, int SRC, bool PER, class Real>
__global__ void __launch_bounds__(kBlock) k_virial(StepArgsT<Real> a) {
  double W[D * D];
  for (int c = 0; c < D * D; ++c) W[c] = 0.0;
  auto outer = [](Vec<D, Real> rij, Vec<D, Real> F, double* w) {
    Real r[D], f[D];
    to_arr(rij, r);
    to_arr(F, f);
#pragma unroll
    for (int p = 0; p < D; ++p)
#pragma unroll
      for (int c = 0; c < D; ++c) w[p * D + c] = 0.5 * ((double)r[p] * (double)f[c]);
  };
  if constexpr (SRC == SRC_NLIST) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    Side<D, Real> me;
    load_side<D, LAW>(a, i, me);
    const int32_t* row = a.nl + i * a.M;
    for (int sl = 0; sl < a.M; ++sl) {
      const int32_t j = row[sl];
      if (j < 0) break;
      if (!may_interact(a, i, j)) continue;
      Vec<D, Real> xold = zero_vec<D, Real>();
      if constexpr (LawTraits<LAW>::hist) {
        if ((a.hist_live[i * a.W32 + (sl >> 5)] >> (sl & 31)) & 1u) xold = ld<D>(a.hist_xi, i * a.M + sl);
      }
      Side<D, Real> b;
      b.x = ld<D>(a.pos_in, j);
      b.r = a.rad[j];
      b.mat = 0;
      fill_partner<D, LAW>(a, b, j);
      const Vec<D, Real> rij = disp_<PER>(me.x, b.x, a.dom);
      const PairOut<D, Real> o = law_eval<D, LAW>(a.law, me, b, rij, dot(rij, rij), xold, a.dt);
      double w[D * D];
      outer(rij, o.F, w);
      for (int c = 0; c < D * D; ++c) W[c] += w[c];
    }
    for (int c = 0; c < D * D; ++c) a.e_out[i * D * D + c] = W[c];
  } else if constexpr (SRC == SRC_CELLS_LANE) {
    __shared__ LaneWalkLds<D * D, double> lds[kBlock / 64];
    const int64_t w0 = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * kBlock + (threadIdx.x & ~63u);
    const int64_t s = w0 + (threadIdx.x & 63);
    const bool on = s < a.n;
    const int64_t i = a.perm[on ? s : 0];
    Side<D, Real> me;
    load_cand<D, SRC_CELLS>(a, on ? s : 0, me.x, me.r);
    lane_walk<D, PER, true>(
        a, on, s, i, me.x, me.r, lds[threadIdx.x >> 6],
        [&](int o, int k, double* out) {
          Vec<D, Real> rij;
          const PairOut<D, Real> r = pair_of_slots<D, LAW, PER>(a, w0 + o, k, rij);
          outer(rij, r.F, out);
        },
        [&](const double* v) {
#pragma unroll
          for (int c = 0; c < D * D; ++c) W[c] += v[c];
        });
    if (on)
      for (int c = 0; c < D * D; ++c) a.e_out[i * D * D + c] = W[c];
  } else {
    constexpr int G = group_lanes<D, SRC>();
    __shared__ int queues[kBlock / G][queue_len<D, SRC>()];
    int* queue = queues[threadIdx.x / G];
    const int64_t s = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * (kBlock / G) + threadIdx.x / G;
    if (s >= a.n) return;
    const int64_t i = SRC == SRC_CELLS ? (int64_t)a.perm[s] : s;
    Side<D, Real> me;
    load_side<D, LAW>(a, i, me);
    walk_candidates<D, SRC, PER, true>(a, s, i, me.x, me.r, queue, [&](int nq) {
      queued_pairs<D, LAW, SRC, PER>(a, me, queue, nq, [&](const PairOut<D, Real>& o, Vec<D, Real> rij, int cnt) {
        double w[D * D];
        outer(rij, o.F, w);
        for (int q = 0; q < cnt; ++q)
#pragma unroll
          for (int c = 0; c < D * D; ++c) W[c] += __shfl(w[c], q, G);
      });
    });
    if ((threadIdx.x & (G - 1)) == 0)
      for (int c = 0; c < D * D; ++c) a.e_out[i * D * D + c] = W[c];
  }
}

// Kinetic energy per particle (utils/thermal.py:83-122), float64.
template <int D, class Real>
__global__ void __launch_bounds__(kBlock) k_kinetic(StepArgsT<Real> a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  // a clump member counts 1/(member count) of its clump (thermal.py:20-77)
  const double cnt = a.clump ? (double)(a.cl_start[a.clump[i] + 1] - a.cl_start[a.clump[i]]) : 1.0;
  const double m = (double)a.mass[i] / cnt;
  double ke = 0.0;  // rotational part
  double v2 = 0.0;
  for (int c = 0; c < D; ++c) {
    const double v = a.vel_in[D * i + c];
    v2 += v * v;
  }
  const double ke_t = 0.5 * m * v2;
  if constexpr (D == 3) {
    // body-frame angular velocity in float64
    const double qw = a.q[4 * i], qx = a.q[4 * i + 1], qy = a.q[4 * i + 2], qz = a.q[4 * i + 3];
    // rotate_back: the rotation by the conjugate (quaternion.py:267-268)
    const double cw = qw, cx = -qx, cy = -qy, cz = -qz;
    const double wx = a.ang_in[3 * i], wy = a.ang_in[3 * i + 1], wz = a.ang_in[3 * i + 2];
    const double tx = 2.0 * (cy * wz - cz * wy), ty = 2.0 * (cz * wx - cx * wz), tz = 2.0 * (cx * wy - cy * wx);
    const double bx = (wx + cw * tx) + (cy * tz - cz * ty);
    const double by = (wy + cw * ty) + (cz * tx - cx * tz);
    const double bz = (wz + cw * tz) + (cx * ty - cy * tx);
    ke += 0.5 * ((double)a.inertia[3 * i] * bx * bx + (double)a.inertia[3 * i + 1] * by * by +
                 (double)a.inertia[3 * i + 2] * bz * bz);
  } else {
    const double w = a.ang_in[i];
    ke += 0.5 * (double)a.inertia[i] * w * w;
  }
  ke = ke / cnt;
  // translational and rotational parts, summed separately
  a.e_out[2 * i] = ke_t;
  a.e_out[2 * i + 1] = ke;
}

// One stage of _step_once on its own (jdem_step_stage).
template <int D>
__global__ void __launch_bounds__(kBlock) k_stage(StepArgs a, int stage) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  Vec<D> x = ld<D>(a.pos_out, i);
  Vec<D> v = ld<D>(a.vel_out, i);
  Ang<D> w = lda<D>(a.ang_out, i);
  Quat q = ldq(a.q, i);
  Vec<D> F = ld<D>(a.force, i);
  Ang<D> T = lda<D>(a.torque, i);
  const Ang<D> I = lda<D>(a.inertia, i);
  const float m = a.mass[i];
  const bool fixed = a.fixed[i] != 0;
  const float freef = fixed ? 0.0f : 1.0f;
  switch (stage) {
    case JDEM_STAGE_DOMAIN_APPLY:
      if (a.dom.kind == JDEM_DOMAIN_REFLECT) reflect_apply<D>(a.dom, x, v, q, F, m, a.rad[i], fixed, a.dt);
      break;
    case JDEM_STAGE_LIN_BEFORE:
      if (a.lin == JDEM_LIN_VERLET) {
        const float s = (a.dt * 0.5f) / m;
        v = v + (F * s) * freef;
        x = x + v * a.dt;
      }
      break;
    case JDEM_STAGE_ROT_BEFORE:
      if (a.rot == JDEM_ROT_VERLET_SPIRAL) vvs_before<D>(q, w, T, I, a.dt, freef);
      break;
    case JDEM_STAGE_FORCE_MANAGER: {
      Vec<D> fp = a.ext_f ? ld<D>(a.ext_f, i) : zero_vec<D>();
      Vec<D> fc = a.ext_fc ? ld<D>(a.ext_fc, i) : zero_vec<D>();
      Vec<D> g;
      if constexpr (D == 3)
        g = Vec<3>{a.g[0], a.g[1], a.g[2]};
      else
        g = Vec<2>{a.g[0], a.g[1]};
      fc = fc + g * (m / 1.0f);
      F = (F + fp) + fc;
      if (a.ext_t) T = T + lda<D>(a.ext_t, i);
      break;
    }
    case JDEM_STAGE_LIN_AFTER:
      if (a.lin == JDEM_LIN_VERLET) {
        const float s = (a.dt * 0.5f) / m;
        v = v + (F * s) * freef;
      } else if (a.lin == JDEM_LIN_EULER) {
        const float s = a.dt / m;
        v = v + (F * s) * freef;
        x = x + v * a.dt;
      }
      break;
    case JDEM_STAGE_ROT_AFTER:
      if (a.rot == JDEM_ROT_VERLET_SPIRAL)
        vvs_after<D>(q, w, T, I, a.dt, freef);
      else if (a.rot == JDEM_ROT_SPIRAL)
        spiral_after<D>(q, w, T, I, a.dt, freef);
      break;
    default:
      break;
  }
  st(a.pos_out, i, x);
  st(a.vel_out, i, v);
  sta(a.ang_out, i, w);
  stq(a.q, i, q);
  st(a.force, i, F);
  sta(a.torque, i, T);
}

// ---------------------------------------------------------------------------
// clumps (rigid bodies of spheres; every member holds its clump's pos_c, q,
// velocities, mass and inertia)
// ---------------------------------------------------------------------------
// State._pos_p_rot = R(q) pos_p and State.pos = pos_c + R(q) pos_p
// (state.py:230-304)
template <int D, class Real>
__global__ void __launch_bounds__(kBlock) k_clump_lab(StepArgsT<Real> a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const QuatT<Real> q = ldq(a.q, i);
  const Vec<D, Real> r = q_rotate(q, ld<D>(a.pos_p, i));
  st(a.ppr, i, r);
  st(a.plab, i, ld<D>(a.pos_in, i) + r);
}

// ForceManager.apply for clumps (force_manager.py:359-412): per member,
// gravity with mass / member count, the lever torque of particle forces,
// the totals; then each member's force and torque are its clump's sums of
// the totals, in ascending member index.
template <int D, class Real>
__global__ void __launch_bounds__(kBlock) k_clump_total(StepArgsT<Real> a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const int c = a.clump[i];
  const Real cnt = (Real)(a.cl_start[c + 1] - a.cl_start[c]);
  const Vec<D, Real> fp = a.ext_f ? ld<D>(a.ext_f, i) : zero_vec<D, Real>();
  Vec<D, Real> fc = a.ext_fc ? ld<D>(a.ext_fc, i) : zero_vec<D, Real>();
  Ang<D, Real> tp = a.ext_t ? lda<D>(a.ext_t, i) : zero_ang<D, Real>();
  Vec<D, Real> g;
  if constexpr (D == 3)
    g = Vec<3, Real>{a.g[0], a.g[1], a.g[2]};
  else
    g = Vec<2, Real>{a.g[0], a.g[1]};
  fc = fc + g * (a.mass[i] / cnt);
  tp = tp + cross_t(ld<D>(a.ppr, i), fp);
  st(a.ftot, i, (ld<D>(a.force, i) + fp) + fc);
  sta(a.ttot, i, lda<D>(a.torque, i) + tp);
}

template <int D, class Real>
__global__ void __launch_bounds__(kBlock) k_clump_sum(StepArgsT<Real> a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const int c = a.clump[i];
  Vec<D, Real> F = zero_vec<D, Real>();
  Ang<D, Real> T = zero_ang<D, Real>();
  for (int k = a.cl_start[c]; k < a.cl_start[c + 1]; ++k) {
    const int32_t m = a.cl_members[k];
    F = F + ld<D>(a.ftot, m);
    T = T + lda<D>(a.ttot, m);
  }
  st(a.force, i, F);
  sta(a.torque, i, T);
}

// ReflectDomain.apply for clumps (reflect.py:160-297).  Per member: its
// overlap past each wall at its lab position; the deepest member of its clump
// per axis takes the impulse with the effective mass of the rigid body; the
// clump's time-of-collision fraction is its members' minimum; the members'
// impulses are summed over the clump into the linear and angular velocity
// changes, and position and orientation are corrected over the remaining
// time.  Matrix products sum in index order.  Scratch per member (rscr):
// [0, D) over_lo, [D, 2D) over_hi, [2D, 3D) wall sign, [3D, 4D) active,
// [4D, 5D) denominator, [5D, 6D) contact velocity, [6D, 7D) contact
// acceleration, 7D alpha minimum, 7D + 1 clump alpha, [7D + 2, 8D + 2)
// impulse / mass, then the angular velocity change (A words).
template <int D, class Real>
JD Real* refl_row(const StepArgsT<Real>& a, int64_t i) {
  return a.rscr + (int64_t)(8 * D + 2 + (D == 3 ? 3 : 1)) * i;
}
// rows of R (body -> lab): row k = R^T e_k = rotate_back(q, e_k)
template <int D, class Real>
JD void rot_rows(QuatT<Real> q, Real R[D][D]) {
#pragma unroll
  for (int k = 0; k < D; ++k) {
    Real e[D];
#pragma unroll
    for (int c = 0; c < D; ++c) e[c] = (c == k) ? Real(1) : Real(0);
    Vec<D, Real> ek;
    from_arr(ek, e);
    Vec<D, Real> rk;
    if constexpr (D == 3)
      rk = q_rotate_back(q, ek);
    else
      rk = q_rotate(q_conj(q), ek);
    to_arr(rk, R[k]);
  }
}
// R^T v (T = true) or R v, summing over j in index order
template <int D, bool T, class Real>
JD void rmul(const Real R[D][D], const Real* v, Real* out) {
#pragma unroll
  for (int i = 0; i < D; ++i) {
    Real acc = (T ? R[0][i] : R[i][0]) * v[0];
#pragma unroll
    for (int j = 1; j < D; ++j) acc = acc + (T ? R[j][i] : R[i][j]) * v[j];
    out[i] = acc;
  }
}

template <int D, class Real>
__global__ void __launch_bounds__(kBlock) k_crefl_over(StepArgsT<Real> a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const Vec<D, Real> r = q_rotate(ldq(a.q, i), ld<D>(a.pos_p, i));
  Real pos[D];
  to_arr(ld<D>(a.pos_in, i) + r, pos);
  const Real rad = a.rad[i];
  Real* s = refl_row<D>(a, i);
#pragma unroll
  for (int c = 0; c < D; ++c) {
    const Real lo = a.dom.anchor[c] + rad;
    const Real hi = (a.dom.anchor[c] + a.dom.box[c]) - rad;
    s[c] = fmax_(Real(0), lo - pos[c]);
    s[D + c] = fmax_(Real(0), pos[c] - hi);
  }
}

template <int D, class Real>
__global__ void __launch_bounds__(kBlock) k_crefl_alpha(StepArgsT<Real> a) {
  constexpr int A = D == 3 ? 3 : 1;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const int c0 = a.clump[i];
  Real mlo[D], mhi[D];
#pragma unroll
  for (int c = 0; c < D; ++c) mlo[c] = mhi[c] = -Real(INFINITY);
  for (int k = a.cl_start[c0]; k < a.cl_start[c0 + 1]; ++k) {
    const Real* sm = refl_row<D>(a, a.cl_members[k]);
#pragma unroll
    for (int c = 0; c < D; ++c) {
      mlo[c] = fmax_(mlo[c], sm[c]);
      mhi[c] = fmax_(mhi[c], sm[D + c]);
    }
  }
  Real* s = refl_row<D>(a, i);
  const QuatT<Real> q = ldq(a.q, i);
  const Vec<D, Real> pp = ld<D>(a.pos_p, i);
  const Vec<D, Real> r = q_rotate(q, pp);
  const Real inv_mass = Real(1) / a.mass[i];
  Real I[A], invI[A];
  to_arr_a(lda<D>(a.inertia, i), I);
#pragma unroll
  for (int k = 0; k < A; ++k) invI[k] = Real(1) / I[k];
  Real R[D][D];
  rot_rows<D>(q, R);
  Real delta[D], ws[D];
#pragma unroll
  for (int c = 0; c < D; ++c) {
    delta[c] = fmax_(mlo[c], mhi[c]);
    const bool dlo = (s[c] > Real(0)) && (s[c] == mlo[c]);
    const bool dhi = (s[D + c] > Real(0)) && (s[D + c] == mhi[c]);
    ws[c] = (dlo ? Real(1) : Real(0)) - (dhi ? Real(1) : Real(0));
    s[2 * D + c] = ws[c];
    s[3 * D + c] = fabs_(ws[c]);
    // effective mass along axis c: 1/m + sum_k invI_k ((pos_p x n'_c)_k)^2
    Vec<D, Real> nc;
    from_arr(nc, R[c]);
    Real x[A];
    to_arr_a(cross_t(pp, nc), x);
    Real drot = (x[0] * x[0]) * invI[0];
#pragma unroll
    for (int k = 1; k < A; ++k) drot = drot + (x[k] * x[k]) * invI[k];
    Real den = inv_mass + drot;
    s[4 * D + c] = (den == Real(0)) ? Real(1) : den;
  }
  const Vec<D, Real> vcs = ld<D>(a.vel_in, i) + cross_wr(lda<D>(a.ang_in, i), r);
  const Vec<D, Real> acl = ld<D>(a.force, i) * inv_mass;
  Ang<D, Real> arot;
  if constexpr (D == 3) {
    Real t[3], w[3], tb[3], wb[3];
    to_arr(lda<3>(a.torque, i), t);
    to_arr(lda<3>(a.ang_in, i), w);
    rmul<3, true>(R, t, tb);
    rmul<3, true>(R, w, wb);
    Vec<3, Real> wbv, tbv, Iv;
    from_arr(wbv, wb);
    from_arr(tbv, tb);
    from_arr(Iv, I);
    const Vec<3, Real> ab = (tbv - cross(wbv, Iv * wbv)) * Vec<3, Real>{invI[0], invI[1], invI[2]};
    Real abv[3], ar[3];
    to_arr(ab, abv);
    rmul<3, false>(R, abv, ar);
    from_arr(arot, ar);
  } else {
    arot = lda<2>(a.torque, i) * Ang1T<Real>{invI[0]};
  }
  const Vec<D, Real> acc = acl + cross_wr(arot, r);
  Real v[D], ac[D];
  to_arr(vcs, v);
  to_arr(acc, ac);
  Real amin = Real(1);
#pragma unroll
  for (int c = 0; c < D; ++c) {
    s[5 * D + c] = v[c];
    s[6 * D + c] = ac[c];
    const Real al = toc_alpha(v[c], ac[c], delta[c], ws[c], a.dt);
    if (fabs_(ws[c]) > Real(0)) amin = fmin_(amin, al);
  }
  s[7 * D] = amin;
}

template <int D, class Real>
__global__ void __launch_bounds__(kBlock) k_crefl_impulse(StepArgsT<Real> a) {
  constexpr int A = D == 3 ? 3 : 1;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const int c0 = a.clump[i];
  Real acl = Real(INFINITY), cnt[D];
#pragma unroll
  for (int c = 0; c < D; ++c) cnt[c] = Real(0);
  for (int k = a.cl_start[c0]; k < a.cl_start[c0 + 1]; ++k) {
    const Real* sm = refl_row<D>(a, a.cl_members[k]);
    acl = fmin_(acl, sm[7 * D]);
#pragma unroll
    for (int c = 0; c < D; ++c) cnt[c] = cnt[c] + sm[3 * D + c];
  }
  Real* s = refl_row<D>(a, i);
  s[7 * D + 1] = acl;
  const QuatT<Real> q = ldq(a.q, i);
  const Real inv_mass = Real(1) / a.mass[i];
  Real I[A];
  to_arr_a(lda<D>(a.inertia, i), I);
  Real R[D][D];
  rot_rows<D>(q, R);
  const Real e = a.dom.restitution;
  const Real dt_factor = (acl - Real(1)) * a.dt;
  Real j[D];
#pragma unroll
  for (int c = 0; c < D; ++c) {
    const Real act = s[3 * D + c];
    const Real weight = act / fmax_(cnt[c], Real(1));
    const Real vc = s[5 * D + c] + dt_factor * s[6 * D + c];
    Real jj = ((-(Real(1) + e)) * vc) / s[4 * D + c];
    const Real closing = ((vc * s[2 * D + c]) < Real(0)) ? Real(1) : Real(0);
    jj = jj * (weight * closing);
    j[c] = jj;
    s[7 * D + 2 + c] = jj * inv_mass;
  }
  Real jb[D];
  rmul<D, true>(R, j, jb);
  Vec<D, Real> jbv;
  from_arr(jbv, jb);
  Real m[A], dw[A];
  to_arr_a(cross_t(ld<D>(a.pos_p, i), jbv), m);
  if constexpr (D == 3) {
    Real mb[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) mb[k] = m[k] * (Real(1) / I[k]);
    rmul<3, false>(R, mb, dw);
  } else {
    dw[0] = m[0] * (Real(1) / I[0]);
  }
#pragma unroll
  for (int k = 0; k < A; ++k) s[8 * D + 2 + k] = dw[k];
}

template <int D, class Real>
__global__ void __launch_bounds__(kBlock) k_crefl_apply(StepArgsT<Real> a) {
  constexpr int A = D == 3 ? 3 : 1;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const int c0 = a.clump[i];
  Real dv[D], dw[A];
#pragma unroll
  for (int c = 0; c < D; ++c) dv[c] = Real(0);
#pragma unroll
  for (int k = 0; k < A; ++k) dw[k] = Real(0);
  for (int k = a.cl_start[c0]; k < a.cl_start[c0 + 1]; ++k) {
    const Real* sm = refl_row<D>(a, a.cl_members[k]);
#pragma unroll
    for (int c = 0; c < D; ++c) dv[c] = dv[c] + sm[7 * D + 2 + c];
#pragma unroll
    for (int kk = 0; kk < A; ++kk) dw[kk] = dw[kk] + sm[8 * D + 2 + kk];
  }
  if (a.fixed[i]) {
#pragma unroll
    for (int c = 0; c < D; ++c) dv[c] = Real(0);
#pragma unroll
    for (int k = 0; k < A; ++k) dw[k] = Real(0);
  }
  const Real dt_rem = (Real(1) - refl_row<D>(a, i)[7 * D + 1]) * a.dt;
  Vec<D, Real> dvv;
  from_arr(dvv, dv);
  Ang<D, Real> dwv;
  if constexpr (D == 3)
    from_arr(dwv, dw);
  else
    dwv = Ang1T<Real>{dw[0]};
  st(a.vel_out, i, ld<D>(a.vel_in, i) + dvv);
  sta(a.ang_out, i, lda<D>(a.ang_in, i) + dwv);
  Vec<3, Real> th;
  if constexpr (D == 3)
    th = dwv * dt_rem;
  else
    th = Vec<3, Real>{Real(0), Real(0), dw[0] * dt_rem};
  stq(a.q, i, q_unit(q_mul(q_from_small_rotvec(th), ldq(a.q, i))));
  st(a.pos_out, i, ld<D>(a.pos_in, i) + dvv * dt_rem);
}

// ---------------------------------------------------------------------------
// dispatch: every collider source and law in float; in double (the float64
// form of the plain step) the laws without history.
// ---------------------------------------------------------------------------
template <class Real>
constexpr bool kIsF32 = std::is_same<Real, float>::value;

#define JDEM_DISPATCH_BODY(KERNEL)                                                               \
  template <int D, int LAW>                                                                      \
  static hipError_t by_src(const StepArgsT<Real>& a, int src, bool per, dim3 g, dim3 b, hipStream_t s) { \
    switch (src) {                                                                               \
      case SRC_NAIVE:                                                                            \
        if (per)                                                                                 \
          hipLaunchKernelGGL((KERNEL<D, LAW, SRC_NAIVE, true, Real>), g, b, 0, s, a);            \
        else                                                                                     \
          hipLaunchKernelGGL((KERNEL<D, LAW, SRC_NAIVE, false, Real>), g, b, 0, s, a);           \
        break;                                                                                   \
      case SRC_CELLS:                                                                            \
        if (per)                                                                                 \
          hipLaunchKernelGGL((KERNEL<D, LAW, SRC_CELLS, true, Real>), g, b, 0, s, a);            \
        else                                                                                     \
          hipLaunchKernelGGL((KERNEL<D, LAW, SRC_CELLS, false, Real>), g, b, 0, s, a);           \
        break;                                                                                   \
      case SRC_CELLS_LANE:                                                                       \
        if (per)                                                                                 \
          hipLaunchKernelGGL((KERNEL<D, LAW, SRC_CELLS_LANE, true, Real>), g, b, 0, s, a);       \
        else                                                                                     \
          hipLaunchKernelGGL((KERNEL<D, LAW, SRC_CELLS_LANE, false, Real>), g, b, 0, s, a);      \
        break;                                                                                   \
      case SRC_NLIST:                                                                            \
        if (per)                                                                                 \
          hipLaunchKernelGGL((KERNEL<D, LAW, SRC_NLIST, true, Real>), g, b, 0, s, a);            \
        else                                                                                     \
          hipLaunchKernelGGL((KERNEL<D, LAW, SRC_NLIST, false, Real>), g, b, 0, s, a);           \
        break;                                                                                   \
      default:                                                                                   \
        return hipErrorInvalidValue;                                                             \
    }                                                                                            \
    return hipGetLastError();                                                                    \
  }                                                                                              \
  template <int D>                                                                               \
  static hipError_t by_law(const StepArgsT<Real>& a, int law, int src, bool per, dim3 g, dim3 b, hipStream_t s) { \
    switch (law) {                                                                               \
      case JDEM_LAW_SPRING:                                                                      \
        return by_src<D, JDEM_LAW_SPRING>(a, src, per, g, b, s);                                 \
      case JDEM_LAW_HERTZ:                                                                       \
        return by_src<D, JDEM_LAW_HERTZ>(a, src, per, g, b, s);                                  \
      case JDEM_LAW_CUNDALL_STRACK:                                                              \
        return by_src<D, JDEM_LAW_CUNDALL_STRACK>(a, src, per, g, b, s);                         \
      case kLawRouted:                                                                           \
        return by_src<D, kLawRouted>(a, src, per, g, b, s);                                      \
      case JDEM_LAW_SPRING_FRICTION:                                                             \
        if constexpr (kIsF32<Real>) return by_src<D, JDEM_LAW_SPRING_FRICTION>(a, src, per, g, b, s); \
        return hipErrorInvalidValue;                                                             \
      case JDEM_LAW_HERTZ_FRICTION:                                                              \
        if constexpr (kIsF32<Real>) return by_src<D, JDEM_LAW_HERTZ_FRICTION>(a, src, per, g, b, s); \
        return hipErrorInvalidValue;                                                             \
      case kLawRoutedHist:                                                                       \
        if constexpr (kIsF32<Real>) return by_src<D, kLawRoutedHist>(a, src, per, g, b, s);     \
        return hipErrorInvalidValue;                                                             \
      default:                                                                                   \
        return hipErrorInvalidValue;                                                             \
    }                                                                                            \
  }                                                                                              \
  static hipError_t run(StepArgsT<Real> a, int dim, int law, int src, bool walks, hipStream_t s) { \
    if (a.n == 0) return hipSuccess;                                                             \
    if (src == SRC_CELLS && walks && a.n >= lane_walk_min(a, dim)) src = SRC_CELLS_LANE;               \
    dim3 g(blocks(a, dim, src)), b(kBlock);                                                      \
    const bool per = a.dom.kind == JDEM_DOMAIN_PERIODIC;                                         \
    return dim == 3 ? by_law<3>(a, law, src, per, g, b, s) : by_law<2>(a, law, src, per, g, b, s); \
  }

// The cell list is walked by one lane per particle from this many particles
// on, by a group of lanes below.  A group needs three to four times the
// instructions, a lane three to four times the serial chain, so the lane wins
// once there are wavefronts for every SIMD.  Time per step (sort included),
// group / lane, us: 3D springs 58 / 64 at 32 k particles, 72 / 64 at 64 k,
// 338 / 182 at 2^20; 3D Cundall-Strack 65 / 74, 86 / 76, 561 / 252; 2D springs
// 42 / 45, 46 / 45, 160 / 104; float64 springs 65 / 65 at 32 k, 90 / 65 at
// 64 k.  More columns (3D, small cells: 81 at search range 4) lengthen the
// chain: 149 / 183 at 64 k, 228 / 199 at 128 k; float64 157 / 169 at 48 k,
// 191 / 175 at 64 k.
template <class Real>
int64_t lane_walk_min(const StepArgsT<Real>& a, int dim) {
  if (dim == 3 && a.grid.sr > 1) return kIsF32<Real> ? 98304 : 65536;
  return kIsF32<Real> ? 49152 : 32768;
}

// particles that a wavefront walks at once
inline int walked_at_once(int dim, int src) {
  return 64 / (dim == 3 ? (src == SRC_NAIVE ? group_lanes<3, SRC_NAIVE>() : group_lanes<3, SRC_CELLS>())
                        : (src == SRC_NAIVE ? group_lanes<2, SRC_NAIVE>() : group_lanes<2, SRC_CELLS>()));
}

template <class Real>
struct StepDispatch {
  // A wavefront of the cell-list or naive step finishes a.pw particles, one
  // per lane: as many as keep kStepWaves wavefronts in flight, since the
  // finishing lanes cost the same for one particle as for 64.
  static constexpr int64_t kStepWaves = 8192;
  static unsigned blocks(StepArgsT<Real>& a, int dim, int src) {
    if (src == SRC_NLIST) return nblocks(a.n);
    int pw = 64;
    if (src != SRC_CELLS_LANE && a.do_force && !a.force_zero)
      while (pw > walked_at_once(dim, src) && a.n < kStepWaves * pw) pw /= 2;
    a.pw = pw;
    return nblocks(a.n, pw * (kBlock / 64));
  }
  JDEM_DISPATCH_BODY(k_step)
};
// Energy and virial: one lane or one group of lanes per particle.
template <class Real>
struct EnergyDispatch {
  static unsigned blocks(StepArgsT<Real>& a, int dim, int src) {
    return src == SRC_NLIST || src == SRC_CELLS_LANE ? nblocks(a.n) : nblocks(a.n, walked_at_once(dim, src) * (kBlock / 64));
  }
  JDEM_DISPATCH_BODY(k_energy)
};
template <class Real>
struct VirialDispatch {
  static unsigned blocks(StepArgsT<Real>& a, int dim, int src) { return EnergyDispatch<Real>::blocks(a, dim, src); }
  JDEM_DISPATCH_BODY(k_virial)
};

template <class Real>
hipError_t kinetic_run(const StepArgsT<Real>& a, int dim, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  if (dim == 3)
    hipLaunchKernelGGL((k_kinetic<3, Real>), dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  else
    hipLaunchKernelGGL((k_kinetic<2, Real>), dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_step(const StepArgs& a, int dim, int law, int src, hipStream_t s) {
  return StepDispatch<float>::run(a, dim, law, src, a.do_force && !a.force_zero, s);
}
hipError_t launch_energy(const StepArgs& a, int dim, int law, int src, hipStream_t s) {
  return EnergyDispatch<float>::run(a, dim, law, src, true, s);
}
hipError_t launch_virial(const StepArgs& a, int dim, int law, int src, hipStream_t s) {
  return VirialDispatch<float>::run(a, dim, law, src, true, s);
}
hipError_t launch_kinetic(const StepArgs& a, int dim, hipStream_t s) { return kinetic_run(a, dim, s); }
hipError_t launch_step(const StepArgs64& a, int dim, int law, int src, hipStream_t s) {
  return StepDispatch<double>::run(a, dim, law, src, a.do_force && !a.force_zero, s);
}
hipError_t launch_energy(const StepArgs64& a, int dim, int law, int src, hipStream_t s) {
  return EnergyDispatch<double>::run(a, dim, law, src, true, s);
}
hipError_t launch_kinetic(const StepArgs64& a, int dim, hipStream_t s) { return kinetic_run(a, dim, s); }
template <class Real>
hipError_t clump_lab_run(const StepArgsT<Real>& a, int dim, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  if (dim == 3)
    hipLaunchKernelGGL((k_clump_lab<3, Real>), dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  else
    hipLaunchKernelGGL((k_clump_lab<2, Real>), dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}
template <class Real>
hipError_t clump_forces_run(const StepArgsT<Real>& a, int dim, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  if (dim == 3) {
    hipLaunchKernelGGL((k_clump_total<3, Real>), dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
    hipLaunchKernelGGL((k_clump_sum<3, Real>), dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  } else {
    hipLaunchKernelGGL((k_clump_total<2, Real>), dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
    hipLaunchKernelGGL((k_clump_sum<2, Real>), dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  }
  return hipGetLastError();
}
template <class Real>
hipError_t clump_reflect_run(const StepArgsT<Real>& a, int dim, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  const dim3 g(nblocks(a.n)), b(kBlock);
  if (dim == 3) {
    hipLaunchKernelGGL((k_crefl_over<3, Real>), g, b, 0, s, a);
    hipLaunchKernelGGL((k_crefl_alpha<3, Real>), g, b, 0, s, a);
    hipLaunchKernelGGL((k_crefl_impulse<3, Real>), g, b, 0, s, a);
    hipLaunchKernelGGL((k_crefl_apply<3, Real>), g, b, 0, s, a);
  } else {
    hipLaunchKernelGGL((k_crefl_over<2, Real>), g, b, 0, s, a);
    hipLaunchKernelGGL((k_crefl_alpha<2, Real>), g, b, 0, s, a);
    hipLaunchKernelGGL((k_crefl_impulse<2, Real>), g, b, 0, s, a);
    hipLaunchKernelGGL((k_crefl_apply<2, Real>), g, b, 0, s, a);
  }
  return hipGetLastError();
}
hipError_t launch_clump_reflect(const StepArgs& a, int dim, hipStream_t s) { return clump_reflect_run(a, dim, s); }
hipError_t launch_clump_reflect(const StepArgs64& a, int dim, hipStream_t s) { return clump_reflect_run(a, dim, s); }
hipError_t launch_clump_lab(const StepArgs& a, int dim, hipStream_t s) { return clump_lab_run(a, dim, s); }
hipError_t launch_clump_lab(const StepArgs64& a, int dim, hipStream_t s) { return clump_lab_run(a, dim, s); }
hipError_t launch_clump_forces(const StepArgs& a, int dim, hipStream_t s) { return clump_forces_run(a, dim, s); }
hipError_t launch_clump_forces(const StepArgs64& a, int dim, hipStream_t s) { return clump_forces_run(a, dim, s); }

hipError_t launch_stage(const StepArgs& a, int dim, int stage, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  if (dim == 3)
    hipLaunchKernelGGL(k_stage<3>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a, stage);
  else
    hipLaunchKernelGGL(k_stage<2>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a, stage);
  return hipGetLastError();
}

}  // namespace jdem
