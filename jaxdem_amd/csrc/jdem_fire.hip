// jdem_fire.hip -- the FIRE energy minimiser on the GPU
// (minimizers/optimizers.py:150-339, minimizers/routines.py:150-383).
//
// An iteration is the force and energy evaluation (jdem_step.hip) between
//   k_fire_terms   per particle: ForceManager's gravity, F = -grad (masked by
//                  ~fixed), v_old = F dt/2 + v; block partials of F . v_old and
//                  the energy in float64, of the largest gradient component
//   k_fire_decide  one block: their sums, the stopping tests (routines.py:
//                  284-314), the downhill / uphill update of dt, alpha, N_good,
//                  N_bad (optimizers.py:250-296)
//   k_fire_move    per particle: velocity mixing, the parameter update and
//                  the new orientation (routines.py:341-360, 37-65)
// Everything about the loop stays on the device (FireDev, FireStop); after a
// stop the decide and move kernels return at once and what else was launched
// recomputes the forces of the final positions.  So the host reads the loop's
// state once per chunk of iterations: with a read per iteration and a kernel
// for each of these terms an iteration of 16 k spheres was 21 launches and
// 130 us, bounded by them; now 10 and 60 us.  The chunks grow with the steps
// done (1, 1, 2, 4, then a quarter of them up to 32), so the evaluations past a
// stop stay below half of those needed.  A neighbour list is checked by the
// host before every evaluation anyway; the stop word comes with that read, and
// nothing is launched past a stop.
// Every float32 expression follows the reference's operation order, so
// positions match the float32 oracle bit for bit while the power decisions
// agree.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "jdem_internal.h"

namespace jdem {

namespace {

// optax.safe_norm(x, 1e-16, axis=-1): the row norm, or 1e-16 where the norm
// is not above it
template <int A>
JD float safe_norm(const float* x) {
  float n2;
  if (A == 3)
    n2 = (x[0] * x[0] + x[1] * x[1]) + x[2] * x[2];
  else if (A == 2)
    n2 = x[0] * x[0] + x[1] * x[1];
  else
    n2 = x[0] * x[0];
  const float n = sqrtf(n2);
  return n <= 1e-16f ? 1e-16f : n;
}

// Quaternion.from_rotvec (quaternion.py:99-127)
JD Quat q_from_rotvec(Vec<3> r) {
  const float n2 = dot(r, r);
  const float safe = fmaxf(n2, 1e-16f);
  const float theta = sqrtf(safe);
  const float half = 0.5f * theta;
  const float ch = cosf(half);
  const float sc = sinf(half) / theta;
  return {ch, r.x * sc, r.y * sc, r.z * sc};
}

// The velocity-mixing update of optimizers.py:297-318 of one leaf: F and v_old
// of a particle -> its new velocity and the parameter update.
template <int A>
JD void fire_mix(const FireDev& s, const float* f, const float* v_old, float* v_new, float* upd) {
  float vh[A];
#pragma unroll
  for (int c = 0; c < A; ++c) vh[c] = v_old[c] * s.vs + (f[c] * s.new_dt) / 2.0f;
  const float vn = safe_norm<A>(vh);
  const float fn = safe_norm<A>(f);
  const float mixr = fn > 1e-16f ? (vn / fn) * s.new_alpha : 0.0f;
#pragma unroll
  for (int c = 0; c < A; ++c) {
    vh[c] = (vh[c] * (1.0f - s.new_alpha) + f[c] * mixr) * s.vs;
    upd[c] = (v_old[c] * s.dt_rev) / 2.0f + (vh[c] * s.new_dt) / 2.0f;
    v_new[c] = vh[c];
  }
}

// The scalars of one update from its power (optimizers.py:250-296).
JD void fire_decide(FireDev& s, const FireP& p, double power) {
  const float cand_inc = fminf(s.dt * p.f_inc, p.dt_max);
  const float cand_dec = fmaxf(s.dt * p.f_dec, p.dt_min);
  if (power > 0.0) {  // downhill (optimizers.py:278-292)
    const int ng = s.n_good + 1;
    s.new_dt = ng > p.n_min ? cand_inc : s.dt;
    s.new_alpha = ng > p.n_min ? s.alpha * p.f_alpha : s.alpha;
    s.n_good = ng;
    s.n_bad = 0;
    s.dt_rev = 0.0f;
    s.vs = 1.0f;
  } else {  // uphill (optimizers.py:258-276)
    int nb = s.n_bad + 1;
    const bool exceeded = nb > p.n_bad_max;
    s.new_dt = exceeded ? p.dt0 : cand_dec;
    s.n_bad = exceeded ? 0 : nb;
    s.new_alpha = p.alpha_init;
    s.n_good = 0;
    s.dt_rev = -s.new_dt;
    s.vs = 0.0f;
  }
  s.power = power;
}

// One parameter leaf of one particle (A components): F, v_old and the
// velocity-mixing update of optimizers.py:245-318.
template <int A>
struct Leaf {
  float f[A], v_old[A];
  JD void load(const float* F, const float* V, int64_t i, float m, float dt) {
#pragma unroll
    for (int c = 0; c < A; ++c) {
      f[c] = -((-F[A * i + c]) * m);  // F = -(grad * mask), grad = -force
      v_old[c] = V[A * i + c] + (f[c] * dt) / 2.0f;
    }
  }
  JD double power() const {
    double p = 0.0;
#pragma unroll
    for (int c = 0; c < A; ++c) p += (double)f[c] * (double)v_old[c];
    return p;
  }
  // returns the update; writes the new velocity
  JD void mix(const FireDev& s, float* V, int64_t i, float* upd) const { fire_mix<A>(s, f, v_old, V + A * i, upd); }
};

// non-negative floats (and the quiet NaN of a NaN component, which makes the
// maximum NaN as jnp.max does) order like their bits
JD unsigned grad_bits(float f) { return f == f ? __float_as_uint(fabsf(f)) : 0x7fc00000u; }

template <int D>
__global__ void __launch_bounds__(kBlock) k_fire_terms(FireArgs a) {
  constexpr int A = D == 3 ? 3 : 1;
  __shared__ double sp[kBlock], se[kBlock];
  __shared__ unsigned sg[kBlock / 64];
  const int tid = threadIdx.x;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + tid;
  double p = 0.0, e = 0.0;
  unsigned g = 0u;
  if (i < a.n) {
    // ForceManager.apply with no external arrays (force_manager.py:341-425)
#pragma unroll
    for (int c = 0; c < D; ++c) {
      const float f = (a.force[D * i + c] + 0.0f) + (0.0f + a.g[c] * (a.mass[i] / 1.0f));
      a.force[D * i + c] = f;
      g = max(g, grad_bits(f));
    }
#pragma unroll
    for (int c = 0; c < A; ++c) g = max(g, grad_bits(a.torque[A * i + c]));
    const float m = a.fixed[i] ? 0.0f : 1.0f;
    const float dt = a.st->dt;
    Leaf<D> lp;
    Leaf<A> lr;
    lp.load(a.force, a.vel_pos, i, m, dt);
    lr.load(a.torque, a.vel_rot, i, m, dt);
    p = lp.power() + lr.power();
    if (a.e_in) e = a.e_in[i];
    if (a.g[0] != 0.0f || a.g[1] != 0.0f || a.g[2] != 0.0f) {  // of gravity (force_manager.py:450-459)
      float gx;
      if (D == 3)
        gx = (a.g[0] * a.pos[3 * i] + a.g[1] * a.pos[3 * i + 1]) + a.g[2] * a.pos[3 * i + 2];
      else
        gx = a.g[0] * a.pos[2 * i] + a.g[1] * a.pos[2 * i + 1];
      e += (double)(-(gx * a.mass[i]));
    }
  }
  sp[tid] = p;
  se[tid] = e;
  for (int off = 32; off > 0; off >>= 1) g = max(g, (unsigned)__shfl_xor((int)g, off));
  if ((tid & 63) == 0) sg[tid >> 6] = g;
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if (tid < off) {
      sp[tid] += sp[tid + off];
      se[tid] += se[tid + off];
    }
    __syncthreads();
  }
  if (tid == 0) {
    for (int w = 1; w < kBlock / 64; ++w) g = max(g, sg[w]);
    a.part[2 * blockIdx.x] = sp[0];
    a.part[2 * blockIdx.x + 1] = se[0];
    a.gpart[blockIdx.x] = g;
  }
}

__global__ void __launch_bounds__(kBlock) k_fire_decide(FireArgs a) {
  if (a.ls->stop) return;
  __shared__ double sp[kBlock], se[kBlock];
  __shared__ unsigned sg[kBlock];
  const int tid = threadIdx.x;
  double p = 0.0, e = 0.0;
  unsigned g = 0u;
  for (int b = tid; b < a.nparts; b += kBlock) {
    p += a.part[2 * b];
    e += a.part[2 * b + 1];
    g = max(g, a.gpart[b]);
  }
  sp[tid] = p;
  se[tid] = e;
  sg[tid] = g;
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if (tid < off) {
      sp[tid] += sp[tid + off];
      se[tid] += se[tid + off];
      sg[tid] = max(sg[tid], sg[tid + off]);
    }
    __syncthreads();
  }
  if (tid != 0) return;
  FireStop& ls = *a.ls;
  const double pe = se[0], gmax = (double)__uint_as_float(sg[0]);
  ls.pe = pe;
  ls.gmax = gmax;
  const double tiny = 2.2250738585072014e-308;  // smallest normal float64
  const bool conv_pe = fabs(pe / a.stop.dN) <= a.stop.pe_tol;
  const double larger = fabs(pe) < fabs(ls.prev) ? fabs(ls.prev) : fabs(pe);
  const double denom = larger < tiny ? tiny : larger;
  const bool conv_rel = fabs(pe - ls.prev) / denom < a.stop.pe_diff_tol;
  if (ls.steps >= a.stop.max_steps || conv_pe || conv_rel || gmax <= a.stop.force_tol) {
    ls.stop = 1;
    if (a.stop_word) *a.stop_word = 1;
    return;
  }
  ls.prev = pe;
  ls.steps += 1;
  FireDev s = *a.st;
  fire_decide(s, a.p, sp[0]);
  s.dt_used = s.dt;  // the update's v_old; the next power takes the new dt
  s.dt = s.new_dt;
  s.alpha = s.new_alpha;
  *a.st = s;
}

template <int D>
__global__ void __launch_bounds__(kBlock) k_fire_move(FireArgs a) {
  if (a.ls->stop) return;
  constexpr int A = D == 3 ? 3 : 1;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const FireDev s = *a.st;
  const bool fixed = a.fixed[i] != 0;
  const float m = fixed ? 0.0f : 1.0f;
  Leaf<D> lp;
  Leaf<A> lr;
  lp.load(a.force, a.vel_pos, i, m, s.dt_used);
  lr.load(a.torque, a.vel_rot, i, m, s.dt_used);
  float up[D], ur[A];
  lp.mix(s, a.vel_pos, i, up);
  lr.mix(s, a.vel_rot, i, ur);
  // updates * mask, then where(mask, params + updates, params)
  if (!fixed)
#pragma unroll
    for (int c = 0; c < D; ++c) a.pos[D * i + c] = a.pos[D * i + c] + up[c] * m;
  float rv[A];
#pragma unroll
  for (int c = 0; c < A; ++c) rv[c] = fixed ? 0.0f : 0.0f + ur[c] * m;
  const Vec<3> r3 = (D == 3) ? Vec<3>{rv[0], rv[A > 1 ? 1 : 0], rv[A > 2 ? 2 : 0]} : Vec<3>{0.0f, 0.0f, rv[0]};
  const float4 q4 = reinterpret_cast<const float4*>(a.q)[i];
  const Quat q = {q4.x, q4.y, q4.z, q4.w};
  const Quat qn = q_unit(q_mul(q_from_rotvec(r3), q));
  reinterpret_cast<float4*>(a.q)[i] = make_float4(qn.w, qn.x, qn.y, qn.z);
}

// ---- precision form ---------------------------------------------------------
// Positions are x = c h + o per axis, c an integer cell and o in [0, h): the
// float32 offset keeps ~1e-7 h of resolution anywhere in the box, where an
// absolute float32 coordinate keeps ~1e-7 L.  The cell edge is the float pair
// h + hlo, so the lattice matches the box to float64 accuracy.  The
// displacement of two spheres in neighbouring cells, (c_i - c_j) h + (o_i -
// o_j), is formed as a float pair too (error-free sums), so it is exact to
// ~1e-14 |r| rather than rounded to ~6e-8 |r|.
//
// The state of a minimisation lives in cell order, (offset, radius), velocity,
// cell and force of sorted slot kk, so every kernel of an iteration streams it
// and only a re-sort permutes it.  An iteration is
//   k_prec_force / k_prec_vforce  force; block partials of energy, max|F| and
//                                 of the power the next update will see
//   k_prec_decide (one block)     sums the partials, stopping tests, FIRE's
//                                 scalars, and the buffers' roles
//   k_prec_move                   the update; raises *moved for a re-sort
//   re-sort (gated by *moved)     keys, counting sort, permute, list build
// The two state buffers swap at every re-sort: word cur says which one holds
// the state, and while *moved is set the kernels after the permute read the
// other one, until k_prec_decide commits the swap.

JD int prec_now(const PrecArgs& a) { return *a.cur ^ (*a.moved ? 1 : 0); }

// x = c h + o with o folded back into [0, h) (c wrapped periodically);
// returns whether the cell changed
template <int D>
JD bool prec_fold(const PrecArgs& a, float* o, int* c) {
  bool moved = false;
#pragma unroll
  for (int q = 0; q < D; ++q) {
    if (!(o[q] >= 0.0f && o[q] < a.h[q])) {
      const float m = floorf(o[q] / a.h[q]);
      o[q] = (o[q] - m * a.h[q]) - m * a.hlo[q];
      if (o[q] < 0.0f) o[q] = 0.0f;  // rounding of o - m h
      if (o[q] >= a.h[q]) o[q] = 0.0f, c[q] += 1;
      c[q] = (c[q] + (int)m) % a.dims[q];
      if (c[q] < 0) c[q] += a.dims[q];
      moved = true;
    }
  }
  return moved;
}

// the caller's arrays -> slot = sphere id, at rest; the largest radius
template <int D>
__global__ void __launch_bounds__(kBlock) k_prec_load(PrecArgs a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  float r = 0.0f;
  if (i < a.n) {
    const float ri = a.rad[i];
    r = ri > 0.0f ? ri : 0.0f;  // -0 and less would order above every radius below
    a.S[0][i] = make_float4(a.off[D * i], a.off[D * i + 1], D == 3 ? a.off[D * i + 2] : 0.0f, ri);
    a.V[0][i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    a.C[0][i] = make_int4(a.cidx[D * i], a.cidx[D * i + 1], D == 3 ? a.cidx[D * i + 2] : 0, (int)i);
  }
  for (int off = 32; off > 0; off >>= 1) r = fmaxf(r, __shfl_xor(r, off));
  // not negative, so the bits order like the values; most waves find the
  // maximum already there
  if ((threadIdx.x & 63) == 0 && __float_as_uint(r) > *a.rmax_bits) atomicMax(a.rmax_bits, __float_as_uint(r));
}

// the state back to the caller's order
template <int D>
__global__ void __launch_bounds__(kBlock) k_prec_store(PrecArgs a) {
  const int64_t kk = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (kk >= a.n) return;
  const int now = prec_now(a);
  const float4 s = a.S[now][kk], f = a.F[kk];
  const int4 c = a.C[now][kk];
  const float o[3] = {s.x, s.y, s.z}, ff[3] = {f.x, f.y, f.z};
  const int cc[3] = {c.x, c.y, c.z};
  const int64_t i = c.w;
#pragma unroll
  for (int q = 0; q < D; ++q) {
    a.off[D * i + q] = o[q];
    a.cidx[D * i + q] = cc[q];
    a.force[D * i + q] = ff[q];
  }
}

// Re-sort: fold (list mode; the stencil folds at every move), keys and the
// sort's count pass.  Keys stay in slot order, which is nearly the new order
// (by sphere id they were scattered: 20 us of atomics and stores for 2^18
// spheres, now 10); a cell's spheres sort by id in the rank pass.
template <int D>
__global__ void __launch_bounds__(kBlock) k_prec_keys(PrecArgs a) {
  if (*a.moved == 0 || (a.stop && *a.stop)) return;  // no sphere changed cell: the last sort stands
  const int64_t kk = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (kk >= a.n) return;
  const int cur = *a.cur;
  int4 c4 = a.C[cur][kk];
  int c[3] = {c4.x, c4.y, c4.z};
  if (a.vl) {  // list mode: cells are kept between list builds
    float4 s = a.S[cur][kk];
    float o[3] = {s.x, s.y, s.z};
    if (prec_fold<D>(a, o, c)) {
      a.S[cur][kk] = make_float4(o[0], o[1], o[2], s.w);
      a.C[cur][kk] = make_int4(c[0], c[1], c[2], c4.w);
    }
  }
  const uint32_t key = D == 3 ? (uint32_t)((c[0] * a.dims[1] + c[1]) * a.dims[2] + c[2])
                              : (uint32_t)(c[0] * a.dims[1] + c[1]);
  a.keys[kk] = key;
  a.arr[kk] = atomicAdd(&a.cnt[key], 1);
}

// (id, old slot) by arrival order within each cell
__global__ void __launch_bounds__(kBlock) k_prec_place(PrecArgs a) {
  if (*a.moved == 0 || (a.stop && *a.stop)) return;
  const int64_t kk = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (kk >= a.n) return;
  a.pairs[a.starts[a.keys[kk]] + a.arr[kk]] = make_uint2((uint32_t)a.C[*a.cur][kk].w, (uint32_t)kk);
}

// each sphere's rank among the ids of its cell, and its state to that slot
__global__ void __launch_bounds__(kBlock) k_prec_permute(PrecArgs a) {
  if (*a.moved == 0 || (a.stop && *a.stop)) return;
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= a.n) return;
  const int cur = *a.cur;
  const uint2 me = a.pairs[j];
  const int64_t s = me.y;
  const uint32_t key = a.keys[s];
  const int32_t b = a.starts[key], e = a.starts[key + 1];
  const float4 p = a.S[cur][s], v = a.V[cur][s];
  const int4 c = a.C[cur][s];
  int32_t r = b;
  for (int32_t m = b; m < e; ++m) r += a.pairs[m].x < me.x ? 1 : 0;
  a.S[cur ^ 1][r] = p;
  a.V[cur ^ 1][r] = v;
  a.C[cur ^ 1][r] = c;
  a.skeys[r] = key;
  if (a.vl) a.B[r] = p;  // offsets at the build
}

// Columns of a stencil of half-width sr around cell c along the last axis,
// walked by a group of kPrecGroup lanes: each lane loads one column's bounds,
// a scan numbers the candidates, and visit(in, k, ox, oy, oz) is called for
// kPrecGroup of them at a time (in: the lane has one; the offsets are those of
// its cell).  Candidates come in stencil order (ox, oy, oz), ascending id
// within a cell.  keep(ox, oy, zlo, zhi) may narrow a column's run.  One lane
// per sphere was a serial chain of 125 cell bounds and their candidates.
constexpr int kPrecGroup = 16;
template <int D, class Keep, class Visit>
JD void prec_columns(const PrecArgs& a, int4 c, int sr, Keep&& keep, Visit&& visit) {
  constexpr int G = kPrecGroup;
  const int l = threadIdx.x & (G - 1);
  const int w = 2 * sr + 1, ncol = D == 3 ? w * w : w;
  const int df = a.dims[D - 1], cf = D == 3 ? c.z : c.y;
  for (int cb = 0; cb < ncol; cb += G) {
    const int col = cb + l;
    int s0 = 0, len0 = 0, s1 = 0, len1 = 0, ox = 0, oy = 0;
    uint32_t kbase = 0;
    if (col < ncol) {
      ox = (D == 3 ? col / w : col) - sr;
      oy = D == 3 ? col % w - sr : 0;
      int cx = c.x + ox, cy = c.y + oy;
      cx = cx < 0 ? cx + a.dims[0] : (cx >= a.dims[0] ? cx - a.dims[0] : cx);
      if (D == 3) cy = cy < 0 ? cy + a.dims[1] : (cy >= a.dims[1] ? cy - a.dims[1] : cy);
      kbase = D == 3 ? (uint32_t)((cx * a.dims[1] + cy) * a.dims[2]) : (uint32_t)(cx * a.dims[1]);
      int zlo = -sr, zhi = sr;
      keep(ox, oy, zlo, zhi);
      if (zlo <= zhi) {
        int z0 = cf + zlo, z1 = cf + zhi;  // cells z0..z1, wrapped into two runs at most
        if (z0 < 0) z0 += df, z1 += df;
        if (z0 >= df) z0 -= df, z1 -= df;
        s0 = a.starts[kbase + z0];
        len0 = a.starts[kbase + min(z1, df - 1) + 1] - s0;
        if (z1 >= df) {
          s1 = a.starts[kbase];
          len1 = a.starts[kbase + z1 - df + 1] - s1;
        }
      }
    }
    int incl = len0 + len1;
#pragma unroll
    for (int d = 1; d < G; d <<= 1) {
      const int t = __shfl_up(incl, d, G);
      if (l >= d) incl += t;
    }
    const int pre = incl - (len0 + len1);
    const int total = __shfl(incl, G - 1, G);
    for (int b = 0; b < total; b += G) {
      const int cand = b + l;
      int q = 0;
#pragma unroll
      for (int st = G / 2; st > 0; st >>= 1) q += __shfl(pre, q + st, G) <= cand ? st : 0;
      const int o = cand - __shfl(pre, q, G), f0 = __shfl(s0, q, G), n0 = __shfl(len0, q, G), f1 = __shfl(s1, q, G);
      const int qx = __shfl(ox, q, G), qy = __shfl(oy, q, G);
      const uint32_t qb = (uint32_t)__shfl((int)kbase, q, G);
      const bool in = cand < total;
      const int k = o < n0 ? f0 + o : f1 + (o - n0);
      int oz = 0;
      if (in) {  // the candidate's cell along the column, from its sorted key
        oz = (int)(a.skeys[k] - qb) - cf;
        oz = oz > sr ? oz - df : (oz < -sr ? oz + df : oz);
      }
      visit(in, k, qx, D == 3 ? qy : oz, D == 3 ? oz : 0);
    }
  }
}

// Verlet list of the precision form (rebuilds only, gated by *moved): the
// partners of the sphere in sorted slot kk0 within r_i + r_j + skin, in
// stencil order (half-width vsr <= 2), each entry the partner's sorted slot
// (low 24 bits) and the cell difference c_i - c_j (high 8 bits, base-5
// digits + 2); slot-major, a row ends at its first -1.  Cells stay fixed until
// the next build (offsets may leave [0, h) by up to skin / 2 meanwhile), so
// the entry's cell difference holds for the list's lifetime.  Cells that lie
// further than the list's reach from the sphere (most of the 125) are left
// out: ListReach narrows each column.  2^18 spheres: 303 -> 69 us (a lane each).
template <int D>
struct ListReach {
  float o[3], h[3], reach2;
  JD void start(const PrecArgs& a, const float* oi, float ri) {
    // no partner lies further than this (a margin over the test's rounding)
    const float reach = ((ri + __uint_as_float(*a.rmax_bits)) + a.vcut) * 1.001f;
    reach2 = reach * reach;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      o[q] = oi[q];
      h[q] = a.h[q];
    }
  }
  JD float gap2(int q, int d) const {  // squared distance along axis q to the cells at offset d
    const float g = d > 0 ? (float)d * h[q] - o[q] : (d < 0 ? o[q] - (float)(d + 1) * h[q] : 0.0f);
    return g > 0.0f ? g * g : 0.0f;
  }
  JD void narrow(int ox, int oy, int& zlo, int& zhi) const {
    const float left = reach2 - (gap2(0, ox) + (D == 3 ? gap2(1, oy) : 0.0f));
    if (left < 0.0f) {
      zlo = 1, zhi = 0;
      return;
    }
    while (zlo < 0 && gap2(D - 1, zlo) > left) ++zlo;
    while (zhi > 0 && gap2(D - 1, zhi) > left) --zhi;
  }
};
template <int D>
JD bool listed(const PrecArgs& a, const float4& si, const float4& sj, int ox, int oy, int oz) {
  const float oi[3] = {si.x, si.y, si.z}, oj[3] = {sj.x, sj.y, sj.z};
  const int o[3] = {ox, oy, oz};
  float d2 = 0.0f;
#pragma unroll
  for (int q = 0; q < D; ++q) {
    const float r = (float)(-o[q]) * a.h[q] + (oi[q] - oj[q]);
    d2 = d2 + r * r;
  }
  const float R = (si.w + sj.w) + a.vcut;
  return d2 < R * R;
}
JD int32_t list_entry(int k, int ox, int oy, int oz) {
  const int code = (2 - ox) + 5 * ((2 - oy) + 5 * (2 - oz));
  return (int32_t)((uint32_t)k | ((uint32_t)code << 24));
}

// A group of lanes per sphere.
template <int D>
__global__ void __launch_bounds__(kBlock) k_prec_vbuild(PrecArgs a) {
  if (*a.moved == 0 || (a.stop && *a.stop)) return;
  constexpr int G = kPrecGroup;
  const int lane = threadIdx.x & 63, l = lane & (G - 1);
  const int64_t kk0 = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * (kBlock / G) + threadIdx.x / G;
  if (kk0 >= a.n) return;
  const int now = prec_now(a);
  const float4* S = a.S[now];
  const float4 si = S[kk0];
  const float oi[3] = {si.x, si.y, si.z};
  ListReach<D> lr;
  lr.start(a, oi, si.w);
  int cnt = 0;
  prec_columns<D>(
      a, a.C[now][kk0], a.vsr, [&](int ox, int oy, int& zlo, int& zhi) { lr.narrow(ox, oy, zlo, zhi); },
      [&](bool in, int k, int ox, int oy, int oz) {
        const bool hit = in && k != (int)kk0 && listed<D>(a, si, S[k], ox, oy, oz);
        const uint64_t m = (__ballot(hit) >> (lane & ~(G - 1))) & ((1ull << G) - 1ull);
        if (hit) {
          const int t = cnt + __popcll(m & ((1ull << l) - 1ull));
          if (t < a.vm) a.vl[(int64_t)t * a.n + kk0] = list_entry(k, ox, oy, oz);
        }
        cnt += __popcll(m);
      });
  if (l == 0) {
    if (cnt < a.vm) a.vl[(int64_t)cnt * a.n + kk0] = -1;
    if (cnt > a.vm) *a.vovf = 1;
  }
}

// One lane per sphere, candidates four at a time: a quarter of the
// instructions, a longer chain.
template <int D>
__global__ void __launch_bounds__(kBlock) k_prec_vbuild_lane(PrecArgs a) {
  if (*a.moved == 0 || (a.stop && *a.stop)) return;
  const int64_t kk0 = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (kk0 >= a.n) return;
  const int now = prec_now(a);
  const float4* __restrict__ S = a.S[now];
  const float4 si = S[kk0];
  const int4 c = a.C[now][kk0];
  const float oi[3] = {si.x, si.y, si.z};
  ListReach<D> lr;
  lr.start(a, oi, si.w);
  const int sr = a.vsr, df = a.dims[D - 1], cf = D == 3 ? c.z : c.y;
  int cnt = 0;
  for (int ox = -sr; ox <= sr; ++ox)
    for (int oy = D == 3 ? -sr : 0; oy <= (D == 3 ? sr : 0); ++oy) {
      int zlo = -sr, zhi = sr;
      lr.narrow(ox, oy, zlo, zhi);
      if (zlo > zhi) continue;
      int cx = c.x + ox, cy = c.y + oy;
      cx = cx < 0 ? cx + a.dims[0] : (cx >= a.dims[0] ? cx - a.dims[0] : cx);
      if (D == 3) cy = cy < 0 ? cy + a.dims[1] : (cy >= a.dims[1] ? cy - a.dims[1] : cy);
      const uint32_t base = D == 3 ? (uint32_t)((cx * a.dims[1] + cy) * a.dims[2]) : (uint32_t)(cx * a.dims[1]);
      int z0 = cf + zlo, z1 = cf + zhi;
      if (z0 < 0) z0 += df, z1 += df;
      if (z0 >= df) z0 -= df, z1 -= df;
      const int k0 = a.starts[base + z0], k0e = a.starts[base + min(z1, df - 1) + 1];
      const int k1 = z1 >= df ? a.starts[base] : 0, k1e = z1 >= df ? a.starts[base + z1 - df + 1] : 0;
      for (int run = 0; run < 2; ++run) {
        const int ke = run ? k1e : k0e;
        for (int kg = run ? k1 : k0; kg < ke; kg += 4) {
          float4 sj[4];
          uint32_t key[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            sj[u] = kg + u < ke ? S[kg + u] : make_float4(0.f, 0.f, 0.f, 0.f);
            key[u] = kg + u < ke ? a.skeys[kg + u] : base;
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (kg + u >= ke) break;
            if (kg + u == (int)kk0) continue;
            int oz = (int)(key[u] - base) - cf;
            oz = oz > sr ? oz - df : (oz < -sr ? oz + df : oz);
            const int qy = D == 3 ? oy : oz, qz = D == 3 ? oz : 0;
            if (!listed<D>(a, si, sj[u], ox, qy, qz)) continue;
            if (cnt < a.vm) a.vl[(int64_t)cnt * a.n + kk0] = list_entry(kg + u, ox, qy, qz);
            ++cnt;
          }
        }
      }
    }
  if (cnt < a.vm) a.vl[(int64_t)cnt * a.n + kk0] = -1;
  if (cnt > a.vm) *a.vovf = 1;
}

// The spring law (spring.py:97-108, 138-147) of one touching pair; float32
// pair arithmetic, float64 energy.  dc: cell difference c_i - c_j (exact in
// float32).  r = rh + rl, both float32: two_sum of the cell term and the
// offset difference, whose own rounding error two_sum recovers too.  delta =
// (R^2 - |r|^2) / (R + |r|) with |r|^2 = sum rh^2 + 2 rh rl and the squares
// split exactly into hi + lo with fma, so the cancellation of R against |r| at
// small overlaps loses nothing; R - |r| directly would keep only ~1e-7 |r| /
// delta of relative accuracy.
struct PrecPair {
  float f[3];
  double e;
};
template <int D>
JD PrecPair prec_pair(const PrecArgs& a, const float* oi, const float* oj, const int* dc, const float* r, float d2,
                      float R) {
  float rl[3] = {0, 0, 0};
#pragma unroll
  for (int q = 0; q < D; ++q) {
    const float b = oi[q] - oj[q];
    const float bv = b - oi[q];
    const float be = (oi[q] - (b - bv)) + (-oj[q] - bv);
    const float c = (float)dc[q] * a.h[q];
    const float t = c + b;
    const float tv = t - c;
    const float te = (c - (t - tv)) + (b - tv);
    rl[q] = (te + be) + (float)dc[q] * a.hlo[q];
  }
  const float inv = 1.0f / sqrtf(d2);
  float sh = 0.0f, sl = 0.0f;
#pragma unroll
  for (int q = 0; q < D; ++q) {
    const float p = r[q] * r[q];
    const float pe = fmaf(r[q], r[q], -p);
    const float t = sh + p;
    const float bp = t - sh;
    sl = sl + ((((sh - (t - bp)) + (p - bp)) + pe) + 2.0f * r[q] * rl[q]);
    sh = t;
  }
  const float RR = R * R;
  const float diff = (RR - sh) + (fmaf(R, R, -RR) - sl);
  const float delta = diff / (R + d2 * inv);
  const float s = (a.k * delta) * inv;
  PrecPair o;
#pragma unroll
  for (int q = 0; q < 3; ++q) o.f[q] = q < D ? s * r[q] : 0.0f;
  const double dd = (double)delta;
  o.e = 0.25 * (double)a.k * dd * dd;
  return o;
}
// r of a pair and whether it touches
template <int D>
JD bool prec_touch(const PrecArgs& a, const float* oi, float ri, float4 sj, const int* dc, float* r, float& d2,
                   float& R) {
  const float osj[3] = {sj.x, sj.y, sj.z};
#pragma unroll
  for (int q = 0; q < D; ++q) r[q] = (float)dc[q] * a.h[q] + (oi[q] - osj[q]);
  d2 = D == 3 ? (r[0] * r[0] + r[1] * r[1]) + r[2] * r[2] : r[0] * r[0] + r[1] * r[1];
  R = ri + sj.w;
  return d2 < R * R && d2 != 0.0f;
}

// The end of a force kernel: the sphere's force, and the block's partials of
// the energy, of max|F| (a NaN component makes it NaN, as jnp.max does; the
// bits of non-negative floats and of that NaN order like the values) and of
// FIRE's power F . v_old, v_old = v + F dt / 2 (optimizers.py:245-256).
struct PrecTerm {
  double e, p;
  unsigned g;
};
template <int D>
JD PrecTerm prec_term(const PrecArgs& a, int now, int64_t kk, const float* F, double e) {
  a.F[kk] = make_float4(F[0], F[1], D == 3 ? F[2] : 0.0f, 0.0f);
  const float4 v4 = a.V[now][kk];
  const float v[3] = {v4.x, v4.y, v4.z};
  const float dt = a.st->dt;
  PrecTerm t = {e, 0.0, 0u};
  float m = 0.0f;
#pragma unroll
  for (int q = 0; q < D; ++q) {
    t.p += (double)F[q] * (double)(v[q] + (F[q] * dt) / 2.0f);
    m = fmaxf(m, fabsf(F[q]));
  }
#pragma unroll
  for (int q = 0; q < D; ++q)
    if (F[q] != F[q]) m = __int_as_float(0x7fc00000);
  t.g = __float_as_uint(m);
  return t;
}
JD void prec_partials(const PrecArgs& a, unsigned block, PrecTerm t) {
  __shared__ double se[kBlock / 64], sp[kBlock / 64];
  __shared__ unsigned sg[kBlock / 64];
  for (int off = 32; off > 0; off >>= 1) {
    t.e += __shfl_xor(t.e, off);
    t.p += __shfl_xor(t.p, off);
    t.g = max(t.g, (unsigned)__shfl_xor((int)t.g, off));
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    se[w] = t.e;
    sp[w] = t.p;
    sg[w] = t.g;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int q = 1; q < kBlock / 64; ++q) {
    t.e += se[q];
    t.p += sp[q];
    t.g = max(t.g, sg[q]);
  }
  a.part_e[block] = t.e;
  a.part_p[block] = t.p;
  a.part_g[block] = t.g;
}

// The force on the 27-cell stencil (9 in 2D), a group of lanes per sphere;
// touching candidates are queued in LDS in stencil order, evaluated one per
// lane and summed in that order.  A block takes kPrecTile spheres.
constexpr int kPrecTile = 64;
template <int D>
__global__ void __launch_bounds__(kBlock) k_prec_force(PrecArgs a) {
  if (a.stop && *a.stop) return;
  constexpr int G = kPrecGroup, Q = 2 * G;
  __shared__ int qk[kBlock / G][Q], qc[kBlock / G][Q];
  const int lane = threadIdx.x & 63, l = lane & (G - 1), grp = threadIdx.x / G;
  const int now = prec_now(a);
  const float4* S = a.S[now];
  const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);
  PrecTerm acc = {0.0, 0.0, 0u};
  for (int p = grp; p < kPrecTile; p += kBlock / G) {
    const int64_t kk0 = (int64_t)tile * kPrecTile + p;
    if (kk0 >= a.n) continue;
    const float4 si = S[kk0];
    const float oi[3] = {si.x, si.y, si.z};
    float F[3] = {0, 0, 0};
    double e = 0.0, w[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    int nq = 0;
    auto flush = [&]() {
      wave_sync();
      for (int h0 = 0; h0 < nq; h0 += G) {
        PrecPair o = {{0, 0, 0}, 0.0};
        float r[3] = {0, 0, 0};
        if (h0 + l < nq) {
          const int code = qc[grp][h0 + l];
          const int dc[3] = {code % 3 - 1, (code / 3) % 3 - 1, code / 9 - 1};
          const float4 sj = S[qk[grp][h0 + l]];
          const float oj[3] = {sj.x, sj.y, sj.z};
          float d2, R;
          prec_touch<D>(a, oi, si.w, sj, dc, r, d2, R);
          o = prec_pair<D>(a, oi, oj, dc, r, d2, R);
        }
        const int cnt = min(G, nq - h0);
        for (int q = 0; q < cnt; ++q) {
          float f[3], rr[3];
#pragma unroll
          for (int c = 0; c < D; ++c) {
            f[c] = __shfl(o.f[c], q, G);
            F[c] = F[c] + f[c];
          }
          e += __shfl(o.e, q, G);
          if (a.w_out) {
#pragma unroll
            for (int c = 0; c < D; ++c) rr[c] = __shfl(r[c], q, G);
#pragma unroll
            for (int c = 0; c < D; ++c)
#pragma unroll
              for (int d = 0; d < D; ++d) w[D * c + d] += 0.5 * (double)rr[c] * (double)f[d];
          }
        }
      }
      wave_sync();
      nq = 0;
    };
    prec_columns<D>(
        a, a.C[now][kk0], 1, [](int, int, int&, int&) {},
        [&](bool in, int k, int ox, int oy, int oz) {
          bool hit = false;
          const int dc[3] = {-ox, -oy, -oz};
          if (in && k != (int)kk0) {
            float r[3], d2, R;
            hit = prec_touch<D>(a, oi, si.w, S[k], dc, r, d2, R);
          }
          const uint64_t m = (__ballot(hit) >> (lane & ~(G - 1))) & ((1ull << G) - 1ull);
          if (hit) {
            const int t = nq + __popcll(m & ((1ull << l) - 1ull));
            qk[grp][t] = k;
            qc[grp][t] = (dc[0] + 1) + 3 * ((dc[1] + 1) + 3 * (dc[2] + 1));
          }
          nq += __popcll(m);
          if (nq > Q - G) flush();
        });
    if (nq > 0) flush();
    if (l == 0) {
      const PrecTerm t = prec_term<D>(a, now, kk0, F, e);
      acc.e += t.e;
      acc.p += t.p;
      acc.g = max(acc.g, t.g);
      if (a.w_out)
        for (int q = 0; q < D * D; ++q) a.w_out[(int64_t)D * D * kk0 + q] = w[q];
    }
  }
  prec_partials(a, tile, acc);
}

// The same over the Verlet list, one lane per sphere, the pair's cell
// difference read from the entry.  With h >= 2 r_max and offsets within
// skin / 2 < h / 2 of [0, h), a contact has |c_i - c_j| <= 2 per axis, so
// (c_i - c_j) h is still exact in float32.  Partners are summed in the
// list's order (the stencil order of the build).  The list is slot-major, so
// a wavefront reads each of its slots in one piece; four entries and their
// spheres are loaded before any is used.  2^18 spheres: 54 -> 19 us, now with
// the partials of the reductions that were kernels of their own.
template <int D>
__global__ void __launch_bounds__(kBlock) k_prec_vforce(PrecArgs a) {
  if (a.stop && *a.stop) return;
  const int now = prec_now(a);
  const float4* __restrict__ S = a.S[now];
  const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);
  const int64_t kk0 = (int64_t)tile * kBlock + threadIdx.x;
  PrecTerm t = {0.0, 0.0, 0u};
  if (kk0 < a.n) {
    const float4 si = S[kk0];
    const float oi[3] = {si.x, si.y, si.z};
    float F[3] = {0, 0, 0};
    double e = 0.0, w[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    constexpr int PF = 4;
    bool done = false;
    for (int t0 = 0; t0 < a.vm && !done; t0 += PF) {
      int32_t ent[PF];
      float4 sj[PF];
#pragma unroll
      for (int u = 0; u < PF; ++u) ent[u] = t0 + u < a.vm ? a.vl[(int64_t)(t0 + u) * a.n + kk0] : -1;
#pragma unroll
      for (int u = 1; u < PF; ++u) ent[u] = ent[u - 1] < 0 ? -1 : ent[u];  // what follows a row's end is stale
#pragma unroll
      for (int u = 0; u < PF; ++u)
        sj[u] = ent[u] >= 0 ? S[ent[u] & 0xFFFFFF] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int u = 0; u < PF; ++u) {
        if (ent[u] < 0) {
          done = true;
          break;
        }
        const int code = (int)((uint32_t)ent[u] >> 24);
        const int dc[3] = {code % 5 - 2, (code / 5) % 5 - 2, code / 25 - 2};
        float r[3] = {0, 0, 0}, d2, R;
        if (!prec_touch<D>(a, oi, si.w, sj[u], dc, r, d2, R)) continue;
        const float oj[3] = {sj[u].x, sj[u].y, sj[u].z};
        const PrecPair o = prec_pair<D>(a, oi, oj, dc, r, d2, R);
#pragma unroll
        for (int q = 0; q < D; ++q) F[q] = F[q] + o.f[q];
        e += o.e;
        if (a.w_out)
          for (int p = 0; p < D; ++p)
            for (int q = 0; q < D; ++q) w[D * p + q] += 0.5 * (double)r[p] * (double)o.f[q];
      }
    }
    t = prec_term<D>(a, now, kk0, F, e);
    if (a.w_out)
      for (int q = 0; q < D * D; ++q) a.w_out[(int64_t)D * D * kk0 + q] = w[q];
  }
  prec_partials(a, tile, t);
}

// The FIRE update of the position leaf (no rotation: the spring law has no
// torque).  Stencil mode folds the offset back into [0, h); list mode keeps
// the cells and asks for a rebuild once a sphere has moved skin / 2.
template <int D>
__global__ void __launch_bounds__(kBlock) k_prec_move(PrecArgs a) {
  if (a.stop && *a.stop) return;
  const int64_t kk = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (kk >= a.n) return;
  const int cur = *a.cur;
  const FireDev s = *a.st;
  const float4 f4 = a.F[kk], v4 = a.V[cur][kk], s4 = a.S[cur][kk];
  const float f[3] = {f4.x, f4.y, f4.z}, v[3] = {v4.x, v4.y, v4.z};
  float o[3] = {s4.x, s4.y, s4.z}, v_old[D], vn[3] = {0, 0, 0}, up[D];
#pragma unroll
  for (int q = 0; q < D; ++q) v_old[q] = v[q] + (f[q] * s.dt_used) / 2.0f;
  fire_mix<D>(s, f, v_old, vn, up);
  a.V[cur][kk] = make_float4(vn[0], vn[1], vn[2], 0.0f);
#pragma unroll
  for (int q = 0; q < D; ++q) o[q] = o[q] + up[q];
  bool moved = false;
  if (a.vl) {
    const float4 b4 = a.B[kk];
    const float b[3] = {b4.x, b4.y, b4.z};
    float d2 = 0.0f;
#pragma unroll
    for (int q = 0; q < D; ++q) {
      const float d = o[q] - b[q];
      d2 = d2 + d * d;
    }
    moved = d2 > a.vtrig;
  } else {
    const int4 c4 = a.C[cur][kk];
    int c[3] = {c4.x, c4.y, c4.z};
    moved = prec_fold<D>(a, o, c);
    if (moved) a.C[cur][kk] = make_int4(c[0], c[1], c[2], c4.w);
  }
  a.S[cur][kk] = make_float4(o[0], o[1], o[2], s4.w);
  if (moved) *a.moved = 1;
}

// Sums of the force kernel's partials (one block); thread 0 holds them.
JD PrecTerm prec_sum_partials(const PrecArgs& a) {
  __shared__ double se[16], sp[16];
  __shared__ unsigned sg[16];
  PrecTerm t = {0.0, 0.0, 0u};
  for (int b = threadIdx.x; b < a.nparts; b += blockDim.x) {
    t.e += a.part_e[b];
    t.p += a.part_p[b];
    t.g = max(t.g, a.part_g[b]);
  }
  for (int off = 32; off > 0; off >>= 1) {
    t.e += __shfl_xor(t.e, off);
    t.p += __shfl_xor(t.p, off);
    t.g = max(t.g, (unsigned)__shfl_xor((int)t.g, off));
  }
  if ((threadIdx.x & 63) == 0) {
    se[threadIdx.x >> 6] = t.e;
    sp[threadIdx.x >> 6] = t.p;
    sg[threadIdx.x >> 6] = t.g;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    for (int q = 1; q < (int)blockDim.x / 64; ++q) {
      t.e += se[q];
      t.p += sp[q];
      t.g = max(t.g, sg[q]);
    }
  return t;
}

// Between two force evaluations: the swap of the state buffers after a
// re-sort, the tests at the top of one iteration of minimize's loop
// (routines.py:284-314: pe_tol on the energy per sphere, pe_diff_tol on the
// relative change, force_tol on max|F|, max_steps) plus a stall test (no new
// low of max|F|, or of the energy by more than 1e-13 of it, for stall_steps
// iterations): sets stop, or counts the update about to run and decides its
// scalars.
__global__ void __launch_bounds__(1024) k_prec_decide(PrecArgs a, PrecStop* ps, PrecStopP p, FireP fp) {
  if (ps->stop) return;
  const PrecTerm t = prec_sum_partials(a);
  if (threadIdx.x != 0) return;
  if (*a.moved) {
    *a.cur ^= 1;
    *a.moved = 0;
  }
  const double pe = t.e, g = (double)__uint_as_float(t.g);
  ps->pe = pe;
  ps->gmax = g;
  if (ps->first) {
    ps->best_g = g;
    ps->best_e = pe;
    ps->best_at = 0;
    ps->first = 0;
  }
  if (ps->steps >= p.max_steps) {
    ps->stop = 1;
    return;
  }
  const double tiny = 2.2250738585072014e-308;
  const bool conv_pe = fabs(pe / p.dN) <= p.pe_tol;
  const double denom = fmax(fmax(fabs(pe), fabs(ps->prev)), tiny);
  const bool conv_rel = fabs(pe - ps->prev) / denom < p.pe_diff_tol;
  if (g < ps->best_g) ps->best_g = g, ps->best_at = ps->steps;
  if (pe < ps->best_e - 1e-13 * fabs(ps->best_e)) ps->best_e = pe, ps->best_at = ps->steps;
  const bool stalled = p.stall_steps > 0 && ps->steps - ps->best_at >= p.stall_steps;
  if (conv_pe || conv_rel || g <= p.force_tol || stalled) {
    ps->stop = 1;
    return;
  }
  ps->prev = pe;
  ps->steps += 1;
  FireDev s = *a.st;
  fire_decide(s, fp, t.p);
  s.dt_used = s.dt;  // the update's v_old; the next power takes the new dt
  s.dt = s.new_dt;
  s.alpha = s.new_alpha;
  *a.st = s;
}

// energy and max|F| of the last evaluation, for a caller that does not step on
__global__ void __launch_bounds__(1024) k_prec_total(PrecArgs a, PrecStop* ps) {
  const PrecTerm t = prec_sum_partials(a);
  if (threadIdx.x != 0) return;
  ps->pe = t.e;
  ps->gmax = (double)__uint_as_float(t.g);
}

// float64 positions <-> integer cell + float32 offset (precision.py
// to_cell_offset / from_cell_offset): the same float64 operations in the same
// order, so the same cells and offsets.
struct PrecBox {
  double L[3], h[3];
  float hi[3];
  long long dims[3];
};
__global__ void __launch_bounds__(kBlock) k_prec_import(const double* __restrict__ pos, int64_t n, int D, PrecBox b,
                                                         int32_t* __restrict__ cidx, float* __restrict__ off) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * D) return;
  const int q = (int)(t % D);
  const double x0 = pos[t];
  const double x = x0 - b.L[q] * floor(x0 / b.L[q]);
  double f = floor(x / b.h[q]);
  long long c = f < 0.0 ? 0 : (f > (double)(b.dims[q] - 1) ? b.dims[q] - 1 : (long long)f);
  float o = (float)(x - (double)c * b.h[q]);
  const bool over = o >= b.hi[q];
  o = over ? 0.0f : (o > 0.0f ? o : (o == o ? 0.0f : o));
  if (over) c = (c + 1) % b.dims[q];
  cidx[t] = (int32_t)c;
  off[t] = o;
}
__global__ void __launch_bounds__(kBlock) k_prec_export(const int32_t* __restrict__ cidx,
                                                         const float* __restrict__ off, int64_t n, int D, PrecBox b,
                                                         double* __restrict__ pos) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * D) return;
  pos[t] = (double)cidx[t] * b.h[t % D] + (double)off[t];
}

}  // namespace

// The list build takes one lane per sphere from this many on.  A FIRE step
// whose list is rebuilt almost every time, group / lane: 58 / 82 us at 32 k
// spheres, 90 / 99 at 128 k, 142 / 126 at 2^18 (277 - 647 with 22 launches per
// step, row-major lists and one lane per 125 cells).
constexpr int64_t kVbuildLane = 163840;

unsigned prec_parts(int64_t n, bool list) { return std::max(1u, nblocks(n, list ? kBlock : kPrecTile)); }
hipError_t launch_prec_load(const PrecArgs& a, hipStream_t s) {
  if (a.dim == 3)
    hipLaunchKernelGGL(k_prec_load<3>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  else
    hipLaunchKernelGGL(k_prec_load<2>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_prec_store(const PrecArgs& a, hipStream_t s) {
  if (a.dim == 3)
    hipLaunchKernelGGL(k_prec_store<3>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  else
    hipLaunchKernelGGL(k_prec_store<2>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_prec_keys(const PrecArgs& a, hipStream_t s) {
  if (a.dim == 3)
    hipLaunchKernelGGL(k_prec_keys<3>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  else
    hipLaunchKernelGGL(k_prec_keys<2>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_prec_permute(const PrecArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_prec_place, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  hipLaunchKernelGGL(k_prec_permute, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  if (a.vl) {
    const bool lane = a.n >= kVbuildLane;
    const dim3 g(nblocks(a.n, lane ? kBlock : kBlock / kPrecGroup));
    if (a.dim == 3 && lane)
      hipLaunchKernelGGL(k_prec_vbuild_lane<3>, g, dim3(kBlock), 0, s, a);
    else if (a.dim == 3)
      hipLaunchKernelGGL(k_prec_vbuild<3>, g, dim3(kBlock), 0, s, a);
    else if (lane)
      hipLaunchKernelGGL(k_prec_vbuild_lane<2>, g, dim3(kBlock), 0, s, a);
    else
      hipLaunchKernelGGL(k_prec_vbuild<2>, g, dim3(kBlock), 0, s, a);
  }
  return hipGetLastError();
}
hipError_t launch_prec_force(const PrecArgs& a, hipStream_t s) {
  const dim3 g(prec_parts(a.n, a.vl != nullptr));
  if (a.vl) {
    if (a.dim == 3)
      hipLaunchKernelGGL(k_prec_vforce<3>, g, dim3(kBlock), 0, s, a);
    else
      hipLaunchKernelGGL(k_prec_vforce<2>, g, dim3(kBlock), 0, s, a);
  } else if (a.dim == 3) {
    hipLaunchKernelGGL(k_prec_force<3>, g, dim3(kBlock), 0, s, a);
  } else {
    hipLaunchKernelGGL(k_prec_force<2>, g, dim3(kBlock), 0, s, a);
  }
  return hipGetLastError();
}
hipError_t launch_prec_update(const PrecArgs& a, PrecStop* ps, const PrecStopP& p, const FireP& fp, hipStream_t s) {
  hipLaunchKernelGGL(k_prec_decide, dim3(1), dim3(1024), 0, s, a, ps, p, fp);
  if (a.dim == 3)
    hipLaunchKernelGGL(k_prec_move<3>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  else
    hipLaunchKernelGGL(k_prec_move<2>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_prec_total(const PrecArgs& a, PrecStop* ps, hipStream_t s) {
  hipLaunchKernelGGL(k_prec_total, dim3(1), dim3(1024), 0, s, a, ps);
  return hipGetLastError();
}
static PrecBox prec_box(int D, const double* L, const double* h, const float* hi, const int32_t* dims) {
  PrecBox b = {};
  for (int q = 0; q < D; ++q) {
    b.L[q] = L[q];
    b.h[q] = h[q];
    b.hi[q] = hi[q];
    b.dims[q] = dims[q];
  }
  return b;
}
hipError_t launch_prec_import(const double* pos, int64_t n, int D, const double* L, const double* h, const float* hi,
                              const int32_t* dims, int32_t* cidx, float* off, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_prec_import, dim3(nblocks(n * D)), dim3(kBlock), 0, s, pos, n, D, prec_box(D, L, h, hi, dims),
                     cidx, off);
  return hipGetLastError();
}
hipError_t launch_prec_export(const int32_t* cidx, const float* off, int64_t n, int D, const double* L,
                              const double* h, const float* hi, const int32_t* dims, double* pos, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_prec_export, dim3(nblocks(n * D)), dim3(kBlock), 0, s, cidx, off, n, D,
                     prec_box(D, L, h, hi, dims), pos);
  return hipGetLastError();
}

hipError_t launch_fire_terms(const FireArgs& a, hipStream_t s) {
  if (a.dim == 3)
    hipLaunchKernelGGL(k_fire_terms<3>, dim3(a.nparts), dim3(kBlock), 0, s, a);
  else
    hipLaunchKernelGGL(k_fire_terms<2>, dim3(a.nparts), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_fire_decide(const FireArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_fire_decide, dim3(1), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_fire_move(const FireArgs& a, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  if (a.dim == 3)
    hipLaunchKernelGGL(k_fire_move<3>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  else
    hipLaunchKernelGGL(k_fire_move<2>, dim3(nblocks(a.n)), dim3(kBlock), 0, s, a);
  return hipGetLastError();
}

}  // namespace jdem
