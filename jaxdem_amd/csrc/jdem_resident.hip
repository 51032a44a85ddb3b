// jdem_resident.hip -- the NeighborList time step on a resident, cell-sorted
// working set (the hot path of System.step with the NeighborList collider,
// system.py:60-82 + neighbor_list.py:58-131, 594-669).
//
// Layout in HBM for the duration of one jdem_system_step call:
//   P4[b] = (x, y, z, r)   V4[b] = (v, m)   W4[b] = (omega)   Q4[b] = q
//   I4[b] = (inertia, bits: species << 16 | mat_id << 1 | fixed)
// 2D records use their free lanes so that the step kernel reads neither I4
// nor old4: P4 = (x, y, x_build, r), V4 = (vx, vy, y_build, m),
// W4 = (omega, inertia, bits, spring offset).  I4 and old4 are kept as in 3D
// for the other kernels.
// in "work" order b: particles sorted by (cell, original id) at every list
// rebuild, so a particle's candidates are its memory neighbours.  orig[b] is
// the original index of work slot b.  The neighbour list is slot-major
// nl[s*N + b] (work indices) and ends at its first -1; one 64-bit live mask
// per particle and 64 slots marks the slots that carry a tangential spring.
// The springs themselves are stored by rank: xi[k*N + b] is the spring of
// the k-th live slot of particle b, so the rows a wavefront touches are the
// first few, densely used ones.  xi is double-buffered (read one, write the
// other) because a step's new ranks can overtake its old ones.  Sorting by (cell, original id) makes each row the
// reference's row (stencil order, ascending original id within a cell), so
// sums and history match the CPU oracle bit for bit.
//
// The caller's arrays (original order, JaxDEM layouts) are read once on entry
// and written once on exit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "jdem_internal.h"

namespace jdem {

// ---------------------------------------------------------------------------
// float4 helpers
// ---------------------------------------------------------------------------
template <int D>
JD Vec<D> xyz(float4 a);
template <>
JD Vec<3> xyz<3>(float4 a) { return {a.x, a.y, a.z}; }
template <>
JD Vec<2> xyz<2>(float4 a) { return {a.x, a.y}; }
JD float4 f4(Vec<3> v, float w) { return make_float4(v.x, v.y, v.z, w); }
JD float4 f4(Vec<2> v, float w) { return make_float4(v.x, v.y, 0.0f, w); }
template <int D>
JD Ang<D> ang4(float4 a);
template <>
JD Vec<3> ang4<3>(float4 a) { return {a.x, a.y, a.z}; }
template <>
JD Ang1 ang4<2>(float4 a) { return {a.x}; }
JD float4 f4a(Vec<3> v) { return make_float4(v.x, v.y, v.z, 0.0f); }
JD float4 f4a(Ang1 v) { return make_float4(v.z, 0.0f, 0.0f, 0.0f); }
JD Quat q4(float4 a) { return {a.x, a.y, a.z, a.w}; }
JD float4 f4q(Quat q) { return make_float4(q.w, q.x, q.y, q.z); }

// ---------------------------------------------------------------------------
// entry / exit conversions
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(kBlock) k_in_state(InOut a) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= a.n) return;
  const int64_t i = a.orig[b];
  const int D = a.dim;
  const int A = D == 3 ? 3 : 1;
  float p[3] = {0, 0, 0}, v[3] = {0, 0, 0}, w[3] = {0, 0, 0}, f[3] = {0, 0, 0}, t[3] = {0, 0, 0}, I[3] = {0, 0, 0},
        o[3] = {0, 0, 0};
  for (int c = 0; c < D; ++c) {
    p[c] = a.pos[D * i + c];
    v[c] = a.vel[D * i + c];
    f[c] = a.force[D * i + c];
    o[c] = a.old_user ? a.old_user[D * i + c] : 0.0f;
  }
  for (int c = 0; c < A; ++c) {
    w[c] = a.ang[A * i + c];
    t[c] = a.torque[A * i + c];
    I[c] = a.inertia[A * i + c];
  }
  const int bits = ((a.species ? a.species[i] : 0) << 16) | ((a.mat_id ? a.mat_id[i] : 0) << 1) | (a.fixed[i] ? 1 : 0);
  if (a.iso_flag && D == 3) {
    const float r = a.rad[i], Is = (0.4f * a.mass[i]) * (r * r);
    if (a.fixed[i] || I[0] != Is || I[1] != Is || I[2] != Is) *a.iso_flag = 0;
  }
  if (D == 2) {
    float ox = o[0], oy = o[1];
    if (a.old_keep) {
      const float4 ok = a.old4[b];
      ox = ok.x;
      oy = ok.y;
    }
    a.P4[b] = make_float4(p[0], p[1], ox, a.rad[i]);
    a.V4[b] = make_float4(v[0], v[1], oy, a.mass[i]);
    a.W4[b] = make_float4(w[0], I[0], __int_as_float(bits), 0.0f);
  } else {
    a.P4[b] = make_float4(p[0], p[1], p[2], a.rad[i]);
    a.V4[b] = make_float4(v[0], v[1], v[2], a.mass[i]);
    a.W4[b] = make_float4(w[0], w[1], w[2], 0.0f);
  }
  a.Q4[b] = reinterpret_cast<const float4*>(a.q)[i];
  a.I4[b] = make_float4(I[0], I[1], I[2], __int_as_float(bits));
  a.F4[b] = make_float4(f[0], f[1], f[2], 0.0f);
  a.T4[b] = make_float4(t[0], t[1], t[2], 0.0f);
  if (!a.old_keep) a.old4[b] = make_float4(o[0], o[1], o[2], 0.0f);
}

// user (N, M) list of original ids -> slot-major work list; history likewise
__global__ void __launch_bounds__(kBlock) k_in_nlist(InOut a) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= a.n) return;
  const int64_t i = a.orig[b];
  const int W32 = (a.M + 31) / 32;
  for (int w = 0; w < a.W64; ++w) a.live[(int64_t)w * a.n + b] = 0ull;
  int rank = 0;
  for (int s = 0; s < a.M; ++s) {
    int32_t j = a.nl_user[i * a.M + s];
    if (j >= a.n) j = -1;  // not a particle of this state: treated as padding
    a.nl[(int64_t)s * a.n + b] = j >= 0 ? a.wpos[j] : -1;
    if (a.xi_user && j >= 0) {
      const bool lv = (a.live_user[i * W32 + (s >> 5)] >> (s & 31)) & 1u;
      if (lv) {
        float x[3] = {0, 0, 0};
        for (int c = 0; c < a.dim; ++c) x[c] = a.xi_user[(i * a.M + s) * a.dim + c];
        a.xi[(int64_t)rank * a.n + b] = make_float4(x[0], x[1], x[2], 0.0f);
        ++rank;
        a.live[(int64_t)(s >> 6) * a.n + b] |= 1ull << (s & 63);
      }
    }
  }
}

__global__ void __launch_bounds__(kBlock) k_out_state(InOut a) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= a.n) return;
  const int64_t i = a.orig[b];
  const int D = a.dim;
  const int A = D == 3 ? 3 : 1;
  const float4 p = a.P4[b], v = a.V4[b], w = a.W4[b], f = a.F4[b], t = a.T4[b], o = a.old4[b];
  const float pp[3] = {p.x, p.y, p.z}, vv[3] = {v.x, v.y, v.z}, ww[3] = {w.x, w.y, w.z}, ff[3] = {f.x, f.y, f.z},
              tt[3] = {t.x, t.y, t.z}, oo[3] = {o.x, o.y, o.z};
  for (int c = 0; c < D; ++c) {
    a.pos[D * i + c] = pp[c];
    a.vel[D * i + c] = vv[c];
    a.force[D * i + c] = ff[c];
    if (a.old_user) a.old_user[D * i + c] = oo[c];
  }
  for (int c = 0; c < A; ++c) {
    a.ang[A * i + c] = ww[c];
    a.torque[A * i + c] = tt[c];
  }
  reinterpret_cast<float4*>(a.q)[i] = a.Q4[b];
}

__global__ void __launch_bounds__(kBlock) k_out_nlist(InOut a) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= a.n) return;
  const int64_t i = a.orig[b];
  const int W32 = (a.M + 31) / 32;
  uint32_t words[8];
  for (int w = 0; w < W32 && w < 8; ++w) words[w] = 0u;
  bool ended = false;  // work rows end at their first -1
  int rank = 0;
  for (int s = 0; s < a.M; ++s) {
    const int32_t j = ended ? -1 : a.nl[(int64_t)s * a.n + b];
    ended = j < 0;
    a.nl_user[i * a.M + s] = j >= 0 ? a.orig[j] : -1;
    if (a.xi_user) {
      const bool lv = j >= 0 && ((a.live[(int64_t)(s >> 6) * a.n + b] >> (s & 63)) & 1ull);
      if (lv) {
        const float4 x = a.xi[(int64_t)rank * a.n + b];
        ++rank;
        const float xx[3] = {x.x, x.y, x.z};
        for (int c = 0; c < a.dim; ++c) a.xi_user[(i * a.M + s) * a.dim + c] = xx[c];
        if ((s >> 5) < 8) words[s >> 5] |= 1u << (s & 31);
      }
    }
  }
  if (a.xi_user)
    for (int w = 0; w < W32 && w < 8; ++w) a.live_user[i * W32 + w] = words[w];
}

// positions at the last build, work order -> the caller's (N, D)
__global__ void __launch_bounds__(kBlock) k_out_old(InOut a) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= a.n) return;
  const int64_t i = a.orig[b];
  const float4 o = a.old4[b];
  const float oo[3] = {o.x, o.y, o.z};
  for (int c = 0; c < a.dim; ++c) a.old_user[a.dim * i + c] = oo[c];
}

// Slot-major rows up to and including their first -1 (every reader of a work
// row stops there), so a working set is copied in proportion to its entries.
__global__ void __launch_bounds__(kBlock) k_copy_rows(const int32_t* __restrict__ src, int32_t* __restrict__ dst,
                                                       int64_t n, int M) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n) return;
  for (int s = 0; s < M; ++s) {
    const int32_t v = src[(int64_t)s * n + b];
    dst[(int64_t)s * n + b] = v;
    if (v < 0) break;
  }
}

// ---------------------------------------------------------------------------
// rebuild: hash in original order, stable sort, permutation of the work set
// ---------------------------------------------------------------------------
template <bool PER>
JD int ccoord(float x, int a, const DomP& dom, const GridP& g) {
  float f;
  if (PER) {
    float t = (x - dom.anchor[a]) / dom.box[a];
    t = t - floorf(t);
    f = floorf(t * (float)g.dims[a]);
  } else {
    f = floorf((x - dom.anchor[a]) / g.cell[a]);
  }
  f = fminf(fmaxf(f, 0.0f), (float)(g.dims[a] - 1));
  return (int)f;
}

// Work-space cell key: the LAST axis varies fastest (z in 3D, y in 2D), so
// the stencil's fastest axis ('ij' meshgrid order, cell_list.py:425-427)
// walks consecutive keys.  Any linearisation gives the same rows (stencil
// order, ascending id within a cell); this one makes a stencil column one
// contiguous range of the sorted work set.
template <int D>
JD uint32_t wkey(const int* c, const GridP& g) {
  if (D == 3) return (uint32_t)((c[0] * g.dims[1] + c[1]) * g.dims[2] + c[2]);
  return (uint32_t)(c[0] * g.dims[1] + c[1]);
}

// keys[orig[b]] = work cell key of P4[b]; wpos[orig[b]] = b; with cnt, the
// element's arrival number in its cell
template <int D, bool PER>
__global__ void __launch_bounds__(kBlock) k_hash_work(const float4* __restrict__ P4, const int32_t* __restrict__ orig,
                                                       int64_t n, DomP dom, GridP g, uint32_t* __restrict__ keys,
                                                       int32_t* __restrict__ wpos, int32_t* __restrict__ cnt,
                                                       int32_t* __restrict__ arr) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n) return;
  const float4 p = P4[b];
  const float x[3] = {p.x, p.y, p.z};
  int c[3] = {0, 0, 0};
#pragma unroll
  for (int a = 0; a < D; ++a) c[a] = ccoord<PER>(x[a], a, dom, g);
  const int32_t i = orig[b];
  const uint32_t k = wkey<D>(c, g);
  keys[i] = k;
  wpos[i] = (int32_t)b;
  if (cnt) arr[i] = atomicAdd(&cnt[k], 1);  // the count pass of the counting sort
}

// seg[b] = the system whose particle range [offsets[s], offsets[s + 1])
// holds b
__global__ void __launch_bounds__(kBlock) k_seg_ids(const int64_t* __restrict__ offsets, int n_seg, int64_t n,
                                                     int32_t* __restrict__ seg) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n) return;
  int lo = 0, hi = n_seg;  // largest s with offsets[s] <= b
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (offsets[mid] <= b)
      lo = mid;
    else
      hi = mid;
  }
  seg[b] = lo;
}

// Dense cell starts: starts[h] = first sorted slot with key >= h, for h in
// [0, n_cells]; an empty cell gets the start of the next occupied one, so
// consecutive cells h1..h2 hold the slots [starts[h1], starts[h2 + 1]).  A
// workgroup takes kStartsChunk cells: its first two wavefronts search the
// slots of the chunk's two ends, 64 ways at a time, and each cell is searched
// between those, which for most chunks of a sparse grid are one and the same
// slot.  So a run of empty cells costs its 4 bytes a cell whatever its length:
// with a full search per cell the step of 200 k disks on 1.6 10^8 cells took
// 1.32 ms, 0.44 here; filled by the thread of the slot behind it, the empty planes of a
// lattice on cells of half its spacing took 1.4 ms at 150 k spheres.
constexpr int kStartsChunk = 16 * kBlock;

// first of the slots [0, n] with key >= h; the whole wavefront calls
JD int64_t wave_lower_bound(const uint32_t* __restrict__ sk, int64_t n, int64_t h) {
  const int lane = threadIdx.x & 63;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t step = (hi - lo + 63) / 64, p = lo + lane * step;
    const int below = __popcll(__ballot(p < hi && (int64_t)sk[p < hi ? p : lo] < h));  // probes 0 .. below - 1
    hi = below == 0 ? lo : min(hi, lo + below * step);
    lo = below == 0 ? lo : lo + (below - 1) * step + 1;
  }
  return lo;
}

__global__ void __launch_bounds__(kBlock) k_cell_starts(const uint32_t* __restrict__ sk, int64_t n, int64_t n_cells,
                                                         int32_t* __restrict__ starts) {
  __shared__ int64_t ends[2];
  const int64_t c0 = (int64_t)blockIdx.x * kStartsChunk, c1 = min(c0 + kStartsChunk, n_cells + 1);
  if (threadIdx.x < 128) {
    const int w = threadIdx.x >> 6;
    const int64_t at = wave_lower_bound(sk, n, w ? c1 - 1 : c0);
    if ((threadIdx.x & 63) == 0) ends[w] = at;
  }
  __syncthreads();
  for (int64_t h = c0 + threadIdx.x; h < c1; h += kBlock) {
    int64_t lo = ends[0], hi = ends[1];
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if ((int64_t)sk[mid] < h)
        lo = mid + 1;
      else
        hi = mid;
    }
    starts[h] = (int32_t)lo;
  }
}

// new work slot b' takes old slot src = wpos[new_orig[b']]; inv[src] = b'
__global__ void __launch_bounds__(kBlock) k_permute(int64_t n, const int32_t* __restrict__ new_orig,
                                                     const int32_t* __restrict__ wpos, const float4* __restrict__ P,
                                                     const float4* __restrict__ V, const float4* __restrict__ W,
                                                     const float4* __restrict__ Q, const float4* __restrict__ I,
                                                     float4* __restrict__ P2, float4* __restrict__ V2,
                                                     float4* __restrict__ W2, float4* __restrict__ Q2,
                                                     float4* __restrict__ I2, int32_t* __restrict__ orig2,
                                                     int32_t* __restrict__ src_out, int32_t* __restrict__ inv_out,
                                                     float4* __restrict__ old2, int dim) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n) return;
  const int32_t i = new_orig[b];
  const int32_t s = wpos[i];
  float4 p = P[s];
  float4 v = V[s];
  if (old2) {
    old2[b] = p;  // the positions of this build
    if (dim == 2) {  // and in the 2D records' free lanes
      p.z = p.x;
      v.z = p.y;
    }
  }
  P2[b] = p;
  V2[b] = v;
  W2[b] = W[s];
  Q2[b] = Q[s];
  I2[b] = I[s];
  orig2[b] = i;
  src_out[b] = s;
  inv_out[s] = (int32_t)b;
}

// Call start, before the first step kernel: a system without a list asks
// for a build (and raises *gate when set), every other flag starts clear.
__global__ void k_seg_init_flags(int n_seg, const int32_t* __restrict__ n_build, int32_t* __restrict__ seg_flag,
                                 int32_t* __restrict__ gate) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n_seg) return;
  const bool unbuilt = n_build[s] == 0;
  seg_flag[s] = unbuilt ? 1 : 0;
  if (unbuilt && gate) *gate = 1;
}

// ---- batch rebuilds in place -----------------------------------------------
// Only the systems that asked for a rebuild are re-sorted and rebuilt, each
// inside its own range of work slots; the others are not touched.  Flagged
// particles are numbered compactly: system s's particles take the compact
// range [cpref[s], cpref[s + 1]) in original order, its cells the compact
// key range starting at ccref[s].
//
// The chain runs after every step and mostly finds nothing to do, so what it
// costs is its launches: plan, keys, scan totals, scan, placement, gather and
// rows, seven where every pass had a kernel of its own (eighteen: 55 us of a
// step of 256 systems of disks, 31 us now).

// Wavefronts (64 work slots) that hold particles of system s.
JD int64_t seg_waves(const int64_t* __restrict__ offsets, int s) {
  const int64_t a = offsets[s], e = offsets[s + 1];
  return e > a ? ((e - 1) >> 6) - (a >> 6) + 1 : 0;
}

// The plan (one block): the gate word moves to go, which the other kernels of
// the chain read, so the next step kernel finds it clear.  If it is set: the
// mode of each system (KEEP when it did not ask for a rebuild, FRESH for its
// first build, REMAP otherwise; its build count grows and its flag is cleared)
// and the exclusive prefix sums over the systems of the flagged particle, cell
// and wavefront counts.
__global__ void __launch_bounds__(1024) k_rebuild_plan(RB r, RBPlan q) {
  const bool go = *q.gate != 0;
  __syncthreads();  // every thread has read the gate
  const int t = threadIdx.x;
  if (t == 0) {
    *q.go = go ? 1 : 0;
    if (go) {
      *q.gate = 0;
      *q.overflow = 0;
      *q.events += 1;
    }
  }
  if (!go) return;
  __shared__ int64_t sp[1024], sc[1024], sw[1024];
  const int per = (r.n_seg + 1023) / 1024;
  const int s0 = t * per, s1 = min(r.n_seg, s0 + per);
  int64_t np = 0, nc = 0, nw = 0;
  for (int s = s0; s < s1; ++s) {
    const int f = q.seg_flag[s] != 0;
    r.seg_mode[s] = f ? (q.n_build[s] > 0 ? SEG_REMAP : SEG_FRESH) : SEG_KEEP;
    if (!f) continue;
    q.n_build[s] += 1;
    q.seg_flag[s] = 0;
    np += r.offsets[s + 1] - r.offsets[s];
    nc += r.segp[s].grid.n_cells;
    nw += seg_waves(r.offsets, s);
  }
  sp[t] = np;
  sc[t] = nc;
  sw[t] = nw;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {  // inclusive scan
    const int64_t ap = t >= off ? sp[t - off] : 0, ac = t >= off ? sc[t - off] : 0, aw = t >= off ? sw[t - off] : 0;
    __syncthreads();
    sp[t] += ap;
    sc[t] += ac;
    sw[t] += aw;
    __syncthreads();
  }
  int64_t p = sp[t] - np, c = sc[t] - nc, w = sw[t] - nw;
  for (int s = s0; s < s1; ++s) {
    r.cpref[s] = p;
    r.ccref[s] = c;
    r.wpref[s] = w;
    if (r.seg_mode[s] != SEG_KEEP) {
      p += r.offsets[s + 1] - r.offsets[s];
      c += r.segp[s].grid.n_cells;
      w += seg_waves(r.offsets, s);
    }
  }
  if (t == 1023) {
    r.cpref[r.n_seg] = sp[t];
    r.ccref[r.n_seg] = sc[t];
    r.wpref[r.n_seg] = sw[t];
  }
}

// The flagged system that holds compact index k of a prefix over the
// systems (cpref, wpref): the last s with pref[s] <= k (systems that are
// not flagged add nothing to the prefix, so the next flagged one shares
// their value and comes after them).
JD int seg_of_compact(const int64_t* __restrict__ pref, int n_seg, int64_t k) {
  int lo = 0, hi = n_seg - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (pref[mid] <= k)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// The compact key of every particle of a flagged system, at its compact
// index, counted; and the springs of the kept systems' slots in the first and
// last wavefront of a flagged system, whose springs are placed anew.
template <int D>
__global__ void __launch_bounds__(kBlock) k_rebuild_keys(RB r) {
  if (*r.go == 0) return;
  const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t fn = r.cpref[r.n_seg];
  for (int64_t k = t0; k < fn; k += stride) {
    const int s = seg_of_compact(r.cpref, r.n_seg, k);
    const int64_t b = r.offsets[s] + (k - r.cpref[s]);
    const SegP& sp = r.segp[s];
    const float4 p = r.P[b];
    const float x[3] = {p.x, p.y, p.z};
    int c[3] = {0, 0, 0};
    const bool per = sp.dom.kind == JDEM_DOMAIN_PERIODIC;
#pragma unroll
    for (int a = 0; a < D; ++a)
      c[a] = per ? ccoord<true>(x[a], a, sp.dom, sp.grid) : ccoord<false>(x[a], a, sp.dom, sp.grid);
    const int64_t i = r.cpref[s] + (r.orig[b] - r.offsets[s]);
    const uint32_t key = (uint32_t)(r.ccref[s] + wkey<D>(c, sp.grid));
    r.keys_c[i] = key;
    r.slot_c[i] = (int32_t)b;
    r.arr[i] = atomicAdd(&r.cnt[key], 1);
  }
  if (!r.live) return;
  for (int64_t t = t0; t < (int64_t)r.n_seg * 128; t += stride) {
    const int s = (int)(t >> 7);
    const int64_t a = r.offsets[s], e = r.offsets[s + 1];
    if (r.seg_mode[s] == SEG_KEEP || e <= a) continue;
    const int64_t b = (((t & 64) ? e - 1 : a) & ~(int64_t)63) + (t & 63);
    if (b >= r.n || r.seg_mode[r.seg[b]] != SEG_KEEP) continue;
    int cnt = 0;
    for (int w = 0; w < r.W64; ++w) cnt += __popcll(r.live[(int64_t)w * r.n + b]);
    const float4* src = r.xi + (b & ~(int64_t)63) * r.M + __float_as_int(r.W[b].w);
    for (int k = 0; k < cnt; ++k) r.keep_xi[(int64_t)k * r.n + b] = src[k];
  }
}

// The rank pass of the sort, then the fields of the particle that goes to
// compact index k, and its live springs with their partners' old slots.
__global__ void __launch_bounds__(kBlock) k_rebuild_gather(RB r) {
  if (*r.go == 0) return;
  const int64_t fn = r.cpref[r.n_seg];
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < fn; j += (int64_t)gridDim.x * blockDim.x) {
    const uint2 me = r.pairs[j];
    const int32_t cs = r.starts[me.x], ce = r.starts[me.x + 1];
    int32_t k = cs;
    for (int32_t m = cs; m < ce; ++m) k += r.pairs[m].y < me.y ? 1 : 0;
    const int32_t ob = r.slot_c[me.y];
    const int s = r.seg[ob];
    r.sk[k] = me.x;
    r.tP[k] = r.P[ob];
    r.tV[k] = r.V[ob];
    r.tW[k] = r.W[ob];
    r.tQ[k] = r.Q[ob];
    r.tI[k] = r.I[ob];
    r.torig[k] = r.orig[ob];
    r.inv[ob] = (int32_t)(r.offsets[s] + (k - r.cpref[s]));
    if (!r.live) continue;
    int q = 0;
    if (r.seg_mode[s] == SEG_REMAP) {
      const float4* src = r.xi + ((int64_t)ob & ~(int64_t)63) * r.M + __float_as_int(r.W[ob].w);
      for (int c = 0; c < r.W64; ++c) {
        uint64_t bits = r.live[(int64_t)c * r.n + ob];
        while (bits) {
          const int sl = c * 64 + __ffsll((unsigned long long)bits) - 1;
          bits &= bits - 1ull;
          r.tnl[(int64_t)q * r.n + k] = r.nl[(int64_t)sl * r.n + ob];
          r.txi[(int64_t)q * r.n + k] = src[q];
          ++q;
        }
      }
    }
    r.tlive[k] = q;
  }
}

// neighbour list in work space (cell_list.py:500-595).  The stencil is
// walked in the reference's 'ij' order (cell_list.py:425-427), last axis
// fastest; a run of stencil cells along that axis is one contiguous range of
// work slots, [starts[h_first], starts[h_last + 1]), split in two where a
// periodic axis wraps.  Candidates within a cell come in ascending original
// id, the order of the reference's stable hash sort.

JD bool bonded_o(const int32_t* bond_id, int bond_w, int64_t i, int32_t j) {
  for (int w = 0; w < bond_w; ++w)
    if (bond_id[i * bond_w + w] == j) return true;
  return false;
}

// Number of set bits of the live words (w0..w3) below slot s.
JD int rank_below(uint64_t w0, uint64_t w1, uint64_t w2, uint64_t w3, int s) {
  const int ws = s >> 6;
  const uint64_t below = (1ull << (s & 63)) - 1ull;
  int r = 0;
  r += ws > 0 ? __popcll(w0) : __popcll(w0 & below);
  if (ws >= 1) r += ws > 1 ? __popcll(w1) : __popcll(w1 & below);
  if (ws >= 2) r += ws > 2 ? __popcll(w2) : __popcll(w2 & below);
  if (ws >= 3) r += __popcll(w3 & below);
  return r;
}

// History of a freshly built row (neighbor_list.py:29-54): the history of
// new pair (b, j) is the old history of the same two particles, zero when
// they were not listed together.  Only live old slots carry history, so each
// one is looked up in the new row (row(s), s < nrow): old slot t of src[b]
// lists old work slot o, now at inv[o].  A pair occurs at most once per row,
// so the lookups are one-to-one.  The first sweep finds the new live slots,
// the second copies each spring from its old rank to its new one.  Rows hold
// at most 256 slots (four live words).
template <class Row>
JD int find_in_row(int32_t tgt, int nrow, Row row) {
  for (int s = 0; s < nrow; ++s)
    if (row(s) == tgt) return s;
  return -1;
}

// exclusive prefix sum over the 64 lanes of a wave; every lane must call it
JD int wave_exclusive_scan(int v, int lane) {
  int incl = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int t = __shfl_up(incl, d);
    if (lane >= d) incl += t;
  }
  return incl - v;
}

// Every lane of the wave must call it (inactive lanes with
// active = false): the new springs are placed per wavefront after a
// wave-wide scan of the new counts.
template <class Row>
JD void remap_row(const NLW& a, int64_t b, bool active, int nrow, Row row, bool remap) {
  if (!a.live) return;
  const int64_t n = a.n;
  uint64_t out0 = 0ull, out1 = 0ull, out2 = 0ull, out3 = 0ull;
  // the old row of the particle now at b: at slot src[b] of the previous
  // buffers
  const bool go = active && remap;
  const int64_t ob = go ? (int64_t)a.src[b] : 0;
  // start of the old springs, read before any lane writes new offsets (old_W
  // and new_W are one buffer when the rebuild does not re-sort)
  const int64_t obase = go ? (ob & ~(int64_t)63) * a.M + __float_as_int(a.old_W[ob].w) : 0;
  // visit(t, o_slot_new): each live old slot t whose partner is listed
  // again, with the rank of t among the live old slots
  auto sweep = [&](auto&& f) {
    int rank_old = 0;
    for (int w = 0; w < a.W64; ++w) {
      uint64_t bits = a.old_live[(int64_t)w * n + ob];
      while (bits) {
        const int t = w * 64 + (__ffsll((unsigned long long)bits) - 1);
        bits &= bits - 1ull;
        const int32_t o = a.old_nl[(int64_t)t * n + ob];
        const int s = o < 0 ? -1 : find_in_row(a.inv[o], nrow, row);
        if (s >= 0) f(s, rank_old);
        ++rank_old;
      }
    }
  };
  if (go)
    sweep([&](int s, int) {
      const uint64_t bit = 1ull << (s & 63);
      const int ws = s >> 6;
      out0 |= ws == 0 ? bit : 0ull;
      out1 |= ws == 1 ? bit : 0ull;
      out2 |= ws == 2 ? bit : 0ull;
      out3 |= ws == 3 ? bit : 0ull;
    });
  const int cnt = __popcll(out0) + __popcll(out1) + __popcll(out2) + __popcll(out3);
  const int off = wave_exclusive_scan(cnt, (int)(threadIdx.x & 63));
  if (active) a.new_W[b].w = __int_as_float(off);
  const int64_t wbase = (b & ~(int64_t)63) * a.M + off;
  if (go)
    sweep([&](int s, int rank_old) {
      const int rank_new = rank_below(out0, out1, out2, out3, s);
      a.xi[wbase + rank_new] = a.old_xi[obase + rank_old];
    });
  if (!active) return;
  a.live[b] = out0;
  if (a.W64 > 1) a.live[n + b] = out1;
  if (a.W64 > 2) a.live[2 * n + b] = out2;
  if (a.W64 > 3) a.live[3 * n + b] = out3;
}

// A row ends at its first -1 (or at M slots); the slots after the
// terminator are not written.
JD void end_row(const NLW& a, int64_t b, bool active, int count) {
  if (active && count < a.M) a.nl[(int64_t)count * a.n + b] = -1;
  if (active && count > a.M) atomicOr(a.overflow, 1);
  remap_row(a, b, active, min(count, a.M), [&](int s) { return a.nl[(int64_t)s * a.n + b]; }, a.remap != 0);
}



// The first kRowLds slots of each row are collected in LDS, slot-major, and
// written out one slot at a time for the whole workgroup, so the stores of a
// slot are contiguous; later slots go straight to memory.
constexpr int kRowLds = 16;

// The neighbours of the particle self, one lane's walk: put(t, k) takes the
// t-th, in candidate order.  Returns how many there are.
template <int D, bool PER, class Put>
JD int lane_row(const float4* __restrict__ P4, const int32_t* __restrict__ orig, int64_t self, uint32_t key,
                const GridP& grid, const DomP& dom, float cutoff_sq, const int32_t* __restrict__ starts,
                const int32_t* __restrict__ bond_id, int bond_w, bool chk_bond, Put&& put) {
  const Vec<D> xi = xyz<D>(P4[self]);
  const int d0 = grid.dims[0], d1 = grid.dims[1], d2 = (D == 3) ? grid.dims[2] : 1;
  int c0, c1, cf;
  if (D == 3) {
    cf = (int)(key % (uint32_t)d2);
    const uint32_t r = key / (uint32_t)d2;
    c1 = (int)(r % (uint32_t)d1);
    c0 = (int)(r / (uint32_t)d1);
  } else {
    cf = (int)(key % (uint32_t)d1);
    c0 = (int)(key / (uint32_t)d1);
    c1 = 0;
  }
  const int sr = grid.sr;
  const int dF = (D == 3) ? d2 : d1;
  int r0a, r0b, r1a, r1b;
  stencil_runs(PER, cf, sr, dF, r0a, r0b, r1a, r1b);
  const int hi0 = PER ? min(sr, d0 - sr - 1) : sr;
  const int lo1 = (D == 3) ? -sr : 0;
  const int hi1 = (D == 3) ? (PER ? min(sr, d1 - sr - 1) : sr) : 0;
  const int64_t ib = chk_bond ? (int64_t)orig[self] : 0;
  int count = 0;
  for (int ox = -sr; ox <= hi0; ++ox) {
    const int cx = stencil_cell(PER, c0, ox, d0);
    if (cx < 0) continue;
    for (int oy = lo1; oy <= hi1; ++oy) {
      int64_t base;
      if (D == 3) {
        const int cy = stencil_cell(PER, c1, oy, d1);
        if (cy < 0) continue;
        base = (int64_t)(cx * d1 + cy) * d2;
      } else {
        base = (int64_t)cx * d1;
      }
      // both runs' bounds are loaded before either is walked
      const int k0 = starts[base + r0a], k0e = starts[base + r0b + 1];
      const int k1 = (r1b >= r1a) ? starts[base + r1a] : 0;
      const int k1e = (r1b >= r1a) ? starts[base + r1b + 1] : 0;
#pragma unroll
      for (int run = 0; run < 2; ++run) {
        const int kb = run ? k1 : k0, ke = run ? k1e : k0e;
        // candidates in groups of four, loaded back to back
        for (int kg = kb; kg < ke; kg += 4) {
          float4 pk[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) pk[u] = (kg + u < ke) ? P4[kg + u] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int k = kg + u;
            if (k >= ke) break;
            if (k == self) continue;
            const float dsq = dist_sq<PER>(xi, xyz<D>(pk[u]), dom);
            if (!(dsq <= cutoff_sq)) continue;
            if (chk_bond && bonded_o(bond_id, bond_w, ib, orig[k])) continue;
            put(count, k);
            ++count;
          }
        }
      }
    }
  }
  return count;
}

template <int D, bool PER>
__global__ void __launch_bounds__(kBlock) k_nlist_work(NLW a) {
  __shared__ int32_t rows[kRowLds][kBlock];
  __shared__ int row_max;
  const int tid = threadIdx.x;
  const int64_t b = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * kBlock + tid;
  if (tid == 0) row_max = 0;
  __syncthreads();
  const bool active = b < a.n;
  int count = 0;
  if (active)
    count = lane_row<D, PER>(a.P4, a.orig, b, a.skeys[b], a.grid, a.dom, a.cutoff_sq, a.starts, a.bond_id, a.bond_w,
                             (!a.isb) && a.bond_w > 0, [&](int t, int k) {
                               if (t < kRowLds)
                                 rows[t][tid] = k;
                               else if (t < a.M)
                                 a.nl[(int64_t)t * a.n + b] = k;
                             });
  if (active) atomicMax(&row_max, min(count, kRowLds));
  __syncthreads();
  const int c = min(count, a.M);
  if (active) {
    const int staged = min(row_max, a.M);
    for (int s = 0; s < staged; ++s)
      if (s < c) a.nl[(int64_t)s * a.n + b] = rows[s][tid];
    if (count < a.M) a.nl[(int64_t)count * a.n + b] = -1;
    if (count > a.M) atomicOr(a.overflow, 1);
  }
  remap_row(a, b, active, c, [&](int s) { return s < kRowLds ? rows[s][tid] : a.nl[(int64_t)s * a.n + b]; },
            a.remap != 0);
}

// The list build with a group of G lanes per particle: k_nlist_work's chain of
// column bounds and candidates is serial per lane, and below ~10^5 particles
// there are not enough wavefronts to hide it (154 us for 37 k spheres of 31
// neighbours, most of a rebuild; here 44 us).  A workgroup builds the rows of
// one wavefront's 64 slots: each lane loads one stencil column's bounds, a
// scan numbers the candidates, G of them are tested at a time and those within
// the cutoff appended in candidate order; the old springs are looked up one
// per lane; the new springs' places are a scan over the 64 slots.
// G = 16 in 3D (9 columns of 6 to 20 candidates), 8 in 2D (3 columns of 7).
template <int D>
constexpr int nlist_group() {
  return D == 3 ? 16 : 8;
}
constexpr int kRowGrp = 64;  // row slots collected in LDS

// position of the r-th set bit of the words (r below their count)
JD int select_bit(const uint64_t* w, int n_words, int r) {
  for (int q = 0; q < n_words; ++q) {
    const int c = __popcll(w[q]);
    if (r < c) {
      uint64_t b = w[q];
      for (; r > 0; --r) b &= b - 1ull;
      return q * 64 + __ffsll((unsigned long long)b) - 1;
    }
    r -= c;
  }
  return -1;
}

struct RowLds {
  int32_t rows[kRowGrp][64];
  int row_cnt[64], new_cnt[64], new_off[64];
};

// The row of the particle at slot b, whose lanes p * G .. p * G + G - 1 of the
// workgroup all call this: its own index among the candidates is self, a
// candidate's slot is its index + shift.  Returns the neighbours found, which
// may be more than the M slots kept.
template <int D, bool PER>
JD int group_row(RowLds& lds, const float4* __restrict__ P4, const int32_t* __restrict__ orig, int self, int shift,
                 uint32_t key, const GridP& grid, const DomP& dom, float cutoff_sq,
                 const int32_t* __restrict__ starts, const int32_t* __restrict__ bond_id, int bond_w, bool chk_bond,
                 int32_t* __restrict__ nl, int64_t n, int M, int64_t b) {
  constexpr int G = nlist_group<D>();
  const int p = threadIdx.x / G, l = threadIdx.x & (G - 1), lane = threadIdx.x & 63;
  const uint64_t below = (1ull << l) - 1ull;
  const Vec<D> xi = xyz<D>(P4[self]);
  const int d0 = grid.dims[0], d1 = grid.dims[1], d2 = (D == 3) ? grid.dims[2] : 1;
  int c0, c1, cf;
  if (D == 3) {
    cf = (int)(key % (uint32_t)d2);
    const uint32_t r = key / (uint32_t)d2;
    c1 = (int)(r % (uint32_t)d1);
    c0 = (int)(r / (uint32_t)d1);
  } else {
    cf = (int)(key % (uint32_t)d1);
    c0 = (int)(key / (uint32_t)d1);
    c1 = 0;
  }
  const int sr = grid.sr, dF = (D == 3) ? d2 : d1;
  int r0a, r0b, r1a, r1b;
  stencil_runs(PER, cf, sr, dF, r0a, r0b, r1a, r1b);
  const int n1 = (D == 3) ? (PER ? min(sr, d1 - sr - 1) : sr) + sr + 1 : 1;
  const int ncol = ((PER ? min(sr, d0 - sr - 1) : sr) + sr + 1) * n1;
  const int64_t ib = chk_bond ? (int64_t)orig[self] : 0;
  int count = 0;
  for (int cb = 0; cb < ncol; cb += G) {
    const int col = cb + l;
    int s0 = 0, len0 = 0, s1 = 0, len1 = 0;
    if (col < ncol) {
      const int cx = stencil_cell(PER, c0, (D == 3 ? col / n1 : col) - sr, d0);
      const int cy = (D == 3) ? stencil_cell(PER, c1, col % n1 - sr, d1) : 0;
      if (cx >= 0 && cy >= 0) {
        const int64_t base = (D == 3) ? ((int64_t)cx * d1 + cy) * d2 : (int64_t)cx * d1;
        s0 = starts[base + r0a];
        len0 = starts[base + r0b + 1] - s0;
        if (r1b >= r1a) {
          s1 = starts[base + r1a];
          len1 = starts[base + r1b + 1] - s1;
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
    for (int c8 = 0; c8 < total; c8 += G) {
      const int cand = c8 + l;
      int q = 0;
#pragma unroll
      for (int st = G / 2; st > 0; st >>= 1) q += __shfl(pre, q + st, G) <= cand ? st : 0;
      const int o = cand - __shfl(pre, q, G), f0 = __shfl(s0, q, G), n_0 = __shfl(len0, q, G),
                f1 = __shfl(s1, q, G);
      const int k = o < n_0 ? f0 + o : f1 + (o - n_0);
      bool hit = false;
      if (cand < total && k != self) {
        const Vec<D> xk = xyz<D>(P4[k]);
        const float dsq = dist_sq<PER>(xi, xk, dom);
        hit = dsq <= cutoff_sq;
        if (hit && chk_bond) hit = !bonded_o(bond_id, bond_w, ib, orig[k]);
      }
      const uint64_t m = (__ballot(hit) >> (lane & ~(G - 1))) & ((1ull << G) - 1ull);
      if (hit) {
        const int t = count + __popcll(m & below);
        if (t < kRowGrp)
          lds.rows[t][p] = k + shift;
        else if (t < M)
          nl[(int64_t)t * n + b] = k + shift;
      }
      count += __popcll(m);
    }
  }
  return count;
}

// The collected slots of the region's rows, 64 consecutive particles at a time
// (after a barrier; row_cnt is -1 where no row was built).
template <int G>
JD void write_rows(const RowLds& lds, int32_t* __restrict__ nl, int64_t n, int64_t region) {
  const int lane = threadIdx.x & 63;
  const int cw = lds.row_cnt[lane];
  for (int s = threadIdx.x >> 6; s < kRowGrp; s += G) {
    if (s < cw) nl[(int64_t)s * n + region + lane] = lds.rows[s][lane];
    if (!__any(s + G < cw)) break;
  }
}

// The history of the new row of c slots at b (as remap_row): the r-th of n_old
// live old springs goes to the slot of the new row that lists its partner
// (slot partner(r) now), if any.  place(lane, off) is called once for each
// slot of the region with the start of its springs; spring(r) gives the r-th
// old one; a slot whose row was not built (built = false) keeps kept springs.
// Every thread of the workgroup calls this.
template <int G, int MW, class Partner, class Spring, class Place, class Kept>
JD void group_springs(RowLds& lds, bool built, int c, int n_old, int n_kept, const int32_t* __restrict__ nl,
                      int64_t n, int M, int W64, int64_t region, float4* __restrict__ xi, uint64_t* __restrict__ live,
                      Partner partner, Spring spring, Place place, Kept kept) {
  const int tid = threadIdx.x, p = tid / G, l = tid & (G - 1);
  const int64_t b = region + p;
  uint64_t out[MW];
#pragma unroll
  for (int w = 0; w < MW; ++w) out[w] = 0ull;
  auto new_slot = [&](int r) {
    const int32_t tgt = partner(r);
    if (tgt < 0) return -1;
    for (int s = 0; s < c; ++s)
      if ((s < kRowGrp ? lds.rows[s][p] : nl[(int64_t)s * n + b]) == tgt) return s;
    return -1;
  };
  const int first = l < n_old ? new_slot(l) : -1;  // kept: rows rarely carry more than G springs
  for (int r = l; r < n_old; r += G) {
    const int s = r == l ? first : new_slot(r);
    if (s >= 0)
#pragma unroll
      for (int w = 0; w < MW; ++w) out[w] |= (s >> 6) == w ? 1ull << (s & 63) : 0ull;
  }
#pragma unroll
  for (int w = 0; w < MW; ++w) {
    if (w >= W64) break;  // uniform
#pragma unroll 1
    for (int d = 1; d < G; d <<= 1) out[w] |= (uint64_t)__shfl_xor((unsigned long long)out[w], d, G);
  }
  if (l == 0) {
    int k = n_kept;
#pragma unroll
    for (int w = 0; w < MW; ++w) k += __popcll(out[w]);
    lds.new_cnt[p] = k;
  }
  __syncthreads();  // the old offsets are read, the counts are there
  if (tid < 64) {
    const int off = wave_exclusive_scan(lds.new_cnt[tid], tid);
    lds.new_off[tid] = off;
    place(tid, off);
  }
  __syncthreads();
  const int64_t wbase = region * M + lds.new_off[p];
  for (int r = l; r < n_old; r += G) {
    const int s = r == l ? first : new_slot(r);
    if (s < 0) continue;
    const int rank = MW == 1 ? __popcll(out[0] & ((1ull << s) - 1ull))
                             : rank_below(out[0], out[MW > 1 ? 1 : 0], out[MW > 2 ? 2 : 0], out[MW > 3 ? 3 : 0], s);
    xi[wbase + rank] = spring(r);
  }
  for (int r = l; r < n_kept; r += G) xi[wbase + r] = kept(r);
  if (built && l == 0)
#pragma unroll
    for (int w = 0; w < MW; ++w)
      if (w < W64) live[(int64_t)w * n + b] = out[w];
}

// One system.  MW: live words of a row (1, or 4 for rows of more than 64
// slots).  Eight waves per SIMD (64 VGPRs) let two 3D workgroups share a CU.
template <int D, bool PER, int MW>
__global__ void __launch_bounds__(64 * nlist_group<D>()) __attribute__((amdgpu_waves_per_eu(8, 8)))
k_nlist_group(NLW a) {
  constexpr int G = nlist_group<D>();
  __shared__ RowLds lds;
  const int tid = threadIdx.x, p = tid / G, l = tid & (G - 1);
  const int64_t n = a.n;
  const int64_t region = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * 64, b = region + p;
  const bool active = b < n;
  int count = 0;
  if (active)
    count = group_row<D, PER>(lds, a.P4, a.orig, (int)b, 0, a.skeys[b], a.grid, a.dom, a.cutoff_sq, a.starts,
                                      a.bond_id, a.bond_w, (!a.isb) && a.bond_w > 0, a.nl, n, a.M, b);
  const int c = min(count, a.M);
  if (l == 0) lds.row_cnt[p] = active ? c : -1;
  __syncthreads();
  write_rows<G>(lds, a.nl, n, region);
  if (active && l == 0) {
    if (count < a.M) a.nl[(int64_t)count * n + b] = -1;
    if (count > a.M) atomicOr(a.overflow, 1);
  }
  if (!a.live) return;
  const bool go = active && a.remap != 0;
  const int64_t ob = go ? (int64_t)a.src[b] : 0;
  const int64_t obase = go ? (ob & ~(int64_t)63) * a.M + __float_as_int(a.old_W[ob].w) : 0;
  uint64_t old[MW];
  int n_old = 0;
#pragma unroll
  for (int w = 0; w < MW; ++w) {
    old[w] = go && w < a.W64 ? a.old_live[(int64_t)w * n + ob] : 0ull;
    n_old += __popcll(old[w]);
  }
  group_springs<G, MW>(
      lds, active, c, n_old, 0, a.nl, n, a.M, a.W64, region, a.xi, a.live,
      [&](int r) {
        const int32_t o = a.old_nl[(int64_t)select_bit(old, MW, r) * n + ob];
        return o < 0 ? -1 : a.inv[o];
      },
      [&](int r) { return a.old_xi[obase + r]; },
      [&](int lane, int off) {
        if (region + lane < n) a.new_W[region + lane].w = __int_as_float(off);
      },
      [&](int) { return make_float4(0.f, 0.f, 0.f, 0.f); });
}

// A batch rebuild of many particles, one lane each: a wavefront builds the rows
// of one region of 64 slots and moves their fields and springs.
template <int D, int MW>
JD void lane_regions(const RB& r, int32_t (*rows)[64 * nlist_group<D>()]) {
  constexpr int G = nlist_group<D>();
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t n = r.n, nreg = r.wpref[r.n_seg];
  const int64_t w0 = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * G + (tid >> 6);
  for (int64_t reg = w0; reg < nreg; reg += (int64_t)gridDim.x * G) {  // uniform over the wavefront
    const int fs = seg_of_compact(r.wpref, r.n_seg, reg);
    const int region = (int)((r.offsets[fs] >> 6) + (reg - r.wpref[fs])) * 64, b = region + lane;
    const int sg = b < n ? r.seg[b] : -1;
    const bool active = b < n && r.seg_mode[sg] != SEG_KEEP;
    const int k = active ? (int)(r.cpref[sg] + (b - r.offsets[sg])) : 0;  // compact index
    int count = 0;
    if (r.M > 0) {
      const int s_last = __builtin_amdgcn_readfirstlane(r.seg[min((int64_t)region + 63, n - 1)]);
      for (int s = __builtin_amdgcn_readfirstlane(r.seg[region]); s <= s_last; ++s) {
        const SegP& sp = r.segp[s];
        const int64_t c0 = r.ccref[s];
        auto row = [&](auto per) {
          return lane_row<D, decltype(per)::value>(r.tP, r.torig, k, r.sk[k] - (uint32_t)c0, sp.grid, sp.dom,
                                                   sp.cutoff_sq, r.starts + c0, r.bond_id, r.bond_w,
                                                   (!r.isb) && r.bond_w > 0, [&](int t, int j) {
                                                     const int32_t slot = (int32_t)(j + (b - k));
                                                     if (t < kRowLds)
                                                       rows[t][tid] = slot;
                                                     else if (t < r.M)
                                                       r.nl[(int64_t)t * n + b] = slot;
                                                   });
        };
        if (active && sg == s)
          count = sp.dom.kind == JDEM_DOMAIN_PERIODIC ? row(std::true_type{}) : row(std::false_type{});
      }
    }
    const int c = min(count, r.M);
    if (active) {
      for (int t = 0; t < min(c, kRowLds); ++t) r.nl[(int64_t)t * n + b] = rows[t][tid];
      if (count < r.M) r.nl[(int64_t)count * n + b] = -1;
      if (count > r.M) atomicOr(r.overflow, 1);
      const float4 x = r.tP[k], v = r.tV[k];
      r.old4[b] = x;  // build position
      r.P[b] = D == 2 ? make_float4(x.x, x.y, x.x, x.w) : x;  // and in the 2D records' free lanes
      r.V[b] = D == 2 ? make_float4(v.x, v.y, x.y, v.w) : v;
      r.Q[b] = r.tQ[k];
      r.I[b] = r.tI[k];
      r.orig[b] = r.torig[k];
      if (!r.live) r.W[b] = r.tW[k];
    }
    if (!r.live) continue;
    const int n_old = active ? r.tlive[k] : 0;
    int n_kept = 0;
    if (b < n && !active)
      for (int w = 0; w < r.W64; ++w) n_kept += __popcll(r.live[(int64_t)w * n + b]);
    // each old spring's slot in the new row (as group_springs)
    auto new_slot = [&](int q) {
      const int32_t o = r.tnl[(int64_t)q * n + k];
      return o < 0 ? -1 : find_in_row(r.inv[o], c, [&](int t) { return t < kRowLds ? rows[t][tid] : r.nl[(int64_t)t * n + b]; });
    };
    uint64_t out[MW];
#pragma unroll
    for (int w = 0; w < MW; ++w) out[w] = 0ull;
    for (int q = 0; q < n_old; ++q) {
      const int t = new_slot(q);
#pragma unroll
      for (int w = 0; w < MW; ++w) out[w] |= t >= 0 && (t >> 6) == w ? 1ull << (t & 63) : 0ull;
    }
    int cnt = n_kept;
#pragma unroll
    for (int w = 0; w < MW; ++w) cnt += __popcll(out[w]);
    const int off = wave_exclusive_scan(cnt, lane);
    if (b >= n) continue;
    const int64_t wbase = (int64_t)region * r.M + off;
    if (!active) {
      r.W[b].w = __int_as_float(off);
      for (int q = 0; q < n_kept; ++q) r.xi[wbase + q] = r.keep_xi[(int64_t)q * n + b];
      continue;
    }
    const float4 w4 = r.tW[k];
    r.W[b] = make_float4(w4.x, w4.y, w4.z, __int_as_float(off));
    for (int q = 0; q < n_old; ++q) {
      const int t = new_slot(q);
      if (t < 0) continue;
      const int rank = MW == 1 ? __popcll(out[0] & ((1ull << t) - 1ull))
                               : rank_below(out[0], out[MW > 1 ? 1 : 0], out[MW > 2 ? 2 : 0], out[MW > 3 ? 3 : 0], t);
      r.xi[wbase + rank] = r.txi[(int64_t)q * n + k];
    }
#pragma unroll
    for (int w = 0; w < MW; ++w)
      if (w < r.W64) r.live[(int64_t)w * n + b] = out[w];
  }
}

// From this many particles to rebuild at once, groups of lanes would only add
// instructions.  A rebuild of all systems of a batch, group / lane, us (the
// whole chain): disks of like size with springs 70 / 81 at 120 k, 99 / 86 at
// 250 k, 184 / 104 at 500 k, 388 / 215 at 10^6; spheres 126 / 155, 217 / 165,
// 454 / 223, 938 / 455; log-normal spheres without springs 141 / 272,
// 238 / 275, 437 / 337, 871 / 644.  Below 10^5 groups take half the time.
constexpr int64_t kRebuildLane = 300000;

// The flagged systems of a batch, from the staged particles: rows, springs
// and the particles' fields in their new slots, over the wavefronts that hold
// a flagged system (one shared by two of them is written twice, alike).
// Groups of lanes or, from kRebuildLane particles on, a lane each: with lanes a
// rebuild of one of eight systems of 1 k to 150 k polydisperse spheres left
// most of the chip idle (this kernel 119 us, 58 with groups).
template <int D, int MW>
__global__ void __launch_bounds__(64 * nlist_group<D>()) __attribute__((amdgpu_waves_per_eu(8, 8)))
k_rebuild_rows(RB r) {
  if (*r.go == 0) return;
  constexpr int G = nlist_group<D>();
  union Lds {
    RowLds group;
    int32_t lanes[kRowLds][64 * G];
  };
  __shared__ Lds both;
  if (r.cpref[r.n_seg] >= kRebuildLane) {
    lane_regions<D, MW>(r, both.lanes);
    return;
  }
  RowLds& lds = both.group;
  const int tid = threadIdx.x, p = tid / G, l = tid & (G - 1), lane = tid & 63;
  const int64_t n = r.n, nreg = r.wpref[r.n_seg];
  for (int64_t reg = xcd_tile(blockIdx.x, gridDim.x); reg < nreg; reg += gridDim.x) {
    const int fs = seg_of_compact(r.wpref, r.n_seg, reg);
    const int region = (int)((r.offsets[fs] >> 6) + (reg - r.wpref[fs])) * 64, b = region + p;
    const int sg = b < n ? r.seg[b] : -1;
    const int mode = b < n ? r.seg_mode[sg] : SEG_FRESH;
    const bool active = b < n && mode != SEG_KEEP;
    const int k = active ? (int)(r.cpref[sg] + (b - r.offsets[sg])) : 0;  // compact index
    int count = 0;
    if (r.M > 0) {
      // system by system (mostly one), so that the grid and domain are uniform
      const int s_last = __builtin_amdgcn_readfirstlane(r.seg[min((int64_t)region + 63, n - 1)]);
      for (int s = __builtin_amdgcn_readfirstlane(r.seg[region]); s <= s_last; ++s) {
        const SegP& sp = r.segp[s];
        const int64_t c0 = r.ccref[s];
        auto row = [&](auto per) {
          return group_row<D, decltype(per)::value>(lds, r.tP, r.torig, k, b - k, r.sk[k] - (uint32_t)c0,
                                                    sp.grid, sp.dom, sp.cutoff_sq, r.starts + c0, r.bond_id, r.bond_w,
                                                    (!r.isb) && r.bond_w > 0, r.nl, n, r.M, b);
        };
        if (active && sg == s)
          count = sp.dom.kind == JDEM_DOMAIN_PERIODIC ? row(std::true_type{}) : row(std::false_type{});
      }
    }
    const int c = min(count, r.M);
    if (l == 0) lds.row_cnt[p] = active ? c : -1;
    __syncthreads();
    write_rows<G>(lds, r.nl, n, region);
    if (active && l == 0) {
      if (count < r.M) r.nl[(int64_t)count * n + b] = -1;
      if (count > r.M) atomicOr(r.overflow, 1);
    }
    {  // the fields, one kind per wavefront
      const int bw = region + lane;
      if (lds.row_cnt[lane] >= 0) {
        const int sw = r.seg[bw];
        const int64_t kw = r.cpref[sw] + (bw - r.offsets[sw]);
        switch (tid >> 6) {
          case 0: {
            const float4 x = r.tP[kw];
            r.old4[bw] = x;  // build position
            r.P[bw] = D == 2 ? make_float4(x.x, x.y, x.x, x.w) : x;  // and in the 2D records' free lanes
            break;
          }
          case 1: {
            const float4 v = r.tV[kw];
            r.V[bw] = D == 2 ? make_float4(v.x, v.y, r.tP[kw].y, v.w) : v;
            break;
          }
          case 2:
            r.Q[bw] = r.tQ[kw];
            break;
          case 3:
            r.I[bw] = r.tI[kw];
            break;
          case 4:
            r.orig[bw] = r.torig[kw];
            break;
          case 5:
            if (!r.live) r.W[bw] = r.tW[kw];
            break;
          default:
            break;
        }
      }
    }
    if (r.live) {
      const int n_old = active ? r.tlive[k] : 0;
      int n_kept = 0;
      if (b < n && !active)
        for (int w = 0; w < r.W64; ++w) n_kept += __popcll(r.live[(int64_t)w * n + b]);
      group_springs<G, MW>(
          lds, active, c, n_old, n_kept, r.nl, n, r.M, r.W64, region, r.xi, r.live,
          [&](int q) {
            const int32_t o = r.tnl[(int64_t)q * n + k];
            return o < 0 ? -1 : r.inv[o];
          },
          [&](int q) { return r.txi[(int64_t)q * n + k]; },
          [&](int ln, int off) {
            const int bw = region + ln;
            if (bw >= n) return;
            if (lds.row_cnt[ln] >= 0) {
              const int sw = r.seg[bw];
              const float4 w = r.tW[r.cpref[sw] + (bw - r.offsets[sw])];
              r.W[bw] = make_float4(w.x, w.y, w.z, __int_as_float(off));
            } else {
              r.W[bw].w = __int_as_float(off);
            }
          },
          [&](int q) { return r.keep_xi[(int64_t)q * n + b]; });
    }
    __syncthreads();  // the next region reuses the LDS
  }
}

__global__ void __launch_bounds__(kBlock) k_copy_f4(float4* __restrict__ d, const float4* __restrict__ s, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = s[i];
}

__global__ void __launch_bounds__(kBlock) k_iota(int32_t* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = (int32_t)i;
}


// ---------------------------------------------------------------------------
// spring layouts: by rank <-> per wavefront
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(kBlock) k_pack_springs(int64_t n, int M, int W64, const float4* __restrict__ rank,
                                                          const uint64_t* __restrict__ live, float4* __restrict__ wave,
                                                          float4* __restrict__ W) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int cnt = 0;
  if (b < n)
    for (int w = 0; w < W64; ++w) cnt += __popcll(live[(int64_t)w * n + b]);
  const int off = wave_exclusive_scan(cnt, threadIdx.x & 63);
  if (b >= n) return;
  float4* dst = wave + (b & ~(int64_t)63) * M + off;
  for (int k = 0; k < cnt; ++k) dst[k] = rank[(int64_t)k * n + b];
  W[b].w = __int_as_float(off);
}

__global__ void __launch_bounds__(kBlock) k_unpack_springs(int64_t n, int M, int W64, const float4* __restrict__ wave,
                                                            const uint64_t* __restrict__ live,
                                                            const float4* __restrict__ W, float4* __restrict__ rank) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n) return;
  int cnt = 0;
  for (int w = 0; w < W64; ++w) cnt += __popcll(live[(int64_t)w * n + b]);
  const float4* src = wave + (b & ~(int64_t)63) * M + __float_as_int(W[b].w);
  for (int k = 0; k < cnt; ++k) rank[(int64_t)k * n + b] = src[k];
}

// ---------------------------------------------------------------------------
// the fused step on the work set
// ---------------------------------------------------------------------------

// Minimum waves per SIMD asked of the compiler: six (80 VGPRs) holds the
// spring-friction law and the integrators; the Cundall-Strack and
// Hertz-friction laws in 3D need five, and one fewer in a segmented batch,
// whose per-system domain takes registers too, or with rows of more than 64
// slots, whose slot masks take four words.
template <int D, int LAW, int PM, int MW>
constexpr int ws_waves() {
  const bool heavy = D == 3 && (LAW == JDEM_LAW_CUNDALL_STRACK || LAW == JDEM_LAW_HERTZ_FRICTION ||
                                LawTraits<LAW>::routed);
  const bool seg3 = D == 3 && PM == 2 && LAW != JDEM_LAW_SPRING && LAW != JDEM_LAW_HERTZ;
  const bool wide = MW > 1 && LawTraits<LAW>::hist;
  const int w = heavy ? (PM == 2 ? 4 : 5) : (seg3 ? 5 : 6);
  return wide ? w - 1 : w;
}

// Domain._displacement for mode PM: 0 / 1 = one non-periodic / periodic
// system, 2 = the domain of the slot's system in a segmented batch.
template <int PM, int D>
JD Vec<D> disp_pm(Vec<D> a, Vec<D> b, const DomP& d) {
  if (PM == 2) return d.kind == JDEM_DOMAIN_PERIODIC ? disp_<true>(a, b, d) : disp_<false>(a, b, d);
  return disp_<PM == 1>(a, b, d);
}

// LDS of the lane-balanced force pass: per 64 particles and wave that works
// on them, kPairCap pair descriptors (more marked slots are taken in several
// chunks) and one round of 64 pair results (force + contact flag, torque,
// spring).
constexpr int kPairCap = 128;
// pass 1 keeps the partner index of a lane's first kStash marked slots in LDS,
// so the pair evaluation need not reload it from the list
constexpr int kStash = 4;

// MW = 64-slot words of a row the kernel handles (1 when M <= 64, else 4):
// the per-lane slot masks then take 2 * MW registers
// BS = workgroup size (the tile width: 256, or 128 for batches when the
// autotuner prefers it)
// NW = waves per 64 particles: 1, or 4 for small systems (below kWsSplit particles), where a
// lane's walk of its row, two dependent loads per four slots, is what a step
// takes and too few waves hide it.  Then the workgroup's waves share the
// rows of 64 particles, four slots in turn each, and the marked pairs; the
// first wave adds up and integrates.
template <int D, int LAW, int PM, int MW, int BS = kBlock, int NW = 1>
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(ws_waves<D, LAW, PM, MW>(), 8))) k_ws_step(WS a) {
  static_assert(NW == 1 || NW == BS / 64, "the waves of a workgroup share 64 particles, or none");
  constexpr int kSets = NW == 1 ? BS / 64 : 1, kCap = kPairCap * NW, kRound = 64 * NW;
  __shared__ int pdesc[kSets][kCap];
  __shared__ int pjx[kSets][kCap];
  __shared__ int pstash[BS / 64][kStash][64];
  __shared__ float4 pres[kSets][3][kRound];
  __shared__ int row_end[64];
  __shared__ uint64_t marks[NW][MW][64];
  auto sync = [] {
    if (NW == 1)
      wave_sync();
    else
      __syncthreads();
  };
  if (a.flag_rd && *a.flag_rd) {
    if (a.flag_wr) *a.flag_wr = *a.flag_rd;
    return;
  }
  // every lane of a wave stays to the end of the force pass, which works
  // wave-wide; a lane past the end reads the last particle and writes nothing
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, set = NW == 1 ? wv : 0;
  const int64_t b0 = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * (BS / NW) + (NW == 1 ? (int)threadIdx.x : lane);
  const bool active = b0 < a.n;
  const int64_t b = active ? b0 : a.n - 1;
  DomP dom;
  float dt, trigger;
  if (PM == 2) {
    const SegP& sp = a.segp[a.seg[b]];
    dom = sp.dom;
    dt = sp.dt;
    trigger = sp.trigger;
  } else {
    dom = a.dom;
    dt = a.dt;
    trigger = a.trigger;
  }
  // the force pass needs only this particle's position and radius; the
  // integration reloads them with the velocities and inertia after it,
  // which keeps them out of the registers the pair evaluation needs
  const float4 p4 = a.P[b];
  Side<D> me;
  me.x = xyz<D>(p4);
  me.r = p4.w;
  Vec<D> F;
  Ang<D> T;
  int spring_off = -1;  // start of this slot's new springs in its wave's region
  if (a.do_force) {
    F = zero_vec<D>();
    T = zero_ang<D>();
    // Pass 1 marks the slots whose pair is within reach of a contact,
    // d^2 <= R^2 * 1.0001 (a margin over the law's own overlap test); pass 2
    // evaluates the law on the marked slots only, in slot order, so a wave
    // runs the law as often as its busiest lane has contacts.  Pass 1 loads
    // PF list entries, then their positions, back to back before using any.
    constexpr int PF = 4;
    uint64_t cm[MW];
#pragma unroll
    for (int q = 0; q < MW; ++q) cm[q] = 0ull;
    int n_marked = 0;
    if (NW > 1) {  // the first -1 that any wave has come to
      if (wv == 0) row_end[lane] = a.M;
      __syncthreads();
    }
    bool done = false;
    for (int s0 = NW == 1 ? 0 : wv * PF; s0 < a.M && !done; s0 += NW * PF) {
      if (NW > 1 && s0 >= *(volatile int*)&row_end[lane]) break;
      int32_t js[PF];
      float4 pjs[PF];
#pragma unroll
      for (int k = 0; k < PF; ++k) js[k] = (s0 + k < a.M) ? a.nl[(int64_t)(s0 + k) * a.n + b] : -1;
      // the row ends at its first -1: what follows is stale
#pragma unroll
      for (int k = 1; k < PF; ++k) js[k] = js[k - 1] < 0 ? -1 : js[k];
      // (a wave of several may have come past the end of the row: what it
      // finds there is dropped below, but must not be read through)
#pragma unroll
      for (int k = 0; k < PF; ++k)
        pjs[k] = (NW == 1 ? js[k] >= 0 : (uint64_t)(int64_t)js[k] < (uint64_t)a.n) ? a.P[js[k]]
                                                                                 : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int k = 0; k < PF; ++k) {
        if (js[k] < 0) {
          done = true;
          if (NW > 1 && s0 + k < a.M) atomicMin(&row_end[lane], s0 + k);
          break;
        }
        const float4 pj = pjs[k];
        const Vec<D> rij = disp_pm<PM>(me.x, xyz<D>(pj), dom);
        const float d_sq = dot(rij, rij);
        const float R = me.r + pj.w;
        if (d_sq > (R * R) * 1.0001f) continue;
        if (n_marked < kStash) pstash[wv][n_marked][lane] = js[k];
        ++n_marked;
        const int s = s0 + k;
        const uint64_t bit = 1ull << (s & 63);
        const int ws = s >> 6;
#pragma unroll
        for (int q = 0; q < MW; ++q) cm[q] |= ws == q ? bit : 0ull;
      }
    }
    const int n_words = LawTraits<LAW>::hist ? a.W64 : (a.M + 63) >> 6;
    int nc = 0;
#pragma unroll
    for (int q = 0; q < MW; ++q) {
      if (!active) cm[q] = 0ull;
      nc += __popcll(cm[q]);
    }
    // all waves' marks up to the row's end; cm keeps this wave's
    uint64_t all[MW];
    if constexpr (NW > 1) {
#pragma unroll
      for (int q = 0; q < MW; ++q) marks[wv][q][lane] = cm[q];
      __syncthreads();
      const int end = row_end[lane];
      nc = 0;
#pragma unroll
      for (int q = 0; q < MW; ++q) {
        const int e = end - q * 64;
        const uint64_t keep = e >= 64 ? ~0ull : (e <= 0 ? 0ull : (1ull << e) - 1ull);
        all[q] = 0ull;
#pragma unroll
        for (int w = 0; w < NW; ++w) all[q] |= marks[w][q][lane];
        all[q] &= keep;
        cm[q] &= keep;
        nc += __popcll(all[q]);
      }
    }
    // Pass 2, lane-balanced: the wave's marked slots are numbered lane by
    // lane (slot order within a lane) and dealt out 64 at a time, one pair
    // per lane, so the law runs ceil(total / 64) times per wave instead of
    // as often as the busiest lane has contacts.  Each owner then adds its
    // pairs' results in slot order: the sums, springs and live bits are
    // those of one lane walking its own row.
    int incl = nc;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int t = __shfl_up(incl, d);
      if (lane >= d) incl += t;
    }
    const int total = __shfl(incl, 63);
    const int off = incl - nc;
    spring_off = off;
    uint64_t ln[MW];
#pragma unroll
    for (int q = 0; q < MW; ++q) ln[q] = 0ull;
    int rank_new = 0;  // springs are stored by rank
    for (int cb = 0; cb < total; cb += kCap) {  // uniform over the waves of a set
      // descriptors of pairs cb .. cb + kCap - 1: owner lane | slot << 6
      // | (old spring's place in the wave's region + 1) << 14, and the
      // partner index
      if (off < cb + kCap && off + nc > cb) {
        // old springs: this slot's start in the wave's spring region
        int idx = off, rank_base = LawTraits<LAW>::hist ? __float_as_int(a.W[b].w) : 0, c = 0;
#pragma unroll
        for (int w = 0; w < MW; ++w) {
          uint64_t cmw = w < n_words ? cm[w] : 0ull;
          const int first = idx;  // of this word's marked slots
          uint64_t live_old = 0ull;
          if constexpr (LawTraits<LAW>::hist)
            if (w < n_words) live_old = a.live[(int64_t)w * a.n + b];
#pragma unroll 1
          while (cmw) {
            const int sl = __ffsll((unsigned long long)cmw) - 1;
            cmw &= cmw - 1ull;
            if constexpr (NW > 1) idx = first + __popcll(all[w] & ((1ull << sl) - 1ull));
            int k = -1;
            if constexpr (LawTraits<LAW>::hist)
              if ((live_old >> sl) & 1ull) k = rank_base + __popcll(live_old & ((1ull << sl) - 1ull));
            if (idx >= cb && idx < cb + kCap) {
              pdesc[set][idx - cb] = lane | ((w * 64 + sl) << 6) | ((k + 1) << 14);
              // the LDS read is unconditional, so the two sources stay two
              // loads (not one flat load through a selected pointer)
              int jj = pstash[wv][min(c, kStash - 1)][lane];
              if (c >= kStash) jj = a.nl[(int64_t)(w * 64 + sl) * a.n + b];
              pjx[set][idx - cb] = jj;
            }
            ++idx;
            ++c;
          }
          if constexpr (NW > 1) idx = first + __popcll(all[w]);
          if constexpr (LawTraits<LAW>::hist) rank_base += __popcll(live_old);
        }
      }
      const int tc = min(total - cb, kCap);
      const int pl = NW == 1 ? lane : (int)threadIdx.x;  // place in the round
      for (int r0 = 0; r0 < tc; r0 += kRound) {
        sync();
        if (r0 + pl < tc) {
          const int dsc = pdesc[set][r0 + pl];
          const int32_t j = pjx[set][r0 + pl];
          const int64_t bo = b0 - lane + (dsc & 63);
          const int k = (dsc >> 14) - 1;
          // every load of the pair is issued before any is used
          const float4 po = a.P[bo], pj = a.P[j];
          float4 vo, vj, wo, wj, xo;
          if constexpr (LawTraits<LAW>::kin) {
            vo = a.V[bo];
            vj = a.V[j];
            wo = a.W[bo];
            wj = a.W[j];
          }
          if constexpr (LawTraits<LAW>::hist) xo = a.xi_rd[(b0 - lane) * a.M + (k >= 0 ? k : 0)];
          DomP dom_o;
          float dt_o;
          if (PM == 2) {
            const SegP& sp = a.segp[a.seg[bo]];
            dom_o = sp.dom;
            dt_o = sp.dt;
          } else {
            dom_o = dom;
            dt_o = dt;
          }
          Side<D> mo, o;
          mo.x = xyz<D>(po);
          mo.r = po.w;
          o.x = xyz<D>(pj);
          o.r = pj.w;
          mo.mat = 0;
          o.mat = 0;
          mo.sp = 0;
          o.sp = 0;
          if (a.law.n_mat > 1 || (LawTraits<LAW>::routed && a.law.n_species > 1)) {
            const int bo_bits = D == 2 ? __float_as_int(a.W[bo].z) : __float_as_int(a.I[bo].w);
            const int j_bits = D == 2 ? __float_as_int(a.W[j].z) : __float_as_int(a.I[j].w);
            mo.mat = (bo_bits >> 1) & kMatMask;
            o.mat = (j_bits >> 1) & kMatMask;
            mo.sp = (int)((unsigned)bo_bits >> 16);
            o.sp = (int)((unsigned)j_bits >> 16);
          }
          if constexpr (LawTraits<LAW>::kin) {
            mo.v = xyz<D>(vo);
            mo.m = vo.w;
            mo.w = ang4<D>(wo);
            o.v = xyz<D>(vj);
            o.m = vj.w;
            o.w = ang4<D>(wj);
          }
          Vec<D> xold = zero_vec<D>();
          if constexpr (LawTraits<LAW>::hist)
            if (k >= 0) xold = xyz<D>(xo);
          const Vec<D> rij = disp_pm<PM>(mo.x, o.x, dom_o);
          const float d_sq = dot(rij, rij);
          const PairOut<D> r = law_eval<D, LAW>(a.law, mo, o, rij, d_sq, xold, dt_o);
          pres[set][0][pl] = f4(r.F, r.contact ? 1.0f : 0.0f);
          if constexpr (LawTraits<LAW>::torque) pres[set][1][pl] = f4a(r.T);
          if constexpr (LawTraits<LAW>::hist) pres[set][2][pl] = f4(r.xi, 0.0f);
        }
        sync();
        const int q0 = cb + r0, q1 = NW > 1 && wv > 0 ? 0 : min(off + nc, q0 + kRound);
#pragma unroll 1
        for (int q = max(off, q0); q < q1; ++q) {
          const float4 fr = pres[set][0][q - q0];
          F = F + xyz<D>(fr);
          if constexpr (LawTraits<LAW>::torque) T = T + ang4<D>(pres[set][1][q - q0]);
          if constexpr (LawTraits<LAW>::hist) {
            if (fr.w != 0.0f) {
              const int sl = (pdesc[set][q - cb] >> 6) & 255;
              // new springs from the slot's marked-pair prefix: the wave's
              // springs fill one contiguous run of its region
              a.xi_wr[(b0 - lane) * a.M + off + rank_new] = pres[set][2][q - q0];
              ++rank_new;
              const uint64_t bit = 1ull << (sl & 63);
              const int ws = sl >> 6;
#pragma unroll
              for (int qq = 0; qq < MW; ++qq) ln[qq] |= ws == qq ? bit : 0ull;
            }
          }
        }
      }
      sync();  // the next chunk's descriptors overwrite these
    }
    if (NW > 1 && wv > 0) return;
    if constexpr (LawTraits<LAW>::hist)
      if (active)
#pragma unroll
        for (int w = 0; w < MW; ++w)
          if (w < n_words) {  // most words are unchanged from the last step: skip their stores
            const int64_t li = (int64_t)w * a.n + b;
            if (a.live[li] != ln[w]) a.live[li] = ln[w];
          }
  } else {
    if (NW > 1 && wv > 0) return;
    F = xyz<D>(a.F[b]);
    T = ang4<D>(a.T[b]);
  }
  if (!active) return;
  const float4 p4b = a.P[b], v4 = a.V[b], w4 = a.W[b];
  float4 i4;
  if constexpr (D == 2) {
    i4 = make_float4(w4.y, 0.0f, 0.0f, w4.z);
  } else if (a.iso && *a.iso) {
    const float Is = (0.4f * v4.w) * (p4b.w * p4b.w);
    i4 = make_float4(Is, Is, Is, __int_as_float(0));
  } else {
    i4 = a.I[b];
  }
  const int bits = __float_as_int(i4.w);
  Vec<D> x = xyz<D>(p4b), v = xyz<D>(v4);
  Ang<D> w = ang4<D>(w4);
  Quat q = q4(a.Q[b]);
  const Ang<D> I = ang4<D>(i4);
  const float m = v4.w;
  const bool fixed = (bits & 1) != 0;
  const float freef = fixed ? 0.0f : 1.0f;
  if (a.do_after) {
    if (a.has_fm) {
      const int64_t i = a.orig[b];
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
    }
    if (a.lin == JDEM_LIN_VERLET) {
      const float s = (dt * 0.5f) / m;
      v = v + (F * s) * freef;
    } else if (a.lin == JDEM_LIN_EULER) {
      const float s = dt / m;
      v = v + (F * s) * freef;
      x = x + v * dt;
    }
    if (a.rot == JDEM_ROT_VERLET_SPIRAL)
      vvs_after<D>(q, w, T, I, dt, freef);
    else if (a.rot == JDEM_ROT_SPIRAL)
      spiral_after<D>(q, w, T, I, dt, freef);
  }
  if (a.do_before) {
    if (dom.kind == JDEM_DOMAIN_REFLECT) reflect_apply<D>(dom, x, v, q, F, m, p4b.w, fixed, dt);
    if (a.lin == JDEM_LIN_VERLET) {
      const float s = (dt * 0.5f) / m;
      v = v + (F * s) * freef;
      x = x + v * dt;
    }
    if (a.rot == JDEM_ROT_VERLET_SPIRAL) vvs_before<D>(q, w, T, I, dt, freef);
  }
  float4 p_out = f4(x, p4b.w), v_out = f4(v, m);
  float4 w_out = f4a(w);
  if constexpr (D == 2) {  // build position, inertia and bits ride along
    p_out.z = p4b.z;
    v_out.z = v4.z;
    w_out.y = w4.y;
    w_out.z = w4.z;
  }
  a.P2[b] = p_out;
  a.V2[b] = v_out;
  // the springs' place travels with the angular velocity (its free lane)
  w_out.w = __int_as_float(spring_off >= 0 ? spring_off : __float_as_int(w4.w));
  a.W2[b] = w_out;
  a.Q[b] = f4q(q);
  if (a.store_ft) {
    a.F[b] = f4(F, 0.0f);
    a.T[b] = f4a(T);
  }
  if (a.do_before && a.check_disp) {
    Vec<D> xb;
    if constexpr (D == 2)
      xb = Vec<2>{p4b.z, v4.z};
    else
      xb = xyz<D>(a.old4[b]);
    const Vec<D> d = x - xb;
    if (dot(d, d) > trigger) {
      *a.flag_wr = a.step_idx + 1;
      if (PM == 2) a.seg_flag[a.seg[b]] = 1;
    }
  }
}

// Below this many spheres four waves share the rows of 64.  A step with one /
// four, us: spring-friction, bidisperse 17 / 9.6 at 10 k, 17.6 / 10.8 at 37 k,
// 18.5 / 13.3 at 70 k, 19.3 / 16.8 at 100 k, 24 / 26 at 200 k; log-normal radii
// 19 / 12, 21 / 14, 21 / 18, 24 / 27.  Rows of disks are short: 8 / 7 below
// 20 k, 8 / 8 at 37 k, 9.3 / 12.5 at 100 k, so one wave takes them all.  Batches
// of eight systems of unequal size: bidisperse 22 / 12 at 10 k, 21 / 14 at 37 k,
// 19 / 15 at 79 k; log-normal 30 / 15, 30 / 17, 32 / 26.
constexpr int64_t kWsSplit = 80000;

template <int D, int LAW, int MW>
void launch_ws_mw(const WS& a, bool per, hipStream_t s) {
  dim3 g(nblocks(a.n)), b(kBlock);
  if constexpr (D == 3) {
    if (a.n < kWsSplit) {
      const dim3 g4(nblocks(a.n, 64));
      if (a.segp)
        hipLaunchKernelGGL((k_ws_step<D, LAW, 2, MW, kBlock, 4>), g4, b, 0, s, a);
      else if (per)
        hipLaunchKernelGGL((k_ws_step<D, LAW, 1, MW, kBlock, 4>), g4, b, 0, s, a);
      else
        hipLaunchKernelGGL((k_ws_step<D, LAW, 0, MW, kBlock, 4>), g4, b, 0, s, a);
      return;
    }
  }
  if (a.segp && a.block == 128)
    hipLaunchKernelGGL((k_ws_step<D, LAW, 2, MW, 128>), dim3(nblocks(a.n, 128)), dim3(128), 0, s, a);
  else if (a.segp)
    hipLaunchKernelGGL((k_ws_step<D, LAW, 2, MW>), g, b, 0, s, a);
  else if (per)
    hipLaunchKernelGGL((k_ws_step<D, LAW, 1, MW>), g, b, 0, s, a);
  else
    hipLaunchKernelGGL((k_ws_step<D, LAW, 0, MW>), g, b, 0, s, a);
}
template <int D, int LAW>
hipError_t launch_ws_law(const WS& a, bool per, hipStream_t s) {
  const int words = max(a.W64, (a.M + 63) >> 6);
  if (words <= 1)
    launch_ws_mw<D, LAW, 1>(a, per, s);
  else
    launch_ws_mw<D, LAW, 4>(a, per, s);
  return hipGetLastError();
}

template <int D>
hipError_t launch_ws_dim(const WS& a, int law, bool per, hipStream_t s) {
  switch (law) {
    case JDEM_LAW_SPRING:
      return launch_ws_law<D, JDEM_LAW_SPRING>(a, per, s);
    case JDEM_LAW_HERTZ:
      return launch_ws_law<D, JDEM_LAW_HERTZ>(a, per, s);
    case JDEM_LAW_CUNDALL_STRACK:
      return launch_ws_law<D, JDEM_LAW_CUNDALL_STRACK>(a, per, s);
    case JDEM_LAW_SPRING_FRICTION:
      return launch_ws_law<D, JDEM_LAW_SPRING_FRICTION>(a, per, s);
    case JDEM_LAW_HERTZ_FRICTION:
      return launch_ws_law<D, JDEM_LAW_HERTZ_FRICTION>(a, per, s);
    case kLawRouted:
      return launch_ws_law<D, kLawRouted>(a, per, s);
    case kLawRoutedHist:
      return launch_ws_law<D, kLawRoutedHist>(a, per, s);
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t ws_launch_pack_springs(int64_t n, int M, int W64, const float4* rank, const uint64_t* live, float4* wave,
                                  float4* W, hipStream_t s) {
  if (n == 0 || M == 0) return hipSuccess;
  hipLaunchKernelGGL(k_pack_springs, dim3(nblocks(n)), dim3(kBlock), 0, s, n, M, W64, rank, live, wave, W);
  return hipGetLastError();
}
hipError_t ws_launch_unpack_springs(int64_t n, int M, int W64, const float4* wave, const uint64_t* live,
                                    const float4* W, float4* rank, hipStream_t s) {
  if (n == 0 || M == 0) return hipSuccess;
  hipLaunchKernelGGL(k_unpack_springs, dim3(nblocks(n)), dim3(kBlock), 0, s, n, M, W64, wave, live, W, rank);
  return hipGetLastError();
}

hipError_t ws_launch_step(const WS& a, int dim, int law, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  const bool per = a.dom.kind == JDEM_DOMAIN_PERIODIC;
  return dim == 3 ? launch_ws_dim<3>(a, law, per, s) : launch_ws_dim<2>(a, law, per, s);
}

}  // namespace jdem

// ---------------------------------------------------------------------------
// launch wrappers of the conversion and rebuild kernels
// ---------------------------------------------------------------------------
namespace jdem {

__global__ void __launch_bounds__(kBlock) k_inverse(const int32_t* __restrict__ orig, int64_t n,
                                                     int32_t* __restrict__ wpos) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b < n) wpos[orig[b]] = (int32_t)b;
}

// NaiveSimulator.create_neighbor_list in work space (descending original id;
// the work order is the original order when the secondary collider is naive)
template <int D, bool PER>
__global__ void __launch_bounds__(kBlock) k_nlist_work_naive(NLW a) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool active = b < a.n;  // every lane reaches end_row (wave-wide scan)
  int count = 0;
  if (active) {
    const Vec<D> xi = xyz<D>(a.P4[b]);
    const bool chk_bond = (!a.isb) && a.bond_w > 0;
    for (int64_t k = a.n - 1; k >= 0; --k) {
      if (k == b) continue;
      const Vec<D> d = disp_<PER>(xi, xyz<D>(a.P4[k]), a.dom);
      if (!(dot(d, d) <= a.cutoff_sq)) continue;
      if (chk_bond && bonded_o(a.bond_id, a.bond_w, a.orig[b], a.orig[k])) continue;
      if (count < a.M) a.nl[(int64_t)count * a.n + b] = (int32_t)k;
      ++count;
    }
  }
  end_row(a, b, active, count);
}

hipError_t ws_launch_in(const InOut& io, bool with_nl, hipStream_t s) {
  dim3 g(nblocks(io.n)), b(kBlock);
  hipLaunchKernelGGL(k_in_state, g, b, 0, s, io);
  if (with_nl) hipLaunchKernelGGL(k_in_nlist, g, b, 0, s, io);
  return hipGetLastError();
}
hipError_t ws_launch_out(const InOut& io, bool with_nl, hipStream_t s) {
  dim3 g(nblocks(io.n)), b(kBlock);
  hipLaunchKernelGGL(k_out_state, g, b, 0, s, io);
  if (with_nl) hipLaunchKernelGGL(k_out_nlist, g, b, 0, s, io);
  return hipGetLastError();
}
hipError_t ws_launch_export(const InOut& io, hipStream_t s) {
  if (io.n == 0) return hipSuccess;
  dim3 g(nblocks(io.n)), b(kBlock);
  if (io.old_user) hipLaunchKernelGGL(k_out_old, g, b, 0, s, io);
  if (io.nl_user && io.M > 0) hipLaunchKernelGGL(k_out_nlist, g, b, 0, s, io);
  return hipGetLastError();
}
hipError_t ws_launch_copy_rows(const int32_t* src, int32_t* dst, int64_t n, int M, hipStream_t s) {
  if (n == 0 || M == 0) return hipSuccess;
  hipLaunchKernelGGL(k_copy_rows, dim3(nblocks(n)), dim3(kBlock), 0, s, src, dst, n, M);
  return hipGetLastError();
}
hipError_t ws_launch_inverse(const int32_t* orig, int64_t n, int32_t* wpos, hipStream_t s) {
  hipLaunchKernelGGL(k_inverse, dim3(nblocks(n)), dim3(kBlock), 0, s, orig, n, wpos);
  return hipGetLastError();
}
hipError_t ws_launch_iota(int32_t* p, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_iota, dim3(nblocks(n)), dim3(kBlock), 0, s, p, n);
  return hipGetLastError();
}
hipError_t ws_launch_copy4(float4* d, const float4* src, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_copy_f4, dim3(nblocks(n)), dim3(kBlock), 0, s, d, src, n);
  return hipGetLastError();
}
hipError_t ws_launch_hash(const float4* P4, const int32_t* orig, int64_t n, int dim, const DomP& dom, const GridP& g,
                          uint32_t* keys, int32_t* wpos, hipStream_t s, const CellSort* cs) {
  dim3 gr(nblocks(n)), b(kBlock);
  const bool per = g.periodic != 0;
  int32_t *cnt = cs ? cs->cnt : nullptr, *arr = cs ? cs->arr : nullptr;
  if (dim == 3) {
    if (per)
      hipLaunchKernelGGL((k_hash_work<3, true>), gr, b, 0, s, P4, orig, n, dom, g, keys, wpos, cnt, arr);
    else
      hipLaunchKernelGGL((k_hash_work<3, false>), gr, b, 0, s, P4, orig, n, dom, g, keys, wpos, cnt, arr);
  } else {
    if (per)
      hipLaunchKernelGGL((k_hash_work<2, true>), gr, b, 0, s, P4, orig, n, dom, g, keys, wpos, cnt, arr);
    else
      hipLaunchKernelGGL((k_hash_work<2, false>), gr, b, 0, s, P4, orig, n, dom, g, keys, wpos, cnt, arr);
  }
  return hipGetLastError();
}
hipError_t ws_launch_seg_ids(const int64_t* offsets, int n_seg, int64_t n, int32_t* seg, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_seg_ids, dim3(nblocks(n)), dim3(kBlock), 0, s, offsets, n_seg, n, seg);
  return hipGetLastError();
}
hipError_t ws_launch_permute(int64_t n, const int32_t* new_orig, const int32_t* wpos, const float4* P,
                             const float4* V, const float4* W, const float4* Q, const float4* I, float4* P2,
                             float4* V2, float4* W2, float4* Q2, float4* I2, int32_t* orig2, int32_t* src,
                             int32_t* inv, hipStream_t s, float4* old2, int dim) {
  hipLaunchKernelGGL(k_permute, dim3(nblocks(n)), dim3(kBlock), 0, s, n, new_orig, wpos, P, V, W, Q, I, P2, V2, W2,
                     Q2, I2, orig2, src, inv, old2, dim);
  return hipGetLastError();
}
hipError_t ws_launch_rebuild_plan(const RB& r, const RBPlan& p, hipStream_t s) {
  hipLaunchKernelGGL(k_rebuild_plan, dim3(1), dim3(1024), 0, s, r, p);
  return hipGetLastError();
}
hipError_t ws_launch_rebuild_keys(const RB& r, hipStream_t s) {
  const dim3 g(std::min<unsigned>(nblocks(r.n), (unsigned)kCappedGrid));
  if (r.dim == 3)
    hipLaunchKernelGGL(k_rebuild_keys<3>, g, dim3(kBlock), 0, s, r);
  else
    hipLaunchKernelGGL(k_rebuild_keys<2>, g, dim3(kBlock), 0, s, r);
  return hipGetLastError();
}
hipError_t ws_launch_rebuild_gather(const RB& r, hipStream_t s) {
  hipLaunchKernelGGL(k_rebuild_gather, dim3(std::min<unsigned>(nblocks(r.n), (unsigned)kCappedGrid)), dim3(kBlock), 0,
                     s, r);
  return hipGetLastError();
}
template <int D>
void launch_rebuild_rows(const RB& r, hipStream_t s) {
  // as many workgroups as are resident at once
  const unsigned resident = 256u * 2048u / (64u * nlist_group<D>());
  const dim3 g(std::min<unsigned>(nblocks(r.n, 64), resident)), b(64 * nlist_group<D>());
  if (r.W64 <= 1)
    hipLaunchKernelGGL((k_rebuild_rows<D, 1>), g, b, 0, s, r);
  else
    hipLaunchKernelGGL((k_rebuild_rows<D, 4>), g, b, 0, s, r);
}
hipError_t ws_launch_rebuild_rows(const RB& r, hipStream_t s) {
  if (r.dim == 3)
    launch_rebuild_rows<3>(r, s);
  else
    launch_rebuild_rows<2>(r, s);
  return hipGetLastError();
}
hipError_t ws_launch_seg_init_flags(int n_seg, const int32_t* n_build, int32_t* seg_flag, hipStream_t s,
                                   int32_t* gate) {
  hipLaunchKernelGGL(k_seg_init_flags, dim3(nblocks(n_seg)), dim3(kBlock), 0, s, n_seg, n_build, seg_flag, gate);
  return hipGetLastError();
}
hipError_t ws_launch_cell_starts(const uint32_t* skeys, int64_t n, int64_t n_cells, int32_t* starts, hipStream_t s) {
  hipLaunchKernelGGL(k_cell_starts, dim3(nblocks(n_cells + 1, kStartsChunk)), dim3(kBlock), 0, s, skeys, n, n_cells, starts);
  return hipGetLastError();
}
// From this many particles on a list is built by one lane per particle, which
// takes fewer instructions but a longer chain.  A rebuild, group / lane, us:
// 3D bidisperse 43 / 86 at 10 k, 58 / 87 at 37 k, 84 / 91 at 100 k, 207 / 154
// at 400 k; log-normal radii 84 / 194, 138 / 211, 374 / 346; disks 43 / 56,
// 58 / 59, 106 / 90.
constexpr int64_t kNlistLane = 100000;

template <int MW>
void launch_nlist_group(const NLW& a, int dim, bool per, hipStream_t s) {
  const dim3 g(nblocks(a.n, 64)), b(64 * (dim == 3 ? nlist_group<3>() : nlist_group<2>()));
  if (dim == 3) {
    if (per)
      hipLaunchKernelGGL((k_nlist_group<3, true, MW>), g, b, 0, s, a);
    else
      hipLaunchKernelGGL((k_nlist_group<3, false, MW>), g, b, 0, s, a);
  } else {
    if (per)
      hipLaunchKernelGGL((k_nlist_group<2, true, MW>), g, b, 0, s, a);
    else
      hipLaunchKernelGGL((k_nlist_group<2, false, MW>), g, b, 0, s, a);
  }
}

hipError_t ws_launch_nlist(const NLW& a, int dim, bool naive, hipStream_t s) {
  dim3 g(nblocks(a.n)), b(kBlock);
  const bool per = naive ? a.dom.kind == JDEM_DOMAIN_PERIODIC : a.grid.periodic != 0;
  if (naive) {
    if (dim == 3) {
      if (per)
        hipLaunchKernelGGL((k_nlist_work_naive<3, true>), g, b, 0, s, a);
      else
        hipLaunchKernelGGL((k_nlist_work_naive<3, false>), g, b, 0, s, a);
    } else {
      if (per)
        hipLaunchKernelGGL((k_nlist_work_naive<2, true>), g, b, 0, s, a);
      else
        hipLaunchKernelGGL((k_nlist_work_naive<2, false>), g, b, 0, s, a);
    }
  } else if (a.n < kNlistLane) {
    if (a.W64 <= 1)
      launch_nlist_group<1>(a, dim, per, s);
    else
      launch_nlist_group<4>(a, dim, per, s);
  } else {
    if (dim == 3) {
      if (per)
        hipLaunchKernelGGL((k_nlist_work<3, true>), g, b, 0, s, a);
      else
        hipLaunchKernelGGL((k_nlist_work<3, false>), g, b, 0, s, a);
    } else {
      if (per)
        hipLaunchKernelGGL((k_nlist_work<2, true>), g, b, 0, s, a);
      else
        hipLaunchKernelGGL((k_nlist_work<2, false>), g, b, 0, s, a);
    }
  }
  return hipGetLastError();
}
// FreeDomain box of float4 positions (free.py:42-58)
__global__ void __launch_bounds__(kBlock) k_box_minmax4(const float4* __restrict__ P, int64_t n,
                                                         float* __restrict__ part) {
  __shared__ float smin[3][kBlock], smax[3][kBlock];
  const int tid = threadIdx.x;
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + tid; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float4 p = P[i];
    const float x[3] = {p.x, p.y, p.z};
    for (int a = 0; a < 3; ++a) {
      lo[a] = fminf(lo[a], x[a] - p.w);
      hi[a] = fmaxf(hi[a], x[a] + p.w);
    }
  }
  for (int a = 0; a < 3; ++a) {
    smin[a][tid] = lo[a];
    smax[a][tid] = hi[a];
  }
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if (tid < off)
      for (int a = 0; a < 3; ++a) {
        smin[a][tid] = fminf(smin[a][tid], smin[a][tid + off]);
        smax[a][tid] = fmaxf(smax[a][tid], smax[a][tid + off]);
      }
    __syncthreads();
  }
  if (tid == 0)
    for (int a = 0; a < 3; ++a) {
      part[6 * blockIdx.x + a] = smin[a][0];
      part[6 * blockIdx.x + 3 + a] = smax[a][0];
    }
}
hipError_t ws_launch_box(const float4* P, int64_t n, float* part, int nparts, hipStream_t s) {
  hipLaunchKernelGGL(k_box_minmax4, dim3(nparts), dim3(kBlock), 0, s, P, n, part);
  return hipGetLastError();
}

}  // namespace jdem
