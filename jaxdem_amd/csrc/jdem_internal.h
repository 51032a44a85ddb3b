// jdem_internal.h -- context, scratch arena and kernel-argument structs shared
// by the translation units of libjdem_hip.so.  Not part of the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <string>
#include <vector>

#include "jdem.h"
#include "jdem_device.h"

namespace jdem {

constexpr int kBlock = 256;
// Workgroups of a launch whose size is known only on the device (gated
// batch rebuilds): its kernels walk the work in turn, so an idle launch
// dispatches this many workgroups instead of one per tile.
constexpr int kCappedGrid = 2048;

// Grid parameters on the device (jdem_grid; jdem_grid_f64 for double).
template <class Real = float>
struct GridPT {
  int dims[3];
  int strides[3];
  Real cell[3];
  int sr;
  int periodic;
  int64_t n_cells;
};
using GridP = GridPT<float>;

// Four scalars of one cell-sorted particle, (x, y, z, r).
struct alignas(16) Double4 {
  double x, y, z, w;
};
template <class Real>
struct Real4Of {
  using T = float4;
};
template <>
struct Real4Of<double> {
  using T = Double4;
};
template <class Real>
using Real4 = typename Real4Of<Real>::T;

// One grow-only device allocation of the context.
struct Buf {
  void* p = nullptr;
  size_t bytes = 0;
};

}  // namespace jdem

struct jdem_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  // scratch, grown on demand and reused across calls
  jdem::Buf pos2, vel2, ang2;          // ping-pong kinematics
  jdem::Buf keys[2], vals[2], hist;    // radix sort
  jdem::Buf cscnt;                     // counting sort: per-cell counts, left clear by every finished sort
  bool cscnt_clear = false;
  jdem::Buf cstart, cend, spos;        // cell tables, sorted (x, r)
  jdem::Buf nl_new, xi_new, live_new;  // neighbour-list rebuild
  jdem::Buf flags;                     // small device words
  jdem::Buf red;                       // reduction partials
  jdem::Buf nl_copy, xi_copy, live_copy;
  // resident NeighborList working set (jdem_resident.hip)
  jdem::Buf wP[2], wV[2], wW[2], wQ[2], wI[2], wF, wT, wOld, wOrig[2], wWpos, wSrc, wInv, wKeys, fireV, fireDev, segp, segid, segflag, wNl[2], wXi[2], wLive[2], wXiRank;
  int32_t* host_flags = nullptr;       // pinned host mirror of flags
  // HIP-event timing (jdem_ctx_set_timing)
  struct TimedSpan {
    hipEvent_t start, stop;
    int kind;  // 0 step kernel, 1 idle step kernel, 2 rebuild
    int64_t step;
  };
  bool timing = false;
  std::vector<hipEvent_t> event_pool;
  std::vector<TimedSpan> spans;
  // Device buffers not in use: released working sets (jdem_resident) and
  // buffers handed over to them leave empty scratch slots that ensure()
  // refills from here before it allocates.
  std::vector<jdem::Buf> pool;
  std::mutex pool_mu;
  // private stream on which captured step graphs are replayed (default priority)
  hipStream_t gstream = nullptr;
  hipEvent_t gevent[2] = {nullptr, nullptr};
  // device copy of the last routed law's terms and species offsets, and the
  // host bytes it was made from
  jdem::Buf route;
  std::vector<char> route_host;
  // clumps: members per clump (CSR), lab positions, levers, member totals
  jdem::Buf cl_start, cl_members, plab, ppr, ftot, ttot, crefl;
  // the precision form's Verlet list
  jdem::Buf pvl;
  // every scratch buffer of the context, for accounting and release
  std::vector<jdem::Buf*> bufs();
  size_t scratch_bytes();
};

// The NeighborList working set kept between calls (include/jdem.h): the
// work order and the buffers of the step kernel's layouts, in work order.
struct jdem_resident {
  jdem_ctx* ctx = nullptr;
  int64_t n = 0;
  int M = 0;
  int W64 = 1;
  int dim = 3;
  bool hist = false;
  jdem::Buf orig;  // int32 (N): original index of work slot b
  jdem::Buf old4;  // float4 (N): positions at the last build
  jdem::Buf nl;    // int32 slot-major (M, N): rows end at their first -1
  jdem::Buf live;  // uint64 (W64, N): slots that carry a spring
  jdem::Buf xi;    // float4 by rank (M, N): k-th live spring of slot b
};

namespace jdem {

// Kernel-side parameters of the ABI's domain and grid structs.
DomP dom_of(const jdem_domain& d);
GridP grid_of(const jdem_grid& g);
DomPT<double> dom_of(const jdem_domain_f64& d);
GridPT<double> grid_of(const jdem_grid_f64& g);

// Ensure b holds at least `bytes`; returns false on allocation failure.
// An empty b is first refilled from the context's pool.
bool ensure(jdem_ctx* ctx, Buf& b, size_t bytes);
// Give b's memory to the context's pool and leave b empty.
void pool_give(jdem_ctx* ctx, Buf& b);
// Free every pooled buffer (after the stream has drained).
void pool_trim(jdem_ctx* ctx);

// Kernel arguments of the fused step / force / energy kernels.
template <class Real = float>
struct StepArgsT {
  int64_t n;
  int bond_w;
  int isb;
  const Real* pos_in;
  const Real* vel_in;
  const Real* ang_in;
  Real* pos_out;
  Real* vel_out;
  Real* ang_out;
  Real* q;
  Real* force;
  Real* torque;
  const Real* rad;
  const Real* mass;
  const Real* inertia;
  const int32_t* mat_id;
  const int32_t* bond_id;
  const uint8_t* fixed;
  const Real* ext_f;
  const Real* ext_fc;
  const Real* ext_t;
  Real g[3];
  int has_fm;
  LawPT<Real> law;
  DomPT<Real> dom;
  Real dt;
  int lin;
  int rot;
  // cell-list source: cells numbered with the last axis fastest, so a stencil
  // column is one run of cstart (n_cells + 1 entries); sorted (x, r)
  const int32_t* perm;
  const int32_t* skeys;
  const int32_t* cstart;
  const Real4<Real>* spos;
  GridPT<Real> grid;
  // particles of one wavefront of a cell-list or naive traversal (a multiple
  // of the particles it walks at once, at most 64)
  int pw;
  // neighbour-list source
  const int32_t* nl;
  int M;
  Real* hist_xi;
  uint32_t* hist_live;
  int W32;
  // phases
  int do_force;
  int force_zero;  // collider "": contact force and torque are zero
  int do_after;
  int do_before;
  int write_kin;
  // neighbour-list displacement check (neighbor_list.py:78-85)
  const Real* old_pos;
  Real trigger;
  int check_disp;
  const int32_t* flag_rd;
  int32_t* flag_wr;
  int32_t step_idx;
  // energy / virial outputs (per particle, float64)
  double* e_out;
  // clumps (null for spheres): ids (the pair mask), R(q) pos_p per member
  // (the torque lever), the members of each clump (CSR: cl_start (N + 1),
  // cl_members (N) in ascending index), body offsets, and the per-member
  // force / torque totals of ForceManager before the clump sum
  const int32_t* clump;
  Real* ppr;
  const int32_t* cl_start;
  const int32_t* cl_members;
  const Real* pos_p;
  Real* plab;
  Real* ftot;
  Real* ttot;
  Real* rscr;  // reflective domain with clumps: per-member scratch (kReflW words)
};
using StepArgs = StepArgsT<float>;
// The float64 form of the plain step (jdem_system_step_f64 and friends).
using StepArgs64 = StepArgsT<double>;
using DomP64 = DomPT<double>;
using GridP64 = GridPT<double>;
using LawP64 = LawPT<double>;

// SRC_CELLS_LANE: the cell list walked by one lane per particle, chosen by
// launch_step for large systems
enum Src { SRC_NAIVE = 1, SRC_CELLS = 2, SRC_NLIST = 3, SRC_CELLS_LANE = 4 };

// launchers (jdem_step.hip)
hipError_t launch_step(const StepArgs& a, int dim, int law, int src, hipStream_t s);
hipError_t launch_energy(const StepArgs& a, int dim, int law, int src, hipStream_t s);
hipError_t launch_virial(const StepArgs& a, int dim, int law, int src, hipStream_t s);
// float64 instances: every collider source, laws without history
hipError_t launch_step(const StepArgs64& a, int dim, int law, int src, hipStream_t s);
hipError_t launch_energy(const StepArgs64& a, int dim, int law, int src, hipStream_t s);
hipError_t launch_kinetic(const StepArgs64& a, int dim, hipStream_t s);
// clumps: lab positions and levers; ForceManager totals; the sum over each
// clump broadcast to its members (both scalar types)
hipError_t launch_clump_lab(const StepArgs& a, int dim, hipStream_t s);
hipError_t launch_clump_lab(const StepArgs64& a, int dim, hipStream_t s);
hipError_t launch_clump_forces(const StepArgs& a, int dim, hipStream_t s);
hipError_t launch_clump_forces(const StepArgs64& a, int dim, hipStream_t s);
// ReflectDomain.apply for clumps (four launches; scratch a.rscr of
// refl_scratch_words(dim) words per member)
hipError_t launch_clump_reflect(const StepArgs& a, int dim, hipStream_t s);
hipError_t launch_clump_reflect(const StepArgs64& a, int dim, hipStream_t s);
inline int refl_scratch_words(int dim) { return 8 * dim + 2 + (dim == 3 ? 3 : 1); }

// launchers (jdem_cells.hip)
// Buffers of one counting sort by cell: per-cell counts, each element's
// arrival number in its cell, (key, id) by arrival, scan totals; sorted keys
// and ids.
struct CellSort {
  int32_t* cnt;
  int32_t* arr;
  uint2* pairs;
  uint32_t* sums;
  uint32_t* sk;
  int32_t* perm;
};
// With cs, the key kernel is the sort's count pass too.
hipError_t launch_hash(const float* pos, int64_t n, int dim, const DomP& dom, const GridP& g, uint32_t* keys,
                       hipStream_t s, const CellSort* cs = nullptr);
hipError_t launch_hash(const double* pos, int64_t n, int dim, const DomP64& dom, const GridP64& g, uint32_t* keys,
                       hipStream_t s, const CellSort* cs = nullptr);
// Buffers of a sort: key and value ping-pong arrays of n entries (the
// counting sort takes k0 and v0 as one array of 2 n words at k0), a histogram
// / scan-sum array and (counting sort) per-cell counts.
struct SortBufs {
  uint32_t* k0;
  uint32_t* k1;
  int32_t* v0;
  int32_t* v1;
  uint32_t* hist;
  int32_t* cur;
};
// uint32 words of SortBufs::hist that a radix sort of n keys uses
size_t radix_hist_words(int64_t n);
// uint32 words of SortBufs::hist that a counting sort over n_cells uses
size_t cell_sort_sum_words(int64_t n_cells);
// The sorts below on caller-given buffers (no allocation).
hipError_t radix_sort_bufs(const SortBufs& sb, const uint32_t* keys_in, int64_t n, int nbits, uint32_t** keys_out,
                           int32_t** vals_out, hipStream_t s);
hipError_t cell_sort_bufs(const SortBufs& sb, const uint32_t* keys_in, int64_t n, int64_t n_cells, uint32_t** keys_out,
                          int32_t** vals_out, int32_t* starts, hipStream_t s);
// Sort (keys, iota) by key; results in (keys_out, vals_out).  nbits = key bits.
hipError_t radix_sort_pairs(jdem_ctx* ctx, const uint32_t* keys_in, int64_t n, int nbits, uint32_t** keys_out,
                            int32_t** vals_out, hipStream_t s);
// The same result as radix_sort_pairs for keys < n_cells, by counting:
// per-cell counts, their exclusive scan (written to starts[0..n_cells],
// starts[n_cells] = n), placement by arrival number, then each element's rank
// among its cell's ids.  Cost grows with n + n_cells.
// cell_sort_begin hands out the buffers (counts clear); a kernel of the caller
// then writes each key, adds 1 to its cell's count and keeps the value the
// atomic returned; cell_sort_end runs the remaining passes on those keys (and,
// with spos, gathers the sorted (x, r)).
hipError_t cell_sort_begin(jdem_ctx* ctx, int64_t n, int64_t n_cells, CellSort* cs, hipStream_t s);
// cell_sort_starts only scans the counts into starts: the caller places its
// elements itself.  Its kernels return at once while *gate == 0 (a device word),
// leaving the previous starts in place.
hipError_t cell_sort_starts(jdem_ctx* ctx, const CellSort& cs, int64_t n_cells, int32_t* starts, hipStream_t s,
                            const int32_t* gate);
hipError_t cell_sort_end(jdem_ctx* ctx, const CellSort& cs, const uint32_t* keys, int64_t n, int64_t n_cells,
                         int32_t* starts, hipStream_t s);
hipError_t cell_sort_end(jdem_ctx* ctx, const CellSort& cs, const uint32_t* keys, int64_t n, int64_t n_cells,
                         int32_t* starts, const float* pos, const float* rad, int dim, float4* spos, hipStream_t s);
hipError_t cell_sort_end(jdem_ctx* ctx, const CellSort& cs, const uint32_t* keys, int64_t n, int64_t n_cells,
                         int32_t* starts, const double* pos, const double* rad, int dim, Double4* spos,
                         hipStream_t s);
hipError_t cell_sort_pairs(jdem_ctx* ctx, const uint32_t* keys_in, int64_t n, int64_t n_cells, uint32_t** keys_out,
                           int32_t** vals_out, int32_t* starts, hipStream_t s);
// The counting sort of a batch rebuild, between cell_sort_begin and the
// caller's rank pass: the first *n_dev of the keys (n bounds it), every key
// below *c_dev (n_cells bounds it), starts of *c_dev + 1 entries, (key, id) at
// their cells in cs.pairs.  The launches are sized by the bounds and capped
// (kCappedGrid workgroups that walk the work in turn), so a rebuild of a few
// systems of a large batch costs what its particles and cells need.
hipError_t cell_sort_dev(const CellSort& cs, const uint32_t* keys, int64_t n, int64_t n_cells, const int64_t* n_dev,
                         const int64_t* c_dev, int32_t* starts, hipStream_t s, const int32_t* gate);
// cend[c] = starts[c + 1] for c < n_cells
hipError_t launch_starts_to_ends(const int32_t* starts, int64_t n_cells, int32_t* cend, hipStream_t s);
// key bits of a grid of n_cells cells (at least 1)
inline int nbits_for_cells(int64_t n_cells) {
  int64_t m = n_cells > 1 ? n_cells - 1 : 1;
  int b = 0;
  while (m > 0) {
    ++b;
    m >>= 1;
  }
  return b;
}
// Device address of the fixed scratch array of jdem_cell_build_noalloc,
// looked up once per device (jdem_noalloc.hip).
int noalloc_init(int device);
// whether cell_sort_pairs is the cheaper sort for n keys below n_cells
inline bool use_cell_sort(int64_t n, int64_t n_cells) { return n > 0 && n_cells <= 4 * n + 65536; }
// The same question where memory may be allocated: a cell costs 16 bytes of
// traffic against 4 with the radix sort, whose launches are two to five per
// eight key bits, so the counting sort stays ahead on grids far sparser than the
// particles (10^6 disks on 27 10^6 cells, five steps: 0.95 ms, 2.2 with the
// radix sort and the cell ranges).
inline bool use_cell_sort_sparse(int64_t n, int64_t n_cells) { return n > 0 && n_cells <= 32 * n + (1 << 20); }
hipError_t launch_fill_i32(int32_t* p, int64_t n, int32_t v, hipStream_t s);
hipError_t launch_cell_ranges(const uint32_t* skeys, int64_t n, int32_t* cstart, int32_t* cend, hipStream_t s);
hipError_t launch_gather_spos(const int32_t* perm, const float* pos, const float* rad, int64_t n, int dim,
                              float4* spos, hipStream_t s);
hipError_t launch_gather_spos(const int32_t* perm, const double* pos, const double* rad, int64_t n, int dim,
                              Double4* spos, hipStream_t s);
template <class Real = float>
struct NLBuildT {
  int64_t n;
  int dim;
  int M;
  Real cutoff_sq;
  int isb;
  int bond_w;
  const int32_t* bond_id;
  const Real* pos;
  const int32_t* perm;
  const int32_t* skeys;
  const int32_t* cstart;
  const int32_t* cend;
  const float4* spos;  // float only: sorted (x, r)
  GridPT<Real> grid;
  DomPT<Real> dom;
  int32_t* nl;
  int32_t* overflow;
  const int32_t* clump;  // clump ids (pairs of one clump are not listed), or null
};
using NLBuild = NLBuildT<float>;
hipError_t launch_nlist_cells(const NLBuild& b, hipStream_t s);
hipError_t launch_nlist_naive(const NLBuild& b, hipStream_t s);
hipError_t launch_nlist_cells(const NLBuildT<double>& b, hipStream_t s);
hipError_t launch_nlist_naive(const NLBuildT<double>& b, hipStream_t s);
hipError_t launch_remap_hist(int64_t n, int M, int W32, int dim, const int32_t* old_nl, const uint32_t* old_live,
                             const float* old_xi, const int32_t* new_nl, uint32_t* new_live, float* new_xi,
                             hipStream_t s);
// pos_p (clumps, or null): the bounding radius is |pos_p| + rad
hipError_t launch_box_minmax(const float* pos, const float* rad, int64_t n, int dim, float* part, int nparts,
                             hipStream_t s, const float* pos_p = nullptr);
hipError_t launch_box_minmax(const double* pos, const double* rad, int64_t n, int dim, double* part, int nparts,
                             hipStream_t s, const double* pos_p = nullptr);
hipError_t launch_sum_f64(const double* in, int64_t n, int stride, int ncomp, double* partial, double* out,
                          int nparts, hipStream_t s);
hipError_t launch_kinetic(const StepArgs& a, int dim, hipStream_t s);
hipError_t launch_stage(const StepArgs& a, int dim, int stage, hipStream_t s);
hipError_t launch_copy_f32(float* dst, const float* src, int64_t n, hipStream_t s);


// ---- resident NeighborList engine (jdem_resident.hip) ----------------------
struct InOut {
  int64_t n;
  int dim;
  int M;
  int W64;  // live words per particle
  // caller arrays (original order)
  float* pos;
  float* vel;
  float* ang;
  float* q;
  float* force;
  float* torque;
  const float* rad;
  const float* mass;
  const float* inertia;
  const int32_t* mat_id;
  const int32_t* species;  // routed laws with species, else null
  const uint8_t* fixed;
  int32_t* nl_user;      // (N, M)
  float* old_user;       // (N, D)
  float* xi_user;        // (N, M, D) or null
  uint32_t* live_user;   // (N, ceil(M/32)) or null
  // work arrays
  const int32_t* orig;  // work -> original
  const int32_t* wpos;  // original -> work
  float4* P4;
  float4* V4;
  float4* W4;
  float4* Q4;
  float4* I4;
  float4* F4;
  float4* T4;
  float4* old4;
  int32_t* nl;
  float4* xi;
  uint64_t* live;
  int old_keep;  // entry: old4 already holds the build positions
  // entry: cleared when some sphere is fixed or its inertia differs from
  // (0.4 m) r^2 in any component (3D; set to 1 before the entry)
  int32_t* iso_flag;
};

// Parameters of one system of a segmented batch (jdem_batch_step).  The
// systems' particles occupy consecutive ranges of the work set in both the
// caller's order and the cell order, because each system owns a consecutive
// range of work cell keys starting at cell_base.
struct SegP {
  DomP dom;
  GridP grid;
  uint32_t cell_base;
  float dt;
  float cutoff_sq;  // (cutoff + skin)^2 of the list build
  float trigger;    // rebuild threshold on |x - x_build|^2
};

struct NLW {
  int64_t n;
  int M;
  float cutoff_sq;
  int isb;
  int bond_w;
  const int32_t* bond_id;  // original indexing
  const int32_t* orig;
  const float4* P4;
  const uint32_t* skeys;  // sorted keys = cell of work slot
  const int32_t* starts;  // (n_cells + 1) first slot of each cell
  GridP grid;
  DomP dom;
  int32_t* nl;
  int32_t* overflow;
  // history carried over from the previous list (null live: no history)
  int W64;
  int remap;                // 0: start with empty history, 1: remap old
  const int32_t* src;       // new work slot -> old work slot
  const int32_t* inv;       // old work slot -> new work slot
  const int32_t* old_nl;
  const float4* old_xi;
  // old and new springs are kept per wavefront (the step kernel's layout), the
  // start of a slot's in old_W[.].w and new_W[.].w
  const float4* old_W;
  float4* new_W;
  const uint64_t* old_live;
  float4* xi;
  uint64_t* live;
};
enum { SEG_KEEP = 0, SEG_FRESH = 1, SEG_REMAP = 2 };

// In-place rebuild of the flagged systems of a batch (jdem_resident.hip).
// Flagged particles have a compact index (system s: [cpref[s], cpref[s + 1]),
// in original order before the sort and in the new slots' order after it),
// their cells a compact key from ccref[s]; wpref counts the wavefronts of
// slots that hold a flagged system.
struct RB {
  int64_t n;
  int n_seg;
  int dim;
  const int32_t* go;  // every kernel but the first returns at once while *go == 0
  int M, W64;
  const int32_t* seg;  // system of each work slot
  const SegP* segp;
  const int64_t* offsets;
  // the plan of this rebuild
  int32_t *seg_mode;  // SEG_KEEP / SEG_FRESH / SEG_REMAP of each system
  int64_t *cpref, *ccref, *wpref;
  // work set (updated in place)
  float4 *P, *V, *W, *Q, *I, *old4;
  int32_t* orig;
  int32_t* nl;
  uint64_t* live;  // null: no history
  float4* xi;      // per wavefront
  float4* keep_xi; // by rank, of the kept systems' slots in a rebuilt wavefront
  // counting sort
  uint32_t* keys_c;
  int32_t* slot_c;  // slot of compact index i before the sort
  int32_t *cnt, *arr;
  const uint2* pairs;
  int32_t* starts;
  // staging, compact index of the new slot
  uint32_t* sk;
  float4 *tP, *tV, *tW, *tQ, *tI;
  int32_t* torig;
  int32_t* tlive;  // live springs, each with its partner's old slot, by rank (stride n)
  int32_t* tnl;
  float4* txi;
  int32_t* inv;  // old slot -> new slot
  int isb;
  int bond_w;
  const int32_t* bond_id;
  int32_t* overflow;
};
// what the first kernel of the chain works on
struct RBPlan {
  int32_t *gate, *go, *overflow, *events, *seg_flag, *n_build;
};
hipError_t ws_launch_rebuild_plan(const RB& r, const RBPlan& p, hipStream_t s);
hipError_t ws_launch_rebuild_keys(const RB& r, hipStream_t s);
hipError_t ws_launch_rebuild_gather(const RB& r, hipStream_t s);
hipError_t ws_launch_rebuild_rows(const RB& r, hipStream_t s);

// Workgroups are dispatched round-robin over the 8 XCDs of the chip, each
// with its own L2: workgroup w runs on XCD w % 8.  xcd_tile maps them so
// that XCD x processes one contiguous run of tiles; in the cell-sorted work
// order, spatial neighbours are then mostly served by the same L2.
__device__ inline unsigned xcd_tile(unsigned w, unsigned nw) {
  const unsigned q = nw / 8u, r = nw % 8u, x = w % 8u, l = w / 8u;
  return (x < r ? x * (q + 1u) : r * (q + 1u) + (x - r) * q) + l;
}

// Cells of the stencil along one axis, in stencil order: the offsets
// -sr..hi (hi = min(sr, dims - sr - 1) on a periodic axis, which drops the
// offsets that would revisit a cell) give at most two runs of consecutive
// cells, [r0a, r0b] then [r1a, r1b] (empty when a > b).
JD void stencil_runs(bool per, int c, int sr, int dims, int& r0a, int& r0b, int& r1a, int& r1b) {
  if (per) {
    const int cnt = sr + min(sr, dims - sr - 1) + 1;  // in [1, dims]
    int start = (c - sr) % dims;
    if (start < 0) start += dims;
    const int last = start + cnt - 1;
    r0a = start;
    r0b = min(last, dims - 1);
    r1a = 0;
    r1b = last - dims;
  } else {
    r0a = max(c - sr, 0);
    r0b = min(c + sr, dims - 1);
    r1a = 0;
    r1b = -1;
  }
}

// Offsets along a slow axis; returns the cell or -1 when it is off the grid.
JD int stencil_cell(bool per, int c, int o, int dims) {
  int x = c + o;
  if (per) {
    x %= dims;
    if (x < 0) x += dims;
    return x;
  }
  return (x < 0 || x >= dims) ? -1 : x;
}

// orders the LDS traffic of one wave around an exchange between its lanes
JD void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct WS {
  int64_t n;
  int M;
  int W64;
  // 3D: device word, nonzero when every sphere is free with inertia (0.4 m) r^2
  // in each component and one material: the kernel computes the inertia
  // record instead of reading it
  const int32_t* iso;
  LawP law;
  DomP dom;
  float dt;
  int lin, rot;
  float g[3];
  int has_fm;
  const float* ext_f;   // original order
  const float* ext_fc;
  const float* ext_t;
  const int32_t* orig;
  const float4* P;
  const float4* V;
  const float4* W;
  float4* P2;
  float4* V2;
  float4* W2;
  float4* Q;
  const float4* I;
  float4* F;
  float4* T;
  const float4* old4;
  const int32_t* nl;
  const float4* xi_rd;  // springs by rank, read
  float4* xi_wr;        // springs by rank, written (another buffer)
  uint64_t* live;
  int do_force, do_after, do_before, store_ft;
  float trigger;
  int check_disp;
  const int32_t* flag_rd;
  int32_t* flag_wr;
  int32_t step_idx;
  // segmented batch (null for one system); seg_flag[s] = 1 when system s
  // needs a rebuild
  const int32_t* seg;
  const SegP* segp;
  int32_t* seg_flag;
  int block;  // workgroup size of a batch's step kernel (256 or 128)
};

hipError_t ws_launch_in(const InOut& io, bool with_nl, hipStream_t s);
hipError_t ws_launch_out(const InOut& io, bool with_nl, hipStream_t s);
// A working set's list, build positions and springs in the caller's layouts
// (io.nl_user / old_user / xi_user / live_user; each may be null).
hipError_t ws_launch_export(const InOut& io, hipStream_t s);
// dst[s*n + b] = src[s*n + b] for the slots of row b up to its first -1
hipError_t ws_launch_copy_rows(const int32_t* src, int32_t* dst, int64_t n, int M, hipStream_t s);
// Tangential springs of the step kernel, per wavefront: the 64 work slots
// of wave w own the region [64 w M, 64 (w + 1) M) of the spring buffer, and
// slot b's springs (in slot order of its live bits) start at offset W[b].w
// (an int in the float bits) of that region.  The entry and the exit keep
// springs by rank instead ([k N + b], k-th live slot).
// pack: by rank -> per wave (offsets = prefix of the live counts);
// unpack: per wave -> by rank.
hipError_t ws_launch_pack_springs(int64_t n, int M, int W64, const float4* rank, const uint64_t* live, float4* wave,
                                  float4* W, hipStream_t s);
hipError_t ws_launch_unpack_springs(int64_t n, int M, int W64, const float4* wave, const uint64_t* live,
                                    const float4* W, float4* rank, hipStream_t s);
hipError_t ws_launch_inverse(const int32_t* orig, int64_t n, int32_t* wpos, hipStream_t s);
hipError_t ws_launch_iota(int32_t* p, int64_t n, hipStream_t s);
hipError_t ws_launch_copy4(float4* d, const float4* src, int64_t n, hipStream_t s);
hipError_t ws_launch_hash(const float4* P4, const int32_t* orig, int64_t n, int dim, const DomP& dom, const GridP& g,
                          uint32_t* keys, int32_t* wpos, hipStream_t s, const CellSort* cs = nullptr);
// seg[b] = system of particle b for the ranges offsets[0..n_seg]
hipError_t ws_launch_seg_ids(const int64_t* offsets, int n_seg, int64_t n, int32_t* seg, hipStream_t s);
hipError_t ws_launch_permute(int64_t n, const int32_t* new_orig, const int32_t* wpos, const float4* P,
                             const float4* V, const float4* W, const float4* Q, const float4* I, float4* P2,
                             float4* V2, float4* W2, float4* Q2, float4* I2, int32_t* orig2, int32_t* src,
                             int32_t* inv, hipStream_t s, float4* old2 = nullptr, int dim = 3);
// batch rebuilds, at the start of a call: the flags of never-built systems
// (and *gate, when one is set)
hipError_t ws_launch_seg_init_flags(int n_seg, const int32_t* n_build, int32_t* seg_flag, hipStream_t s,
                                   int32_t* gate = nullptr);
hipError_t ws_launch_cell_starts(const uint32_t* skeys, int64_t n, int64_t n_cells, int32_t* starts, hipStream_t s);
hipError_t ws_launch_nlist(const NLW& a, int dim, bool naive, hipStream_t s);
hipError_t ws_launch_step(const WS& a, int dim, int law, hipStream_t s);
hipError_t ws_launch_box(const float4* P, int64_t n, float* part, int nparts, hipStream_t s);

// ---- FIRE minimiser (jdem_fire.hip) -----------------------------------------
struct FireP {
  float dt0, alpha_init, f_inc, f_dec, f_alpha;
  float dt_max, dt_min;  // dt0 * dt_{max,min}_scale, rounded once to float
  int n_min, n_bad_max;
};
// Optimiser scalars, kept on the device between the kernels of an iteration.
struct FireDev {
  float dt, alpha;
  int n_good, n_bad;
  float new_dt, new_alpha, dt_rev, vs;
  double power;
  float dt_used;  // dt of the update just decided (dt is the next one's)
};
// Where a FIRE loop decided on the device stands, and its tests (routines.py:
// 284-314).
struct FireStop {
  double pe, prev, gmax;
  long long steps;
  int32_t stop;
};
struct FireStopP {
  double pe_tol, pe_diff_tol, force_tol, dN;
  long long max_steps;
};
struct FireArgs {
  int64_t n;
  int dim;
  FireP p;
  FireDev* st;
  FireStop* ls;
  int32_t* stop_word;  // set with ls->stop (null: none)
  FireStopP stop;
  float* force;
  const float* torque;
  const uint8_t* fixed;
  float* vel_pos;
  float* vel_rot;
  float* pos;
  float* q;
  const double* e_in;  // pair energy of each particle (null: none)
  double* part;        // block partials: power and energy, largest gradient component
  unsigned* gpart;
  int nparts;
  float g[3];
  const float* mass;
};
// The same of the precision form, which also tests for a stall.
struct PrecStop {
  double pe, prev, best_g, best_e, gmax;
  long long best_at, steps;
  int32_t stop;
  int32_t first;
};
struct PrecStopP {
  double pe_tol, pe_diff_tol, force_tol, dN;
  long long max_steps, stall_steps;
};
hipError_t launch_fire_terms(const FireArgs& a, hipStream_t s);
hipError_t launch_fire_decide(const FireArgs& a, hipStream_t s);
hipError_t launch_fire_move(const FireArgs& a, hipStream_t s);

// ---- precision form: integer cell + float32 offset (jdem_fire.hip) ----------
struct PrecArgs {
  int64_t n;
  int dim;
  int dims[3];   // cells per axis (periodic)
  float h[3];    // cell edges: h + hlo as an unevaluated float pair
  float hlo[3];
  // caller's arrays, by sphere
  int32_t* cidx; // (N, D) cell of each sphere
  float* off;    // (N, D) position inside the cell, [0, h)
  const float* rad;
  float* force;  // (N, D)
  float k;
  // state by cell-sorted slot; S, V, C swap at a re-sort (word *cur)
  float4* S[2];  // offset, radius
  float4* V[2];  // FIRE velocity
  int4* C[2];    // cell, sphere id
  float4* F;
  float4* B;     // list mode: offsets at the build
  int32_t* cur;
  int32_t* moved;        // a re-sort is due (or, until the next decision, done)
  const int32_t* stop;   // when set, every kernel returns at once once *stop is set
  unsigned* rmax_bits;   // largest radius
  // sort
  uint32_t* keys;        // cell key of each slot
  int32_t* cnt;
  int32_t* arr;
  uint2* pairs;
  uint32_t* skeys;       // keys in the new order
  const int32_t* starts; // first sorted position of each cell (n_cells + 1)
  // partials of a force evaluation
  FireDev* st;
  int nparts;
  double* part_e;
  double* part_p;
  unsigned* part_g;
  double* w_out;         // (N, D*D) half the pair virials by slot, or null
  // Verlet list (vl set): *moved is raised when a sphere has moved skin / 2
  // since the build; the fold of the offsets, the sort and the list build run
  // only then
  int32_t* vl;           // (vm, N) slot-major: partner slot | cell difference << 24, -1 ends a row
  int vm;
  int vsr;               // stencil half-width of the list build (1 or 2)
  float vcut;            // list reach beyond r_i + r_j (the skin)
  float vtrig;           // (skin / 2)^2
  int32_t* vovf;         // set when a row would exceed vm
};
// blocks (partials) of a force evaluation
unsigned prec_parts(int64_t n, bool list);
hipError_t launch_prec_load(const PrecArgs& a, hipStream_t s);
hipError_t launch_prec_store(const PrecArgs& a, hipStream_t s);
hipError_t launch_prec_keys(const PrecArgs& a, hipStream_t s);
// placement and permute into the new order and, in list mode, the list build
hipError_t launch_prec_permute(const PrecArgs& a, hipStream_t s);
hipError_t launch_prec_force(const PrecArgs& a, hipStream_t s);
// stopping tests and FIRE scalars from the last evaluation, then the update
hipError_t launch_prec_update(const PrecArgs& a, PrecStop* ps, const PrecStopP& p, const FireP& fp, hipStream_t s);
// ps->pe, ps->gmax of the last evaluation
hipError_t launch_prec_total(const PrecArgs& a, PrecStop* ps, hipStream_t s);
hipError_t launch_prec_import(const double* pos, int64_t n, int D, const double* L, const double* h, const float* hi,
                              const int32_t* dims, int32_t* cidx, float* off, hipStream_t s);
hipError_t launch_prec_export(const int32_t* cidx, const float* off, int64_t n, int D, const double* L,
                              const double* h, const float* hi, const int32_t* dims, double* pos, hipStream_t s);

inline unsigned nblocks(int64_t n, int b = kBlock) { return (unsigned)((n + b - 1) / b); }

}  // namespace jdem
