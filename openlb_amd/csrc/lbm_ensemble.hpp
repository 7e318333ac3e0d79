// Kernels of the lattice ensemble: many independent blocks of uneven extent,
// each with its own padded PS columns, dynamics ids, parameters and walls,
// advanced together by one launch per time step.
//
// The launch covers the concatenated 256-cell chunks of every active lattice.
// A chunk finds its lattice through `chunk_lattice` and reads that lattice's
// entry from the table with uniform (scalar) loads, then runs exactly the
// cell body of the single-block kernel.  The shifts and step counters live on
// the device in two copies: a step reads one and the first workgroup of each
// lattice writes the other, advanced by one step, so a sequence of steps needs
// no host involvement, can be captured in a HIP graph, and takes one launch per
// step.  A call starts and ends on the first copy (an odd number of steps is
// followed by a copy), so that a call a program captures can be replayed.
// (An advance kernel of its own, one thread per lattice, took 5-9 us
// per step behind the step kernel: 96 FP16 cavities 148 + 8.9 us, the solve
// server's two ensembles 26 + 16 + 2 x 5.2 us.)  The copy a step reads also
// gives the pass its direction (chunk_of_block).
#pragma once

#include "lbm_kernels.hpp"

namespace lbmh {

constexpr int kEnsembleWalls = 64;  // wall-table entries per lattice (ids 0..63)

template <int Q>
struct EnsembleEntry {
  void* pop;                // column 0
  uint64_t stride;          // elements between columns
  const uint8_t* ids;       // per core cell dynamics id
  const double* walls;      // [id][4] rho, ux, uy, uz
  const uint32_t* info;     // [id] packed LocalInfo
  const void* force;        // per-cell FORCE [3][ncore] in the arithmetic type, or null (bp.force)
  uint32_t n_padded, ncore, nx, ny, nz, sx, sy;
  FastDiv div_z, div_y;
  uint32_t periodic;
  uint32_t chunk_begin;     // first chunk of this lattice in the launch
  BulkParams<double> bp;
  uint32_t dmod[Q];         // (c_i . projection) mod n_padded
};

// What a step changes of a lattice besides its populations.
template <int Q>
struct MemberState {
  int64_t steps_left;       // 0: idle, < 0: unbounded
  int64_t steps_done;
  uint32_t stepped;         // 1 if the last step moved this lattice (its post-processors run)
  uint32_t pad_;
  uint32_t shift[Q];        // PS shifts, in [0, n_padded)
};

// Address ranges of the arenas, so that a workgroup can refuse an entry that does not fit.
struct EnsembleLimits {
  uint64_t pop_begin, pop_end;
  uint64_t ids_begin, ids_end;
  uint32_t members;         // table slots
};

// Whole-member arguments of the single-block cell body, from a table entry.
template <int Q, typename S>
__device__ __forceinline__ StepArgs<Q, typename StorageTraits<S>::V> member_args(
    const EnsembleEntry<Q>& e, const MemberState<Q>& st, bool local)
{
  using V = typename StorageTraits<S>::V;
  StepArgs<Q, V> a;
  a.pop = e.pop;
  a.stride = e.stride;
  a.n_padded = e.n_padded;
#pragma unroll
  for (int i = 0; i < Q; ++i) a.shift[i] = st.shift[i];
  a.ids = e.ids;
  a.ncore = e.ncore;
  a.nx = e.nx;
  a.ny = e.ny;
  a.nz = e.nz;
  a.sx = e.sx;
  a.sy = e.sy;
  a.div_z = e.div_z;
  a.div_y = e.div_y;
  a.periodic = e.periodic;
  a.xcd_group = 0;
  a.reverse = 0;
  a.walls = e.walls;
  a.info = local ? e.info : nullptr;
  a.force = static_cast<const V*>(e.force);
  a.bp.omega = V(e.bp.omega);
  a.bp.omega2 = V(e.bp.omega2);
  a.bp.guo = V(e.bp.guo);
  for (int d = 0; d < 3; ++d) {
    a.bp.force[d] = V(e.bp.force[d]);
    a.bp.half_force[d] = V(e.bp.half_force[d]);
  }
  a.bp.sm_a = V(e.bp.sm_a);
  a.bp.sm_b = V(e.bp.sm_b);
  a.bp.sm_k = V(e.bp.sm_k);
  a.bp.tau = V(e.bp.tau);
  a.bp.half_tau = V(e.bp.half_tau);
  return a;
}

// uniform guard: every column and the id range of the entry inside the arenas
template <int Q, typename S>
__device__ __forceinline__ bool entry_fits(const EnsembleEntry<Q>& e, const EnsembleLimits& limits)
{
  const uint64_t pop = reinterpret_cast<uint64_t>(e.pop), ids = reinterpret_cast<uint64_t>(e.ids);
  return !(e.stride < e.n_padded || pop < limits.pop_begin || pop + uint64_t(Q) * e.stride * sizeof(S) > limits.pop_end ||
           ids < limits.ids_begin || ids + e.ncore > limits.ids_end);
}

// Streaming of a lattice, by the threads of its first workgroup: rotate its
// columns and count the step if it stepped, into the copy the next step reads.
template <int Q>
__device__ __forceinline__ void advance_member(const EnsembleEntry<Q>& e, const MemberState<Q>& st, MemberState<Q>& next)
{
  const uint32_t i = threadIdx.x;
  const bool step = st.steps_left != 0;
  if (i < uint32_t(Q)) {
    const uint32_t s = st.shift[i], d = e.dmod[i];
    next.shift[i] = !step ? s : (s >= d ? s - d : s + (e.n_padded - d));
  }
  if (i == 0) {
    next.stepped = step ? 1u : 0u;
    next.steps_left = st.steps_left > 0 ? st.steps_left - 1 : st.steps_left;
    next.steps_done = st.steps_done + (step ? 1 : 0);
  }
}

// The states of all members from one copy to the other, `words` 32-bit words.
static __global__ __launch_bounds__(kBlock) void ensemble_settle_kernel(uint32_t* __restrict__ to,
                                                                        const uint32_t* __restrict__ from, uint32_t words)
{
  const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
  if (k < words) to[k] = from[k];
}

// LOCAL = kLocalFlat when some member has local boundaries: their inner edges
// and corners are left to ensemble_local_kernel.
template <int Q, typename S, int KIND, int LOCAL = kLocalNone>
__global__ __launch_bounds__(kBlock) void ensemble_step_kernel(const EnsembleEntry<Q>* __restrict__ table,
                                                               const MemberState<Q>* __restrict__ state,
                                                               MemberState<Q>* __restrict__ next, uint32_t reverse,
                                                               const uint32_t* __restrict__ chunk_lattice,
                                                               uint32_t xcd_group, EnsembleLimits limits)
{
  const uint32_t b = chunk_of_block(blockIdx.x, gridDim.x, xcd_group, reverse);
  const uint32_t lat = chunk_lattice[b];
  if (lat >= limits.members) return;
  const EnsembleEntry<Q>& e = table[lat];
  const MemberState<Q>& st = state[lat];
  if (b == e.chunk_begin) advance_member(e, st, next[lat]);
  if (st.steps_left == 0) return;
  if (!entry_fits<Q, S>(e, limits)) return;
  const auto a = member_args<Q, S>(e, st, LOCAL != kLocalNone);
  collide_stream_cell<Q, S, KIND, true, LOCAL>(a, (b - e.chunk_begin) * kBlock + threadIdx.x);
}

// The local-boundary cells of every stepping member: list entries are
// (member, core cell) pairs.
template <int Q, typename S, int KIND>
__global__ __launch_bounds__(64) void ensemble_local_kernel(const EnsembleEntry<Q>* __restrict__ table,
                                                            const MemberState<Q>* __restrict__ state,
                                                            const uint2* __restrict__ cells, uint32_t count,
                                                            EnsembleLimits limits)
{
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= count) return;
  const uint2 lc = cells[k];
  if (lc.x >= limits.members) return;
  const EnsembleEntry<Q>& e = table[lc.x];
  const MemberState<Q>& st = state[lc.x];
  if (st.steps_left == 0 || !entry_fits<Q, S>(e, limits) || lc.y >= e.ncore) return;
  const auto a = member_args<Q, S>(e, st, true);
  collide_stream_cell<Q, S, KIND, true, kLocalCollide>(a, lc.y);
}

// Plane, edge or corner post-processors (KIND) of the members that stepped
// last (or of member `only` when only >= 0: initialize()).  Eight lanes per
// (member, cell) entry, as outer_post_kernel.  The SCRATCH plane pass
// computes entry k's populations into scratch[k * Q ...] and
// ensemble_plane_store_kernel writes them afterwards: pressure faces read the
// velocity of their face neighbours from populations the pass rewrites
// (plane_scratch_kernel / plane_store_kernel of a lattice).  The two are
// separate instantiations, as the lattice's kernels are, so that each
// compiles the reconstruction exactly as the lattice does.
template <int Q, typename S, int KIND, bool SCRATCH = false>
__global__ __launch_bounds__(64) void ensemble_post_kernel(const EnsembleEntry<Q>* __restrict__ table,
                                                           const MemberState<Q>* __restrict__ state,
                                                           const uint2* __restrict__ cells, uint32_t count,
                                                           EnsembleLimits limits, int only, int forced,
                                                           typename StorageTraits<S>::V* scratch = nullptr)
{
  using V = typename StorageTraits<S>::V;
  __shared__ V nb[64 / kPostLanes][kPostSlots][4];
  const int slot = int(threadIdx.x % kPostLanes), j = int(threadIdx.x / kPostLanes);
  const uint32_t k = blockIdx.x * (64 / kPostLanes) + uint32_t(j);
  bool valid = k < count;
  uint2 lc = make_uint2(0, 0);
  PostArgs<Q> a;
  if (valid) {
    lc = cells[k];
    valid = lc.x < limits.members;
  }
  if (valid) {
    const EnsembleEntry<Q>& e = table[lc.x];
    const MemberState<Q>& st = state[lc.x];
    valid = (only >= 0 ? int(lc.x) == only : st.stepped != 0) && entry_fits<Q, S>(e, limits) && lc.y < e.ncore;
    if (valid) {
      a.pop = e.pop;
      a.stride = e.stride;
      a.n_padded = e.n_padded;
#pragma unroll
      for (int i = 0; i < Q; ++i) a.shift[i] = st.shift[i];
      a.ids = e.ids;
      a.walls = e.walls;
      a.info = e.info;
      a.cells = nullptr;
      a.recs = nullptr;
      a.remote = nullptr;
      // a forced bulk neighbour reports u + F/2 (the member's uniform FORCE)
      a.forced = uint32_t(forced);
      a.force = nullptr;
      a.half_force[0] = e.bp.half_force[0];
      a.half_force[1] = e.bp.half_force[1];
      a.half_force[2] = e.bp.half_force[2];
      a.count = 0;
      a.nx = int(e.nx);
      a.ny = int(e.ny);
      a.nz = int(e.nz);
      a.sx = e.sx;
      a.sy = e.sy;
      a.periodic = e.periodic;
      a.div_z = e.div_z;
      a.div_y = e.div_y;
      a.omega = e.bp.omega;
    }
  }
  if (valid && slot < kPostSlots) post_gather<Q, S, KIND>(a, lc.y, slot, nb[j][slot]);
  __syncthreads();
  if (valid && slot == 0) {
    if constexpr (SCRATCH)
      post_finish<Q, S, KIND>(a, lc.y, int(a.ids[lc.y]), nb[j], scratch + uint64_t(k) * Q);
    else
      post_finish<Q, S, KIND>(a, lc.y, int(a.ids[lc.y]), nb[j]);
  }
}

// Second half of a two-phase plane pass: entry k's populations from scratch.
template <int Q, typename S>
__global__ __launch_bounds__(64) void ensemble_plane_store_kernel(const EnsembleEntry<Q>* __restrict__ table,
                                                                  const MemberState<Q>* __restrict__ state,
                                                                  const uint2* __restrict__ cells, uint32_t count,
                                                                  const typename StorageTraits<S>::V* scratch,
                                                                  EnsembleLimits limits, int only)
{
  using V = typename StorageTraits<S>::V;
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= count) return;
  const uint2 lc = cells[k];
  if (lc.x >= limits.members) return;
  const EnsembleEntry<Q>& e = table[lc.x];
  const MemberState<Q>& st = state[lc.x];
  if (!((only >= 0 ? int(lc.x) == only : st.stepped != 0) && entry_fits<Q, S>(e, limits) && lc.y < e.ncore)) return;
  int x, y, z;
  core_coords(e.div_z, e.div_y, int(e.ny), int(e.nz), lc.y, x, y, z);
  const uint32_t n = uint32_t(x + 1) * e.sx + uint32_t(y + 1) * e.sy + uint32_t(z + 1);
  S* pop = static_cast<S*>(e.pop);
#pragma unroll
  for (int i = 0; i < Q; ++i)
    store_pop<S, V>(column_at(pop + uint64_t(i) * e.stride, wrap_index(n, st.shift[i], e.n_padded)),
                    scratch[uint64_t(k) * Q + i]);
}

}  // namespace lbmh
