// C ABI of lattice ensembles (declarations in include/lbmh.h).
//
// Members live in two device arenas (populations, dynamics ids) carved at
// creation, so admitting or retiring a member never calls hipMalloc/hipFree
// (hipFree would also wait for the whole device).  The member table and the
// chunk -> member map are device arrays; the host keeps the arena bookkeeping
// and rebuilds the map when membership changes.  Shifts and step counters are
// advanced on the device, so a step loop can be captured in a HIP graph.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <new>
#include <tuple>
#include <vector>

#include "boundary_classify.hpp"
#include "checkpoint.hpp"
#include "launch_shape.hpp"
#include "lbm_fields.hpp"
#include "lbm_ensemble.hpp"
#include "lbmh.h"
#include "lbmh_common.hpp"
#include "result_copy.hpp"

using namespace lbmh;

namespace {

constexpr uint64_t kAlign = 256;

uint64_t align_up(uint64_t v) { return (v + kAlign - 1) / kAlign * kAlign; }

// First-fit allocator over [0, capacity) with coalescing of free ranges.
class Arena {
 public:
  explicit Arena(uint64_t capacity = 0) : capacity_(capacity)
  {
    if (capacity) free_[0] = capacity;
  }
  bool alloc(uint64_t bytes, uint64_t* off)
  {
    bytes = align_up(bytes);
    for (auto it = free_.begin(); it != free_.end(); ++it) {
      if (it->second >= bytes) {
        *off = it->first;
        const uint64_t rest = it->second - bytes, start = it->first + bytes;
        free_.erase(it);
        if (rest) free_[start] = rest;
        used_ += bytes;
        return true;
      }
    }
    return false;
  }
  void release(uint64_t off, uint64_t bytes)
  {
    bytes = align_up(bytes);
    used_ -= bytes;
    auto it = free_.emplace(off, bytes).first;
    auto next = std::next(it);
    if (next != free_.end() && it->first + it->second == next->first) {
      it->second += next->second;
      free_.erase(next);
    }
    if (it != free_.begin()) {
      auto prev = std::prev(it);
      if (prev->first + prev->second == it->first) {
        prev->second += it->second;
        free_.erase(it);
      }
    }
  }
  uint64_t used() const { return used_; }
  uint64_t capacity() const { return capacity_; }

 private:
  uint64_t capacity_ = 0, used_ = 0;
  std::map<uint64_t, uint64_t> free_;
};

struct Member {
  bool active = false;
  int n[3] = {0, 0, 0};
  int periodic[3] = {0, 0, 0};
  uint64_t pop_off = 0, pop_bytes = 0;   // bytes in the population arena
  uint64_t ids_off = 0, ids_bytes = 0;
  uint32_t ncore = 0;
  lbmh_bulk_params params{};
  // local boundaries: host ids, per-id descriptors, cell lists (core indices)
  std::vector<uint8_t> h_ids;
  uint32_t info[kEnsembleWalls] = {};
  bool id_defined[kEnsembleWalls] = {};
  std::vector<uint32_t> local, edges, corners, planes;
  bool pressure_planes = false;  // InterpolatedPressure faces: its planes run the two-phase pass
};

}  // namespace

struct lbmh_ensemble {
  int device = 0, q = 19, storage = LBMH_F32, kind = LBMH_BGK;
  int max_members = 0;
  void* d_pop = nullptr;
  uint8_t* d_ids = nullptr;
  double* d_walls = nullptr;
  void* d_table = nullptr;
  uint32_t* d_chunk = nullptr;
  uint32_t chunk_capacity = 0, total_chunks = 0;
  size_t entry_bytes = 0;
  Arena pop_arena, id_arena;
  std::vector<Member> members;
  std::vector<unsigned char> h_table;   // host mirror of the member table
  // steps left and done and PS shifts of every member: two copies of
  // max_members records on the device behind the table, the first current
  // between calls (each step reads one and writes the other), and a host
  // mirror of it
  char* d_state = nullptr;
  size_t state_bytes = 0;               // one record
  std::vector<unsigned char> h_state;
  lbmh_launch_config launch{0, 4};  // used once launch_chosen, else step_launch()
  bool launch_chosen = false;     // set by lbmh_ensemble_set_launch_config / _autotune: keep it
  uint64_t version = 1;
  hipStream_t capture_stream = nullptr;
  hipGraphExec_t graph = nullptr;
  uint64_t graph_version = 0;
  int64_t graph_steps = 0;
  // local boundaries: per-member id descriptors and (member, cell) lists
  uint32_t* d_info = nullptr;
  uint2* d_local = nullptr;
  uint2* d_edges = nullptr;
  uint2* d_corners = nullptr;
  uint2* d_planes = nullptr;    // plane cells of members without pressure planes: one pass
  uint2* d_pplanes = nullptr;   // plane cells of members with pressure planes: two-phase pass
  size_t boundary_capacity = 0;
  // the two-phase plane pass's populations, boundary_capacity x Q values,
  // allocated with the first member that has InterpolatedPressure faces
  void* d_plane_scratch = nullptr;
  uint32_t n_local = 0, n_edges = 0, n_corners = 0, n_planes = 0, n_pplanes = 0;
  bool has_local = false;            // some member ever had local boundaries
};

namespace {

template <int Q>
EnsembleEntry<Q>& entry(lbmh_ensemble* E, int m)
{
  return *reinterpret_cast<EnsembleEntry<Q>*>(E->h_table.data() + size_t(m) * E->entry_bytes);
}

template <int Q>
MemberState<Q>& state(lbmh_ensemble* E, int m)
{
  return *reinterpret_cast<MemberState<Q>*>(E->h_state.data() + size_t(m) * E->state_bytes);
}

// The device's copy k of member m's state.
char* device_state(lbmh_ensemble* E, uint32_t k, int m = 0)
{
  return E->d_state + (size_t(k) * size_t(E->max_members) + size_t(m)) * E->state_bytes;
}

EnsembleLimits limits_of(const lbmh_ensemble* E)
{
  const uint64_t pop = reinterpret_cast<uint64_t>(E->d_pop), ids = reinterpret_cast<uint64_t>(E->d_ids);
  return EnsembleLimits{pop, pop + E->pop_arena.capacity(), ids, ids + E->id_arena.capacity(), uint32_t(E->max_members)};
}

template <typename F>
int with_q(const lbmh_ensemble* E, F&& f)
{
  return E->q == 19 ? f(std::integral_constant<int, 19>()) : f(std::integral_constant<int, 27>());
}

template <typename F>
int with_types(int q, int storage, F&& f)
{
  if (q == 19) {
    if (storage == LBMH_F64) return f(std::integral_constant<int, 19>(), double());
    if (storage == LBMH_F32) return f(std::integral_constant<int, 19>(), float());
    return f(std::integral_constant<int, 19>(), _Float16());
  }
  if (storage == LBMH_F64) return f(std::integral_constant<int, 27>(), double());
  if (storage == LBMH_F32) return f(std::integral_constant<int, 27>(), float());
  return f(std::integral_constant<int, 27>(), _Float16());
}

template <typename F>
int with_types(const lbmh_ensemble* E, F&& f)
{
  return with_types(E->q, E->storage, std::forward<F>(f));
}

// The members' states as the device holds them; the table only changes here on
// the host.  (Copies above 16 KB take another way through the runtime: repeated
// on their own 9 us against 12 to 18 below, but 80 to 120 us between kernels and
// other copies, 18 to 28 below, so reads are not made larger than they need be.)
int pull_state(lbmh_ensemble* E)
{
  LBMH_HIP(hipDeviceSynchronize());
  LBMH_HIP(hipMemcpy(E->h_state.data(), device_state(E, 0), E->h_state.size(), hipMemcpyDeviceToHost));
  return LBMH_OK;
}

// The state of member m alone.
int pull_state(lbmh_ensemble* E, int m)
{
  LBMH_HIP(hipDeviceSynchronize());
  LBMH_HIP(hipMemcpy(E->h_state.data() + size_t(m) * E->state_bytes, device_state(E, 0, m), E->state_bytes,
                     hipMemcpyDeviceToHost));
  return LBMH_OK;
}

// Assign chunk ranges to active members in slot order and upload table + map.
int push_table(lbmh_ensemble* E)
{
  std::vector<uint32_t> map;
  map.reserve(E->total_chunks);
  const int rc = with_q(E, [&](auto qc) -> int {
    constexpr int Q = decltype(qc)::value;
    for (int m = 0; m < E->max_members; ++m) {
      EnsembleEntry<Q>& e = entry<Q>(E, m);
      if (!E->members[m].active) {
        e.chunk_begin = 0;
        std::memset(&state<Q>(E, m), 0, sizeof(MemberState<Q>));
        continue;
      }
      e.chunk_begin = uint32_t(map.size());
      const uint32_t chunks = grid_for(e.ncore, kBlock);
      map.insert(map.end(), chunks, uint32_t(m));
    }
    return LBMH_OK;
  });
  if (rc != LBMH_OK) return rc;
  if (map.size() > E->chunk_capacity) return fail(LBMH_E_MEMORY, "chunk map capacity exceeded");
  E->total_chunks = uint32_t(map.size());
  // table and both copies of the states (a slot without a member has no
  // workgroup to carry its state over) in one copy
  std::vector<unsigned char> all = E->h_table;
  all.resize(size_t(E->d_state - static_cast<char*>(E->d_table)));
  for (int k = 0; k < 2; ++k) all.insert(all.end(), E->h_state.begin(), E->h_state.end());
  LBMH_HIP(hipMemcpy(E->d_table, all.data(), all.size(), hipMemcpyHostToDevice));
  if (!map.empty()) LBMH_HIP(hipMemcpy(E->d_chunk, map.data(), map.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
  E->version += 1;
  return LBMH_OK;
}

int check_member(const lbmh_ensemble* E, int m)
{
  if (!E) return fail(LBMH_E_INVALID, "null ensemble");
  if (m < 0 || m >= E->max_members || !E->members[m].active) return fail(LBMH_E_INVALID, "no such member");
  return LBMH_OK;
}

// Concatenate the local-boundary lists of the active members into the device lists.
int rebuild_lists(lbmh_ensemble* E)
{
  std::vector<uint2> all[5];
  for (int m = 0; m < E->max_members; ++m) {
    const Member& mem = E->members[m];
    if (!mem.active) continue;
    const std::vector<uint32_t>* src[4] = {&mem.local, &mem.edges, &mem.corners, &mem.planes};
    for (int k = 0; k < 4; ++k) {
      const int to = (k == 3 && mem.pressure_planes) ? 4 : k;
      for (uint32_t c : *src[k]) all[to].push_back(make_uint2(uint32_t(m), c));
    }
  }
  for (int k = 0; k < 5; ++k)
    if (all[k].size() > E->boundary_capacity) return fail(LBMH_E_MEMORY, "boundary list capacity exceeded");
  uint2* dst[5] = {E->d_local, E->d_edges, E->d_corners, E->d_planes, E->d_pplanes};
  for (int k = 0; k < 5; ++k)
    if (!all[k].empty()) LBMH_HIP(hipMemcpy(dst[k], all[k].data(), all[k].size() * sizeof(uint2), hipMemcpyHostToDevice));
  E->n_local = uint32_t(all[0].size());
  E->n_edges = uint32_t(all[1].size());
  E->n_corners = uint32_t(all[2].size());
  E->n_planes = uint32_t(all[3].size());
  E->n_pplanes = uint32_t(all[4].size());
  E->version += 1;
  return LBMH_OK;
}

template <int Q>
CoreGeom geom_of(const EnsembleEntry<Q>& e)
{
  CoreGeom g;
  g.ncore = e.ncore;
  g.nx = e.nx;
  g.ny = e.ny;
  g.nz = e.nz;
  g.sx = e.sx;
  g.sy = e.sy;
  g.n_padded = e.n_padded;
  g.stride = e.stride;
  g.div_z = e.div_z;
  g.div_y = e.div_y;
  return g;
}

template <int Q>
Shifts<Q> shifts_of(const MemberState<Q>& st)
{
  Shifts<Q> s;
  for (int i = 0; i < Q; ++i) s.s[i] = st.shift[i];
  return s;
}

// PostStream stage of the local boundaries: edges, then corners, of the
// members that stepped (only < 0) or of member `only`.
template <int Q, typename S>
int launch_post(lbmh_ensemble* E, const EnsembleEntry<Q>* table, const MemberState<Q>* st, const EnsembleLimits& limits,
                hipStream_t stream, int only)
{
  const int forced = (E->kind == LBMH_FORCED_BGK || E->kind == LBMH_FORCED_TRT) ? 1 : 0;
  if (E->n_planes) {
    hipLaunchKernelGGL((ensemble_post_kernel<Q, S, kPostPlane>), dim3(grid_for(E->n_planes, 64 / kPostLanes)), dim3(64),
                       0, stream, table, st, E->d_planes, E->n_planes, limits, only,
                       forced);
    LBMH_HIP(hipGetLastError());
  }
  if (E->n_pplanes) {
    // members with pressure faces: every plane cell into the workspace, then stored
    using V = typename StorageTraits<S>::V;
    V* scratch = static_cast<V*>(E->d_plane_scratch);
    hipLaunchKernelGGL((ensemble_post_kernel<Q, S, kPostPlane, true>), dim3(grid_for(E->n_pplanes, 64 / kPostLanes)),
                       dim3(64), 0, stream, table, st, E->d_pplanes, E->n_pplanes,
                       limits, only, forced, scratch);
    LBMH_HIP(hipGetLastError());
    hipLaunchKernelGGL((ensemble_plane_store_kernel<Q, S>), dim3(grid_for(E->n_pplanes, 64)), dim3(64), 0, stream,
                       table, st, E->d_pplanes, E->n_pplanes, static_cast<const V*>(scratch), limits, only);
    LBMH_HIP(hipGetLastError());
  }
  if (E->n_edges) {
    hipLaunchKernelGGL((ensemble_post_kernel<Q, S, kPostEdge>), dim3(grid_for(E->n_edges, 64 / kPostLanes)), dim3(64), 0,
                       stream, table, st, E->d_edges, E->n_edges, limits, only, forced);
    LBMH_HIP(hipGetLastError());
  }
  if (E->n_corners) {
    hipLaunchKernelGGL((ensemble_post_kernel<Q, S, kPostCorner>), dim3(grid_for(E->n_corners, 64 / kPostLanes)), dim3(64), 0,
                       stream, table, st, E->d_corners, E->n_corners, limits, only,
                       forced);
    LBMH_HIP(hipGetLastError());
  }
  return LBMH_OK;
}

// Launch shape of a step: the chosen one, else by what the members hold.
// LDS reservation as for a single block: 40 KB in FP32 and 48 KB in FP64, none
// in FP16 and while the members fit the caches (up to 64 MB; 12 FP32 cavities,
// 38 MB, 15.6 us capped, 15.0 us not).  With local-boundary members the step
// kernel collides their flat faces too, in divergent waves that need more
// occupancy: 24 KB (FP32, 96 local-velocity cavities 458 us per step against
// 509 us; velocity-inlet ducts 266 against 269 us).  XCD groups of 32 keep a
// small member's chunks, and the lines they share, on one XCD (group 8 -> 32:
// 12 FP16 cavities 11.4 -> 11.2 us, 16 FP32 ducts 60.6 -> 59.7 us, 40 FP64
// cavities 142.1 -> 140.7 us, 96 FP32 cavities 236 -> 237 us).
lbmh_launch_config step_launch(const lbmh_ensemble* E)
{
  if (E->launch_chosen) return E->launch;
  lbmh_launch_config c{0, 32};
  if (E->storage == LBMH_F16) return c;
  if (E->has_local) c.lds_bytes = 24576;
  else if (E->pop_arena.used() >= 64000000u) c.lds_bytes = E->storage == LBMH_F64 ? 49152 : 40960;
  return c;
}

template <int Q, typename S, int LOCAL>
int launch_step_kernel(int kind, const EnsembleEntry<Q>* table, const MemberState<Q>* st, MemberState<Q>* next,
                       uint32_t reverse, const uint32_t* chunk_member, uint32_t chunks, const lbmh_launch_config& launch,
                       const EnsembleLimits& limits, hipStream_t stream)
{
  const unsigned lds = unsigned(launch.lds_bytes);
  const uint32_t group = uint32_t(launch.xcd_group);
#define LBMH_ENSEMBLE_STEP(KIND_)                                                                               \
  hipLaunchKernelGGL((ensemble_step_kernel<Q, S, KIND_, LOCAL>), dim3(chunks), dim3(kBlock), lds, stream, table, st, \
                     next, reverse, chunk_member, group, limits)
  switch (kind) {
  case LBMH_BGK: LBMH_ENSEMBLE_STEP(kBGK); break;
  case LBMH_FORCED_BGK: LBMH_ENSEMBLE_STEP(kForcedBGK); break;
  case LBMH_TRT: LBMH_ENSEMBLE_STEP(kTRT); break;
  case LBMH_FORCED_TRT: LBMH_ENSEMBLE_STEP(kForcedTRT); break;
  default: LBMH_ENSEMBLE_STEP(kSmagorinsky); break;
  }
#undef LBMH_ENSEMBLE_STEP
  LBMH_HIP(hipGetLastError());
  return LBMH_OK;
}

// The boundary cells of a `local` step collide with their BGK mixin whatever the bulk kind.
template <int Q, typename S>
int launch_step_kernel(int kind, bool local, const EnsembleEntry<Q>* table, const MemberState<Q>* st,
                       MemberState<Q>* next, uint32_t reverse, const uint32_t* chunk_member, uint32_t chunks,
                       const lbmh_launch_config& launch, const EnsembleLimits& limits, hipStream_t stream)
{
  return local ? launch_step_kernel<Q, S, kLocalFlat>(kind, table, st, next, reverse, chunk_member, chunks, launch,
                                                      limits, stream)
               : launch_step_kernel<Q, S, kLocalNone>(kind, table, st, next, reverse, chunk_member, chunks, launch,
                                                      limits, stream);
}

int launch_steps(lbmh_ensemble* E, int64_t n, hipStream_t stream)
{
  const lbmh_launch_config launch = step_launch(E);
  return with_types(E, [&](auto qc, auto s) -> int {
    constexpr int Q = decltype(qc)::value;
    using S = decltype(s);
    auto* table = static_cast<EnsembleEntry<Q>*>(E->d_table);
    const EnsembleLimits limits = limits_of(E);
    const bool local = E->has_local;
    for (int64_t k = 0; k < n; ++k) {
      const uint32_t cur = uint32_t(k & 1);
      const auto* st = reinterpret_cast<const MemberState<Q>*>(device_state(E, cur));
      auto* next = reinterpret_cast<MemberState<Q>*>(device_state(E, cur ^ 1u));
      if (E->total_chunks) {
        const int rc = launch_step_kernel<Q, S>(E->kind, local, table, st, next, cur, E->d_chunk, E->total_chunks,
                                                launch, limits, stream);
        if (rc != LBMH_OK) return rc;
      }
      if (local && E->n_local) {
#define LBMH_ENSEMBLE_LOCAL(KIND_)                                                                              \
  hipLaunchKernelGGL((ensemble_local_kernel<Q, S, KIND_>), dim3(grid_for(E->n_local, 64)), dim3(64), 0, stream,      \
                     table, st, E->d_local, E->n_local, limits)
        switch (E->kind) {
        case LBMH_BGK: LBMH_ENSEMBLE_LOCAL(kBGK); break;
        case LBMH_FORCED_BGK: LBMH_ENSEMBLE_LOCAL(kForcedBGK); break;
        case LBMH_TRT: LBMH_ENSEMBLE_LOCAL(kTRT); break;
        case LBMH_FORCED_TRT: LBMH_ENSEMBLE_LOCAL(kForcedTRT); break;
        default: LBMH_ENSEMBLE_LOCAL(kSmagorinsky); break;
        }
#undef LBMH_ENSEMBLE_LOCAL
        LBMH_HIP(hipGetLastError());
      }
      const int rc = launch_post<Q, S>(E, table, static_cast<const MemberState<Q>*>(next), limits, stream, -1);
      if (rc != LBMH_OK) return rc;
    }
    if (n & 1) {
      const uint32_t words = uint32_t(E->h_state.size() / sizeof(uint32_t));
      hipLaunchKernelGGL(ensemble_settle_kernel, dim3(grid_for(words, kBlock)), dim3(kBlock), 0, stream,
                         reinterpret_cast<uint32_t*>(device_state(E, 0)),
                         reinterpret_cast<const uint32_t*>(device_state(E, 1)), words);
      LBMH_HIP(hipGetLastError());
    }
    return LBMH_OK;
  });
}

}  // namespace

int lbmh::launch_block_table_step(const BlockTableStep& t, hipStream_t stream)
{
  return with_types(t.q, t.storage, [&](auto qc, auto s) -> int {
    constexpr int Q = decltype(qc)::value;
    using S = decltype(s);
    // the blocks are the caller's own allocations, not ranges of an arena
    const EnsembleLimits limits{0, ~uint64_t(0), 0, ~uint64_t(0), t.blocks};
    return launch_step_kernel<Q, S>(t.kind, t.local, static_cast<const EnsembleEntry<Q>*>(t.table),
                                    static_cast<const MemberState<Q>*>(t.state), static_cast<MemberState<Q>*>(t.next),
                                    t.reverse, t.chunk_block, t.chunks, t.launch, limits, stream);
  });
}

extern "C" {

int lbmh_ensemble_create(const lbmh_ensemble_desc* d, lbmh_ensemble** out)
{
  if (!d || !out) return fail(LBMH_E_INVALID, "null argument");
  *out = nullptr;
  if (d->q != 19 && d->q != 27) return fail(LBMH_E_INVALID, "q must be 19 or 27");
  if (d->storage < LBMH_F64 || d->storage > LBMH_F16) return fail(LBMH_E_INVALID, "unknown storage type");
  if (d->bulk_kind < LBMH_BGK || d->bulk_kind > LBMH_SMAGORINSKY) return fail(LBMH_E_INVALID, "unknown bulk kind");
  if (d->max_members < 1 || d->max_members > (1 << 20)) return fail(LBMH_E_INVALID, "max_members out of range");
  if (d->population_bytes < kAlign || d->cell_capacity < 1) return fail(LBMH_E_INVALID, "arena sizes must be positive");
  auto* E = new (std::nothrow) lbmh_ensemble();
  if (!E) return fail(LBMH_E_MEMORY, "host allocation failed");
  ResultPool::get().retain();
  E->device = d->device;
  E->q = d->q;
  E->storage = d->storage;
  E->kind = d->bulk_kind;
  E->max_members = d->max_members;
  // the device indexes table[m] with this exact stride
  E->entry_bytes = E->q == 19 ? sizeof(EnsembleEntry<19>) : sizeof(EnsembleEntry<27>);
  E->members.resize(size_t(E->max_members));
  E->h_table.assign(E->entry_bytes * size_t(E->max_members), 0);
  E->state_bytes = E->q == 19 ? sizeof(MemberState<19>) : sizeof(MemberState<27>);
  E->h_state.assign(E->state_bytes * size_t(E->max_members), 0);
  E->pop_arena = Arena(align_up(d->population_bytes));
  E->id_arena = Arena(align_up(d->cell_capacity) + kAlign * size_t(E->max_members));
  E->chunk_capacity = uint32_t(d->cell_capacity / kBlock + size_t(E->max_members) + 1);
  DeviceGuard guard(E->device);
  hipError_t e = device_alloc(&E->d_pop, E->pop_arena.capacity());
  if (e == hipSuccess) e = device_alloc((void**)&E->d_ids, E->id_arena.capacity());
  if (e == hipSuccess) e = device_alloc((void**)&E->d_walls, sizeof(double) * 4 * kEnsembleWalls * E->max_members);
  const size_t state_at = align_up(E->h_table.size()), table_bytes = state_at + 2 * E->h_state.size();
  if (e == hipSuccess) e = device_alloc(&E->d_table, table_bytes);
  E->d_state = static_cast<char*>(E->d_table) + state_at;
  if (e == hipSuccess) e = device_alloc((void**)&E->d_chunk, sizeof(uint32_t) * E->chunk_capacity);
  E->boundary_capacity = d->boundary_capacity ? d->boundary_capacity : d->cell_capacity / 4 + 64;
  if (e == hipSuccess) e = device_alloc((void**)&E->d_info, sizeof(uint32_t) * kEnsembleWalls * E->max_members);
  if (e == hipSuccess) e = hipMemset(E->d_info, 0, sizeof(uint32_t) * kEnsembleWalls * E->max_members);
  for (uint2** list : {&E->d_local, &E->d_edges, &E->d_corners, &E->d_planes, &E->d_pplanes})
    if (e == hipSuccess) e = device_alloc((void**)list, sizeof(uint2) * E->boundary_capacity);
  if (e == hipSuccess) e = hipMemset(E->d_table, 0, table_bytes);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&E->capture_stream, hipStreamNonBlocking);
  if (e != hipSuccess) {
    const int rc = hip_fail(e, "lbmh_ensemble_create");
    lbmh_ensemble_destroy(E);
    return e == hipErrorOutOfMemory ? fail(LBMH_E_MEMORY, g_error) : rc;
  }
  *out = E;
  return LBMH_OK;
}

int lbmh_ensemble_destroy(lbmh_ensemble* E)
{
  if (!E) return LBMH_OK;
  DeviceGuard guard(E->device);
  (void)hipDeviceSynchronize();
  if (E->graph) (void)hipGraphExecDestroy(E->graph);
  if (E->capture_stream) (void)hipStreamDestroy(E->capture_stream);
  if (E->d_pop) (void)hipFree(E->d_pop);
  if (E->d_ids) (void)hipFree(E->d_ids);
  if (E->d_walls) (void)hipFree(E->d_walls);
  if (E->d_table) (void)hipFree(E->d_table);
  if (E->d_chunk) (void)hipFree(E->d_chunk);
  if (E->d_info) (void)hipFree(E->d_info);
  if (E->d_local) (void)hipFree(E->d_local);
  if (E->d_edges) (void)hipFree(E->d_edges);
  if (E->d_corners) (void)hipFree(E->d_corners);
  if (E->d_planes) (void)hipFree(E->d_planes);
  if (E->d_pplanes) (void)hipFree(E->d_pplanes);
  if (E->d_plane_scratch) (void)hipFree(E->d_plane_scratch);
  delete E;
  ResultPool::get().release();
  return LBMH_OK;
}

int lbmh_ensemble_member_bytes(const lbmh_ensemble* E, const int extent[3], size_t* pop_bytes, size_t* id_bytes)
{
  if (!E || !extent) return fail(LBMH_E_INVALID, "null argument");
  for (int d = 0; d < 3; ++d)
    if (extent[d] < 1) return fail(LBMH_E_INVALID, "extent must be >= 1");
  const uint64_t npad = uint64_t(extent[0] + 2) * (extent[1] + 2) * (extent[2] + 2);
  const uint64_t elem = storage_size(E->storage);
  const uint64_t stride = align_up(npad * elem) / elem;
  if (pop_bytes) *pop_bytes = size_t(align_up(stride * elem * E->q));
  if (id_bytes) *id_bytes = size_t(align_up(uint64_t(extent[0]) * extent[1] * extent[2]));
  return LBMH_OK;
}

int lbmh_ensemble_add(lbmh_ensemble* E, const int extent[3], const int periodic[3], const uint8_t* ids,
                      const lbmh_bulk_params* params, int64_t steps, int* member)
{
  if (!E || !extent || !periodic || !ids || !params || !member) return fail(LBMH_E_INVALID, "null argument");
  *member = -1;
  for (int d = 0; d < 3; ++d)
    if (extent[d] < 1) return fail(LBMH_E_INVALID, "extent must be >= 1");
  const uint64_t sx = uint64_t(extent[0]) + 2, sy = uint64_t(extent[1]) + 2, sz = uint64_t(extent[2]) + 2;
  const uint64_t npad = sx * sy * sz;
  if (npad >= (uint64_t(1) << 31)) return fail(LBMH_E_INVALID, "padded cell count must be below 2^31");
  if (npad * storage_size(E->storage) >= (uint64_t(1) << 31))
    return fail(LBMH_E_INVALID, "a population column must stay below 2 GiB (padded cells x bytes per population)");
  const uint32_t ncore = uint32_t(uint64_t(extent[0]) * extent[1] * extent[2]);
  for (uint32_t c = 0; c < ncore; ++c)
    if (ids[c] >= kEnsembleWalls) return fail(LBMH_E_INVALID, "ensemble dynamics ids must be below 64");
  if (!valid_bulk_params(E->kind, *params)) return LBMH_E_INVALID;
  int slot = -1;
  for (int m = 0; m < E->max_members; ++m)
    if (!E->members[m].active) {
      slot = m;
      break;
    }
  if (slot < 0) return fail(LBMH_E_MEMORY, "no free member slot");
  size_t pop_bytes = 0, id_bytes = 0;
  lbmh_ensemble_member_bytes(E, extent, &pop_bytes, &id_bytes);
  Member mem;
  if (!E->pop_arena.alloc(pop_bytes, &mem.pop_off)) return fail(LBMH_E_MEMORY, "population arena full");
  if (!E->id_arena.alloc(id_bytes, &mem.ids_off)) {
    E->pop_arena.release(mem.pop_off, pop_bytes);
    return fail(LBMH_E_MEMORY, "id arena full");
  }
  mem.pop_bytes = pop_bytes;
  mem.ids_bytes = id_bytes;
  mem.active = true;
  mem.ncore = ncore;
  mem.params = *params;
  for (int d = 0; d < 3; ++d) {
    mem.n[d] = extent[d];
    mem.periodic[d] = periodic[d] ? 1 : 0;
  }
  DeviceGuard guard(E->device);
  auto undo = [&](int rc) {
    E->pop_arena.release(mem.pop_off, mem.pop_bytes);
    E->id_arena.release(mem.ids_off, mem.ids_bytes);
    return rc;
  };
  int rc = pull_state(E);
  if (rc != LBMH_OK) return undo(rc);
  hipError_t e = hipMemset(static_cast<char*>(E->d_pop) + mem.pop_off, 0, pop_bytes);
  if (e == hipSuccess) e = hipMemcpy(E->d_ids + mem.ids_off, ids, ncore, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    std::vector<double> walls(4 * kEnsembleWalls, 0.0);
    for (int w = 0; w < kEnsembleWalls; ++w) walls[4 * w] = 1.0;
    e = hipMemcpy(E->d_walls + size_t(slot) * 4 * kEnsembleWalls, walls.data(), walls.size() * sizeof(double),
                  hipMemcpyHostToDevice);
  }
  if (e == hipSuccess) e = hipMemcpy(E->d_info + size_t(slot) * kEnsembleWalls, mem.info, sizeof(mem.info),
                                     hipMemcpyHostToDevice);
  mem.h_ids.assign(ids, ids + ncore);
  if (e != hipSuccess) return undo(hip_fail(e, "lbmh_ensemble_add"));
  const uint64_t elem = storage_size(E->storage);
  with_q(E, [&](auto qc) -> int {
    constexpr int Q = decltype(qc)::value;
    EnsembleEntry<Q>& en = entry<Q>(E, slot);
    std::memset(&en, 0, sizeof(en));
    en.pop = static_cast<char*>(E->d_pop) + mem.pop_off;
    en.stride = align_up(npad * elem) / elem;
    en.ids = E->d_ids + mem.ids_off;
    en.walls = E->d_walls + size_t(slot) * 4 * kEnsembleWalls;
    en.info = E->d_info + size_t(slot) * kEnsembleWalls;
    en.n_padded = uint32_t(npad);
    en.ncore = ncore;
    en.nx = uint32_t(extent[0]);
    en.ny = uint32_t(extent[1]);
    en.nz = uint32_t(extent[2]);
    en.sx = uint32_t(sy * sz);
    en.sy = uint32_t(sz);
    en.div_z = FastDiv(uint32_t(extent[2]));
    en.div_y = FastDiv(uint32_t(extent[1]));
    en.periodic = uint32_t(mem.periodic[0] | (mem.periodic[1] << 1) | (mem.periodic[2] << 2));
    MemberState<Q>& st = state<Q>(E, slot);
    std::memset(&st, 0, sizeof(st));
    st.steps_left = steps;
    en.bp = derive_bulk_params<double>(E->q, *params);
    for (int i = 0; i < Q; ++i) {
      const int64_t dist = neighbor_distance<Q>(i, int64_t(sy * sz), int64_t(sz));
      int64_t dm = dist % int64_t(npad);
      if (dm < 0) dm += int64_t(npad);
      en.dmod[i] = uint32_t(dm);
    }
    return LBMH_OK;
  });
  E->members[slot] = mem;
  rc = push_table(E);
  if (rc != LBMH_OK) {
    E->members[slot].active = false;
    return undo(rc);
  }
  *member = slot;
  return LBMH_OK;
}

int lbmh_ensemble_remove(lbmh_ensemble* E, int m)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  DeviceGuard guard(E->device);
  rc = pull_state(E);
  if (rc != LBMH_OK) return rc;
  Member& mem = E->members[m];
  E->pop_arena.release(mem.pop_off, mem.pop_bytes);
  E->id_arena.release(mem.ids_off, mem.ids_bytes);
  mem = Member();
  with_q(E, [&](auto qc) -> int {
    constexpr int Q = decltype(qc)::value;
    std::memset(&entry<Q>(E, m), 0, sizeof(EnsembleEntry<Q>));
    return LBMH_OK;
  });
  rc = push_table(E);
  if (rc != LBMH_OK) return rc;
  return rebuild_lists(E);
}

int lbmh_ensemble_set_wall(lbmh_ensemble* E, int m, int id, double rho, const double u[3])
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  if (!u) return fail(LBMH_E_INVALID, "null velocity");
  if (id < LBMH_ID_FIRST_WALL || id >= kEnsembleWalls) return fail(LBMH_E_INVALID, "ensemble wall id must be in [3, 63]");
  DeviceGuard guard(E->device);
  const double w[4] = {rho, u[0], u[1], u[2]};
  LBMH_HIP(hipDeviceSynchronize());
  LBMH_HIP(hipMemcpy(E->d_walls + (size_t(m) * kEnsembleWalls + id) * 4, w, sizeof(w), hipMemcpyHostToDevice));
  Member& mem = E->members[m];
  mem.id_defined[id] = true;
  mem.info[id] = pack_local_info(kMovingWall, 0, 0, 0);
  LBMH_HIP(hipMemcpy(E->d_info + size_t(m) * kEnsembleWalls + id, &mem.info[id], sizeof(uint32_t), hipMemcpyHostToDevice));
  return LBMH_OK;
}

int lbmh_ensemble_set_local_boundary(lbmh_ensemble* E, int m, int id, int kind, double rho, const double u[3])
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  if (!u) return fail(LBMH_E_INVALID, "null velocity");
  if (kind < LBMH_LOCAL_VELOCITY || kind > LBMH_INTERP_PRESSURE) return fail(LBMH_E_INVALID, "unknown local boundary kind");
  if (id < 2 || id >= kEnsembleWalls) return fail(LBMH_E_INVALID, "ensemble boundary id must be in [2, 63]");
  if ((kind == LBMH_LOCAL_PRESSURE || kind == LBMH_INTERP_PRESSURE) && !(rho > 0))
    return fail(LBMH_E_INVALID, "pressure boundary density must be positive");
  Member& mem = E->members[m];
  const int n[3] = {mem.n[0], mem.n[1], mem.n[2]};
  bool used[kEnsembleWalls] = {};
  for (uint8_t v : mem.h_ids) used[v] = true;
  for (int w = 0; w < kEnsembleWalls; ++w) used[w] = used[w] || mem.id_defined[w];
  used[0] = used[1] = used[2] = true;
  std::map<std::tuple<int, int, int, int>, int> entry_ids;
  std::vector<uint8_t> next = mem.h_ids;
  std::vector<uint32_t> cells, edges, corners, planes;
  uint32_t info[kEnsembleWalls];
  double walls[kEnsembleWalls][4];
  std::memcpy(info, mem.info, sizeof(info));
  int free_id = kEnsembleWalls - 1;
  for (int x = 0; x < n[0]; ++x)
    for (int y = 0; y < n[1]; ++y)
      for (int z = 0; z < n[2]; ++z) {
        const uint32_t c = uint32_t((int64_t(x) * n[1] + y) * n[2] + z);
        if (mem.h_ids[c] != id) continue;
        int type, nrm[3];
        classify_boundary_cell(n, mem.periodic, mem.h_ids.data(), x, y, z, type, nrm);
        const bool flat = type == kTypeFlat && (nrm[0] || nrm[1] || nrm[2]);
        const uint32_t k = local_kind(kind, type, flat);
        if (k == kInvalidKind) {
          return fail(LBMH_E_INVALID, kind == LBMH_LOCAL_PRESSURE ? "local pressure boundary on a non-flat wall cell"
                                                                 : "interpolated boundary on a wall cell without normal");
        }
        int a = nrm[0], b = nrm[1], cc = nrm[2];
        if (k == kOuterEdge || k == kInnerEdge) {
          const int plane = nrm[0] == 0 ? 0 : (nrm[1] == 0 ? 1 : 2);
          a = plane;
          b = nrm[(plane + 1) % 3];
          cc = nrm[(plane + 2) % 3];
        }
        const auto key = std::make_tuple(int(k), a, b, cc);
        auto it = entry_ids.find(key);
        if (it == entry_ids.end()) {
          while (free_id >= 3 && used[free_id]) --free_id;
          if (free_id < 3) return fail(LBMH_E_INVALID, "no free ensemble dynamics ids left (ids 3..63)");
          used[free_id] = true;
          info[free_id] = pack_local_info(k, a, b, cc);
          walls[free_id][0] = rho;
          for (int d = 0; d < 3; ++d) walls[free_id][d + 1] = u[d];
          it = entry_ids.emplace(key, free_id).first;
        }
        next[c] = uint8_t(it->second);
        if (k == kInnerEdge || k == kInnerCorner || k == kDeadWall) cells.push_back(c);
        if (k == kFdVelocity || k == kFdPressure) planes.push_back(c);
        if (k == kOuterEdge) edges.push_back(c);
        if (k == kOuterCorner) corners.push_back(c);
      }
  if (entry_ids.empty()) return LBMH_OK;
  DeviceGuard guard(E->device);
  LBMH_HIP(hipDeviceSynchronize());
  if (kind == LBMH_INTERP_PRESSURE && !planes.empty() && !E->d_plane_scratch) {
    const size_t elem = E->storage == LBMH_F64 ? sizeof(double) : sizeof(float);
    LBMH_HIP(device_alloc(&E->d_plane_scratch, elem * size_t(E->q) * E->boundary_capacity));
  }
  if (kind == LBMH_INTERP_PRESSURE && !planes.empty()) mem.pressure_planes = true;
  for (const auto& kv : entry_ids) {
    const int w = kv.second;
    mem.id_defined[w] = true;
    LBMH_HIP(hipMemcpy(E->d_walls + (size_t(m) * kEnsembleWalls + w) * 4, walls[w], sizeof(walls[w]),
                       hipMemcpyHostToDevice));
  }
  std::memcpy(mem.info, info, sizeof(info));
  mem.h_ids.swap(next);
  mem.local.insert(mem.local.end(), cells.begin(), cells.end());
  mem.edges.insert(mem.edges.end(), edges.begin(), edges.end());
  mem.corners.insert(mem.corners.end(), corners.begin(), corners.end());
  mem.planes.insert(mem.planes.end(), planes.begin(), planes.end());
  LBMH_HIP(hipMemcpy(E->d_info + size_t(m) * kEnsembleWalls, mem.info, sizeof(mem.info), hipMemcpyHostToDevice));
  LBMH_HIP(hipMemcpy(E->d_ids + mem.ids_off, mem.h_ids.data(), mem.ncore, hipMemcpyHostToDevice));
  E->has_local = true;
  return rebuild_lists(E);
}

int lbmh_ensemble_initialize(lbmh_ensemble* E, int m)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  if (!E->n_edges && !E->n_corners && !E->n_planes && !E->n_pplanes) return LBMH_OK;
  DeviceGuard guard(E->device);
  rc = with_types(E, [&](auto qc, auto s) -> int {
    constexpr int Q = decltype(qc)::value;
    using S = decltype(s);
    const EnsembleLimits limits = limits_of(E);
    return launch_post<Q, S>(E, static_cast<EnsembleEntry<Q>*>(E->d_table),
                             reinterpret_cast<const MemberState<Q>*>(device_state(E, 0)), limits, nullptr, m);
  });
  if (rc != LBMH_OK) return rc;
  LBMH_HIP(hipDeviceSynchronize());
  return LBMH_OK;
}

int lbmh_ensemble_set_steps(lbmh_ensemble* E, int m, int64_t steps)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  DeviceGuard guard(E->device);
  rc = pull_state(E);
  if (rc != LBMH_OK) return rc;
  return with_q(E, [&](auto qc) -> int {
    constexpr int Q = decltype(qc)::value;
    MemberState<Q>& st = state<Q>(E, m);
    st.steps_left = steps;
    char* dst = device_state(E, 0, m) + offsetof(MemberState<Q>, steps_left);
    LBMH_HIP(hipMemcpy(dst, &st.steps_left, sizeof(int64_t), hipMemcpyHostToDevice));
    return LBMH_OK;
  });
}

int lbmh_ensemble_status(lbmh_ensemble* E, int m, int64_t* done, int64_t* left)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  DeviceGuard guard(E->device);
  rc = pull_state(E, m);
  if (rc != LBMH_OK) return rc;
  return with_q(E, [&](auto qc) -> int {
    constexpr int Q = decltype(qc)::value;
    const MemberState<Q>& st = state<Q>(E, m);
    if (done) *done = st.steps_done;
    if (left) *left = st.steps_left;
    return LBMH_OK;
  });
}

int lbmh_ensemble_status_all(lbmh_ensemble* E, int64_t* done, int64_t* left)
{
  if (!E || !done || !left) return fail(LBMH_E_INVALID, "null argument");
  DeviceGuard guard(E->device);
  const int rc = pull_state(E);
  if (rc != LBMH_OK) return rc;
  return with_q(E, [&](auto qc) -> int {
    constexpr int Q = decltype(qc)::value;
    for (int m = 0; m < E->max_members; ++m) {
      const MemberState<Q>& st = state<Q>(E, m);
      const bool on = E->members[m].active;
      done[m] = on ? st.steps_done : 0;
      left[m] = on ? st.steps_left : 0;
    }
    return LBMH_OK;
  });
}

int lbmh_ensemble_ini_equilibrium(lbmh_ensemble* E, int m, const double* rho_u)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  if (!rho_u) return fail(LBMH_E_INVALID, "null moments");
  DeviceGuard guard(E->device);
  rc = pull_state(E, m);
  if (rc != LBMH_OK) return rc;
  const Member& mem = E->members[m];
  DeviceBuffer staging;
  const size_t bytes = size_t(4) * mem.ncore * sizeof(double);
  LBMH_HIP(device_alloc(&staging.p, bytes));
  LBMH_HIP(hipMemcpy(staging.p, rho_u, bytes, hipMemcpyHostToDevice));
  const int forced = (E->kind == LBMH_FORCED_BGK || E->kind == LBMH_FORCED_TRT) ? 1 : 0;
  rc = with_types(E, [&](auto qc, auto s) -> int {
    constexpr int Q = decltype(qc)::value;
    using S = decltype(s);
    const EnsembleEntry<Q>& en = entry<Q>(E, m);
    const MemberState<Q>& st = state<Q>(E, m);
    S* pop = static_cast<S*>(en.pop);
    hipLaunchKernelGGL((ini_equilibrium_kernel<Q, S>), dim3(grid_for(mem.ncore, 256)), dim3(256), 0, 0,
                       (const double*)staging.p, E->d_ids + mem.ids_off, pop, geom_of(en), shifts_of(st),
                       mem.params.force[0] * 0.5, mem.params.force[1] * 0.5, mem.params.force[2] * 0.5, forced,
                       nullptr);
    LBMH_HIP(hipGetLastError());
    return LBMH_OK;
  });
  if (rc != LBMH_OK) return rc;
  LBMH_HIP(hipDeviceSynchronize());
  return LBMH_OK;
}

int lbmh_ensemble_upload(lbmh_ensemble* E, int m, const void* host, int dtype)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  if (!host || dtype < LBMH_F64 || dtype > LBMH_F16) return fail(LBMH_E_INVALID, "bad host buffer or dtype");
  DeviceGuard guard(E->device);
  rc = pull_state(E, m);
  if (rc != LBMH_OK) return rc;
  const Member& mem = E->members[m];
  DeviceBuffer staging;
  const size_t bytes = size_t(E->q) * mem.ncore * storage_size(dtype);
  LBMH_HIP(device_alloc(&staging.p, bytes));
  LBMH_HIP(hipMemcpy(staging.p, host, bytes, hipMemcpyHostToDevice));
  rc = with_types(E, [&](auto qc, auto s) -> int {
    constexpr int Q = decltype(qc)::value;
    using S = decltype(s);
    const EnsembleEntry<Q>& en = entry<Q>(E, m);
    const MemberState<Q>& st = state<Q>(E, m);
    S* pop = static_cast<S*>(en.pop);
    const dim3 grid(grid_for(mem.ncore, 256));
    if (dtype == LBMH_F64)
      hipLaunchKernelGGL((scatter_populations<Q, double, S>), grid, dim3(256), 0, 0, (const double*)staging.p, pop, geom_of(en), shifts_of(st));
    else if (dtype == LBMH_F32)
      hipLaunchKernelGGL((scatter_populations<Q, float, S>), grid, dim3(256), 0, 0, (const float*)staging.p, pop, geom_of(en), shifts_of(st));
    else
      hipLaunchKernelGGL((scatter_populations<Q, _Float16, S>), grid, dim3(256), 0, 0, (const _Float16*)staging.p, pop, geom_of(en), shifts_of(st));
    LBMH_HIP(hipGetLastError());
    return LBMH_OK;
  });
  if (rc != LBMH_OK) return rc;
  LBMH_HIP(hipDeviceSynchronize());
  return LBMH_OK;
}

int lbmh_ensemble_download(lbmh_ensemble* E, int m, void* host, int dtype)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  if (!host || dtype < LBMH_F64 || dtype > LBMH_F16) return fail(LBMH_E_INVALID, "bad host buffer or dtype");
  DeviceGuard guard(E->device);
  rc = pull_state(E, m);
  if (rc != LBMH_OK) return rc;
  const Member& mem = E->members[m];
  ResultBuffer staging;
  const size_t bytes = size_t(E->q) * mem.ncore * storage_size(dtype);
  rc = staging.allocate(E->device, bytes);
  if (rc != LBMH_OK) return rc;
  rc = with_types(E, [&](auto qc, auto s) -> int {
    constexpr int Q = decltype(qc)::value;
    using S = decltype(s);
    const EnsembleEntry<Q>& en = entry<Q>(E, m);
    const MemberState<Q>& st = state<Q>(E, m);
    const S* pop = static_cast<const S*>(en.pop);
    const dim3 grid(grid_for(mem.ncore, 256));
    if (dtype == LBMH_F64)
      hipLaunchKernelGGL((gather_populations<Q, double, S>), grid, dim3(256), 0, 0, (double*)staging.p, pop, geom_of(en), shifts_of(st));
    else if (dtype == LBMH_F32)
      hipLaunchKernelGGL((gather_populations<Q, float, S>), grid, dim3(256), 0, 0, (float*)staging.p, pop, geom_of(en), shifts_of(st));
    else
      hipLaunchKernelGGL((gather_populations<Q, _Float16, S>), grid, dim3(256), 0, 0, (_Float16*)staging.p, pop, geom_of(en), shifts_of(st));
    LBMH_HIP(hipGetLastError());
    return LBMH_OK;
  });
  if (rc != LBMH_OK) return rc;
  return staging.to_host(host, bytes);
}

namespace {

// The member as one block for the checkpoint code; its wall table comes from
// the device into `walls`.  Call after pull_state.
int member_block(lbmh_ensemble* E, int m, CheckpointBlock& b, std::vector<double>& walls)
{
  const Member& mem = E->members[m];
  walls.resize(size_t(4) * kEnsembleWalls);
  LBMH_HIP(hipMemcpy(walls.data(), E->d_walls + size_t(m) * 4 * kEnsembleWalls, walls.size() * sizeof(double),
                     hipMemcpyDeviceToHost));
  b.q = E->q;
  b.storage = E->storage;
  b.kind = E->kind;
  for (int d = 0; d < 3; ++d) {
    b.n[d] = mem.n[d];
    b.periodic[d] = mem.periodic[d];
    b.force[d] = mem.params.force[d];
  }
  b.ids = mem.h_ids.data();
  b.walls = walls.data();
  b.info = mem.info;
  b.n_ids = kEnsembleWalls;
  return with_q(E, [&](auto qc) -> int {
    constexpr int Q = decltype(qc)::value;
    const EnsembleEntry<Q>& en = entry<Q>(E, m);
    const MemberState<Q>& st = state<Q>(E, m);
    b.n_padded = en.n_padded;
    b.stride = en.stride;
    b.d_pop = en.pop;
    for (int i = 0; i < Q; ++i) {
      b.shift[i] = st.shift[i];
      b.dist[i] = neighbor_distance<Q>(i, int64_t(en.sx), int64_t(en.sy));
    }
    return LBMH_OK;
  });
}

}  // namespace

int lbmh_ensemble_checkpoint_size(lbmh_ensemble* E, int m, int real, size_t* bytes)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  if (!bytes) return fail(LBMH_E_INVALID, "null argument");
  if (real != LBMH_F64 && real != LBMH_F32) return fail(LBMH_E_INVALID, "checkpoint value type must be F64 or F32");
  DeviceGuard guard(E->device);
  rc = pull_state(E);
  if (rc != LBMH_OK) return rc;
  CheckpointBlock b;
  std::vector<double> walls;
  rc = member_block(E, m, b, walls);
  if (rc != LBMH_OK) return rc;
  *bytes = checkpoint_bytes(b, real);
  return LBMH_OK;
}

int lbmh_ensemble_checkpoint_save(lbmh_ensemble* E, int m, int real, void* buffer, size_t bytes)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  DeviceGuard guard(E->device);
  rc = pull_state(E, m);
  if (rc != LBMH_OK) return rc;
  CheckpointBlock b;
  std::vector<double> walls;
  rc = member_block(E, m, b, walls);
  if (rc != LBMH_OK) return rc;
  return checkpoint_save(b, real, buffer, bytes);
}

int lbmh_ensemble_checkpoint_load(lbmh_ensemble* E, int m, int real, const void* buffer, size_t bytes)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  DeviceGuard guard(E->device);
  rc = pull_state(E);
  if (rc != LBMH_OK) return rc;
  CheckpointBlock b;
  std::vector<double> walls;
  rc = member_block(E, m, b, walls);
  if (rc != LBMH_OK) return rc;
  int64_t shift[27];
  rc = checkpoint_load(b, real, buffer, bytes, shift);
  if (rc != LBMH_OK) return rc;
  // only the member's shifts change in the table
  return with_q(E, [&](auto qc) -> int {
    constexpr int Q = decltype(qc)::value;
    MemberState<Q>& st = state<Q>(E, m);
    for (int i = 0; i < Q; ++i) st.shift[i] = uint32_t(shift[i]);
    char* dst = device_state(E, 0, m) + offsetof(MemberState<Q>, shift);
    LBMH_HIP(hipMemcpy(dst, st.shift, sizeof(st.shift), hipMemcpyHostToDevice));
    return LBMH_OK;
  });
}

int lbmh_ensemble_field_export(lbmh_ensemble* E, int m, int field, int overlap, const double conversion[3],
                               float* host, size_t floats)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  if (!host) return fail(LBMH_E_INVALID, "null argument");
  if (field < LBMH_FIELD_DENSITY || field > LBMH_FIELD_PHYS_PRESSURE) return fail(LBMH_E_INVALID, "unknown field");
  if (overlap < 0 || overlap > 1) return fail(LBMH_E_INVALID, "overlap must be 0 or 1 (the block's padding)");
  if ((field == LBMH_FIELD_PHYS_VELOCITY || field == LBMH_FIELD_PHYS_PRESSURE) && !conversion)
    return fail(LBMH_E_INVALID, "physical fields need the unit conversion factors");
  const Member& mem = E->members[m];
  const uint64_t points = uint64_t(mem.n[0] + 2 * overlap) * (mem.n[1] + 2 * overlap) * (mem.n[2] + 2 * overlap);
  const size_t want = size_t(points) * field_components(field);
  if (floats != want)
    return fail(LBMH_E_INVALID, "field buffer holds " + std::to_string(floats) + " floats, the export " +
                                    std::to_string(want));
  if (points > 0xffffffffull || !field_export_grid_fits(field_export_blocks(mem.n[0], mem.n[1], mem.n[2], overlap)))
    return fail(LBMH_E_INVALID, "member too large for one export (its 32z x 8x tiles exceed 2^32 work-items)");
  DeviceGuard guard(E->device);
  rc = pull_state(E, m);
  if (rc != LBMH_OK) return rc;
  ResultBuffer out;
  rc = out.allocate(E->device, want * sizeof(float));
  if (rc != LBMH_OK) return rc;
  FieldConversion conv{0.0, 0.0, 0.0};
  if (conversion) conv = FieldConversion{conversion[0], conversion[1], conversion[2]};
  const int forced = (E->kind == LBMH_FORCED_BGK || E->kind == LBMH_FORCED_TRT) ? 1 : 0;
  const double* F = mem.params.force;
  rc = with_types(E, [&](auto qc, auto s) -> int {
    constexpr int Q = decltype(qc)::value;
    using S = decltype(s);
    const EnsembleEntry<Q>& en = entry<Q>(E, m);
    const MemberState<Q>& st = state<Q>(E, m);
    PostArgs<Q> a;
    a.pop = static_cast<S*>(en.pop);
    a.stride = en.stride;
    a.n_padded = en.n_padded;
    for (int i = 0; i < Q; ++i) a.shift[i] = st.shift[i];
    a.ids = en.ids;
    a.walls = E->d_walls + size_t(m) * kEnsembleWalls * 4;
    a.info = E->d_info + size_t(m) * kEnsembleWalls;
    a.cells = nullptr;
    a.remote = nullptr;
    a.forced = 0;
    a.force = nullptr;
    a.count = 0;
    a.nx = int(en.nx);
    a.ny = int(en.ny);
    a.nz = int(en.nz);
    a.sx = en.sx;
    a.sy = en.sy;
    a.periodic = en.periodic;
    a.div_z = en.div_z;
    a.div_y = en.div_y;
    a.omega = en.bp.omega;
    hipLaunchKernelGGL((field_export_kernel<Q, S>), dim3(uint32_t(field_export_blocks(a.nx, a.ny, a.nz, overlap))),
                       dim3(kExportTileZ * kExportTileX), 0, 0, a,
                       overlap, field, conv, forced, F[0] * 0.5, F[1] * 0.5, F[2] * 0.5,
                       nullptr, static_cast<float*>(out.p), uint32_t(points));
    LBMH_HIP(hipGetLastError());
    return LBMH_OK;
  });
  if (rc != LBMH_OK) return rc;
  return out.to_host(host, want * sizeof(float));
}

int lbmh_ensemble_moments(lbmh_ensemble* E, int m, double* rho_u)
{
  int rc = check_member(E, m);
  if (rc != LBMH_OK) return rc;
  if (!rho_u) return fail(LBMH_E_INVALID, "null output");
  DeviceGuard guard(E->device);
  rc = pull_state(E, m);
  if (rc != LBMH_OK) return rc;
  const Member& mem = E->members[m];
  ResultBuffer out;
  const size_t bytes = size_t(4) * mem.ncore * sizeof(double);
  rc = out.allocate(E->device, bytes);
  if (rc != LBMH_OK) return rc;
  const int forced = (E->kind == LBMH_FORCED_BGK || E->kind == LBMH_FORCED_TRT) ? 1 : 0;
  rc = with_types(E, [&](auto qc, auto s) -> int {
    constexpr int Q = decltype(qc)::value;
    using S = decltype(s);
    const EnsembleEntry<Q>& en = entry<Q>(E, m);
    const MemberState<Q>& st = state<Q>(E, m);
    const S* pop = static_cast<const S*>(en.pop);
    hipLaunchKernelGGL((moments_kernel<Q, S>), dim3(grid_for(mem.ncore, 256)), dim3(256), 0, 0, (double*)out.p,
                       E->d_ids + mem.ids_off, pop, geom_of(en), shifts_of(st), mem.params.force[0] * 0.5,
                       mem.params.force[1] * 0.5, mem.params.force[2] * 0.5, forced, nullptr);
    LBMH_HIP(hipGetLastError());
    return LBMH_OK;
  });
  if (rc != LBMH_OK) return rc;
  return out.to_host(rho_u, bytes);
}

int lbmh_ensemble_step(lbmh_ensemble* E, int64_t n, void* stream)
{
  if (!E) return fail(LBMH_E_INVALID, "null ensemble");
  if (n < 0) return fail(LBMH_E_INVALID, "negative step count");
  DeviceGuard guard(E->device);
  return launch_steps(E, n, static_cast<hipStream_t>(stream));
}

int lbmh_ensemble_step_graph(lbmh_ensemble* E, int64_t n, void* stream)
{
  if (!E) return fail(LBMH_E_INVALID, "null ensemble");
  if (n < 0) return fail(LBMH_E_INVALID, "negative step count");
  DeviceGuard guard(E->device);
  hipStream_t s = static_cast<hipStream_t>(stream);
  constexpr int64_t kGraphSteps = 32;
  if (n >= kGraphSteps && (!E->graph || E->graph_version != E->version)) {
    if (E->graph) {
      LBMH_HIP(hipGraphExecDestroy(E->graph));
      E->graph = nullptr;
    }
    LBMH_HIP(hipStreamBeginCapture(E->capture_stream, hipStreamCaptureModeThreadLocal));
    const int rc = launch_steps(E, kGraphSteps, E->capture_stream);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(E->capture_stream, &g);
    if (rc != LBMH_OK) {
      if (g) (void)hipGraphDestroy(g);
      return rc;
    }
    if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
    const hipError_t ei = hipGraphInstantiate(&E->graph, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ei != hipSuccess) return hip_fail(ei, "hipGraphInstantiate");
    E->graph_version = E->version;
    E->graph_steps = kGraphSteps;
  }
  int64_t done = 0;
  if (E->graph && E->graph_version == E->version) {
    for (; done + E->graph_steps <= n; done += E->graph_steps) LBMH_HIP(hipGraphLaunch(E->graph, s));
  }
  return launch_steps(E, n - done, s);
}

int lbmh_ensemble_set_launch_config(lbmh_ensemble* E, const lbmh_launch_config* cfg)
{
  if (!E || !cfg) return fail(LBMH_E_INVALID, "null argument");
  if (cfg->lds_bytes < 0 || cfg->lds_bytes > 65536) return fail(LBMH_E_INVALID, "lds_bytes must be in [0, 65536]");
  if (cfg->xcd_group < 0 || cfg->xcd_group > 64) return fail(LBMH_E_INVALID, "xcd_group must be in [0, 64]");
  E->launch = *cfg;
  E->launch_chosen = true;
  E->version += 1;
  return LBMH_OK;
}

int lbmh_ensemble_autotune(lbmh_ensemble* E, int trial_steps, lbmh_launch_config* chosen)
{
  if (!E) return fail(LBMH_E_INVALID, "null ensemble");
  if (trial_steps < 1) return fail(LBMH_E_INVALID, "trial_steps must be >= 1");
  DeviceGuard guard(E->device);
  // The trials run real steps: the members' populations and their
  // states (shifts, step counters) are copied aside first and put back after each
  // candidate, so every candidate times the same members and the ensemble
  // ends as it began.
  uint64_t end = 0;
  for (const Member& m : E->members)
    if (m.active) end = std::max(end, m.pop_off + m.pop_bytes);
  struct Scratch {
    void* pop = nullptr;
    void* state = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    ~Scratch()
    {
      if (pop) (void)hipFree(pop);
      if (state) (void)hipFree(state);
      if (e0) (void)hipEventDestroy(e0);
      if (e1) (void)hipEventDestroy(e1);
    }
  } sc;
  const size_t state_bytes = E->h_state.size();
  LBMH_HIP(hipDeviceSynchronize());
  if (end) {
    const hipError_t e = device_alloc(&sc.pop, end);
    if (e != hipSuccess) return fail(LBMH_E_MEMORY, "autotune needs device memory for a copy of the members' populations");
    LBMH_HIP(hipMemcpy(sc.pop, E->d_pop, end, hipMemcpyDeviceToDevice));
  }
  LBMH_HIP(device_alloc(&sc.state, state_bytes));
  LBMH_HIP(hipMemcpy(sc.state, E->d_state, state_bytes, hipMemcpyDeviceToDevice));
  LBMH_HIP(hipEventCreate(&sc.e0));
  LBMH_HIP(hipEventCreate(&sc.e1));
  auto restore = [&]() -> int {
    LBMH_HIP(hipDeviceSynchronize());
    if (end) LBMH_HIP(hipMemcpy(E->d_pop, sc.pop, end, hipMemcpyDeviceToDevice));
    LBMH_HIP(hipMemcpy(E->d_state, sc.state, state_bytes, hipMemcpyDeviceToDevice));
    return LBMH_OK;
  };
  const lbmh_launch_config before = E->launch;
  const bool before_chosen = E->launch_chosen;
  E->launch_chosen = false;
  const lbmh_launch_config standard = step_launch(E);
  E->launch_chosen = before_chosen;
  const std::vector<lbmh_launch_config> shapes =
      tuning_shapes(step_launch(E), standard, {4, 8, 16, 32}, {0, 16384, 24576, 32768, 40960, 49152}, E->total_chunks);
  lbmh_launch_config best = before;
  const int rc = fastest_shape(shapes, [&](const lbmh_launch_config& shape, float* ms) -> int {
    E->launch = shape;
    E->launch_chosen = true;  // time exactly this shape
    auto timed = [&]() -> int {
      const int rw = launch_steps(E, 1, nullptr);
      if (rw != LBMH_OK) return rw;
      LBMH_HIP(hipEventRecord(sc.e0, nullptr));
      const int rt = launch_steps(E, trial_steps, nullptr);
      if (rt != LBMH_OK) return rt;
      LBMH_HIP(hipEventRecord(sc.e1, nullptr));
      LBMH_HIP(hipEventSynchronize(sc.e1));
      LBMH_HIP(hipEventElapsedTime(ms, sc.e0, sc.e1));
      return LBMH_OK;
    };
    const int rt = timed(), rr = restore();
    return rt != LBMH_OK ? rt : rr;
  }, best);
  if (rc != LBMH_OK) {
    E->launch = before;
    E->launch_chosen = before_chosen;
    E->version += 1;
    return rc;
  }
  E->launch = best;
  E->launch_chosen = true;
  E->version += 1;  // a captured step loop is rebuilt with the chosen shape
  if (chosen) *chosen = best;
  return LBMH_OK;
}

int lbmh_ensemble_usage(const lbmh_ensemble* E, int* members, size_t* cells, size_t* used, size_t* capacity)
{
  if (!E) return fail(LBMH_E_INVALID, "null ensemble");
  int count = 0;
  size_t ncells = 0;
  for (const Member& m : E->members)
    if (m.active) {
      ++count;
      ncells += m.ncore;
    }
  if (members) *members = count;
  if (cells) *cells = ncells;
  if (used) *used = size_t(E->pop_arena.used() + E->id_arena.used());
  if (capacity) *capacity = size_t(E->pop_arena.capacity() + E->id_arena.capacity());
  return LBMH_OK;
}

}  // extern "C"
