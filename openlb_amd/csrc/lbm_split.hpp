// Kernels of a split lattice's time step: every block of a SuperLattice in one
// launch per phase, from tables that hold for the whole call.
//
// The collision of all blocks is the ensemble's step kernel (lbm_ensemble.hpp)
// over a table of the blocks; it also advances the blocks' shifts on the device,
// from one copy of their states to the other, so the following launches need
// nothing from the host.  Each workgroup of the kernels below takes one job: a
// run of entries of one halo, one block's post-processor list, or one halo's
// remote neighbours.  Everything but the entries is then uniform over the
// workgroup and read with scalar loads.
//
// With one launch per block and phase, and the descriptor tables of the halos
// and of each post-processor stage sent from the host in every step, the 101^3
// LocalVelocity cavity on 2x2x2 blocks took 440 us per step; it takes 87 us, of
// which the collision is 42 us, the halos 17 us, and the edge and corner
// processors with their remote neighbours 28 us.
#pragma once

#include "lbm_ensemble.hpp"
#include "lbm_local.hpp"

namespace lbmh {

struct SplitJob {
  uint32_t item;    // index into the kernel's table
  uint32_t first;   // first entry of this workgroup
};

// One halo: the overlap cells of block dst that copy core cells of block src.
struct SplitHalo {
  void* dst;
  const void* src;
  const uint2* pairs;
  uint64_t dst_stride, src_stride;
  uint32_t dst_n, src_n;
  uint32_t dst_block, src_block;
  uint32_t count;
  uint32_t pad_ = 0;  // here and below: no unnamed bytes, the tables are compared whole
};

// The copies of halo_copy_kernel before the streaming: `state` is the copy the
// collision read.  blockIdx.y is the population.
template <int Q, typename S>
__global__ __launch_bounds__(256) void split_halo_kernel(const SplitHalo* __restrict__ halos,
                                                         const MemberState<Q>* __restrict__ state,
                                                         const SplitJob* __restrict__ jobs)
{
  const SplitJob job = jobs[blockIdx.x];
  const SplitHalo& h = halos[job.item];
  const uint32_t i = blockIdx.y, k = job.first + threadIdx.x;
  if (k >= h.count) return;
  const uint2 p = h.pairs[k];
  S* dst = static_cast<S*>(h.dst) + uint64_t(i) * h.dst_stride;
  const S* src = static_cast<const S*>(h.src) + uint64_t(i) * h.src_stride;
  dst[wrap_index(p.x, state[h.dst_block].shift[i], h.dst_n)] = src[wrap_index(p.y, state[h.src_block].shift[i], h.src_n)];
}

// A block's momenta evaluation, read through the shifts of its state.
template <int Q>
struct SplitPost {
  PostArgs<Q> a;
  uint32_t block;
  uint32_t pad_ = 0;
};

template <int Q>
__device__ __forceinline__ PostArgs<Q> split_post_args(const SplitPost<Q>& s, const MemberState<Q>* state)
{
  PostArgs<Q> a = s.a;
#pragma unroll
  for (int i = 0; i < Q; ++i) a.shift[i] = state[s.block].shift[i];
  return a;
}

// One post-processor kind (outer_post_kernel) of all blocks after the
// streaming: `state` is the copy the collision wrote.
template <int Q, typename S, int KIND>
__global__ __launch_bounds__(64) void split_post_kernel(const SplitPost<Q>* __restrict__ posts,
                                                        const MemberState<Q>* __restrict__ state,
                                                        const SplitJob* __restrict__ jobs)
{
  const SplitJob job = jobs[blockIdx.x];
  const PostArgs<Q> a = split_post_args<Q>(posts[job.item], state);
  outer_post_cells<Q, S, KIND>(a, job.first);
}

// The remote neighbours of one halo that a post-processor stage reads.
template <int Q>
struct SplitRemote {
  SplitPost<Q> src;
  const RemotePair* pairs;
  void* out;
  uint32_t count;
  uint32_t pad_ = 0;
};

template <int Q, typename S>
__global__ __launch_bounds__(64) void split_remote_kernel(const SplitRemote<Q>* __restrict__ remotes,
                                                          const MemberState<Q>* __restrict__ state,
                                                          const SplitJob* __restrict__ jobs)
{
  const SplitJob job = jobs[blockIdx.x];
  const SplitRemote<Q>& d = remotes[job.item];
  const uint32_t k = job.first + threadIdx.x;
  if (k >= d.count) return;
  const PostArgs<Q> a = split_post_args<Q>(d.src, state);
  remote_moments<Q, S>(a, d.pairs[k], d.out);
}

}  // namespace lbmh
