// Device helpers of the layers run one launch each by owner workgroups
// (sorted_queue.hip, rank_owner.hip).
#pragma once
#include "common.hpp"
#include "kernels.hpp"

namespace mgbfs {

// Nibble-packed permutations: generators by value, shift groups.
struct NibbleAction {
  PackedGenerators gens;
  __device__ __forceinline__ uint32_t count() const { return gens.count; }
  __device__ __forceinline__ uint64_t child(uint64_t key, uint32_t g) const {
    return apply_groups(key, gens, static_cast<int>(g));
  }
  __device__ __forceinline__ uint32_t mask(uint32_t g) const { return gens.child_mask[g]; }
};

// How a finished layer leaves the session; every workgroup of the next
// launch comes to the same answer from the same totals.
__device__ __forceinline__ uint32_t owner_state(const OwnerCtl& c, const OwnerRules& rules) {
  const uint32_t N = static_cast<uint32_t>(c.counts), children = static_cast<uint32_t>(c.counts >> 32);
  if (c.error || N > rules.rows) return kLayerRejected;
  if (N == 0) return kLayerEmpty;
  const bool few = children < rules.low && !c.imported;
  return c.spill || few || children > rules.high ? kLayerStop : kLayerNext;
}

__device__ __forceinline__ void owner_publish(const OwnerCtl& c, uint32_t state, LayerRecord* rec, uint64_t seq) {
  rec->N = static_cast<uint32_t>(c.counts);
  rec->children = c.counts >> 32;
  rec->unique = c.unique;
  rec->ticks = wall_clock64();
  rec->state = state;
  __hip_atomic_store(&rec->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace mgbfs
