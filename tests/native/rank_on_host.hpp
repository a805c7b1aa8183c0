// The owner bitmap engine (rank_engine.hip) with its kernels restated on the
// host, for checks on a HIP runtime in host memory.
#pragma once
#include <vector>
#include "fake_hip.hpp"
#include "device_cache.hip"
#include "engine.hip"
#include "rank_engine.hip"
// rank_owner.hip for its plans; its wrappers under other names.
#define rank_seed device_rank_seed
#define rank_layer device_rank_layer
#define rank_block device_rank_block
#define rank_export device_rank_export
#define rank_report device_rank_report
#include "rank_owner.hip"
#undef rank_seed
#undef rank_layer
#undef rank_block
#undef rank_export
#undef rank_report

using fake::require;

namespace mgbfs {

hipError_t fill_u32(uint32_t* dst, uint32_t value, uint64_t count, hipStream_t s) {
  require(fake::holds(dst, 4 * count), "fill");
  std::fill(dst, dst + count, value);
  return fake::launch(s);
}
hipError_t zero_u32x3(uint32_t* a, uint64_t na, uint32_t* b, uint64_t nb, uint32_t*, uint64_t, hipStream_t s,
                      unsigned long long*) {
  require(fake::holds(a, 4 * na) && fake::holds(b, 4 * nb), "zero");
  std::fill(a, a + na, 0u);
  std::fill(b, b + nb, 0u);
  return fake::launch(s);
}
hipError_t owner_begin(uint32_t* counts, uint32_t words, OwnerCtl* ctl, uint32_t F, hipStream_t s, LayerRecord*,
                       const LayerCounters*) {
  std::fill(counts, counts + words, 0u);
  ctl[0] = ctl[1] = OwnerCtl{};
  ctl[0].counts = F;
  ctl[0].imported = 1;
  return fake::launch(s);
}
static uint32_t state_of(const OwnerCtl& c) {
  if (c.error) return kLayerRejected;
  if (static_cast<uint32_t>(c.counts) == 0) return kLayerEmpty;
  return c.spill ? kLayerStop : kLayerNext;
}
static void publish(const OwnerCtl& c, LayerRecord* rec, uint64_t seq) {
  rec->N = static_cast<uint32_t>(c.counts);
  rec->state = state_of(c);
  rec->seq = seq;
}
hipError_t rank_seed(const RankPlan& p, uint64_t key, uint32_t* bitmap, uint32_t* list, uint32_t* ends, hipStream_t s) {
  const Place at = place_of(rank_of(bytes_of(key)), p.owners, p.magic);
  bitmap[static_cast<uint64_t>(at.owner) * p.slice_words + (at.position >> 5)] = 1u << (at.position & 31u);
  list[static_cast<uint64_t>(at.owner) * p.list_cap] = at.position << 4;
  ends[at.owner] = 1;
  return fake::launch(s);
}
hipError_t rank_layer(const RankLayer& a, const RankGenerators& gens, hipStream_t s) {
  const RankPlan& p = a.plan;
  const uint64_t W = p.owners;
  require(a.out_cap != 0 && fake::holds(a.out, 4 * W * a.out_cap), "children sent to memory that is not the engine's");
  if (a.claim) {
    require(fake::holds(a.in, 4 * W * a.in_cap), "messages read from memory that is not the engine's");
    const OwnerCtl before = *a.before;
    const bool run = !before.halt && state_of(before) == kLayerNext;
    if (!before.halt) publish(before, a.rec, a.seq);
    if (!run) a.now->halt = 1;
    *a.after = OwnerCtl{};
    if (!run) return fake::launch(s);
  }
  uint64_t N = 0;
  for (uint32_t f = 0; f < W; ++f) {
    uint32_t* list = a.list + f * static_cast<uint64_t>(p.list_cap);
    const uint32_t start = a.ends_before[f];
    uint32_t end = a.claim ? start : a.ends_now[f];
    if (a.claim) {
      uint32_t* slice = a.bitmap + f * static_cast<uint64_t>(p.slice_words);
      for (uint32_t k = 0; k < a.in_count[f * p.count_stride]; ++k) {
        const uint32_t m = a.in[f * static_cast<uint64_t>(a.in_cap) + k], q = m >> 4;
        if ((slice[q >> 5] >> (q & 31u)) & 1u) continue;
        slice[q >> 5] |= 1u << (q & 31u);
        list[end++] = m;
      }
      a.in_count[f * p.count_stride] = 0;
      a.ends_now[f] = end;
      N += end - start;
    }
  }
  for (uint32_t f = 0; f < W; ++f)
    for (uint32_t r = a.ends_before[f]; r < a.ends_now[f]; ++r) {
      const uint32_t m = a.list[f * static_cast<uint64_t>(p.list_cap) + r], tag = m & 15u;
      const Bytes parent = unrank((m >> 4) * p.owners + f, p.degree);
      for (uint32_t g = 0; g < gens.count; ++g) {
        if (g + 1 == tag) continue;
        const Place to = place_of(rank_of(child_of(parent, gens.of[g])), p.owners, p.magic);
        uint32_t& n = a.out_count[to.owner * p.count_stride];
        if (n < a.out_cap) a.out[to.owner * static_cast<uint64_t>(a.out_cap) + n++] = (to.position << 4) | gens.of[g].tag;
        else a.now->spill = 1;
      }
    }
  if (a.claim) a.now->counts += N;
  return fake::launch(s);
}
static uint32_t block_runs;  // searches by one workgroup (not restated)
hipError_t rank_block(const RankBlock& a, const RankGenerators&, hipStream_t s) {
  ++block_runs;
  a.rec->N = 1;
  a.sizes[0] = 0;
  a.rec->seq = a.seq;
  return fake::launch(s);
}
hipError_t rank_report(const OwnerCtl* ctl, const OwnerRules&, LayerRecord* rec, uint64_t seq, hipStream_t s) {
  if (!ctl->halt) publish(*ctl, rec, seq);
  return fake::launch(s);
}
hipError_t rank_export(const RankPlan& p, const uint32_t* list, const uint32_t* lo, const uint32_t* hi, uint64_t limit,
                       uint64_t* keys, hipStream_t s) {
  uint64_t at = 0;
  for (uint32_t f = 0; f < p.owners; ++f)
    for (uint32_t r = lo[f]; r < hi[f] && at < limit; ++r)
      keys[at++] = key_of(unrank((list[f * static_cast<uint64_t>(p.list_cap) + r] >> 4) * p.owners + f, p.degree));
  require(at == limit, "a sample of the layer's size");
  return fake::launch(s);
}

}  // namespace mgbfs

using namespace mgbfs;

// Layer sizes by a plain search over keys.
static std::vector<uint64_t> plain(const Graph& g) {
  const uint32_t n = g.elements;
  std::vector<uint8_t> seen(factorial_u64(n), 0);
  std::vector<uint64_t> layer{g.start_key()}, sizes;
  auto rank = [&](uint64_t key) { return rank_of(bytes_of(key)); };
  seen[rank(layer[0])] = 1;
  while (!layer.empty()) {
    sizes.push_back(layer.size());
    std::vector<uint64_t> next;
    for (uint64_t key : layer)
      for (uint32_t k = 0; k < g.generators; ++k) {
        uint64_t child = 0;
        for (uint32_t i = 0; i < n; ++i) child |= ((key >> (4 * g.perms[k * n + i])) & 15u) << (4 * i);
        if (!seen[rank(child)]) {
          seen[rank(child)] = 1;
          next.push_back(child);
        }
      }
    layer.swap(next);
  }
  return sizes;
}
