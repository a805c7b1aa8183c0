// Permutation bitmap by owners: layers of permutations of degree 3 to 12,
// one launch each, without global atomics on the bitmap.
//
// A claim in the shared bitmap (bitmap_kernels.hip) is a global atomic, and
// those run at 27 G/s on the whole chip whatever their locality (plain
// random loads at 60 to 270 G/s), and push the bitmap's lines out of L2 for
// the loads that share them: 31 G probes/s when half of them claim.  Here
// the bitmap is cut into one slice per workgroup, rank r's bit at position
// r / W of slice r mod W (W prime, so that layers spread evenly).  A launch
// per layer:
//
//   every owner loads its slice into LDS, claims the positions sent to it,
//   appends the new ones to its list (discovery order, each state once per
//   search), stores the slice, and sends the children of the new states to
//   their owners for the next launch.
//
// A message is four bytes: the position in the slice and the parent edge's
// tag (the generator leading back, skipped on expansion); a state is
// rebuilt from its rank when it is expanded.
//
// Whole LRX searches, one shared bitmap -> owners: degree 12 33.0 -> 10.6
// ms, 11 4.77 -> 1.32 ms, 10 2.04 -> 0.48 ms, 9 1.44 -> 0.31 ms, 8 0.77 ->
// 0.23 ms (less by one workgroup, below); [L, X] of degree 10 3.41 -> 0.65 ms.  S_11's
// widest layer (3.05 M states, 6.1 M messages) takes 61 us, 445 VALU
// instructions a state: half of the wave cycles wait at the routing's
// barriers, global traffic (30 MB of messages and states, 10 MB of slices)
// would take 10 us.  Layers below 100 children an owner take 6 to 13 us.
#include <algorithm>
#include "common.hpp"
#include "kernels.hpp"
#include "owner_device.hpp"
#include "rank_device.hpp"

namespace mgbfs {

namespace {

constexpr uint32_t kBlockRunThreads = 1024;
constexpr uint32_t kBlockRunWords = 1264;  // 8! bits, rounded up

__global__ void rank_seed_kernel(RankPlan p, uint64_t start_key, uint32_t* bitmap, uint32_t* list, uint32_t* ends) {
  if (threadIdx.x != 0) return;
  const Place at = place_of(rank_of(bytes_of(start_key)), p.owners, p.magic);
  bitmap[static_cast<uint64_t>(at.owner) * p.slice_words + (at.position >> 5)] = 1u << (at.position & 31u);
  list[static_cast<uint64_t>(at.owner) * p.list_cap] = at.position << 4;
  ends[at.owner] = 1;  // of layer 0; the others are 0
}

// One layer of one owner (see the file header).  claim: messages of this
// layer into the slice and the list; otherwise the layer is in the list
// already and only its children are sent (the start layer, or after a
// message slab was full).  The slice and the routing tile share LDS: two
// workgroups per CU.
__global__ __launch_bounds__(kRouteThreads)
    __attribute__((amdgpu_waves_per_eu(4))) void rank_layer_kernel(RankLayer a, RankGenerators gens) {
  __shared__ alignas(16) char lds[sizeof(TileLds)];
  __shared__ RankGenerator gen[kMaxGenerators];
  __shared__ uint32_t rows, made;
  const RankPlan p = a.plan;
  const uint32_t f = blockIdx.x;
  if (a.claim) {
    const OwnerCtl before = *a.before;
    const uint32_t state = owner_state(before, a.rules);
    const bool run = !before.halt && state == kLayerNext;
    if (f == 0 && threadIdx.x == 0) {
      if (!before.halt) owner_publish(before, state, a.rec, a.seq);
      if (!run) a.now->halt = 1;
      *a.after = OwnerCtl{};
    }
    if (!run) return;
  }
  const uint32_t c = a.claim ? a.in_count[f * p.count_stride] : 0u;
  const uint32_t start = a.ends_before[f];
  uint32_t* list = a.list + static_cast<uint64_t>(f) * p.list_cap;
  if (threadIdx.x == 0) {
    rows = a.claim ? start : a.ends_now[f];
    made = 0;
  }
  __syncthreads();
  if (c)
    rank_claim(lds, &rows, p, a.bitmap + static_cast<uint64_t>(f) * p.slice_words,
               a.in + static_cast<uint64_t>(f) * a.in_cap, c, list);
  const uint32_t end = rows;
  if (threadIdx.x == 0 && a.claim) {
    a.in_count[f * p.count_stride] = 0;
    a.ends_now[f] = end;
  }
  if (end != start) {
    __syncthreads();  // the slice is stored, the list is in place
    for (uint32_t i = threadIdx.x; i < kMaxGenerators * sizeof(RankGenerator) / 4; i += kRouteThreads)
      reinterpret_cast<uint32_t*>(gen)[i] = reinterpret_cast<const uint32_t*>(gens.of)[i];
    const RankOut o{a.out, a.out_count, a.out_cap, a.out_dump, &a.now->spill, 1u, gens.count, a.slots};
    uint32_t mine = wave_incl_scan(rank_send(lds, gen, p, f, list, start, end, o));
    if ((threadIdx.x & (kWave - 1)) == kWave - 1 && mine) atomicAdd(&made, mine);
    __syncthreads();
  }
  if (threadIdx.x == 0 && (end != start || made)) {
    const uint32_t N = a.claim ? end - start : 0u;
    atomicAdd(&a.now->counts, static_cast<unsigned long long>(N) | (static_cast<unsigned long long>(made) << 32));
  }
}

// Small searches by one workgroup: the bitmap (5 KB at degree 8) in LDS, no
// messages, layer after layer in one launch.  Threads take children one each
// while a layer has at most one for every thread, and parents otherwise
// (rebuilt once).  251 owners -> one workgroup, whole searches: LRX 4 54 -> 14
// us, 7 162 -> 38, 8 228 -> 120 (29 layers of 4 us: two dependent LDS steps,
// the list's round trip through L2 and 1.4 parents a thread).
__global__ __launch_bounds__(kBlockRunThreads) void rank_block_kernel(RankBlock a, RankGenerators gens) {
  __shared__ alignas(16) uint32_t bits[kBlockRunWords];
  __shared__ RankGenerator gen[kMaxGenerators];
  __shared__ uint32_t rows;
  const RankPlan p = a.plan;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const unsigned long long began = wall_clock64();
  for (uint32_t i = threadIdx.x; i < p.slice_words; i += kBlockRunThreads) bits[i] = a.bitmap[i];
  for (uint32_t i = threadIdx.x; i < kMaxGenerators * sizeof(RankGenerator) / 4; i += kBlockRunThreads)
    reinterpret_cast<uint32_t*>(gen)[i] = reinterpret_cast<const uint32_t*>(gens.of)[i];
  uint32_t start = a.depth ? a.ends[(a.depth - 1) & 3u] : 0u, end = a.ends[a.depth & 3u];
  if (threadIdx.x == 0) rows = end;
  __syncthreads();
  // Claims a child and appends it (whole waves come here).
  auto claim = [&](bool valid, const Bytes& parent, uint32_t g) {
    const RankGenerator& by = gen[g];
    const uint32_t r = rank_of(child_of(parent, by)), bit = 1u << (r & 31u);
    const bool fresh = valid && !(atomicOr(&bits[r >> 5], bit) & bit);
    const uint64_t b = __ballot(fresh);
    uint32_t at = 0;
    if (lane == 0 && b) at = atomicAdd(&rows, static_cast<uint32_t>(__popcll(b)));
    at = __shfl(at, 0, kWave) + static_cast<uint32_t>(__popcll(b & ((1ull << lane) - 1)));
    if (fresh) a.list[at] = (r << 4) | by.tag;
  };
  uint32_t d = a.depth, run = 0;
  while (d < a.target) {
    const bool all = d == 0 || !a.tagged;
    const uint32_t S = all ? gens.count : gens.count - 1, n = end - start;
    if (n * S <= kBlockRunThreads) {
      if (threadIdx.x / kWave * kWave < n * S) {
        const uint32_t i = min(threadIdx.x, n * S - 1), at = i / S, j = i - at * S;
        const uint32_t m = a.list[start + at], tag = m & 15u;
        const uint32_t g = all ? j : j + (j + 1 >= tag ? 1u : 0u);
        claim(threadIdx.x < n * S && !(all && g + 1 == tag), unrank(m >> 4, p.degree), g);
      }
    } else {
      for (uint32_t i = threadIdx.x; i / kWave * kWave < n; i += kBlockRunThreads) {
        const uint32_t m = a.list[start + min(i, n - 1)], tag = m & 15u;
        const Bytes parent = unrank(m >> 4, p.degree);
        for (uint32_t j = 0; j < S; ++j) {
          const uint32_t g = all ? j : j + (j + 1 >= tag ? 1u : 0u);
          claim(i < n && !(all && g + 1 == tag), parent, g);
        }
      }
    }
    __syncthreads();
    start = end;
    end = rows;
    ++d;
    if (threadIdx.x == 0) {
      a.ends[d & 3u] = end;
      a.sizes[run] = end - start;
    }
    ++run;
    if (end == start) break;
    __syncthreads();  // everyone has read the list's length
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < p.slice_words; i += kBlockRunThreads) a.bitmap[i] = bits[i];
  if (threadIdx.x == 0) {
    a.rec->N = run;
    a.rec->stamps[0] = began;
    a.rec->ticks = wall_clock64();
    __hip_atomic_store(&a.rec->seq, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// States [first, last) of a layer, as packed keys in any order: owner f's
// part of the layer is list rows [lo[f], hi[f]).
__global__ __launch_bounds__(kRouteThreads) void rank_export_kernel(RankPlan p, const uint32_t* list,
                                                                    const uint32_t* lo, const uint32_t* hi,
                                                                    uint64_t limit, uint64_t* keys) {
  __shared__ uint32_t sums[kRouteThreads / kWave];
  const uint32_t f = blockIdx.x;
  uint32_t before = 0;
  for (uint32_t j = threadIdx.x; j < f; j += kRouteThreads) before += hi[j] - lo[j];
  before = wave_incl_scan(before);
  if ((threadIdx.x & (kWave - 1)) == kWave - 1) sums[threadIdx.x / kWave] = before;
  __syncthreads();
  before = 0;
#pragma unroll
  for (uint32_t w = 0; w < kRouteThreads / kWave; ++w) before += sums[w];
  const uint32_t n = hi[f] - lo[f];
  const uint32_t* from = list + static_cast<uint64_t>(f) * p.list_cap + lo[f];
  for (uint32_t i = threadIdx.x; i < n; i += kRouteThreads)
    if (before + i < limit) keys[before + i] = key_of(unrank((from[i] >> 4) * p.owners + f, p.degree));
}

__global__ void rank_report_kernel(const OwnerCtl* ctl, OwnerRules rules, LayerRecord* rec, uint64_t seq) {
  if (threadIdx.x != 0 || ctl->halt) return;
  owner_publish(*ctl, owner_state(*ctl, rules), rec, seq);
}

}  // namespace

hipError_t rank_seed(const RankPlan& p, uint64_t start_key, uint32_t* bitmap, uint32_t* list, uint32_t* ends,
                     hipStream_t stream) {
  hipLaunchKernelGGL(rank_seed_kernel, dim3(1), dim3(64), 0, stream, p, start_key, bitmap, list, ends);
  return hipGetLastError();
}

hipError_t rank_layer(const RankLayer& a, const RankGenerators& gens, hipStream_t stream) {
  const RankPlan& p = a.plan;
  if (p.owners == 0 || p.owners > kOwnersMax || p.degree < 3 || p.degree > kRankDegree || gens.count == 0 ||
      gens.count > kMaxGenerators || a.slots == 0 || a.slots > gens.count || a.slots + 1 < gens.count ||
      p.slice_words % 4 || p.slice_words * 4ull > sizeof(TileLds) || !a.out || a.out_cap == 0 || a.out_cap % 4 ||
      (a.claim && (!a.in || a.in_cap == 0)) || a.in_cap % 4)
    return hipErrorInvalidValue;
  RankLayer b = a;
  b.out_dump = route_dump_index(static_cast<uint64_t>(p.owners) * a.out_cap, kTile);
  hipLaunchKernelGGL(rank_layer_kernel, dim3(p.owners), dim3(kRouteThreads), 0, stream, b, gens);
  return hipGetLastError();
}

hipError_t rank_block(const RankBlock& a, const RankGenerators& gens, hipStream_t stream) {
  const RankPlan& p = a.plan;
  if (p.owners != 1 || p.degree < 3 || p.degree > kRankBlockDegree || p.slice_words > kBlockRunWords ||
      gens.count == 0 || gens.count > kMaxGenerators || a.target <= a.depth || a.target - a.depth > kRankBlockLayers ||
      (a.tagged && gens.count < 2))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(rank_block_kernel, dim3(1), dim3(kBlockRunThreads), 0, stream, a, gens);
  return hipGetLastError();
}

hipError_t rank_export(const RankPlan& p, const uint32_t* list, const uint32_t* lo, const uint32_t* hi, uint64_t limit,
                       uint64_t* keys, hipStream_t stream) {
  hipLaunchKernelGGL(rank_export_kernel, dim3(p.owners), dim3(kRouteThreads), 0, stream, p, list, lo, hi, limit, keys);
  return hipGetLastError();
}

hipError_t rank_report(const OwnerCtl* ctl, const OwnerRules& rules, LayerRecord* rec, uint64_t seq,
                       hipStream_t stream) {
  hipLaunchKernelGGL(rank_report_kernel, dim3(1), dim3(64), 0, stream, ctl, rules, rec, seq);
  return hipGetLastError();
}

RankGenerators rank_generators(const PackedGenerators& gens, const uint8_t* tags) {
  RankGenerators r{};
  r.count = gens.count;
  for (uint32_t g = 0; g < gens.count; ++g) {
    r.of[g].tag = tags[g];
    r.tagged += tags[g] != 0;
    for (uint32_t i = 0; i < kRankDegree; ++i) {
      const uint32_t at = 8 * (i % 4), s = i < gens.degree ? gens.src[g][i] : kRankDegree;
      r.of[g].low[i / 4] |= (s < 8 ? s : kNoByte) << at;
      r.of[g].high[i / 4] |= (s >= 8 && s < kRankDegree ? s - 8 : 4 + i % 4) << at;
    }
  }
  return r;
}

RankPlan rank_plan(uint32_t degree, uint32_t owners) {
  RankPlan p{};
  p.degree = degree;
  // Enough owners that a slice fits LDS and every CU has one (two at degree
  // 11 and 12, where throughput counts); primes, so that rank mod owners
  // spreads whole layers.
  p.owners = owners ? owners : (degree <= 10 ? 251 : (degree == 11 ? 509 : 1021));
  // Message counters apart: next to each other, the reservations of all
  // owners queue on a few cache lines (whole LRX searches, 1 / 8 / 16 / 32
  // words: degree 10 0.67 / 0.59 / 0.51 / 0.48 ms, 11 1.79 / 1.59 / 1.32 /
  // 1.34, 12 10.83 / 10.57 / 11.11 / 11.22, where tiles are many and the
  // lines touched count).
  p.count_stride = degree <= 10 ? 32 : (degree == 11 ? 16 : 8);
  p.magic = p.owners == 1 ? ~0u : static_cast<uint32_t>((1ull << 32) / p.owners);
  const uint64_t positions = (factorial_u64(degree) + p.owners - 1) / p.owners;
  p.slice_words = static_cast<uint32_t>((positions + 127) / 128 * 4);
  p.list_cap = static_cast<uint32_t>(positions);
  return p;
}

}  // namespace mgbfs
