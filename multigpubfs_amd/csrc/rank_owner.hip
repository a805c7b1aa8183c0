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
// Whole LRX searches, one shared bitmap -> owners: degree 12 33.0 -> 21.0
// ms, 11 4.77 -> 2.73 ms, 10 2.04 -> 0.81 ms, 9 1.44 -> 0.53 ms, 8 0.77 ->
// 0.34 ms, 3 0.16 -> 0.04 ms; [L, X] of degree 10 3.44 -> 1.08 ms.  S_11's
// widest layer (3.05 M states, 6.1 M messages) takes 166 us: 711 VALU
// instructions a state are a third of that, and the routing's barriers at
// four waves a SIMD most of the rest (64% of wave cycles wait); global
// traffic (30 MB of messages, 10 MB of slices) would take 10 us.
#include <algorithm>
#include "common.hpp"
#include "kernels.hpp"
#include "owner_device.hpp"
#include "sorted_device.hpp"

namespace mgbfs {

namespace {

constexpr int kRankItems = 8;  // child slots per thread and tile

// Lexicographic rank of a nibble-packed permutation of 0..n-1, n <= 12.
__host__ __device__ __forceinline__ uint32_t rank_of(uint64_t key, uint32_t n) {
  uint32_t seen = 0, r = 0;
#pragma unroll
  for (uint32_t i = 0; i < kRankDegree; ++i)
    if (i < n) {
      const uint32_t s = nib(key, i);
#if defined(__HIP_DEVICE_COMPILE__)
      const uint32_t below = static_cast<uint32_t>(__popc(seen & ((1u << s) - 1u)));
#else
      const uint32_t below = static_cast<uint32_t>(__builtin_popcount(seen & ((1u << s) - 1u)));
#endif
      seen |= 1u << s;
      r = r * (n - i) + s - below;
    }
  return r;
}

// Its inverse: digits by division (radix 2 up to n, constants once
// unrolled), symbols picked out of the packed list of unused ones.
__host__ __device__ __forceinline__ uint64_t unrank(uint32_t r, uint32_t n) {
  uint32_t digit[kRankDegree] = {};
#pragma unroll
  for (uint32_t radix = 2; radix <= kRankDegree; ++radix)
    if (radix <= n) {
      digit[radix - 1] = r % radix;  // of position n - radix
      r /= radix;
    }
  uint64_t unused = 0xba9876543210ull, key = 0;
#pragma unroll
  for (uint32_t radix = kRankDegree; radix >= 1; --radix)
    if (radix <= n) {
      const uint32_t at = 4 * digit[radix - 1];
      const uint64_t low = (1ull << at) - 1;
      key |= ((unused >> at) & 15u) << (4 * (n - radix));
      unused = (unused & low) | ((unused >> 4) & ~low);
    }
  return key;
}

struct Place {
  uint32_t owner, position;
};
__host__ __device__ __forceinline__ Place place_of(uint32_t rank, uint32_t owners, uint32_t magic) {
  uint32_t q = static_cast<uint32_t>((static_cast<uint64_t>(rank) * magic) >> 32);  // exact or one less (wide.hpp: mod32)
  uint32_t f = rank - q * owners;
  if (f >= owners) {
    f -= owners;
    ++q;
  }
  return Place{f, q};
}

__global__ void rank_seed_kernel(RankPlan p, uint64_t start_key, uint32_t* bitmap, uint32_t* list, uint32_t* ends) {
  if (threadIdx.x != 0) return;
  const Place at = place_of(rank_of(start_key, p.degree), p.owners, p.magic);
  bitmap[static_cast<uint64_t>(at.owner) * p.slice_words + (at.position >> 5)] = 1u << (at.position & 31u);
  list[static_cast<uint64_t>(at.owner) * p.list_cap] = at.position << 4;
  ends[at.owner] = 1;  // of layer 0; the others are 0
}

// One layer of one owner (see the file header).  claim: messages of this
// layer into the slice and the list; otherwise the layer is in the list
// already and only its children are sent (the start layer, or after a
// message slab was full).  A slice is loaded only when enough messages
// arrive (one per 32-byte sector or so); a few go to the bitmap directly.
// The slice and the routing tile share LDS: two workgroups per CU.
__global__ __launch_bounds__(kRouteThreads) void rank_layer_kernel(RankLayer a, NibbleAction act) {
  __shared__ alignas(16) char lds[sizeof(TileLds)];
  __shared__ uint32_t rows, made;
  const RankPlan p = a.plan;
  const uint32_t f = blockIdx.x;
  const uint32_t lane = threadIdx.x & (kWave - 1);
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
  const uint32_t c = a.claim ? a.in_count[f] : 0u;
  const uint32_t start = a.ends_before[f];
  uint32_t* list = a.list + static_cast<uint64_t>(f) * p.list_cap;
  if (threadIdx.x == 0) {
    rows = a.claim ? start : a.ends_now[f];
    made = 0;
  }
  __syncthreads();
  if (c) {
    uint32_t* slice = a.bitmap + static_cast<uint64_t>(f) * p.slice_words;
    uint32_t* bits = reinterpret_cast<uint32_t*>(lds);
    const bool staged = c >= p.slice_words / 8;
    if (staged) {
      for (uint32_t i = threadIdx.x; i < p.slice_words / 4; i += kRouteThreads)
        reinterpret_cast<uint4*>(bits)[i] = reinterpret_cast<const uint4*>(slice)[i];
      __syncthreads();
    }
    const uint32_t* in = a.in + static_cast<uint64_t>(f) * a.in_cap;
    const uint32_t rounds = (c + 4 * kRouteThreads - 1) / (4 * kRouteThreads);
    for (uint32_t k = 0; k < rounds; ++k) {
      const uint32_t i = 4 * (k * kRouteThreads + threadIdx.x);
      uint4 m = make_uint4(0, 0, 0, 0);
      if (i < c) m = reinterpret_cast<const uint4*>(in)[i / 4];
      const uint32_t msg[4] = {m.x, m.y, m.z, m.w};
      uint32_t fresh = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (i + j < c) {
          const uint32_t q = msg[j] >> 4, bit = 1u << (q & 31u);
          const uint32_t old = staged ? atomicOr(&bits[q >> 5], bit)
                                      : __hip_atomic_fetch_or(&slice[q >> 5], bit, __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_WORKGROUP);
          if (!(old & bit)) fresh |= 1u << j;
        }
      uint64_t b[4];
      uint32_t total = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        b[j] = __ballot((fresh >> j) & 1u);
        total += static_cast<uint32_t>(__popcll(b[j]));
      }
      uint32_t at = 0;
      if (lane == 0 && total) at = atomicAdd(&rows, total);
      at = __shfl(at, 0, kWave);
      const uint64_t below = (1ull << lane) - 1;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if ((fresh >> j) & 1u) list[at + __popcll(b[j] & below)] = msg[j];
        at += static_cast<uint32_t>(__popcll(b[j]));
      }
    }
    __syncthreads();
    if (staged && rows != start)
      for (uint32_t i = threadIdx.x; i < p.slice_words / 4; i += kRouteThreads)
        reinterpret_cast<uint4*>(slice)[i] = reinterpret_cast<const uint4*>(bits)[i];
  }
  const uint32_t end = rows;
  if (threadIdx.x == 0 && a.claim) {
    a.in_count[f] = 0;
    a.ends_now[f] = end;
  }
  if (end != start) {
    __syncthreads();  // the slice is stored, the list is in place
    TileLds& t = *reinterpret_cast<TileLds*>(lds);
    clear_tile_counters(t);
    __syncthreads();
    const uint32_t G = act.count();
    const uint32_t P = kRankItems * kRouteThreads / G / kWave * kWave;
    const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(threadIdx.x)) / kWave;
    const RunCursors runs{a.out_count, 1, a.out_cap, &a.now->spill, 1u};
    const uint64_t cap = a.out_cap;
    uint32_t mine = 0;
    for (uint32_t p0 = start; p0 < end; p0 += P) {
      // The tile's parents are rebuilt once, into the LDS words that the
      // routing places children in only after they have been read.
      const uint32_t count = min(P, end - p0), padded = (count + kWave - 1) / kWave * kWave;
      __syncthreads();
      for (uint32_t i = threadIdx.x; i < count; i += kRouteThreads) {
        const uint32_t m = list[p0 + i];
        t.s[i] = unrank((m >> 4) * p.owners + f, p.degree) | (static_cast<uint64_t>(m & 15u) << 60);
      }
      __syncthreads();
      uint64_t v[kRankItems];
      uint32_t valid = 0;
#pragma unroll
      for (int k = 0; k < kRankItems; ++k) {
        const uint32_t s = (k * (kRouteThreads / kWave) + wave) * kWave;  // the wave's first slot
        const uint32_t g = s / padded, m = s - g * padded + lane;
        v[k] = 0;
        if (g < G) {  // uniform
          const uint64_t h = t.s[m < count ? m : 0u];
          if (m < count && static_cast<uint32_t>(h >> 60) != g + 1) valid |= 1u << k;
          const Place to = place_of(rank_of(act.child(h & ((1ull << 60) - 1), g), p.degree), p.owners, p.magic);
          v[k] = (static_cast<uint64_t>(to.owner) << 32) | (to.position << 4) | act.gens.child_tag[g];
        }
      }
      // (Masked: rows past the tile's end hold words of another kind.)
      route_regs(t, v, valid, [](uint64_t h) { return static_cast<uint32_t>(h >> 32) & ((1u << kMaxPassBits) - 1u); }, runs,
                 [cap](uint32_t b) { return b * cap; }, a.out, a.out_dump, [] {});
      mine += __popc(valid);
    }
    mine = wave_incl_scan(mine);
    if (lane == kWave - 1 && mine) atomicAdd(&made, mine);
    __syncthreads();
  }
  if (threadIdx.x == 0 && (end != start || made)) {
    const uint32_t N = a.claim ? end - start : 0u;
    atomicAdd(&a.now->counts, static_cast<unsigned long long>(N) | (static_cast<unsigned long long>(made) << 32));
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
    if (before + i < limit) keys[before + i] = unrank((from[i] >> 4) * p.owners + f, p.degree);
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

hipError_t rank_layer(const RankLayer& a, const PackedGenerators& gens, hipStream_t stream) {
  const RankPlan& p = a.plan;
  if (p.owners == 0 || p.owners > kOwnersMax || p.degree < 3 || p.degree > kRankDegree || gens.count == 0 ||
      gens.count > kMaxGenerators || p.slice_words % 4 || p.slice_words * 4ull > sizeof(TileLds) || a.out_cap % 4 ||
      a.in_cap % 4)
    return hipErrorInvalidValue;
  RankLayer b = a;
  b.out_dump = route_dump_index(static_cast<uint64_t>(p.owners) * a.out_cap, kTile);
  hipLaunchKernelGGL(rank_layer_kernel, dim3(p.owners), dim3(kRouteThreads), 0, stream, b, NibbleAction{gens});
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

RankPlan rank_plan(uint32_t degree) {
  RankPlan p{};
  p.degree = degree;
  // Enough owners that a slice fits LDS and every CU has one (two at degree
  // 11 and 12, where throughput counts); primes, so that rank mod owners
  // spreads whole layers.
  p.owners = degree <= 10 ? 251 : (degree == 11 ? 509 : 1021);
  p.magic = static_cast<uint32_t>((1ull << 32) / p.owners);
  const uint64_t positions = (factorial_u64(degree) + p.owners - 1) / p.owners;
  p.slice_words = static_cast<uint32_t>((positions + 127) / 128 * 4);
  p.list_cap = static_cast<uint32_t>(positions);
  return p;
}

}  // namespace mgbfs
