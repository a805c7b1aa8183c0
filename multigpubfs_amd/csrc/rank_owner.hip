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
// 0.23 ms, 3 0.16 -> 0.03 ms; [L, X] of degree 10 3.41 -> 0.65 ms.  S_11's
// widest layer (3.05 M states, 6.1 M messages) takes 61 us, 445 VALU
// instructions a state: half of the wave cycles wait at the routing's
// barriers, global traffic (30 MB of messages and states, 10 MB of slices)
// would take 10 us.  Layers below 100 children an owner take 6 to 13 us.
#include <algorithm>
#include "common.hpp"
#include "kernels.hpp"
#include "owner_device.hpp"
#include "sorted_device.hpp"

namespace mgbfs {

namespace {

// A permutation of 0..n-1, n <= 12, as bytes (0 past n).
struct Bytes {
  uint32_t w[3];
};

// Bytes of (hi, lo) by selector: byte j of the result is byte sel_j of the
// eight (0 to 3 from lo), 0 for kNoByte.
constexpr uint32_t kNoByte = 0x0cu;
__host__ __device__ __forceinline__ uint32_t pick_bytes(uint32_t hi, uint32_t lo, uint32_t sel) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_perm(hi, lo, sel);
#else
  const uint64_t x = (static_cast<uint64_t>(hi) << 32) | lo;
  uint32_t r = 0;
  for (uint32_t j = 0; j < 4; ++j) {
    const uint32_t s = (sel >> (8 * j)) & 255u;
    if (s < 8) r |= (static_cast<uint32_t>(x >> (8 * s)) & 255u) << (8 * j);
  }
  return r;
#endif
}

// Child bytes i = parent byte src[i]: word j of the child picks from words 0
// and 1, then from word 2 and that (six byte permutes, whatever the
// generator, so every lane may use another one).
__host__ __device__ __forceinline__ Bytes child_of(const Bytes& p, const RankGenerator& g) {
  Bytes c;
#pragma unroll
  for (int j = 0; j < 3; ++j) c.w[j] = pick_bytes(pick_bytes(p.w[1], p.w[0], g.low[j]), p.w[2], g.high[j]);
  return c;
}

__host__ __device__ constexpr uint32_t rank_factorial(uint32_t n) { return n < 2 ? 1u : n * rank_factorial(n - 1); }

// Rank of a permutation: the sum of i! times the number of smaller symbols
// before position i.  The weights don't depend on the degree and the bytes
// past it add nothing.  24-bit products (full rate) up to position 10;
// position 11 joins it in one factor.
__host__ __device__ __forceinline__ uint32_t rank_of(const Bytes& p) {
  uint32_t seen = 0, r = 0, below = 0;
#pragma unroll
  for (uint32_t i = 0; i < kRankDegree; ++i) {
    const uint32_t s = (p.w[i / 4] >> (8 * (i % 4))) & 255u;
    const uint32_t under = seen & ((1u << s) - 1u);
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t d = static_cast<uint32_t>(__popc(under));
#else
    const uint32_t d = static_cast<uint32_t>(__builtin_popcount(under));
#endif
    seen |= 1u << s;
    if (i < 10) r += d * rank_factorial(i);
    else if (i == 10) below = d;
    else r += (below + 11u * d) * rank_factorial(10);
  }
  return r;
}

// floor(x / d) by a 24-bit product, exact for the x < 11,880 and x < 40,320
// that occur (shown for all of them in rank_check.cpp).
template <uint32_t D>
__host__ __device__ __forceinline__ uint32_t quotient(uint32_t x) {
  constexpr uint32_t kShift = D >= 9 ? 17 : 18;
  constexpr uint32_t kMagic = ((1u << kShift) + D - 1) / D;
  return D == 2 ? x >> 1 : (x * kMagic) >> kShift;
}

// Its inverse: the digits 8 to 11 from the quotient by 8!, the others from
// the remainder; then from the last position down, each digit picks out of
// the ascending list of symbols left (four words' worth while more than
// eight are left).
__host__ __device__ __forceinline__ Bytes unrank(uint32_t r, uint32_t n) {
  uint32_t d[kRankDegree] = {};
  uint32_t hi = r / rank_factorial(8), lo = r - hi * rank_factorial(8), q;
  q = quotient<2>(lo), d[1] = lo - 2 * q, lo = q;
  q = quotient<3>(lo), d[2] = lo - 3 * q, lo = q;
  q = quotient<4>(lo), d[3] = lo - 4 * q, lo = q;
  q = quotient<5>(lo), d[4] = lo - 5 * q, lo = q;
  q = quotient<6>(lo), d[5] = lo - 6 * q, lo = q;
  q = quotient<7>(lo), d[6] = lo - 7 * q, d[7] = q;
  q = quotient<9>(hi), d[8] = hi - 9 * q, hi = q;
  q = quotient<10>(hi), d[9] = hi - 10 * q, hi = q;
  q = quotient<11>(hi), d[10] = hi - 11 * q, d[11] = q;
  Bytes p{};
  uint64_t left = 0xba9876543210ull;
#pragma unroll
  for (uint32_t i = 11; i >= 8; --i)
    if (i < n) {
      const uint64_t above = ~0ull << (4 * d[i]);
      p.w[2] |= (static_cast<uint32_t>(left >> (4 * d[i])) & 15u) << (8 * (i - 8));
      left = (left & ~above) | ((left >> 4) & above);
    }
  uint32_t few = static_cast<uint32_t>(left);
#pragma unroll
  for (uint32_t i = 7; i < 8; --i)
    if (i < n) {
      const uint32_t above = ~0u << (4 * d[i]);
      p.w[i / 4] |= ((few >> (4 * d[i])) & 15u) << (8 * (i % 4));
      few = (few & ~above) | ((few >> 4) & above);
    }
  return p;
}

__host__ __device__ __forceinline__ Bytes bytes_of(uint64_t key) {
  Bytes p{};
#pragma unroll
  for (uint32_t i = 0; i < kRankDegree; ++i) p.w[i / 4] |= (static_cast<uint32_t>(key >> (4 * i)) & 15u) << (8 * (i % 4));
  return p;
}

__host__ __device__ __forceinline__ uint64_t key_of(const Bytes& p) {
  uint64_t key = 0;
#pragma unroll
  for (uint32_t i = 0; i < kRankDegree; ++i)
    key |= static_cast<uint64_t>((p.w[i / 4] >> (8 * (i % 4))) & 15u) << (4 * i);
  return key;
}

// Owners with at most this many children send each by itself (a slot of the
// receiver by a global atomic), others through a routing tile.
constexpr uint32_t kDirectChildren = 128;
constexpr int kSmallItems = 4;  // children per thread of a small routing tile

struct Place {
  uint32_t owner, position;
};
__host__ __device__ __forceinline__ Place place_of(uint32_t rank, uint32_t owners, uint32_t magic) {
  // Exact or one less (wide.hpp: mod32).
  uint32_t q = static_cast<uint32_t>((static_cast<uint64_t>(rank) * magic) >> 32);
  uint32_t f = rank - q * owners;
  if (f >= owners) {
    f -= owners;
    ++q;
  }
  return Place{f, q};
}

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
// message slab was full).  A slice is loaded only when enough messages
// arrive (one per 32-byte sector or so); a few go to the bitmap directly.
// The slice and the routing tile share LDS: two workgroups per CU.
//
// Expansion: a thread rebuilds a parent and makes its children one after
// the other into its kTilePerThread slots.  Where every state but the start
// carries a tag (a.slots = generators - 1), the generator leading back has
// no slot: slot j takes generator j, or j + 1 from the tag's on, so lanes
// use different generators.  (With a slot per generator and uniform ones, a
// third of an LRX tile was empty.)
__global__ __launch_bounds__(kRouteThreads) __attribute__((amdgpu_waves_per_eu(4))) void rank_layer_kernel(RankLayer a, RankGenerators gens) {
  __shared__ alignas(16) char lds[sizeof(TileLds)];
  __shared__ RankGenerator gen[kMaxGenerators];
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
  const uint32_t c = a.claim ? a.in_count[f * p.count_stride] : 0u;
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
    a.in_count[f * p.count_stride] = 0;
    a.ends_now[f] = end;
  }
  if (end != start) {
    __syncthreads();  // the slice is stored, the list is in place
    TileLds& t = *reinterpret_cast<TileLds*>(lds);
    for (uint32_t i = threadIdx.x; i < kMaxGenerators * sizeof(RankGenerator) / 4; i += kRouteThreads)
      reinterpret_cast<uint32_t*>(gen)[i] = reinterpret_cast<const uint32_t*>(gens.of)[i];
    const uint32_t S = a.slots;
    const bool all = S == gens.count;
    uint32_t mine = 0;
    // Child i of the parents from row p0 on, with its owner in the high word;
    // false: the edge back to where its parent came from.
    auto child_at = [&](uint32_t p0, uint32_t i, uint64_t& v) {
      const uint32_t at = i / S, j = i - at * S, m = list[p0 + at], tag = m & 15u;
      const uint32_t g = all ? j : j + (j + 1 >= tag ? 1u : 0u);
      const RankGenerator& by = gen[g];
      const Place to = place_of(rank_of(child_of(unrank((m >> 4) * p.owners + f, p.degree), by)), p.owners, p.magic);
      v = (static_cast<uint64_t>(to.owner) << 32) | (to.position << 4) | by.tag;
      return !(all && g + 1 == tag);
    };
    if ((end - start) * S <= kDirectChildren) {
      __syncthreads();
      uint64_t v;
      if (threadIdx.x < (end - start) * S && child_at(start, threadIdx.x, v)) {
        const uint32_t to = static_cast<uint32_t>(v >> 32), off = atomicAdd(&a.out_count[to * p.count_stride], 1u);
        if (off < a.out_cap) a.out[to * a.out_cap + off] = static_cast<uint32_t>(v);
        else atomicOr(&a.now->spill, 1u);
        mine = 1;
      }
    } else {
      clear_tile_counters(t);
      __syncthreads();
      const uint32_t P = kTilePerThread / S * kRouteThreads;  // parents per tile
      const RunCursors runs{a.out_count, p.count_stride, a.out_cap, &a.now->spill, 1u};
      const uint64_t cap = a.out_cap;
      // (Masked: rows past a tile's end hold words of another kind.)
      auto owner = [](uint64_t h) { return static_cast<uint32_t>(h >> 32) & ((1u << kMaxPassBits) - 1u); };
      auto slab = [cap](uint32_t b) { return b * cap; };
      uint32_t p0 = start;
      for (; (end - p0) * S > kSmallItems * kRouteThreads; p0 += min(P, end - p0)) {
        uint64_t v[kTilePerThread];
        uint32_t valid = 0, j = 0, at = p0 + threadIdx.x, tag = 0;
        Bytes parent{};
#pragma unroll
        for (int k = 0; k < kTilePerThread; ++k) {
          v[k] = 0;
          if (static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(at)) < end && k < P / kRouteThreads * S) {  // uniform
            if (j == 0) {  // uniform: the next parent
              const uint32_t m = at < end ? list[at] : 0u;
              tag = m & 15u;
              parent = unrank((m >> 4) * p.owners + f, p.degree);
            }
            const uint32_t g = all ? j : j + (j + 1 >= tag ? 1u : 0u);
            if (at < end && !(all && g + 1 == tag)) valid |= 1u << k;
            const RankGenerator& by = gen[g];
            const Place to = place_of(rank_of(child_of(parent, by)), p.owners, p.magic);
            v[k] = (static_cast<uint64_t>(to.owner) << 32) | (to.position << 4) | by.tag;
            if (++j == S) {
              j = 0;
              at += kRouteThreads;
            }
          }
          // One child after the other: left free, the scheduler brings every
          // generator's words in at once and spills.
          asm volatile("" : "+v"(v[k]) : : "memory");
        }
        route_regs(t, v, valid, owner, runs, slab, a.out, a.out_dump, [] {});
        mine += __popc(valid);
      }
      if (p0 < end) {  // a small tile: one child per slot
        const uint32_t n = (end - p0) * S;
        uint64_t v[kSmallItems];
        uint32_t valid = 0;
#pragma unroll
        for (int k = 0; k < kSmallItems; ++k) {
          const uint32_t i = k * kRouteThreads + threadIdx.x;
          v[k] = 0;
          if (i < n && child_at(p0, i, v[k])) valid |= 1u << k;
          asm volatile("" : "+v"(v[k]) : : "memory");
        }
        route_regs(t, v, valid, owner, runs, slab, a.out, a.out_dump, [] {});
        mine += __popc(valid);
      }
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
      p.slice_words % 4 || p.slice_words * 4ull > sizeof(TileLds) || a.out_cap % 4 || a.in_cap % 4)
    return hipErrorInvalidValue;
  RankLayer b = a;
  b.out_dump = route_dump_index(static_cast<uint64_t>(p.owners) * a.out_cap, kTile);
  hipLaunchKernelGGL(rank_layer_kernel, dim3(p.owners), dim3(kRouteThreads), 0, stream, b, gens);
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

RankGenerators rank_generators(const PackedGenerators& gens) {
  RankGenerators r{};
  r.count = gens.count;
  for (uint32_t g = 0; g < gens.count; ++g) {
    r.of[g].tag = gens.child_tag[g];
    r.tagged += gens.child_tag[g] != 0;
    for (uint32_t i = 0; i < kRankDegree; ++i) {
      const uint32_t at = 8 * (i % 4), s = i < gens.degree ? gens.src[g][i] : kRankDegree;
      r.of[g].low[i / 4] |= (s < 8 ? s : kNoByte) << at;
      r.of[g].high[i / 4] |= (s >= 8 && s < kRankDegree ? s - 8 : 4 + i % 4) << at;
    }
  }
  return r;
}

RankPlan rank_plan(uint32_t degree) {
  RankPlan p{};
  p.degree = degree;
  // Enough owners that a slice fits LDS and every CU has one (two at degree
  // 11 and 12, where throughput counts); primes, so that rank mod owners
  // spreads whole layers.
  p.owners = degree <= 10 ? 251 : (degree == 11 ? 509 : 1021);
  // Message counters apart: next to each other, the reservations of all
  // owners queue on a few cache lines (whole LRX searches, 1 / 8 / 16 / 32
  // words: degree 10 0.67 / 0.59 / 0.51 / 0.48 ms, 11 1.79 / 1.59 / 1.32 /
  // 1.34, 12 10.83 / 10.57 / 11.11 / 11.22, where tiles are many and the
  // lines touched count).
  p.count_stride = degree <= 10 ? 32 : (degree == 11 ? 16 : 8);
  p.magic = static_cast<uint32_t>((1ull << 32) / p.owners);
  const uint64_t positions = (factorial_u64(degree) + p.owners - 1) / p.owners;
  p.slice_words = static_cast<uint32_t>((positions + 127) / 128 * 4);
  p.list_cap = static_cast<uint32_t>(positions);
  return p;
}

}  // namespace mgbfs
