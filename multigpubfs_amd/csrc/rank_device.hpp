// Device code of permutation layers by owners of a bitmap (rank_owner.hip,
// batch_kernels.hip): ranks, children, and the two halves of an owner's
// layer.
#pragma once
#include "common.hpp"
#include "kernels.hpp"
#include "sorted_device.hpp"

namespace mgbfs {

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

// An owner's messages (c of them) into its slice and its list: the new ones
// are appended from `rows` on (LDS, the list's length, set before).  The
// slice is loaded only when enough messages arrive (one per 32-byte sector
// or so); a few go to the bitmap directly.  lds: the routing tile's.
__device__ __forceinline__ void rank_claim(char* lds, uint32_t* rows, const RankPlan& p, uint32_t* slice,
                                           const uint32_t* in, uint32_t c, uint32_t* list) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t start = *rows;
  __syncthreads();
  uint32_t* bits = reinterpret_cast<uint32_t*>(lds);
  const bool staged = c >= p.slice_words / 8;
  if (staged) {
    for (uint32_t i = threadIdx.x; i < p.slice_words / 4; i += kRouteThreads)
      reinterpret_cast<uint4*>(bits)[i] = reinterpret_cast<const uint4*>(slice)[i];
    __syncthreads();
  }
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
    if (lane == 0 && total) at = atomicAdd(rows, total);
    at = __shfl(at, 0, kWave);
    const uint64_t below = (1ull << lane) - 1;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if ((fresh >> j) & 1u) list[at + __popcll(b[j] & below)] = msg[j];
      at += static_cast<uint32_t>(__popcll(b[j]));
    }
  }
  __syncthreads();
  if (staged && *rows != start)
    for (uint32_t i = threadIdx.x; i < p.slice_words / 4; i += kRouteThreads)
      reinterpret_cast<uint4*>(slice)[i] = reinterpret_cast<const uint4*>(bits)[i];
}

// Where an owner's children go.
struct RankOut {
  uint32_t* out;    // owners x cap messages
  uint32_t* count;  // count_stride words apart
  uint32_t cap, dump;
  uint32_t* error;  // err_bit is set when a slab is full
  uint32_t err_bit;
  uint32_t generators, slots;
};

// The children of list rows [start, end) of owner f, end > start, to their
// owners; returns this thread's share of their number.  gen: in LDS, set by
// the caller before (the first barrier here covers it).
//
// A thread rebuilds a parent and makes its children one after the other into
// its kTilePerThread slots.  Where every state but the start carries a tag
// (slots = generators - 1), the generator leading back has no slot: slot j
// takes generator j, or j + 1 from the tag's on, so lanes use different
// generators.  (With a slot per generator and uniform ones, a third of an LRX
// tile was empty.)
__device__ __forceinline__ uint32_t rank_send(char* lds, const RankGenerator* gen, const RankPlan& p, uint32_t f,
                                              const uint32_t* list, uint32_t start, uint32_t end, const RankOut& o) {
  TileLds& t = *reinterpret_cast<TileLds*>(lds);
  const uint32_t S = o.slots;
  const bool all = S == o.generators;
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
      const uint32_t to = static_cast<uint32_t>(v >> 32), off = atomicAdd(&o.count[to * p.count_stride], 1u);
      if (off < o.cap) o.out[static_cast<uint64_t>(to) * o.cap + off] = static_cast<uint32_t>(v);
      else atomicOr(o.error, o.err_bit);
      mine = 1;
    }
  } else {
    clear_tile_counters(t);
    __syncthreads();
    const uint32_t P = kTilePerThread / S * kRouteThreads;  // parents per tile
    const RunCursors runs{o.count, p.count_stride, o.cap, o.error, o.err_bit};
    const uint64_t cap = o.cap;
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
      route_regs(t, v, valid, owner, runs, slab, o.out, o.dump, [] {});
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
      route_regs(t, v, valid, owner, runs, slab, o.out, o.dump, [] {});
      mine += __popc(valid);
    }
  }
  return mine;
}

}  // namespace mgbfs
