// Device machinery of the sorted backend shared by its layer kernels
// (sorted_kernels.hip) and its queued layers (sorted_queue.hip): bucket
// arithmetic, the LDS routing tile and the stored-value layout.
#pragma once
#include "common.hpp"
#include "kernels.hpp"

namespace mgbfs {

constexpr int kRouteThreads = 512;
constexpr int kTile = 8192;                            // elements per LDS routing tile
constexpr int kTilePerThread = kTile / kRouteThreads;  // 16 elements held in registers
static_assert(kRouteDump >= kTile, "a dropped run fits the dump area");

constexpr uint64_t kEmpty = ~0ull;  // never a stored value: tag bit tagbits-2 stays clear

// Index of h among n equal ranges of its top 32 bits: floor(top32 * n / 2^32).
// Monotone in h, so a bank ordered by its top bits is ordered by any such
// index, and with n' = n << b every range of n' nests in one range of n.
__device__ __forceinline__ uint32_t range_index(uint64_t h, uint32_t n) {
  return __umulhi(static_cast<uint32_t>(h >> 32), n);
}

// Inclusive prefix sum over the 64 lanes of a wave: DPP row shifts by 1, 2,
// 4 and 8 (lanes shifted in from outside the 16-lane row read 0) give each
// row's prefix; row broadcasts of lane 15 into rows 1 and 3, then of lane
// 31 into rows 2 and 3, carry the row totals.  No lane predicates, no LDS.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  int x = static_cast<int>(v);
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);   // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);   // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return static_cast<uint32_t>(x);
}

// ------------------------------------------------------------ expansion

// Shared tile machinery.  Each thread holds up to PER tile elements in
// registers (bit k of `valid` marks v[k]); they are ranked within their
// bucket by LDS atomics and placed bucket-contiguously in t.s.  Bucket b's
// run of n elements is reserved in its slab (which starts at slab_base(b))
// through runs.cursor(b); kDropRun: the slab is full and the run is
// dropped.  The run is then written contiguously.  Run offsets stay 32-bit
// so two 512-thread tiles fit one CU's LDS.
constexpr uint32_t kDropRun = ~0u;

struct TileLds {
  uint64_t s[kTile + kWave];  // + one parking slot per lane for invalid elements
  alignas(8) uint32_t off[1u << kMaxPassBits];
  // Bucket counters, then one spare counter per lane that ranks invalid
  // elements (its values are never used).
  alignas(8) uint32_t lhist[(1u << kMaxPassBits) + kWave];
  alignas(8) uint32_t lstart[1u << kMaxPassBits];
  alignas(16) uint32_t wave_sums[kRouteThreads / kWave];
};
static_assert((1u << kMaxPassBits) == 2 * kRouteThreads, "each routing thread owns two bucket counters");

// Clears every bucket counter (two per thread); entries at or above a
// pass's bucket count stay zero, so the tile scan runs over all of them.
__device__ __forceinline__ void clear_tile_counters(TileLds& t) {
  reinterpret_cast<uint2*>(t.lhist)[threadIdx.x] = make_uint2(0u, 0u);
}

// Exclusive scan of all bucket counters into t.lstart; thread t owns
// buckets 2t and 2t+1, returns their counts in c and clears them (no other
// thread reads them: the next tile's increments come after later barriers).
// Returns the tile's total; start receives the two buckets' starts.
__device__ __forceinline__ uint32_t tile_scan(TileLds& t, uint2& c, uint2& start) {
  c = reinterpret_cast<const uint2*>(t.lhist)[threadIdx.x];
  reinterpret_cast<uint2*>(t.lhist)[threadIdx.x] = make_uint2(0u, 0u);
  const uint32_t s = c.x + c.y;
  const uint32_t incl = wave_incl_scan(s);
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(threadIdx.x)) / kWave;  // uniform
  if (lane == kWave - 1) t.wave_sums[wave] = incl;
  __syncthreads();
  uint32_t before = 0, total = 0;
#pragma unroll
  for (uint32_t w = 0; w < kRouteThreads / kWave; ++w) {
    const uint32_t ws = t.wave_sums[w];
    before += w < wave ? ws : 0u;
    total += ws;
  }
  const uint32_t run = before + incl - s;
  start = make_uint2(run, run + c.x);
  reinterpret_cast<uint2*>(t.lstart)[threadIdx.x] = start;
  __syncthreads();
  return total;
}

// Destination indexing.  When the output array (plus a kTile-entry dump
// area at index `dump`) has fewer than 2^32 entries, t.off[b] holds bucket
// b's 32-bit destination index minus the run's LDS start, so the write-out
// is one add per element; a dropped run is pointed into the dump area (the
// layer is redone anyway, the writes only have to stay in bounds).
// Otherwise (dump = kWideOut) t.off[b] is the run's slab offset and the
// write-out computes 64-bit addresses and skips dropped runs.
constexpr uint32_t kWideOut = ~0u;

// Run cursors of a routing pass: cursor(b) counts the entries reserved in
// bucket b's slab; settle(off, n) checks a run reserved at off against the
// slab capacity (kDropRun and the error bit when it does not fit, or when
// n = 0).
struct RunCursors {
  uint32_t* base;
  uint64_t stride;  // cursor of bucket b at base[b * stride]
  uint32_t cap;
  uint32_t* error;
  uint32_t err_bit;
  __device__ __forceinline__ uint32_t* cursor(uint32_t b) const { return base + static_cast<uint64_t>(b) * stride; }
  __device__ __forceinline__ uint32_t settle(uint32_t off, uint32_t n) const {
    if (n == 0) return kDropRun;
    if (static_cast<uint64_t>(off) + n > cap) {
      atomicOr(error, err_bit);
      return kDropRun;
    }
    return off;
  }
};

// `between` runs after the tile is placed in LDS and before its write-out:
// the caller issues the next tile's loads there (v is no longer read), so
// they are in flight during the write-out.
// The output may be narrower than the tile's words (Out): their low part is
// written.
template <int PER, typename BucketFn, typename BaseFn, typename BetweenFn, typename Out>
__device__ __forceinline__ void route_regs(TileLds& t, const uint64_t (&v)[PER], uint32_t valid,
                                           BucketFn bkt, const RunCursors& runs, BaseFn slab_base,
                                           Out* __restrict__ out, uint32_t dump, BetweenFn between) {
  // No branches per element: an invalid element takes its rank from the
  // lane's spare counter and is parked in the lane's slot past the tile.
  const uint32_t lane = threadIdx.x & (kWave - 1);
  uint32_t rank[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    uint32_t b = bkt(v[k]);
    asm volatile("" : "+v"(b));  // keeps the choice below a select, not a branch
    rank[k] = atomicAdd(&t.lhist[((valid >> k) & 1u) ? b : (1u << kMaxPassBits) + lane], 1u);
  }
  __syncthreads();
  uint2 n, st;
  const uint32_t ne = tile_scan(t, n, st);
  // Run reservations first: both atomics go out before the LDS placement
  // and their offsets are checked after it, so the round trips overlap the
  // placement.  (A check right after each atomic branches on its result and
  // waits for it there.)  Buckets without a run issue no atomic: a tile's
  // children cluster into few buckets.
  const uint32_t b0 = 2 * threadIdx.x, b1 = b0 + 1;
  uint32_t off0 = 0, off1 = 0;
  if (n.x) off0 = atomicAdd(runs.cursor(b0), n.x);
  if (n.y) off1 = atomicAdd(runs.cursor(b1), n.y);
  // All bucket starts are read first (in bounds for any element) and pinned,
  // so the reads go out together instead of one guarded read per element.
  uint32_t pos[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) pos[k] = t.lstart[bkt(v[k])];
#pragma unroll
  for (int k = 0; k < PER; ++k) asm volatile("" : "+v"(pos[k]));
  // The element predicates are taken afresh from the mask here: reusing the
  // rank step's keeps 2 x PER SGPRs live across the scan, and they spill.
  uint32_t vmask = valid;
  asm volatile("" : "+v"(vmask));
#pragma unroll
  for (int k = 0; k < PER; ++k) t.s[((vmask >> k) & 1u) ? pos[k] + rank[k] : kTile + lane] = v[k];
  asm volatile("" : "+v"(off0), "+v"(off1));  // the offsets are used only from here on
  off0 = runs.settle(off0, n.x);
  off1 = runs.settle(off1, n.y);
  if (dump != kWideOut) {
    auto dest = [&](uint32_t b, uint32_t off, uint32_t start) {
      return (off == kDropRun ? dump : static_cast<uint32_t>(slab_base(b)) + off) - start;
    };
    reinterpret_cast<uint2*>(t.off)[threadIdx.x] = make_uint2(dest(b0, off0, st.x), dest(b1, off1, st.y));
  } else {
    reinterpret_cast<uint2*>(t.off)[threadIdx.x] = make_uint2(off0, off1);
  }
  __syncthreads();
  between();
  if (dump != kWideOut) {
    // Rows go out in rounds of kRound per thread: the round's rows are read
    // at once (rows at or past ne hold stale entries whose bucket index is
    // still in range), then their run offsets, then the rows below ne are
    // stored.  A loop over single rows waits on two dependent LDS reads per
    // row; a single round of all kTilePerThread rows costs the registers of
    // the second workgroup per CU.
    constexpr int kRound = kTilePerThread / 2;
    for (uint32_t r = 0; r < kTile && r < ne; r += kRound * kRouteThreads) {
      uint64_t h[kRound];
      uint32_t o[kRound];
#pragma unroll
      for (int u = 0; u < kRound; ++u) h[u] = t.s[r + threadIdx.x + u * kRouteThreads];
#pragma unroll
      for (int u = 0; u < kRound; ++u) o[u] = t.off[bkt(h[u])];
#pragma unroll
      for (int u = 0; u < kRound; ++u) {
        const uint32_t j = r + threadIdx.x + u * kRouteThreads;
        if (j < ne) out[o[u] + j] = static_cast<Out>(h[u]);  // 32-bit index arithmetic, wraps as intended
      }
    }
  } else {
    for (uint32_t j = threadIdx.x; j < ne; j += kRouteThreads) {
      const uint64_t h = t.s[j];
      const uint32_t b = bkt(h);
      const uint32_t off = t.off[b];
      if (off != kDropRun) out[slab_base(b) + off + (j - t.lstart[b])] = static_cast<Out>(h);
    }
  }
  // No barrier here: the next tile's placement and scan come after its
  // first barrier, which every thread reaches only after its write-out.
}

// A parent's key for the shift-group expansion: keyunmix without its final
// mask, so bits above the key's 4n bits are left as the multiply leaves
// them.  Every shift group keeps only destination nibbles whose source
// nibble lies below n, so those bits never reach a child.
__device__ __forceinline__ uint64_t parent_key(uint64_t h, const SortedLayout& L) {
  uint64_t x = h >> L.tagbits;
  x ^= x >> L.km.shift;
  return x * L.km.i1;
}

// The stored value (keymix(child) << tagbits) | tag.  The layout's key
// width is at least 32 bits, so keymix's mask is applied to the high word
// only (its low word is all ones).
__device__ __forceinline__ uint64_t stored_value(uint64_t child, uint64_t tag, const SortedLayout& L) {
  uint64_t x = child * L.km.m1;
  x &= (static_cast<uint64_t>(static_cast<uint32_t>(L.km.mask >> 32)) << 32) | 0xffffffffull;
  x ^= x >> L.km.shift;
  return (x << L.tagbits) | tag;
}

}  // namespace mgbfs
