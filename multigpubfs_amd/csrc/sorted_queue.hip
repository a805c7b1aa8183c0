// Small and medium layers of the sorted backend, run ahead of the host.
//
// A layer of the general path (sorted_engine.hip) costs about ten launches,
// eight timing events (4.5 us each on the stream), two copies and a host
// wait: 83 us per layer of S_8, of which the kernels' work is a few.  Two
// forms take over the layers whose work is smaller than that:
//
//   block_run    : one workgroup runs layer after layer without leaving the
//       kernel, current and next layer in one LDS table.
//   owner layers : one launch per layer.  Every workgroup owns a range of
//       the stored values for the whole session: it selects its new states
//       from the candidates sent to it, keeps them in its slab, and sends
//       their children to their owners' slabs for the next launch.  The
//       host queues layers ahead and follows the records they leave in
//       pinned memory.  A dependent launch costs 3 us here, a grid-wide
//       barrier with 256 workgroups 7 to 15 us, so the launches are the
//       barriers.
//
// A session of owner layers starts from the dense bank (import) and ends by
// writing the last two layers back as banks (export).  Anything unusual (an
// overflow, a layer above the banks) is rejected, not handled: the layer's
// parents are intact and the general path redoes it.
#include <algorithm>
#include "common.hpp"
#include "kernels.hpp"
#include "owner_device.hpp"
#include "sorted_device.hpp"
#include "wide.hpp"

namespace mgbfs {

namespace {

constexpr int kBlockThreads = 1024;
constexpr uint32_t kNoBank = 3;

struct BlockLds {
  alignas(16) uint64_t table[kBlockSlots];
  uint32_t fresh;     // new states inserted
  uint32_t known;     // current-layer states some child reached
  uint32_t children;
  uint32_t rows;      // survivors written
};

// Lanes adding to an LDS counter together: one atomic for the active lanes.
__device__ __forceinline__ void add_active(uint32_t* counter, bool mine) {
  const uint64_t b = __ballot(mine);
  const uint64_t active = __ballot(true);
  const uint32_t lane = threadIdx.x & (kWave - 1);
  if (b && lane == static_cast<uint32_t>(__builtin_ctzll(active))) atomicAdd(counter, static_cast<uint32_t>(__popcll(b)));
}

// Inserts state value v; true when it was new.  A state already there keeps
// its entry: duplicates OR their back-edge masks into it (merge), and an
// entry of a retained layer (mark set) gets a low tag bit, so reached ones
// can be counted.  Terminates while the table has an empty slot.
__device__ __forceinline__ bool block_insert(uint64_t* table, uint32_t slot_mask, const SortedLayout& L, uint64_t mark,
                                             bool merge, uint64_t v) {
  uint32_t slot = static_cast<uint32_t>(v >> L.tagbits) & slot_mask;
  while (true) {
    const uint64_t old = atomicCAS(reinterpret_cast<unsigned long long*>(&table[slot]), kEmpty, v);
    if (old == kEmpty) return true;
    if ((old | L.tagmask) == (v | L.tagmask)) {
      const uint64_t add = merge ? v & L.tagmask : ((old & mark) ? 1ull : 0ull);
      if (add) atomicOr(reinterpret_cast<unsigned long long*>(&table[slot]), add);
      return false;
    }
    slot = (slot + 1) & slot_mask;
  }
}

// One workgroup, layer after layer.  Per layer: the retained layer(s) go
// into the LDS table marked, then every child is inserted; the unmarked
// entries are the next layer and go to its bank (any order: the bank has a
// single fine bucket).  Bound by LDS atomic round trips (each thread takes
// F / 1024 parents in turn) and five barriers; 16,384 slots of the CU's
// 160 KB are one workgroup's share, so one layer may hold up to about
// 10,000 old and new states together.
template <typename Action>
__global__ __launch_bounds__(kBlockThreads) void block_run_kernel(BlockRun r, Action act) {
  __shared__ BlockLds t;
  const SortedLayout L = r.L;
  const uint64_t mark = 1ull << (L.tagbits - 1);
  const uint32_t G = act.count();
  uint64_t* const b0 = r.bank[0];
  uint64_t* const b1 = r.bank[1];
  uint64_t* const b2 = r.bank[2];
  auto bank_of = [&](uint32_t b) { return b == 0 ? b0 : (b == 1 ? b1 : b2); };
  uint32_t cur = r.cur, prev = r.prev, F = r.F, Fp = r.prev_count, done = 0;
  LayerRecord* rec = r.rec;
  if (threadIdx.x == 0) {
    rec->stamps[0] = wall_clock64();
    rec->compacted = r.counters->compacted;
  }
  while (true) {
    const bool masked = L.prune && r.depth + done > 0;
    const uint64_t* from = bank_of(cur);
    const uint32_t nxt = (cur != 0 && prev != 0) ? 0u : ((cur != 1 && prev != 1) ? 1u : 2u);
    const uint32_t old = !L.prune && prev < kNoBank ? Fp : 0u;
    // Slots: at most half full when every child is new, up to kBlockSlots.
    const uint64_t most = static_cast<uint64_t>(F) * (masked && G > 1 ? G - 1 : G) + F + old;
    uint32_t slots = 256;
    while (slots < 2 * most && slots < kBlockSlots) slots <<= 1;
    const uint32_t slot_mask = slots - 1;
    const uint32_t room = kBlockFill - (F + old);  // new states accepted
    for (uint32_t i = threadIdx.x; i < slots / 2; i += kBlockThreads)
      reinterpret_cast<ulonglong2*>(t.table)[i] = make_ulonglong2(kEmpty, kEmpty);
    if (threadIdx.x == 0) t.fresh = t.known = t.children = t.rows = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < F; i += kBlockThreads)
      block_insert(t.table, slot_mask, L, mark, false, (from[i] & ~L.tagmask) | mark);
    if (old) {
      const uint64_t* before = bank_of(prev);
      for (uint32_t i = threadIdx.x; i < old; i += kBlockThreads)
        block_insert(t.table, slot_mask, L, mark, false, (before[i] & ~L.tagmask) | mark);
    }
    __syncthreads();
    uint32_t children = 0;
    for (uint32_t i = threadIdx.x; i < F; i += kBlockThreads) {
      const uint64_t h = from[i];
      const uint32_t skip = masked ? static_cast<uint32_t>(h & L.tagmask) : 0u;
      const uint64_t key = keyunmix(h >> L.tagbits, L.km);
      for (uint32_t g = 0; g < G; ++g) {
        const uint64_t child = act.child(key, g);
        if ((skip >> g) & 1u) continue;
        ++children;
        // Every wave looks before each child, so at most one insertion per
        // lane passes the limit: the table keeps empty slots.
        if (*const_cast<volatile uint32_t*>(&t.fresh) > room) continue;
        const uint64_t v = (keymix(child, L.km) << L.tagbits) | act.mask(g);
        add_active(&t.fresh, block_insert(t.table, slot_mask, L, mark, L.prune != 0, v));
      }
    }
    for (int off = kWave / 2; off; off >>= 1) children += __shfl_xor(children, off, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) atomicAdd(&t.children, children);
    __syncthreads();
    const uint32_t N = t.fresh;
    const bool reject = N > room || N > r.rows;
    if (!reject) {
      uint64_t* to = bank_of(nxt);
      const uint32_t lane = threadIdx.x & (kWave - 1);
      for (uint32_t i = threadIdx.x; i < slots / 2; i += kBlockThreads) {
        const ulonglong2 p = reinterpret_cast<const ulonglong2*>(t.table)[i];
        const bool ox = p.x != kEmpty, oy = p.y != kEmpty;
        const bool sx = ox && !(p.x & mark), sy = oy && !(p.y & mark);
        add_active(&t.known, ox && !sx && (p.x & L.tagmask) != mark);
        add_active(&t.known, oy && !sy && (p.y & L.tagmask) != mark);
        // Rows for the wave's survivors: one atomic, ballot ranks.
        const uint64_t bx = __ballot(sx), by = __ballot(sy);
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(&t.rows, static_cast<uint32_t>(__popcll(bx) + __popcll(by)));
        base = __shfl(base, 0, kWave);
        const uint64_t below = (1ull << lane) - 1;
        if (sx) to[base + __popcll(bx & below)] = p.x;
        if (sy) to[base + __popcll(bx) + __popcll(by & below)] = p.y;
      }
    }
    __syncthreads();
    // The next layer's children by this one's per parent (the start state's
    // children carry masks, it does not: all but one of each parent's then).
    const uint32_t per = masked || !L.prune ? t.children : (G > 1 ? G - 1 : 1) * F;
    const bool leave = N > kBlockParents || static_cast<uint64_t>(N) * per > static_cast<uint64_t>(kBlockChildren) * F;
    const uint32_t state = reject ? kLayerRejected
                                  : (N == 0 ? kLayerEmpty
                                            : (leave || done + 1 == r.max_layers ? kLayerStop : kLayerNext));
    if (!reject && N != 0) {
      prev = cur;
      Fp = F;
      cur = nxt;
      F = N;
    }
    if (threadIdx.x == 0) {
      if (state != kLayerNext && (done || state == kLayerStop)) {
        // One fine bucket per bank: {0, rows}.
        uint32_t* oc = cur == 0 ? r.off[0] : (cur == 1 ? r.off[1] : r.off[2]);
        oc[0] = 0;
        oc[1] = F;
        if (prev < kNoBank) {
          uint32_t* op = prev == 0 ? r.off[0] : (prev == 1 ? r.off[1] : r.off[2]);
          op[0] = 0;
          op[1] = Fp;
        }
      }
      LayerRecord* o = rec + done;
      o->N = N;
      o->children = t.children;
      o->unique = N + t.known;
      o->ticks = wall_clock64();
      o->state = state;
      if (state != kLayerNext) __threadfence_system();
      __hip_atomic_store(&o->seq, r.seq + done, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (state != kLayerNext) return;
    ++done;
    __syncthreads();  // counters and table are reused
  }
}

__global__ void sorted_start_kernel(uint64_t stored, uint64_t* bank, uint32_t* off, uint64_t* control) {
  if (threadIdx.x == 0) {
    bank[0] = stored;
    off[0] = 0;
    off[1] = 1;
  }
  if (threadIdx.x < 8) control[threadIdx.x] = 0;
}

__global__ void stamp_record_kernel(LayerRecord* rec, const LayerCounters* counters, uint64_t seq) {
  if (threadIdx.x != 0) return;
  rec->compacted = counters->compacted;
  __hip_atomic_store(&rec->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ------------------------------------------------------------ owner layers

__global__ __launch_bounds__(kBlockThreads) void owner_begin_kernel(uint32_t* counts, uint32_t words, OwnerCtl* ctl,
                                                                     uint32_t F, LayerRecord* rec,
                                                                     const LayerCounters* counters) {
  for (uint32_t i = blockIdx.x * kBlockThreads + threadIdx.x; i < words; i += gridDim.x * kBlockThreads) counts[i] = 0;
  if (blockIdx.x) return;
  if (rec && threadIdx.x == 0) {
    rec->stamps[0] = wall_clock64();
    rec->compacted = counters->compacted;
  }
  if (threadIdx.x < 2) {
    OwnerCtl c{};
    c.counts = threadIdx.x == 0 ? F : 0u;
    c.imported = threadIdx.x == 0;
    ctl[threadIdx.x] = c;
  }
}

// A routing tile holds kSendItems x 512 child slots, generator-major over P
// parents (a multiple of 64, so the lanes of a wave share their generator).
constexpr int kSendItems = 8;

__device__ __forceinline__ uint32_t tile_parents(uint32_t G) {
  return kSendItems * kRouteThreads / G / kWave * kWave;
}

// Children of parents[0, count) (count <= tile_parents) routed into the
// slabs of their buckets; returns this thread's number of children.  Called
// by the whole workgroup with cleared tile counters.
template <typename Action, typename BucketFn, typename BaseFn>
__device__ __forceinline__ uint32_t send_tile(TileLds& t, const uint64_t* parents, uint32_t count, bool masked,
                                              const Action& act, const SortedLayout& L, BucketFn bkt,
                                              const RunCursors& runs, BaseFn slab_base, uint64_t* out, uint32_t dump) {
  const uint32_t G = act.count();
  const uint32_t P = (count + kWave - 1) / kWave * kWave;
  const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(threadIdx.x)) / kWave;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  uint64_t v[kSendItems];
  uint32_t gen[kSendItems];
  uint32_t valid = 0;
#pragma unroll
  for (int k = 0; k < kSendItems; ++k) {
    const uint32_t s = (k * (kRouteThreads / kWave) + wave) * kWave;  // the wave's first slot
    const uint32_t g = s / P, m = s - g * P + lane;
    const bool live = g < G && m < count;
    gen[k] = g < G ? g : G;
    v[k] = live ? parents[m] : 0;
    valid |= live ? 1u << k : 0u;
  }
#pragma unroll
  for (int k = 0; k < kSendItems; ++k) {
    const uint32_t g = gen[k];
    if (g < G) {  // uniform
      if (masked && ((v[k] >> g) & 1u)) valid &= ~(1u << k);  // tag bit g: leads back
      const uint64_t child = act.child(keyunmix(v[k] >> L.tagbits, L.km), g);
      v[k] = (keymix(child, L.km) << L.tagbits) | act.mask(g);
    }
  }
  route_regs(t, v, valid, bkt, runs, slab_base, out, dump, [] {});
  return __popc(valid);
}

// The same to the owners' slabs.
template <typename Action>
__device__ __forceinline__ uint32_t owner_send(TileLds& t, const uint64_t* parents, uint32_t count, bool masked,
                                               const Action& act, const SortedLayout& L, uint32_t owners,
                                               const OwnerSlabs& out, uint32_t* spill) {
  return send_tile(
      t, parents, count, masked, act, L, [owners](uint64_t h) { return range_index(h, owners); },
      RunCursors{out.count, kCountStride, kUniqueCap, spill, 1u},
      [](uint32_t b) { return static_cast<uint64_t>(b) * kSlabStride; }, out.data, owners * kSlabStride);
}

// The general path's expansion (expand_scatter_kernel) for wide keys: tiles
// of contiguous parents dealt to blocks round-robin, children to the lane
// slabs.  One instantiation serves every generator count: 4,096 child slots
// per tile instead of 8,192 children, at 90 registers.
template <typename Action>
__global__ __launch_bounds__(kRouteThreads) void expand_wide_kernel(const uint64_t* __restrict__ bank, uint64_t F,
                                                                    Action act, SortedLayout L, bool masked,
                                                                    uint32_t nsub, uint32_t K2, uint32_t NB, uint32_t P,
                                                                    uint32_t cap, uint32_t stride, uint32_t err_bit,
                                                                    uint32_t* __restrict__ cursors,
                                                                    uint32_t* __restrict__ error,
                                                                    uint64_t* __restrict__ out, uint32_t dump) {
  __shared__ TileLds t;
  clear_tile_counters(t);
  __syncthreads();
  const uint32_t part = blockIdx.x % P;
  const uint64_t parents = tile_parents(act.count()), tiles = (F + parents - 1) / parents;
  for (uint64_t tile = blockIdx.x; tile < tiles; tile += NB) {
    const uint64_t p0 = tile * parents;
    const uint32_t n = static_cast<uint32_t>(F - p0 < parents ? F - p0 : parents);
    send_tile(
        t, bank + p0, n, masked, act, L, [nsub, K2](uint64_t h) { return range_index(h, nsub) >> K2; },
        RunCursors{cursors + part, P, cap, error, err_bit},
        [=](uint32_t b) { return (static_cast<uint64_t>(b) * P + part) * stride; }, out, dump);
  }
}

// Dense banks -> owner slabs of the retained layer(s), and the children of
// the current one.  Block ranges: tiles of the current bank, of the
// previous one, then tiles of parents.
template <typename Action>
__global__ __launch_bounds__(kRouteThreads) void owner_import_kernel(OwnerImport im, Action act, SortedLayout L,
                                                                     uint32_t owners, uint32_t cur_tiles,
                                                                     uint32_t prev_tiles) {
  __shared__ TileLds t;
  clear_tile_counters(t);
  __syncthreads();
  constexpr uint32_t kCopy = kSendItems * kRouteThreads;
  if (blockIdx.x < cur_tiles + prev_tiles) {
    const bool first = blockIdx.x < cur_tiles;
    const uint64_t* from = first ? im.cur : im.prev;
    const uint32_t n = first ? im.F : im.prev_count;
    const OwnerSlabs to = first ? im.own : im.own_prev;
    const uint32_t t0 = (first ? blockIdx.x : blockIdx.x - cur_tiles) * kCopy;
    uint64_t v[kSendItems];
    uint32_t valid = 0;
#pragma unroll
    for (int k = 0; k < kSendItems; ++k) {
      const uint32_t i = t0 + k * kRouteThreads + threadIdx.x;
      v[k] = i < n ? from[i] : 0;
      valid |= i < n ? 1u << k : 0u;
    }
    const RunCursors runs{to.count, kCountStride, kUniqueCap, &im.ctl->error, kErrBucketCap};
    auto slab_base = [](uint32_t b) { return static_cast<uint64_t>(b) * kSlabStride; };
    auto bkt = [owners](uint64_t h) { return range_index(h, owners); };
    route_regs(t, v, valid, bkt, runs, slab_base, to.data, owners * kSlabStride, [] {});
    return;
  }
  const uint32_t P = tile_parents(act.count());
  const uint32_t p0 = (blockIdx.x - cur_tiles - prev_tiles) * P;
  uint32_t made = owner_send(t, im.cur + p0, min(P, im.F - p0), im.masked != 0, act, L, owners, im.cand, &im.ctl->spill);
  made = wave_incl_scan(made);
  if ((threadIdx.x & (kWave - 1)) == kWave - 1 && made)
    atomicAdd(&im.ctl->counts, static_cast<unsigned long long>(made) << 32);
}

// Marks h's state in the table if it is there (see probe_value in
// sorted_kernels.hip: each slot matches at most one retained state).
__device__ __forceinline__ void owner_mark(uint64_t* table, uint32_t slot_mask, const SortedLayout& L, uint64_t mark,
                                           uint64_t h) {
  const uint64_t key = h | L.tagmask;
  uint32_t slot = static_cast<uint32_t>(h >> L.tagbits) & slot_mask;
  for (uint32_t probe = 0; probe <= slot_mask; ++probe) {
    const uint64_t v = table[slot];
    if (v == kEmpty) return;
    if ((v | L.tagmask) == key) {
      table[slot] = v | mark;
      return;
    }
    slot = (slot + 1) & slot_mask;
  }
}

// One layer of one owner: its candidates into an LDS table (duplicates
// merge), the retained layers' states mark theirs, the unmarked entries are
// the owner's part of the new layer; then the children of those go out.
// Small layers are bound by the chain of dependent steps (candidate load,
// LDS rounds, slab write and re-read, cursor atomics, child stores; about
// 12 us with the launch), large ones by the same VALU and LDS work as the
// general path's kernels, without its 40 bytes a state of compaction and
// bank reload.  The routing tile reuses the table's LDS (two workgroups per
// CU).
template <typename Action>
__global__ __launch_bounds__(kRouteThreads) void owner_layer_kernel(OwnerLayer a, Action act, SortedLayout L) {
  __shared__ alignas(16) char lds[sizeof(TileLds) > kUniqueSlots * 8 ? sizeof(TileLds) : kUniqueSlots * 8];
  __shared__ uint32_t rows, occupied, made;
  uint64_t* table = reinterpret_cast<uint64_t*>(lds);
  const uint32_t f = blockIdx.x;
  const OwnerCtl before = *a.before;
  uint32_t c = a.in.count[f * kCountStride];
  const uint32_t ncur = a.cur.count[f * kCountStride], nprev = a.prev.data ? a.prev.count[f * kCountStride] : 0u;
  const uint32_t state = owner_state(before, a.rules);
  const bool run = !before.halt && state == kLayerNext;
  if (f == 0 && threadIdx.x == 0) {
    if (!before.halt) owner_publish(before, state, a.rec, a.seq);
    if (!run) a.now->halt = 1;
    *a.after = OwnerCtl{};
  }
  if (!run) return;
  const uint64_t base = static_cast<uint64_t>(f) * kSlabStride;
  const uint64_t* cand = a.in.data + base;
  const uint64_t* cur = a.cur.data + base;
  uint64_t* next = a.next.data + base;
  if (c > kUniqueCap) {  // the sender flagged it; this layer cannot be selected
    if (threadIdx.x == 0) {
      atomicOr(&a.now->error, kErrBucketCap);
      a.next.count[f * kCountStride] = 0;
    }
    c = 0;
  }
  if (c == 0) {
    __syncthreads();  // every thread has read the count
    if (threadIdx.x == 0) {
      a.in.count[f * kCountStride] = 0;
      a.next.count[f * kCountStride] = 0;
    }
    return;
  }
  // The first candidates and retained states are loaded before the table is
  // cleared; later ones in chunks of kChunk per thread.
  constexpr int kChunk = 4;
  auto load = [&](uint64_t (&v)[kChunk], const uint64_t* from, uint32_t at, uint32_t n) {
#pragma unroll
    for (int k = 0; k < kChunk; ++k) {
      const uint32_t i = at + k * kRouteThreads + threadIdx.x;
      v[k] = from[i < n ? i : 0u];
    }
  };
  uint64_t v[kChunk], w[kChunk];
  load(v, cand, 0, c);
  load(w, cur, 0, ncur);
  uint32_t slots = 64;
  while (slots < 2 * c && slots < kUniqueSlots) slots <<= 1;
  const uint32_t slot_mask = slots - 1;
  for (uint32_t i = threadIdx.x; i < slots / 2; i += kRouteThreads)
    reinterpret_cast<ulonglong2*>(table)[i] = make_ulonglong2(kEmpty, kEmpty);
  if (threadIdx.x == 0) rows = occupied = made = 0;
  __syncthreads();
  const uint64_t mark = 1ull << (L.tagbits - 1);
  for (uint32_t at = 0; at < c; at += kChunk * kRouteThreads) {
    if (at) load(v, cand, at, c);
#pragma unroll
    for (int k = 0; k < kChunk; ++k)
      if (at + k * kRouteThreads + threadIdx.x < c) block_insert(table, slot_mask, L, mark, L.prune != 0, v[k]);
  }
  __syncthreads();
  for (uint32_t at = 0; at < ncur; at += kChunk * kRouteThreads) {
    if (at) load(w, cur, at, ncur);
#pragma unroll
    for (int k = 0; k < kChunk; ++k)
      if (at + k * kRouteThreads + threadIdx.x < ncur) owner_mark(table, slot_mask, L, mark, w[k]);
  }
  if (nprev) {
    const uint64_t* prev = a.prev.data + base;
    for (uint32_t at = 0; at < nprev; at += kChunk * kRouteThreads) {
      load(w, prev, at, nprev);
#pragma unroll
      for (int k = 0; k < kChunk; ++k)
        if (at + k * kRouteThreads + threadIdx.x < nprev) owner_mark(table, slot_mask, L, mark, w[k]);
    }
  }
  __syncthreads();
  const uint32_t lane = threadIdx.x & (kWave - 1);
  uint32_t occ = 0;
  for (uint32_t i = threadIdx.x; i < slots / 2; i += kRouteThreads) {  // whole waves: slots / 2 is 32 or a multiple of 64
    const ulonglong2 p = reinterpret_cast<const ulonglong2*>(table)[i];
    const bool ox = p.x != kEmpty, oy = p.y != kEmpty;
    const bool sx = ox && !(p.x & mark), sy = oy && !(p.y & mark);
    occ += (ox ? 1u : 0u) + (oy ? 1u : 0u);
    const uint64_t bx = __ballot(sx), by = __ballot(sy);
    uint32_t at = 0;
    if (lane == 0) at = atomicAdd(&rows, static_cast<uint32_t>(__popcll(bx) + __popcll(by)));
    at = __shfl(at, 0, kWave);
    const uint64_t below = (1ull << lane) - 1;
    if (sx) next[at + __popcll(bx & below)] = p.x;
    if (sy) next[at + __popcll(bx) + __popcll(by & below)] = p.y;
  }
  occ = wave_incl_scan(occ);
  if (lane == kWave - 1 && occ) atomicAdd(&occupied, occ);
  __syncthreads();
  const uint32_t N = rows;
  TileLds& t = *reinterpret_cast<TileLds*>(lds);
  clear_tile_counters(t);
  __syncthreads();
  uint32_t mine = 0;
  const uint32_t P = tile_parents(act.count());
  for (uint32_t p0 = 0; p0 < N; p0 += P)
    mine += owner_send(t, next + p0, min(P, N - p0), L.prune != 0, act, L, a.rules.owners, a.out, &a.now->spill);
  mine = wave_incl_scan(mine);
  if (lane == kWave - 1 && mine) atomicAdd(&made, mine);
  __syncthreads();
  if (threadIdx.x == 0) {
    a.in.count[f * kCountStride] = 0;
    a.next.count[f * kCountStride] = N;
    atomicAdd(&a.now->counts, static_cast<unsigned long long>(N) | (static_cast<unsigned long long>(made) << 32));
    atomicAdd(&a.now->unique, static_cast<unsigned long long>(occupied));
  }
}

__global__ void owner_report_kernel(const OwnerCtl* ctl, OwnerRules rules, LayerRecord* rec, uint64_t seq) {
  if (threadIdx.x != 0 || ctl->halt) return;
  owner_publish(*ctl, owner_state(*ctl, rules), rec, seq);
}

// Blocks [0, owners) write the current layer's bank, the others the
// previous one's; every block sums the counts of the owners before its own.
__global__ __launch_bounds__(kRouteThreads) void owner_export_kernel(OwnerSlabs cur, uint64_t* bank, uint32_t* off,
                                                                     OwnerSlabs prev, uint64_t* prev_bank,
                                                                     uint32_t* prev_off, uint32_t owners) {
  __shared__ uint32_t sums[kRouteThreads / kWave];
  const bool second = blockIdx.x >= owners;
  const uint32_t f = second ? blockIdx.x - owners : blockIdx.x;
  const OwnerSlabs s = second ? prev : cur;
  uint64_t* to = second ? prev_bank : bank;
  uint32_t* offsets = second ? prev_off : off;
  uint32_t before = 0;
  for (uint32_t j = threadIdx.x; j < f; j += kRouteThreads) before += s.count[j * kCountStride];
  before = wave_incl_scan(before);
  if ((threadIdx.x & (kWave - 1)) == kWave - 1) sums[threadIdx.x / kWave] = before;
  __syncthreads();
  before = 0;
#pragma unroll
  for (uint32_t w = 0; w < kRouteThreads / kWave; ++w) before += sums[w];
  const uint32_t n = s.count[f * kCountStride];
  if (threadIdx.x == 0) {
    offsets[f] = before;
    if (f + 1 == owners) offsets[owners] = before + n;
  }
  const uint64_t* from = s.data + static_cast<uint64_t>(f) * kSlabStride;
  for (uint32_t i = threadIdx.x; i < n; i += kRouteThreads) to[before + i] = from[i];
}

}  // namespace

// Calls f with the action the reference stands for.
template <typename F>
static hipError_t with_action(const ActionRef& act, F f) {
  if (act.count == 0 || act.count > kMaxGenerators || (!act.wide && !act.nibble)) return hipErrorInvalidValue;
  if (act.wide) f(WideAction{act.wide, act.count});
  else f(NibbleAction{*act.nibble});
  return hipGetLastError();
}

hipError_t sorted_block_run(const BlockRun& run, const ActionRef& act, hipStream_t stream) {
  if (run.cur > 2 || run.prev > kNoBank || run.prev == run.cur || run.F == 0 || run.max_layers == 0 || !run.rec || !run.counters ||
      run.F > kBlockParents || (run.prev < kNoBank && !run.L.prune && run.prev_count > kBlockParents))
    return hipErrorInvalidValue;
  return with_action(act, [&](auto a) {
    hipLaunchKernelGGL(block_run_kernel<decltype(a)>, dim3(1), dim3(kBlockThreads), 0, stream, run, a);
  });
}

hipError_t sorted_start(uint64_t stored, uint64_t* bank, uint32_t* off, uint64_t* control, hipStream_t stream) {
  hipLaunchKernelGGL(sorted_start_kernel, dim3(1), dim3(64), 0, stream, stored, bank, off, control);
  return hipGetLastError();
}

hipError_t stamp_record(LayerRecord* rec, const LayerCounters* counters, uint64_t seq, hipStream_t stream) {
  hipLaunchKernelGGL(stamp_record_kernel, dim3(1), dim3(64), 0, stream, rec, counters, seq);
  return hipGetLastError();
}

hipError_t owner_begin(uint32_t* counts, uint32_t words, OwnerCtl* ctl, uint32_t F, hipStream_t stream,
                       LayerRecord* rec, const LayerCounters* counters) {
  const uint32_t blocks = std::min<uint32_t>(16, (words + 4 * kBlockThreads - 1) / (4 * kBlockThreads));
  hipLaunchKernelGGL(owner_begin_kernel, dim3(blocks), dim3(kBlockThreads), 0, stream, counts, words, ctl, F, rec, counters);
  return hipGetLastError();
}

hipError_t owner_import(const OwnerImport& im, const ActionRef& act, const SortedLayout& L, uint32_t owners,
                        hipStream_t stream) {
  if (!im.cur || im.F == 0 || owners == 0 || owners > kOwnersMax || act.count == 0 || act.count > kMaxGenerators)
    return hipErrorInvalidValue;
  const uint32_t copy = kSendItems * kRouteThreads;
  const uint32_t cur_tiles = (im.F + copy - 1) / copy;
  const uint32_t prev_tiles = im.prev ? (im.prev_count + copy - 1) / copy : 0u;
  const uint32_t P = kSendItems * kRouteThreads / act.count / kWave * kWave;
  const uint32_t tiles = cur_tiles + prev_tiles + (im.F + P - 1) / P;
  return with_action(act, [&](auto a) {
    hipLaunchKernelGGL(owner_import_kernel<decltype(a)>, dim3(tiles), dim3(kRouteThreads), 0, stream, im, a, L, owners,
                       cur_tiles, prev_tiles);
  });
}

hipError_t owner_layer(const OwnerLayer& a, const ActionRef& act, const SortedLayout& L, hipStream_t stream) {
  if (a.rules.owners == 0 || a.rules.owners > kOwnersMax) return hipErrorInvalidValue;
  return with_action(act, [&](auto x) {
    hipLaunchKernelGGL(owner_layer_kernel<decltype(x)>, dim3(a.rules.owners), dim3(kRouteThreads), 0, stream, a, x, L);
  });
}

hipError_t sorted_expand_route_wide(const uint64_t* bank, uint64_t F, const ActionRef& act, const SortedLayout& L,
                                    bool masked, uint32_t nsub, uint32_t K2, uint32_t NB, uint32_t P, uint32_t cap,
                                    uint32_t stride, uint32_t err_bit, uint32_t* cursors, uint32_t* error,
                                    uint64_t* out, uint64_t out_entries, hipStream_t stream) {
  if (F == 0 || nsub == 0 || K2 > kMaxPassBits || (nsub & ((1u << K2) - 1u)) || (nsub >> K2) > (1u << kMaxPassBits) ||
      NB == 0 || P == 0 || cap == 0 || stride < cap || !act.wide || act.count == 0 || act.count > kMaxGenerators)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(expand_wide_kernel<WideAction>, dim3(NB), dim3(kRouteThreads), 0, stream, bank, F,
                     WideAction{act.wide, act.count}, L, masked, nsub, K2, NB, P, cap, stride, err_bit, cursors, error,
                     out, route_dump_index(out_entries, kTile));
  return hipGetLastError();
}

hipError_t owner_report(const OwnerCtl* ctl, const OwnerRules& rules, LayerRecord* rec, uint64_t seq,
                        hipStream_t stream) {
  hipLaunchKernelGGL(owner_report_kernel, dim3(1), dim3(64), 0, stream, ctl, rules, rec, seq);
  return hipGetLastError();
}

hipError_t owner_export(const OwnerSlabs& cur, uint64_t* bank, uint32_t* off, const OwnerSlabs& prev,
                        uint64_t* prev_bank, uint32_t* prev_off, uint32_t owners, hipStream_t stream) {
  hipLaunchKernelGGL(owner_export_kernel, dim3(2 * owners), dim3(kRouteThreads), 0, stream, cur, bank, off, prev,
                     prev_bank, prev_off, owners);
  return hipGetLastError();
}

}  // namespace mgbfs
