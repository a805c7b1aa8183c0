// Small and medium layers of the sorted backend, run ahead of the host.
//
// A layer of the general path (sorted_engine.hip) costs about ten launches,
// eight timing events (4.5 us each on the stream), two copies and a host
// wait: 83 us per layer of S_8, of which the kernels' work is a few.  Two
// forms take over the layers whose work is smaller than that:
//
//   block_run     : one workgroup runs layer after layer without leaving
//       the kernel, current and next layer in one LDS table.
//   queued layers : three launches per layer (expand, unique, compact),
//       their geometry read from the device, so the host queues layers
//       ahead and only follows the records they leave in pinned memory.
//       A dependent launch costs 3 us here, a grid-wide barrier with 256
//       workgroups 7 to 15 us, so separate launches beat a persistent grid.
//
// Both leave banks and offset tables as the general path does, and anything
// unusual (an overflow, a layer above the banks) is rejected, not handled:
// the layer's parents are intact and the general path redoes it.
#include <algorithm>
#include "common.hpp"
#include "kernels.hpp"
#include "sorted_device.hpp"

namespace mgbfs {

namespace {

constexpr int kBlockThreads = 1024;
constexpr uint32_t kNoBank = 3;

// Nibble-packed permutations: generators by value, shift groups.
struct NibbleAction {
  PackedGenerators gens;
  __device__ __forceinline__ uint32_t count() const { return gens.count; }
  __device__ __forceinline__ uint64_t child(uint64_t key, uint32_t g) const {
    return apply_groups(key, gens, static_cast<int>(g));
  }
  __device__ __forceinline__ uint32_t mask(uint32_t g) const { return gens.child_mask[g]; }
};

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
      o->cand = t.children;
      o->unique = N + t.known;
      o->ticks = wall_clock64();
      o->state = state;
      o->nbo = 1;
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

__global__ __launch_bounds__(kQueueSub) void queue_begin_kernel(QueueCtl* ctl, QueueCtl first, uint32_t* scount,
                                                                 LayerRecord* rec, uint64_t seq) {
  scount[threadIdx.x] = 0;
  if (threadIdx.x == 0) {
    *ctl = first;
    rec->ticks = wall_clock64();
    __hip_atomic_store(&rec->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Children of the current bank into sub-bucket slabs.  A tile holds ITEMS x
// 512 child slots, generator-major over P parents (a multiple of 64, so a
// wave's slots share their generator): four items per thread give a layer
// of 50,000 states 37 workgroups or more instead of 12 with a full tile.
template <typename Action, int ITEMS>
__global__ __launch_bounds__(kRouteThreads) void queue_expand_kernel(const uint64_t* __restrict__ bank,
                                                                     QueueCtl* ctl, Action act, SortedLayout L,
                                                                     uint32_t* __restrict__ scount,
                                                                     uint64_t* __restrict__ out) {
  __shared__ TileLds t;
  const uint32_t F = ctl->F, nsub = ctl->nsub, G = act.count();
  const bool masked = ctl->masked != 0;
  const uint32_t P = ITEMS * kRouteThreads / G / kWave * kWave;
  const uint32_t tiles = (F + P - 1) / P;
  if (blockIdx.x >= tiles) return;
  clear_tile_counters(t);
  __syncthreads();
  const RunCursors runs{scount, 1, kUniqueCap, &ctl->error, kErrBucketCap};
  auto slab_base = [=](uint32_t b) { return static_cast<uint64_t>(b) * kSlabStride; };
  auto bkt = [nsub](uint64_t h) { return range_index(h, nsub); };
  const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(threadIdx.x)) / kWave;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint32_t t0 = tile * P;
    uint64_t v[ITEMS];
    uint32_t gen[ITEMS];
    uint32_t valid = 0;
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
      const uint32_t s = (k * (kRouteThreads / kWave) + wave) * kWave;  // the wave's first slot
      const uint32_t g = s / P, m = t0 + (s - g * P) + lane;
      gen[k] = g;
      const bool live = g < G && m < F;
      valid |= live ? 1u << k : 0u;
      v[k] = bank[m < F ? m : F - 1];
    }
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
      const uint32_t g = gen[k] < G ? gen[k] : 0u;
      if (masked && ((v[k] >> g) & 1u)) valid &= ~(1u << k);  // tag bit g: leads back
      const uint64_t child = act.child(keyunmix(v[k] >> L.tagbits, L.km), g);
      v[k] = (keymix(child, L.km) << L.tagbits) | act.mask(g);
    }
    route_regs(t, v, valid, bkt, runs, slab_base, out, kQueueSub * kSlabStride, [] {});
  }
}

// One workgroup per sub-bucket: survivors (at the start of their slab, fine
// bucket order) -> the next bank, whose offsets come from the survivor
// totals of the sub-buckets before (at most 1,024, summed by every
// workgroup) and the sub-bucket's own fine counts; three scan launches
// saved.  Workgroup 0 sizes the next layer and reports this one.
__global__ __launch_bounds__(kRouteThreads) void queue_compact_kernel(
    const uint64_t* __restrict__ cand, const uint32_t* __restrict__ fine_counts, const uint32_t* __restrict__ totals,
    uint32_t* __restrict__ scount, const QueueCtl* __restrict__ ctl, QueueCtl* __restrict__ next, QueueRules rules,
    uint64_t* __restrict__ bank, uint32_t* __restrict__ off, LayerRecord* rec, uint64_t seq) {
  __shared__ uint32_t sums[2][kRouteThreads / kWave];
  const uint32_t f = blockIdx.x, F = ctl->F, nsub = ctl->nsub, fb = ctl->fb;
  if (threadIdx.x == 0) scount[f] = 0;  // the next layer's cursors
  if (F == 0) {
    if (f == 0 && threadIdx.x == 0) next->F = 0;
    return;
  }
  if (f >= nsub) return;
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  uint32_t before = 0, all = 0;
#pragma unroll
  for (uint32_t j = threadIdx.x; j < kQueueSub; j += kRouteThreads) {
    const uint32_t c = j < nsub ? totals[j] : 0u;
    all += c;
    before += j < f ? c : 0u;
  }
  before = wave_incl_scan(before);
  all = wave_incl_scan(all);
  if (lane == kWave - 1) {
    sums[0][wave] = before;
    sums[1][wave] = all;
  }
  __syncthreads();
  before = all = 0;
#pragma unroll
  for (uint32_t w = 0; w < kRouteThreads / kWave; ++w) {
    before += sums[0][w];
    all += sums[1][w];
  }
  const uint32_t error = ctl->error;
  const bool reject = error != 0 || all > rules.rows;
  if (!reject && all != 0) {
    // Offsets of the fine buckets: wave 0 scans the counts, 64 at a time.
    const uint32_t fine = 1u << fb;
    if (wave == 0) {
      uint32_t run = before;
      for (uint32_t j = lane; j < ((fine + kWave - 1) & ~(kWave - 1u)); j += kWave) {
        const uint32_t c = j < fine ? fine_counts[(f << fb) + j] : 0u;
        const uint32_t incl = wave_incl_scan(c);
        if (j < fine) off[(f << fb) + j] = run + incl - c;
        run += __shfl(incl, kWave - 1, kWave);
      }
      if (f == nsub - 1 && lane == 0) off[nsub << fb] = all;
    }
    const uint32_t mine = totals[f];
    const uint64_t* src = cand + static_cast<uint64_t>(f) * kSlabStride;
    for (uint32_t i = threadIdx.x; i < mine; i += kRouteThreads) bank[before + i] = src[i];
  }
  if (f != 0 || threadIdx.x != 0) return;
  const uint64_t C = ctl->cand;
  QueueCtl n{};
  n.masked = rules.prune;
  n.nbo_cur = nsub << fb;
  n.nbo_prev = ctl->nbo_cur;
  // Children of the next layer: this layer's children per parent plus 10%
  // when parents carry masks (both layers then skip every back-edge).
  const uint64_t most = static_cast<uint64_t>(all) * rules.kids;
  uint64_t guess = most;
  if (rules.prune && ctl->masked) {
    const uint64_t g = static_cast<uint64_t>(static_cast<double>(all) * (static_cast<double>(C) / F) * 1.1);
    guess = g < most ? g : most;
  }
  n.nsub = queue_sub_buckets(guess);
  n.range_inv = range_inverse(n.nsub);
  n.fb = queue_fine_bits(n.nsub, rules.margin);
  uint32_t state = kLayerNext;
  if (reject) state = kLayerRejected;
  else if (all == 0) state = kLayerEmpty;
  else if (guess <= rules.low || guess > kQueueSub * static_cast<uint64_t>(kQueueTarget)) state = kLayerStop;
  n.F = state == kLayerNext ? all : 0u;
  *next = n;
  rec->N = all;
  rec->cand = C;
  rec->unique = ctl->unique;
  rec->ticks = wall_clock64();
  rec->state = state;
  rec->nbo = nsub << fb;
  __hip_atomic_store(&rec->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

hipError_t sorted_block_run(const BlockRun& run, const PackedGenerators& gens, hipStream_t stream) {
  if (run.cur > 2 || run.prev > kNoBank || run.prev == run.cur || run.F == 0 || run.max_layers == 0 || !run.rec ||
      run.F + (run.prev < kNoBank && !run.L.prune ? run.prev_count : 0u) > kBlockFill / 2)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(block_run_kernel<NibbleAction>, dim3(1), dim3(kBlockThreads), 0, stream, run, NibbleAction{gens});
  return hipGetLastError();
}

hipError_t sorted_start(uint64_t stored, uint64_t* bank, uint32_t* off, uint64_t* control, hipStream_t stream) {
  hipLaunchKernelGGL(sorted_start_kernel, dim3(1), dim3(64), 0, stream, stored, bank, off, control);
  return hipGetLastError();
}

hipError_t sorted_queue_begin(QueueCtl* ctl, const QueueCtl& first, uint32_t* scount, LayerRecord* rec, uint64_t seq,
                              hipStream_t stream) {
  hipLaunchKernelGGL(queue_begin_kernel, dim3(1), dim3(kQueueSub), 0, stream, ctl, first, scount, rec, seq);
  return hipGetLastError();
}

hipError_t sorted_queue_expand(const uint64_t* bank, QueueCtl* ctl, const PackedGenerators& gens,
                               const SortedLayout& L, uint32_t* scount, uint64_t* out, uint32_t items, uint32_t grid,
                               hipStream_t stream) {
  if (grid == 0 || gens.count == 0 || gens.count > kMaxGenerators) return hipErrorInvalidValue;
  const NibbleAction act{gens};
  if (items == 4)
    hipLaunchKernelGGL((queue_expand_kernel<NibbleAction, 4>), dim3(grid), dim3(kRouteThreads), 0, stream, bank, ctl,
                       act, L, scount, out);
  else if (items == 8)
    hipLaunchKernelGGL((queue_expand_kernel<NibbleAction, 8>), dim3(grid), dim3(kRouteThreads), 0, stream, bank, ctl,
                       act, L, scount, out);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t sorted_queue_compact(const uint64_t* cand, const uint32_t* fine_counts, const uint32_t* totals,
                                uint32_t* scount, const QueueCtl* ctl, QueueCtl* next, const QueueRules& rules,
                                uint64_t* bank, uint32_t* off, LayerRecord* rec, uint64_t seq, hipStream_t stream) {
  hipLaunchKernelGGL(queue_compact_kernel, dim3(kQueueSub), dim3(kRouteThreads), 0, stream, cand, fine_counts, totals,
                     scount, ctl, next, rules, bank, off, rec, seq);
  return hipGetLastError();
}

}  // namespace mgbfs
