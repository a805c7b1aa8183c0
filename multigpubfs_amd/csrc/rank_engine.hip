// Host runtime of the permutation bitmap by owners (rank_owner.hip).
// RankRun: one search in memory that its owner gives it; layers are queued
// ahead of the host, which follows their records, and a full message slab
// stops the queue after its layer.  RankBitmapEngine: the bitmap backend for
// degrees 3 to 12 when no row capacity is asked for; after a full slab it
// sends that layer's children again with twice the room.
#include <algorithm>
#include <cstring>
#include <vector>
#include "engine.hpp"
#include "kernels.hpp"
#include "rank_run.hpp"

namespace mgbfs {

// ------------------------------------------------------------ one search

RankRecords::RankRecords() {
  MGBFS_HIP(hipHostMalloc(reinterpret_cast<void**>(&rec), sizeof(LayerRecord) * kRing + 8 * kKeys + 4 * kRankBlockLayers,
                          hipHostMallocDefault));
  keys = reinterpret_cast<uint64_t*>(rec + kRing);
  sizes = reinterpret_cast<uint32_t*>(keys + kKeys);
  std::memset(rec, 0, sizeof(LayerRecord) * kRing);
}
RankRecords::~RankRecords() {
  if (rec) (void)hipHostFree(rec);
}

uint64_t RankRun::words_bytes(const RankPlan& p) {
  return (2 * p.count_stride + kEnds) * 4ull * p.owners + 16 + sizeof(OwnerCtl) * (RankRecords::kRing + 1);
}

uint32_t RankRun::first_cap(const RankPlan& p, uint32_t generators) {
  if (p.owners == 1) return 0;
  const uint64_t fifth = static_cast<uint64_t>(p.list_cap) * generators / 5;
  return std::min(last_cap(p, generators), static_cast<uint32_t>((fifth * (p.degree <= 10 ? 2 : 1) + 1027) / 4 * 4));
}
uint32_t RankRun::last_cap(const RankPlan& p, uint32_t generators) {
  return static_cast<uint32_t>(std::min<uint64_t>(static_cast<uint64_t>(p.list_cap) * generators + 3, 1u << 30) / 4 * 4);
}

static RankGenerators generators_of(const Graph& g) {
  PackedGenerators gens = g.packed_generators();
  if (gens.count <= 14) {
    const std::vector<int> inv = inverse_index(gens);
    for (uint32_t a = 0; a < gens.count; ++a) gens.child_tag[a] = inv[a] >= 0 ? static_cast<uint8_t>(inv[a] + 1) : 0;
  }
  return rank_generators(gens, gens.child_tag);
}

// Children per state but the start: where all have a tag, not the one back.
static uint32_t slots_of(const RankGenerators& gens) {
  return gens.tagged == gens.count && gens.count > 1 ? gens.count - 1 : gens.count;
}

// A child takes the one workgroup 1.4 ns, a layer over 251 owners 8 us: LRX 8
// (81 thousand children, 29 layers) 120 against 228 us, but seven children a
// state in 10 layers 221 against 90.  Degree 7 stays below the line with any
// generators.
uint32_t RankRun::owners_for(const Graph& g) {
  return g.elements <= kRankBlockDegree && factorial_u64(g.elements) * slots_of(generators_of(g)) <= 100000 ? 1 : 0;
}

void RankRun::set_graph(const Graph& g) {
  gens_ = generators_of(g);
  start_key_ = g.start_key();
}

void RankRun::start(hipStream_t stream) {
  const uint64_t W = plan.owners;
  MGBFS_HIP(zero_u32x3(memory.bitmap, W * plan.slice_words, memory.words, (2 * plan.count_stride + kEnds) * W, nullptr, 0,
                       stream));
  MGBFS_HIP(rank_seed(plan, start_key_, memory.bitmap, memory.list, ends(0), stream));
  layers.assign(1, 1);
  sent_ = false;
  seconds = 0.0;
}

OwnerCtl* RankRun::ctl(uint64_t layer) {
  const uint64_t at = ((2 * plan.count_stride + kEnds) * 4ull * plan.owners + 15) / 16 * 16;
  return reinterpret_cast<OwnerCtl*>(reinterpret_cast<char*>(memory.words) + at) + layer % RankRecords::kRing;
}

// Layer d is in the list: sends its children.  Its control block is the
// one the next layer's launch reads.
void RankRun::send(uint64_t d, hipStream_t stream) {
  MGBFS_HIP(owner_begin(counts(0), 2 * plan.count_stride * plan.owners, ctl(d), static_cast<uint32_t>(layers.back()), stream));
  MGBFS_HIP(fill_u32(reinterpret_cast<uint32_t*>(ctl(d + 1)), 0u, sizeof(OwnerCtl) / 4, stream));
  parity_ = 0;
  RankLayer a = layer_args(d, nullptr, 0);
  a.claim = 0;
  a.slots = gens_.count;  // the start has no tag
  a.out = memory.messages[0];
  a.out_count = counts(0);
  MGBFS_HIP(rank_layer(a, gens_, stream));
  sent_ = true;
}

// Arguments of layer d's launch (buffers of the current parity).
RankLayer RankRun::layer_args(uint64_t d, LayerRecord* rec, uint64_t seq) {
  RankLayer a{};
  a.plan = plan;
  a.claim = 1;
  a.slots = slots_of(gens_);
  a.in = memory.messages[parity_];
  a.in_count = counts(parity_);
  a.in_cap = memory.cap;
  a.out = memory.messages[parity_ ^ 1u];
  a.out_count = counts(parity_ ^ 1u);
  a.out_cap = memory.cap;
  a.bitmap = memory.bitmap;
  a.list = memory.list;
  a.ends_before = d ? ends(d - 1) : ends(kEnds - 1);  // zeros before the start layer
  a.ends_now = ends(d);
  a.before = d ? ctl(d - 1) : nullptr;
  a.now = ctl(d);
  a.after = ctl(d + 1);
  a.rules = OwnerRules{plan.owners, ~0u, 0u, ~0u};
  a.rec = rec;
  a.seq = seq;
  return a;
}

// The record of layer d, numbered base + d, is written by the launch of
// layer d + 1, or by a report after the last.
int RankRun::run(uint64_t target, RankRecords& records, hipStream_t stream) {
  if (plan.owners == 1) return run_block(target, records, stream);
  constexpr uint32_t kRing = RankRecords::kRing;
  const uint64_t d0 = layers.size() - 1, base = records.base += 1ull << 32;
  auto rec = [&](uint64_t d) { return records.rec + d % kRing; };
  if (!sent_) send(d0, stream);
  uint64_t queued = d0, ticks = 0;
  for (uint64_t d = d0;; ++d) {
    for (; queued < target && queued <= d + kAheadLayers; ++queued) {
      const RankLayer a = layer_args(queued + 1, rec(queued), base + queued);
      MGBFS_HIP(rank_layer(a, gens_, stream));
      parity_ ^= 1u;
      if (queued + 1 == target) MGBFS_HIP(rank_report(ctl(target), a.rules, rec(target), base + target, stream));
    }
    const LayerRecord& got = await(*rec(d), base + d, stream);
    if (d != d0) {
      seconds += static_cast<double>(got.ticks - ticks) * tick_seconds;
      if (got.state == kLayerRejected) throw std::runtime_error("BITMAP_LAYER");
      if (got.state == kLayerEmpty) return MGBFS_COMPLETE;
      layers.push_back(got.N);
    }
    ticks = got.ticks;
    if (got.state == kLayerStop) {
      sent_ = false;
      return kSendAgain;
    }
    if (d == target) return MGBFS_LAYER;
  }
}

// As run(), by one workgroup.
int RankRun::run_block(uint64_t target, RankRecords& records, hipStream_t stream) {
  while (layers.size() - 1 < target) {
    const uint64_t depth = layers.size() - 1, seq = records.base += 1ull << 32;
    RankBlock a{};
    a.plan = plan;
    a.tagged = slots_of(gens_) != gens_.count;
    a.bitmap = memory.bitmap;
    a.list = memory.list;
    a.ends = ends(0);
    a.depth = static_cast<uint32_t>(depth);
    a.target = static_cast<uint32_t>(std::min<uint64_t>(target, depth + kRankBlockLayers));
    a.sizes = records.sizes;
    a.rec = records.rec;
    a.seq = seq;
    MGBFS_HIP(rank_block(a, gens_, stream));
    const LayerRecord& got = await(*records.rec, seq, stream);
    seconds += static_cast<double>(got.ticks - got.stamps[0]) * tick_seconds;
    for (uint64_t i = 0; i < got.N; ++i) {
      if (records.sizes[i] == 0) return MGBFS_COMPLETE;
      layers.push_back(records.sizes[i]);
    }
  }
  return MGBFS_LAYER;
}

const LayerRecord& RankRun::await(const LayerRecord& rec, uint64_t seq, hipStream_t stream) {
  auto there = [&] { return __atomic_load_n(&rec.seq, __ATOMIC_ACQUIRE) == seq; };
  while (true) {
    for (uint32_t spin = 0; spin < (1u << 18); ++spin)
      if (there()) return rec;
    const hipError_t e = hipStreamQuery(stream);
    if (e == hipErrorNotReady) continue;
    MGBFS_HIP(e);
    if (!there()) throw std::runtime_error("BITMAP_LAYER_RECORD");
  }
}

void RankRun::export_layer(uint64_t back, uint64_t limit, uint64_t* keys, hipStream_t stream) {
  const uint64_t d = layers.size() - 1 - back;
  MGBFS_HIP(rank_export(plan, memory.list, d ? ends(d - 1) : ends(kEnds - 1), ends(d), limit, keys, stream));
}

// ------------------------------------------------------------ groups

// A transitive group with a p-cycle, p prime and more than half the degree, is
// primitive (no block of a system can be moved within p points without
// meeting itself), and a primitive group with a p-cycle, p <= degree - 3,
// holds the alternating group (Jordan).  An element has a p-cycle when a
// power of it is one; in the whole group one in p has.  So: transitivity, then
// random products of the generators (each of a few kept ones multiplied by
// another) until one shows it.
bool reaches_whole_group(const Graph& g) {
  const uint32_t n = g.elements, G = g.generators;
  uint32_t p = 0;
  for (uint32_t q : {5u, 7u})
    if (2 * q > n && q + 3 <= n) p = q;
  if (g.kind != 0 || n > kRankDegree || !p || !G) return false;
  uint32_t reached = 1;
  for (uint32_t before = 0; before != reached;) {
    before = reached;
    for (uint32_t k = 0; k < G; ++k)
      for (uint32_t i = 0; i < n; ++i)
        if ((reached >> i) & 1u) reached |= 1u << g.perms[k * n + i];
  }
  if (reached != (1u << n) - 1) return false;
  bool commute = true;  // a transitive commutative group has n elements
  for (uint32_t a = 0; a < G; ++a)
    for (uint32_t b = 0; b < a && commute; ++b)
      for (uint32_t i = 0; i < n && commute; ++i)
        commute = g.perms[a * n + g.perms[b * n + i]] == g.perms[b * n + g.perms[a * n + i]];
  if (commute) return false;
  constexpr uint32_t kKept = 8, kWarm = 32, kTries = 64;
  uint8_t kept[kKept][kRankDegree];
  for (uint32_t k = 0; k < kKept; ++k)
    for (uint32_t i = 0; i < n; ++i) kept[k][i] = static_cast<uint8_t>(g.perms[(k % G) * n + i]);
  uint32_t random = 1;
  for (uint32_t t = 0; t < kWarm + kTries; ++t) {
    random = random * 1664525u + 1013904223u;
    const uint32_t a = random >> 29, b = (a + 1 + ((random >> 16) % (kKept - 1))) % kKept;
    uint8_t product[kRankDegree];
    for (uint32_t i = 0; i < n; ++i) product[i] = kept[a][kept[b][i]];
    for (uint32_t i = 0; i < n; ++i) kept[a][i] = product[i];
    if (t < kWarm) continue;
    for (uint32_t i = 0, seen = 0; i < n; ++i) {
      uint32_t length = 0;
      for (uint32_t j = i; !((seen >> j) & 1u); j = product[j], ++length) seen |= 1u << j;
      if (length == p) return true;
    }
  }
  return false;
}

// ------------------------------------------------------------ backend

class RankBitmapEngine final : public Engine {
 public:
  RankBitmapEngine(const Graph& g, const mgbfs_engine_options& o) : n_(g.elements), run_(g) {
    device_ = o.device;
    backend = MGBFS_BACKEND_BITMAP;
    set_graph(g);
    MGBFS_HIP(hipSetDevice(device_));
    MGBFS_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    int khz = 0;
    MGBFS_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device_));
    run_.tick_seconds = khz > 0 ? 1e-3 / khz : 0.0;
    take_plan(run_.plan);
    reset();
    ensure_messages(wanted_);
  }
  ~RankBitmapEngine() override {
    (void)hipSetDevice(device_);
    if (stream_) (void)hipStreamSynchronize(stream_);
    if (stream_) (void)hipStreamDestroy(stream_);
  }

  void reset() override {
    MGBFS_HIP(hipSetDevice(device_));
    run_.start(stream_);
    wanted_ = std::max(run_.memory.cap, RankRun::first_cap(run_.plan, run_.generators()));
    layers = run_.layers;
    candidates = unique_candidates = 0;
    kernel_seconds = 0.0;
    launches = 0;
    streamed_bytes = 0;
    terminal = false;
  }

  int advance(uint64_t* next_count, uint32_t* fatal) override {
    if (terminal) throw std::runtime_error("ENGINE_TERMINAL");
    (void)fatal;
    const int s = run_layers(1);
    *next_count = s == MGBFS_LAYER ? layers.back() : 0;
    return s;
  }
  int run_to_end() override {
    int s = MGBFS_LAYER;
    while (!terminal) s = run_layers(~0u);
    return s;
  }
  void rebind(const Graph& g) override {
    if (g.elements != n_ || !g.packable() || !g.distinct_perm()) throw std::runtime_error("ENGINE_REBIND_SHAPE");
    MGBFS_HIP(hipSetDevice(device_));
    const RankPlan p = rank_plan(n_, RankRun::owners_for(g));
    if (p.owners != run_.plan.owners) take_plan(p);
    else ensure_messages(RankRun::first_cap(p, g.generators));  // or the old graph stays
    set_graph(g);
    reset();
    ensure_messages(wanted_);
  }
  void layer_keys(std::vector<uint64_t>& out) override { export_layer(0, layers.back(), out); }
  void sample(uint32_t which, uint64_t limit, std::vector<int64_t>& rows, uint64_t& count) override {
    std::vector<uint64_t> keys;
    if (which == 0) export_layer(0, std::min(limit, layers.back()), keys);
    else if (layers.size() >= 2) export_layer(1, std::min(limit, layers[layers.size() - 2]), keys);
    rows.resize(keys.size() * n_);
    for (size_t k = 0; k < keys.size(); ++k)
      for (uint32_t i = 0; i < n_; ++i) rows[k * n_ + i] = static_cast<int64_t>((keys[k] >> (4u * i)) & 15u);
    count = keys.size();
  }
  const char* name() const override { return "PERMUTATION_BITMAP_LEHMER"; }

 private:
  void set_graph(const Graph& g) {
    run_.set_graph(g);
    history_layers = g.inverse_closed ? 3 : 0;
  }
  // Bitmap, lists and words of a plan, for a reset.  The old ones go when all
  // are there (plans change at the smallest degrees only).
  void take_plan(const RankPlan& p) {
    DeviceBuffer bitmap, list, words;
    bitmap.allocate(4ull * p.owners * p.slice_words);
    list.allocate(4ull * p.owners * p.list_cap);
    words.allocate(RankRun::words_bytes(p));
    MGBFS_HIP(hipStreamSynchronize(stream_));
    run_.drop_messages();
    for (auto& m : messages_) m.release();
    bitmap_ = std::move(bitmap);
    list_ = std::move(list);
    words_ = std::move(words);
    run_.plan = p;
    run_.memory.bitmap = bitmap_.as<uint32_t>();
    run_.memory.list = list_.as<uint32_t>();
    run_.memory.words = words_.as<uint32_t>();
  }
  void update_bytes() {
    device_bytes = bitmap_.bytes() + list_.bytes() + words_.bytes() + messages_[0].bytes() + messages_[1].bytes();
  }
  // Message buffers of `cap` entries per owner.  The old ones go first (two
  // pairs of the worst case need not fit), so they are out of the run's reach
  // before they are freed: when the new ones cannot be had, the run has none,
  // and its next call asks again.
  void ensure_messages(uint32_t cap) {
    if (cap > run_.memory.cap) {
      const uint64_t entries = static_cast<uint64_t>(run_.plan.owners) * cap + kRouteDump;
      MGBFS_HIP(hipStreamSynchronize(stream_));
      run_.drop_messages();
      for (auto& m : messages_) m.release();
      update_bytes();
      for (auto& m : messages_) m.allocate(entries * 4);
      for (int i = 0; i < 2; ++i) run_.memory.messages[i] = messages_[i].as<uint32_t>();
      run_.memory.cap = cap;
    }
    update_bytes();
  }
  int run_layers(uint32_t most) {
    MGBFS_HIP(hipSetDevice(device_));
    const uint64_t target = layers.size() - 1 + most;  // depth to reach
    while (true) {
      ensure_messages(wanted_);
      const int s = run_.run(target, records_, stream_);
      take_layers(s == MGBFS_COMPLETE);
      if (s != RankRun::kSendAgain) return s;
      const uint32_t last = RankRun::last_cap(run_.plan, run_.generators());
      if (run_.memory.cap >= last) throw std::runtime_error("BITMAP_MESSAGES");
      wanted_ = static_cast<uint32_t>(std::min<uint64_t>(2ull * run_.memory.cap, last));
      if (layers.size() - 1 == target) return MGBFS_LAYER;  // its children are sent by the next call
    }
  }
  // The run's new layers: every layer expanded by its launches, an empty one
  // at the end too.
  void take_layers(bool complete) {
    const size_t before = layers.size();
    layers = run_.layers;
    kernel_seconds = run_.seconds;
    terminal = complete;
    for (size_t d = before; d < layers.size() + (terminal ? 1 : 0); ++d) {
      candidates += layers[d - 1] * run_.generators();
      streamed_bytes += 8 * (layers[d - 1] + (d < layers.size() ? layers[d] : 0));
      ++launches;
    }
  }
  // States of the current layer (back = 0) or the one before.
  void export_layer(uint64_t back, uint64_t limit, std::vector<uint64_t>& out) {
    MGBFS_HIP(hipSetDevice(device_));
    out.resize(limit);
    if (!limit) return;
    if (limit <= RankRecords::kKeys) {  // written to pinned memory by the kernel
      run_.export_layer(back, limit, records_.keys, stream_);
      MGBFS_HIP(hipStreamSynchronize(stream_));
      std::copy(records_.keys, records_.keys + limit, out.begin());
      return;
    }
    // Through the idle message buffer where it holds them: a layer that was
    // found is also read where no more device memory is left.
    uint64_t room = 0;
    uint64_t* to = run_.spare(&room);
    DeviceBuffer keys;
    if (limit > room) {
      keys.allocate(limit * 8);
      to = keys.as<uint64_t>();
    }
    run_.export_layer(back, limit, to, stream_);
    MGBFS_HIP(hipMemcpyAsync(out.data(), to, limit * 8, hipMemcpyDeviceToHost, stream_));
    MGBFS_HIP(hipStreamSynchronize(stream_));
  }

  uint32_t n_;
  RankRun run_;
  RankRecords records_;
  DeviceBuffer bitmap_, list_, words_, messages_[2];
  uint32_t wanted_ = 0;  // messages per owner that the next layers need
};

uint64_t rank_bitmap_bytes(const Graph& g) {
  const RankPlan p = rank_plan(g.elements, RankRun::owners_for(g));
  const uint64_t messages = p.owners == 1 ? 0 : p.owners * static_cast<uint64_t>(RankRun::last_cap(p, g.generators)) + kRouteDump;
  return p.owners * (4ull * p.slice_words + 4ull * p.list_cap) + RankRun::words_bytes(p) + 2 * 4 * messages;
}

// All degrees that ranks and slices are made for: faster from the smallest to
// degree 12 (figures in rank_owner.hip).  A capacity bounds the rows of a
// layer and a message buffer is not one, so a set capacity keeps the shared
// bitmap; so does a budget that does not hold the messages of every layer
// (degree 12 with three generators: 13.5 GB, of which 4.3 are used).  The
// buffers are made for the whole group, 0.3 GB at degree 11 and 4.3 at 12, so
// generators that are not seen to reach it keep the other form there (two
// swaps of S_12, four states: 76 to 140 ms to create, run and drop an engine
// in a process that has used some memory, against 1.7).
bool rank_bitmap_takes(const Graph& g, const mgbfs_engine_options& o, uint64_t held) {
  if (g.elements < 3 || g.elements > kRankDegree || o.capacity || g.generators > kMaxGenerators) return false;
  if (g.elements >= 11 && !reaches_whole_group(g)) return false;
  if (!o.vram_budget) MGBFS_HIP(hipSetDevice(o.device));
  return rank_bitmap_bytes(g) <= vram_budget(o) + (o.vram_budget ? 0 : held);
}

// Inverse-closed graphs whose backend the library picks run by owners of the
// bitmap (sorted -> owners, warm: LRX 4 0.037 -> 0.014 ms, 7 0.145 -> 0.038,
// 8 0.36 -> 0.12, 9 0.42 -> 0.31, 10 0.65 -> 0.48, 11 2.5 -> 1.3, 12 13.5 ->
// 10.5; Coxeter 6 0.11 -> 0.02, 11 5.5 -> 3.0, 12 96 -> 33; four random
// generators with inverses, 11 5.1 -> 1.9).
// A set that is only declared closed keeps the sorted backend's retention.
bool rank_bitmap_for_auto(const Graph& g, const mgbfs_engine_options& o, uint64_t held) {
  if (o.backend != MGBFS_BACKEND_AUTO || !g.inverse_closed || !g.packable() || !g.distinct_perm() ||
      (o.flags & ~MGBFS_FLAG_MAX_CAPACITY) || !rank_bitmap_takes(g, o, held))
    return false;
  for (int at : inverse_index(g.packed_generators()))
    if (at < 0) return false;
  return true;
}

Engine* make_rank_bitmap_engine(const Graph& g, const mgbfs_engine_options& o) { return new RankBitmapEngine(g, o); }

}  // namespace mgbfs
