// Host runtime of the permutation bitmap by owners (rank_owner.hip): the
// bitmap backend for degrees 3 to 12 when no row capacity is asked for.
// Layers are queued ahead of the host, which follows their records; a full
// message slab stops the queue after its layer, and the host sends that
// layer's children again with twice the room.
#include <algorithm>
#include <cstring>
#include <vector>
#include "engine.hpp"
#include "kernels.hpp"

namespace mgbfs {

namespace {

constexpr uint32_t kRing = 64;   // control blocks and records
constexpr uint32_t kAheadLayers = 4;
constexpr uint32_t kEnds = 4;    // list ends kept: of the last layers
constexpr int kSendAgain = -1;

}  // namespace

class RankBitmapEngine final : public Engine {
 public:
  RankBitmapEngine(const Graph& g, const mgbfs_engine_options& o) : n_(g.elements), plan_(rank_plan(g.elements)) {
    device_ = o.device;
    backend = MGBFS_BACKEND_BITMAP;
    set_graph(g);
    MGBFS_HIP(hipSetDevice(device_));
    MGBFS_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    int khz = 0;
    MGBFS_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device_));
    tick_seconds_ = khz > 0 ? 1e-3 / khz : 0.0;
    const uint64_t W = plan_.owners;
    bitmap_.allocate(W * plan_.slice_words * 4);
    list_.allocate(W * plan_.list_cap * 4);
    // Counts of both message buffers, then the list ends, then the controls.
    words_.allocate((2 * plan_.count_stride + kEnds) * W * 4 + 16 + sizeof(OwnerCtl) * (kRing + 1));
    keys_.allocate(kKeys * 8);
    MGBFS_HIP(hipHostMalloc(reinterpret_cast<void**>(&rec_), sizeof(LayerRecord) * kRing, hipHostMallocDefault));
    std::memset(rec_, 0, sizeof(LayerRecord) * kRing);
    ensure_messages(first_cap(plan_, g.generators));
    reset();
  }
  ~RankBitmapEngine() override {
    (void)hipSetDevice(device_);
    if (stream_) (void)hipStreamSynchronize(stream_);
    if (rec_) (void)hipHostFree(rec_);
    if (stream_) (void)hipStreamDestroy(stream_);
  }

  // Device bytes with message buffers that hold every layer.
  static uint64_t most_bytes(const Graph& g) {
    const RankPlan p = rank_plan(g.elements);
    return p.owners * (4ull * p.slice_words + 4ull * p.list_cap + 8ull * last_cap(p, g.generators)) + (1u << 20);
  }

  void reset() override {
    MGBFS_HIP(hipSetDevice(device_));
    const uint64_t W = plan_.owners;
    MGBFS_HIP(zero_u32x3(bitmap_.as<uint32_t>(), W * plan_.slice_words, words_.as<uint32_t>(), (2 * plan_.count_stride + kEnds) * W, nullptr,
                         0, stream_));
    MGBFS_HIP(rank_seed(plan_, start_key_, bitmap_.as<uint32_t>(), list_.as<uint32_t>(), ends(0), stream_));
    layers.assign(1, 1);
    sent_ = false;
    candidates = unique_candidates = 0;
    kernel_seconds = 0.0;
    launches = 0;
    streamed_bytes = 0;
    terminal = false;
    update_bytes();
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
    set_graph(g);
    reset();
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
  static constexpr uint64_t kKeys = 1024;
  // Messages per owner at first: a fifth of all children there can be (the
  // widest LRX layer sends 15% of them).
  static uint32_t first_cap(const RankPlan& p, uint32_t generators) {
    return std::min(last_cap(p, generators),
                    static_cast<uint32_t>((static_cast<uint64_t>(p.list_cap) * generators / 5 + 1027) / 4 * 4));
  }
  // ... and at most: a state is a child of `generators` states.
  static uint32_t last_cap(const RankPlan& p, uint32_t generators) {
    return static_cast<uint32_t>(std::min<uint64_t>(static_cast<uint64_t>(p.list_cap) * generators + 3, 1u << 30) / 4 * 4);
  }
  void set_graph(const Graph& g) {
    gens_ = g.packed_generators();
    if (gens_.count <= 14) {
      const std::vector<int> inv = inverse_index(gens_);
      for (uint32_t a = 0; a < gens_.count; ++a) gens_.child_tag[a] = inv[a] >= 0 ? static_cast<uint8_t>(inv[a] + 1) : 0;
    }
    rank_gens_ = rank_generators(gens_);
    history_layers = g.inverse_closed ? 3 : 0;
    start_key_ = g.start_key();
  }
  uint32_t* counts(uint32_t parity) { return words_.as<uint32_t>() + parity * plan_.count_stride * plan_.owners; }
  uint32_t* ends(uint64_t layer) { return words_.as<uint32_t>() + (2 * plan_.count_stride + layer % kEnds) * plan_.owners; }
  OwnerCtl* ctl(uint64_t layer) {
    const uint64_t at = ((2 * plan_.count_stride + kEnds) * 4ull * plan_.owners + 15) / 16 * 16;
    return reinterpret_cast<OwnerCtl*>(words_.as<char>() + at) + layer % kRing;
  }
  void ensure_messages(uint32_t cap) {
    if (cap <= cap_) return;
    const uint64_t entries = static_cast<uint64_t>(plan_.owners) * cap + kRouteDump;
    MGBFS_HIP(hipStreamSynchronize(stream_));
    for (auto& m : messages_) m.release();
    for (auto& m : messages_) m.allocate(entries * 4);
    cap_ = cap;
    update_bytes();
  }
  // Layer d is in the list: sends its children.  Its control block is the
  // one the next layer's launch reads.
  void send(uint64_t d) {
    MGBFS_HIP(owner_begin(counts(0), 2 * plan_.count_stride * plan_.owners, ctl(d), static_cast<uint32_t>(layers.back()), stream_));
    MGBFS_HIP(fill_u32(reinterpret_cast<uint32_t*>(ctl(d + 1)), 0u, sizeof(OwnerCtl) / 4, stream_));
    parity_ = 0;
    RankLayer a = layer_args(d);
    a.claim = 0;
    a.slots = gens_.count;  // the start has no tag
    a.out = messages_[0].as<uint32_t>();
    a.out_count = counts(0);
    MGBFS_HIP(rank_layer(a, rank_gens_, stream_));
    sent_ = true;
  }
  // Arguments of layer d's launch (buffers of the current parity).
  RankLayer layer_args(uint64_t d) {
    RankLayer a{};
    a.plan = plan_;
    a.claim = 1;
    a.slots = rank_gens_.tagged == gens_.count && gens_.count > 1 ? gens_.count - 1 : gens_.count;
    a.in = messages_[parity_].as<uint32_t>();
    a.in_count = counts(parity_);
    a.in_cap = cap_;
    a.out = messages_[parity_ ^ 1u].as<uint32_t>();
    a.out_count = counts(parity_ ^ 1u);
    a.out_cap = cap_;
    a.bitmap = bitmap_.as<uint32_t>();
    a.list = list_.as<uint32_t>();
    a.ends_before = d ? ends(d - 1) : ends(kEnds - 1);  // zeros before the start layer
    a.ends_now = ends(d);
    a.before = d ? ctl(d - 1) : nullptr;
    a.now = ctl(d);
    a.after = ctl(d + 1);
    a.rules = OwnerRules{plan_.owners, ~0u, 0u, ~0u};
    a.rec = rec_ + (d ? d - 1 : 0) % kRing;
    a.seq = base_ + (d ? d - 1 : 0);
    return a;
  }
  int run_layers(uint32_t most) {
    MGBFS_HIP(hipSetDevice(device_));
    ensure_messages(first_cap(plan_, gens_.count));
    const uint64_t target = layers.size() - 1 + most;  // depth to reach
    while (true) {
      const int s = session(target);
      if (s != kSendAgain) return s;
      const uint32_t last = last_cap(plan_, gens_.count);
      if (cap_ >= last) throw std::runtime_error("BITMAP_MESSAGES");
      ensure_messages(std::min(2 * cap_, last));
      if (layers.size() - 1 == target) return MGBFS_LAYER;  // its children are sent by the next call
    }
  }
  // Layers up to depth `target`, or the end, or a layer whose children did
  // not fit the message slabs (kSendAgain: whatever was queued after it did
  // nothing).  The record of layer d, numbered base_ + d, is written by the
  // launch of layer d + 1, or by a report after the last.
  int session(uint64_t target) {
    const uint64_t d0 = layers.size() - 1;
    base_ += 1ull << 32;
    if (!sent_) send(d0);
    uint64_t queued = d0, ticks = 0;
    for (uint64_t d = d0;; ++d) {
      for (; queued < target && queued <= d + kAheadLayers; ++queued) {
        const RankLayer a = layer_args(queued + 1);
        MGBFS_HIP(rank_layer(a, rank_gens_, stream_));
        parity_ ^= 1u;
        if (queued + 1 == target)
          MGBFS_HIP(rank_report(ctl(target), a.rules, rec_ + target % kRing, base_ + target, stream_));
      }
      const LayerRecord& rec = await(rec_[d % kRing], base_ + d);
      if (d != d0) {
        kernel_seconds += static_cast<double>(rec.ticks - ticks) * tick_seconds_;
        candidates += layers.back() * gens_.count;
        streamed_bytes += 8 * (layers.back() + rec.N);
        ++launches;
        if (rec.state == kLayerRejected) throw std::runtime_error("BITMAP_LAYER");
        if (rec.state == kLayerEmpty) {
          terminal = true;
          return MGBFS_COMPLETE;
        }
        layers.push_back(rec.N);
      }
      ticks = rec.ticks;
      if (rec.state == kLayerStop) {
        sent_ = false;
        return kSendAgain;
      }
      if (d == target) return MGBFS_LAYER;
    }
  }
  const LayerRecord& await(const LayerRecord& rec, uint64_t seq) {
    auto there = [&] { return __atomic_load_n(&rec.seq, __ATOMIC_ACQUIRE) == seq; };
    while (true) {
      for (uint32_t spin = 0; spin < (1u << 18); ++spin)
        if (there()) return rec;
      const hipError_t e = hipStreamQuery(stream_);
      if (e == hipErrorNotReady) continue;
      MGBFS_HIP(e);
      if (!there()) throw std::runtime_error("BITMAP_LAYER_RECORD");
    }
  }
  // States of the current layer (back = 0) or the one before.
  void export_layer(uint64_t back, uint64_t limit, std::vector<uint64_t>& out) {
    MGBFS_HIP(hipSetDevice(device_));
    const uint64_t d = layers.size() - 1 - back;
    DeviceBuffer large;
    if (limit > kKeys) large.allocate(limit * 8);
    uint64_t* keys = limit > kKeys ? large.as<uint64_t>() : keys_.as<uint64_t>();
    out.resize(limit);
    if (!limit) return;
    MGBFS_HIP(rank_export(plan_, list_.as<uint32_t>(), d ? ends(d - 1) : ends(kEnds - 1), ends(d), limit, keys, stream_));
    MGBFS_HIP(hipMemcpyAsync(out.data(), keys, limit * 8, hipMemcpyDeviceToHost, stream_));
    MGBFS_HIP(hipStreamSynchronize(stream_));
  }
  void update_bytes() {
    device_bytes = bitmap_.bytes() + list_.bytes() + words_.bytes() + keys_.bytes() + messages_[0].bytes() +
                   messages_[1].bytes();
  }

  uint32_t n_;
  RankPlan plan_;
  PackedGenerators gens_{};
  RankGenerators rank_gens_{};
  uint64_t start_key_ = 0;
  DeviceBuffer bitmap_, list_, words_, keys_, messages_[2];
  uint32_t cap_ = 0, parity_ = 0;  // messages per owner; the buffer holding the current layer's children
  bool sent_ = false;              // ... which are complete
  uint64_t base_ = 0;
  double tick_seconds_ = 0.0;
  LayerRecord* rec_ = nullptr;     // pinned
};

// All degrees that ranks and slices are made for: faster from the smallest to
// degree 12 (figures in rank_owner.hip).  A capacity bounds the rows of a
// layer and a message buffer is not one, so a set capacity keeps the shared
// bitmap; so does a budget that does not hold the messages of every layer
// (degree 12 with three generators: 13.5 GB, of which 4.3 are used).
bool rank_bitmap_takes(const Graph& g, const mgbfs_engine_options& o) {
  if (g.elements < 3 || g.elements > kRankDegree || o.capacity || g.generators > kMaxGenerators) return false;
  MGBFS_HIP(hipSetDevice(o.device));
  return RankBitmapEngine::most_bytes(g) <= vram_budget(o);
}

// Inverse-closed graphs whose backend the library picks run by owners of the
// bitmap from degree 8 on (sorted -> owners, warm: LRX 8 0.36 -> 0.23 ms, 9
// 0.47 -> 0.31, 10 0.65 -> 0.48, 11 2.9 -> 1.3, 12 13.7 -> 10.5; Coxeter 11
// 5.5 -> 3.0, 12 96 -> 33; four random generators with inverses, 11 4.9 ->
// 1.8); below, the sorted backend's single workgroup does (LRX 7 0.145
// against 0.162 ms, 4 0.036 against 0.054).
// A set that is only declared closed keeps the sorted backend's retention.
bool rank_bitmap_for_auto(const Graph& g, const mgbfs_engine_options& o) {
  if (o.backend != MGBFS_BACKEND_AUTO || !g.inverse_closed || g.elements < 8 || !g.packable() || !g.distinct_perm() ||
      (o.flags & ~MGBFS_FLAG_MAX_CAPACITY) || !rank_bitmap_takes(g, o))
    return false;
  for (int at : inverse_index(g.packed_generators()))
    if (at < 0) return false;
  return true;
}

Engine* make_rank_bitmap_engine(const Graph& g, const mgbfs_engine_options& o) { return new RankBitmapEngine(g, o); }

}  // namespace mgbfs
