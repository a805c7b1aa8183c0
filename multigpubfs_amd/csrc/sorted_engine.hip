// Host runtime of the sort-unique backend with rotating VRAM banks.
//
// Layer loop (one host readback per layer, plus a retry when a slab
// overflows): expand+route into owner-lane slabs -> partition into
// sub-bucket slabs -> unique_diff -> scan of fine counts -> compact into
// the next bank (queued before the host reads N) -> read N -> rotate.
// Retention is exact for inverse-closed generator sets: every neighbour of
// layer d lies in layer d-1, d or d+1 (graph_definition.py:84-92; retention
// rule history_layers = 3, crates/mgbfs-runtime/src/generic_distributed_run.rs:40).
// With back-edge masks (G <= tagbits - 2) each stored state carries the set
// of generators leading back to layer d-1 -- the OR over all the duplicate
// candidates that discovered it -- and expansion skips them, so every child
// lies in layer d or d+1 and only the current bank is probed.  Otherwise
// nothing is skipped and both retained banks are probed.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include "engine.hpp"
#include "kernels.hpp"
#include "sorted_plan.hpp"
#include "wide.hpp"

namespace mgbfs {

namespace {

// Phases: expand, partition, unique, compact.  Layers run ahead of the host
// (sorted_queue.hip) are one kernel each and count in the first.
constexpr uint32_t kPhaseCount = 4;
constexpr size_t kCtlOffset = 64;       // in control_: the owner layers' control ring, then their slab counts
constexpr uint32_t kOwnerRing = 64;     // owner layers' control blocks and records
constexpr uint32_t kOwnerAhead = 3;     // layers queued beyond the one whose record the host waits for
constexpr uint32_t kOwnerBuffers = 5;   // slab arrays: two of candidates, three of layers
constexpr uint32_t kBlockLayers = 126;  // layers per one-workgroup launch at most
constexpr uint64_t kAheadRows = 1ull << 22;  // bank rows reserved for layers run ahead
constexpr int kAheadNone = -1;          // run_ahead(): the next layer is one for the general path

}  // namespace

class SortedEngine final : public Engine {
 public:
  // wide: the graph's packed code when it is outside the nibble encoding.
  SortedEngine(const Graph& g, const mgbfs_engine_options& o, const WideCode* wide) : n_(g.elements) {
    if (wide) wide_ = std::make_unique<WideCode>(*wide);
    device_ = o.device;
    backend = MGBFS_BACKEND_SORTED;
    history_layers = 3;
    if (!g.inverse_closed) throw std::runtime_error("SORTED_REQUIRES_INVERSE_CLOSED");
    MGBFS_HIP(hipSetDevice(device_));
    MGBFS_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    budget_ = vram_budget(o);
    bound_ = state_space_bound(g);
    cap_limit_ = o.capacity ? o.capacity : ~0ull;
    // The segmented tables hold no layer beyond the state bound (and a quarter,
    // by which their arenas grow): such a layer goes there and ends the run.
    if (wide_ && bound_) cap_limit_ = std::min(cap_limit_, bound_ + bound_ / 4);
    flags_ = o.flags;
    // Stored-value layout and parent-edge tags.
    const uint32_t key_bits = wide_ ? std::max(32u, wide_->key_bits()) : sorted_key_bits(n_);
    layout_.km = make_keymix(key_bits, wide_ != nullptr);
    layout_.tagbits = 64 - key_bits;
    layout_.tagmask = layout_.tagbits ? ((1ull << layout_.tagbits) - 1) : 0;
    set_generators(g);
    // One workgroup per sub-bucket: persistent grids of 2 or 8 workgroups
    // per CU, prefetching the next sub-bucket's bounds, measured slower
    // (127 and 122 vs 120 ms per S13 BFS).
    unique_grid_ = 1u << kMaxBucketBits;
    control_.allocate(kCtlOffset + sizeof(OwnerCtl) * kOwnerRing + 4 * kOwnerBuffers * kOwnersMax * kCountStride);
    fine_counts_.allocate(((1ull << kMaxBucketBits) + 1) * 4);
    for (int b = 0; b < 3; ++b) off_[b].allocate(((1ull << kMaxBucketBits) + 1) * 4);
    const size_t rec_bytes = sizeof(LayerRecord) * (kBlockLayers + 1);
    MGBFS_HIP(hipHostMalloc(reinterpret_cast<void**>(&rec_), rec_bytes, hipHostMallocDefault));
    std::memset(rec_, 0, rec_bytes);
    int khz = 0;
    MGBFS_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device_));
    tick_seconds_ = khz > 0 ? 1e-3 / khz : 0.0;
    // Test flags that force a mechanism of the general path keep to it.
    general_only_ = flags_ & (MGBFS_FLAG_TEST_COARSE_BUCKETS | MGBFS_FLAG_TEST_TIGHT_SLABS |
                              MGBFS_FLAG_TEST_WIDE_ROUTING | MGBFS_FLAG_TEST_SORTED_CAP);
    update_bytes();
    reset();
  }

  ~SortedEngine() override {
    (void)hipSetDevice(device_);
    if (stream_) (void)hipStreamSynchronize(stream_);
    if (rec_) (void)hipHostFree(rec_);
    if (stream_) (void)hipStreamDestroy(stream_);
  }

  void reset() override {
    MGBFS_HIP(hipSetDevice(device_));
    if (!grow_bank(0, 1024)) throw std::runtime_error("SORTED_VRAM_CAPACITY");
    cur_ = 0;
    prev_ = -1;
    slack_ = (flags_ & MGBFS_FLAG_TEST_TIGHT_SLABS) ? 0 : 1;
    last_ratio_ = 0.0;
    for (int b = 0; b < 3; ++b) count_[b] = 0;
    count_[0] = 1;
    nbo_[0] = 1;  // the start bank has one fine bucket
    block_rejected_ = owner_rejected_ = 0;
    start_bank();
    compacted_ = 0;
    layers.assign(1, 1);
    candidates = unique_candidates = 0;
    kernel_seconds = 0.0;
    launches = 0;
    streamed_bytes = 0;
    for (auto& t : phase_seconds) t = 0.0;
    for (auto& b : phase_bytes) b = 0;
    retries = 0;
    terminal = false;
    update_bytes();
  }

  int advance(uint64_t* next_count, uint32_t* fatal) override {
    if (terminal) throw std::runtime_error("ENGINE_TERMINAL");
    MGBFS_HIP(hipSetDevice(device_));
    const int s = run_ahead(1);
    if (s == kAheadNone) return advance_general(next_count, fatal);
    *next_count = s == MGBFS_LAYER ? layers.back() : 0;
    return s;
  }

  int run_to_end() override {
    int s = MGBFS_LAYER;
    if (!terminal) MGBFS_HIP(hipSetDevice(device_));
    while (!terminal) {
      s = run_ahead(kBlockLayers);
      if (s != kAheadNone) continue;
      uint64_t nc;
      uint32_t f;
      s = advance_general(&nc, &f);
      if (s == kAdvanceHandover) return s;
    }
    return s;
  }

 private:
  // One layer with its geometry set by the host: every size, owner lanes
  // above 2^10 sub-buckets, retries after overflows.
  int advance_general(uint64_t* next_count, uint32_t* fatal) {
    const uint64_t F = count_[cur_];
    const uint32_t G = gens_.count;
    // Every parent yields at most G children, at most G-1 when it carries a
    // back-edge mask (every state but the start does); the slabs, the
    // sub-bucket count and the 32-bit candidate bound use that bound.
    const bool masked = layout_.prune && layers.size() > 1;
    const uint64_t Cmax = masked ? F * (G > 1 ? G - 1 : 1) : F * G;
    // Beyond 32-bit candidate counts the run continues on the segmented
    // backend (a test flag lowers the limit to 2^18 children).
    if (Cmax > ((flags_ & MGBFS_FLAG_TEST_SORTED_CAP) ? (1ull << 18) : 0xfffffff0ull)) return kAdvanceHandover;
    const int nxt = next_bank();
    uint64_t Cest = Cmax;
    // Masked layers skip every back-edge, so the previous layer's measured
    // children per parent (plus 10%) predicts this one closely; a low guess
    // costs one retry of the layer (slab or sub-bucket overflow).
    if (masked && last_ratio_ > 0)
      Cest = std::min<uint64_t>(Cest, static_cast<uint64_t>(static_cast<double>(F) * last_ratio_ * 1.1) + 4096);
    const uint64_t kMaxSub = 1ull << kMaxBucketBits;
    uint64_t want = sub_buckets_for(Cest, wide_ ? kTargetBucketWide : kTargetBucket);
    // Test hook: start eight times coarse so large layers exercise the
    // bucket-overflow retry path.
    if ((flags_ & MGBFS_FLAG_TEST_COARSE_BUCKETS) && want >= 8) want >>= 3;
    const bool probe_prev = prev_ >= 0 && !layout_.prune;
    while (true) {
      const SortedGeometry geo = sorted_geometry(want, F, Cest, slack_, margin_);
      const uint32_t K2 = geo.K2, nsub = geo.nsub, NB1 = geo.NB1, P = geo.P, lcap = geo.lcap;
      const uint64_t lslabs = geo.lslabs, lane_entries = geo.lane_entries, sub_entries = geo.sub_entries;
      if (!ensure_slabs(lane_entries + kRouteDump, sub_entries + kRouteDump)) {
        return out_of_room(fatal, kErrFutureCap);
      }
      ensure_u32(lcount_, lslabs);
      ensure_u32(scount_, nsub);
      ensure_u32(scan_ws_, scan_workspace_words(1ull << kMaxBucketBits) + 16);
      const uint32_t fb = geo.fb, nbo = geo.nbo;
      // Counters (unique, error, candidates), sub-bucket and lane cursors.
      // The kernels stamp their start times: eight timing events took 4.5 us
      // each on the stream.
      MGBFS_HIP(zero_u32x3(reinterpret_cast<uint32_t*>(control_.as<uint64_t>()), 6, scount_.as<uint32_t>(), nsub,
                           lcount_.as<uint32_t>(), K2 ? lslabs : 0, stream_, &counters()->stamps[0]));
      uint64_t* sub = sub_.as<uint64_t>();
      const uint32_t stride = K2 ? lcap : kSlabStride, full = K2 ? kErrLaneSlab : kErrBucketCap;
      uint32_t* cursors = K2 ? lcount_.as<uint32_t>() : scount_.as<uint32_t>();
      uint64_t* routed_to = K2 ? lane_.as<uint64_t>() : sub;
      const uint64_t routed_entries = routed(K2 ? lane_entries : sub_entries);
      if (wide_)
        MGBFS_HIP(sorted_expand_route_wide(bank_[cur_].as<uint64_t>(), F, action(), layout_, masked, nsub, K2, NB1, P,
                                           lcap, stride, full, cursors, error_word(), routed_to, routed_entries,
                                           stream_));
      else
        MGBFS_HIP(sorted_expand_route(bank_[cur_].as<uint64_t>(), F, gens_, layout_, masked, nsub, K2, NB1, P, lcap,
                                      stride, full, cursors, error_word(), routed_to, routed_entries, stream_));
      if (K2)
        MGBFS_HIP(sorted_partition(lane_.as<uint64_t>(), lcount_.as<uint32_t>(), lcap, P, nsub, K2,
                                   scount_.as<uint32_t>(), error_word(), sub, routed(sub_entries), stream_,
                                   &counters()->stamps[1]));
      auto* control = reinterpret_cast<unsigned long long*>(control_.as<uint64_t>());
      MGBFS_HIP(sorted_unique_diff(
          sub, scount_.as<uint32_t>(), nsub, bank_[cur_].as<uint64_t>(), off_[cur_].as<uint32_t>(), nbo_[cur_],
          probe_prev ? bank_[prev_].as<uint64_t>() : nullptr, probe_prev ? off_[prev_].as<uint32_t>() : nullptr,
          probe_prev ? nbo_[prev_] : 0, fb, fine_counts_.as<uint32_t>(), error_word(), control, control + 2,
          layout_.tagbits, layout_.prune != 0, unique_grid_, stream_, &counters()->stamps[2]));
      // The scan reports the layer (N, error word, counters) in pinned memory.
      const uint64_t seq = seq_++;
      MGBFS_HIP(exclusive_scan_u32(fine_counts_.as<uint32_t>(), nbo, off_[nxt].as<uint32_t>(),
                                   scan_ws_.as<uint32_t>(), stream_, counters(), rec_, seq));
      // The compaction is queued before the host has read N or the error
      // word; it writes nothing unless the layer is clean and fits the bank
      // as allocated now, and the host relaunches it after growing the bank.
      // The host wakes on the record alone, so its turnaround and the next
      // layer's launches overlap the compaction.
      const uint64_t early_rows = bank_cap_[nxt];
      if (early_rows) compact(sub, nsub, fb, nxt);
      const LayerRecord rec = await(rec_[0], seq);
      const uint32_t err = rec.state;
      const uint64_t C = rec.children, N = rec.N;
      account(rec, F, probe_prev ? count_[prev_] : 0, K2 != 0);
      if (err & kErrLaneSlab) {  // lane slab overflow: retry with twice the slack
        slack_ = slack_ ? 2 * slack_ : 1;
        ++retries;
        continue;
      }
      if (err & kErrBucketCap) {  // a sub-bucket overflowed: twice as many
        if (want < kMaxSub) {
          want = std::min(kMaxSub, 2 * want);
          ++retries;
          continue;
        }
      }
      if (err) return out_of_room(fatal, err);
      candidates += C;
      last_ratio_ = masked ? static_cast<double>(C) / static_cast<double>(F) : 0.0;
      unique_candidates += rec.unique;
      if (N == 0) {
        *next_count = 0;
        terminal = true;
        return MGBFS_COMPLETE;
      }
      if (N > cap_limit_ || !grow_bank(nxt, N)) return out_of_room(fatal, kErrFutureCap);
      if (N > early_rows) compact(sub, nsub, fb, nxt);
      phase_bytes[3] += 16 * N;
      streamed_bytes += 16 * N;
      launches += 1;
      nbo_[nxt] = nbo;
      count_[nxt] = N;
      prev_ = cur_;
      cur_ = nxt;
      layers.push_back(N);
      *next_count = N;
      update_bytes();
      return MGBFS_LAYER;
    }
  }

 public:
  // Another inverse-closed graph of the same degree reuses every bank and slab.
  void rebind(const Graph& g) override {
    if (wide_ || g.elements != n_ || !g.packable() || !g.inverse_closed) throw std::runtime_error("ENGINE_REBIND_SHAPE");
    set_generators(g);
    reset();
  }

  bool handover(PackedHandover& h) override {
    MGBFS_HIP(hipStreamSynchronize(stream_));
    settle();
    lane_.release();
    sub_.release();
    owner_.release();
    lane_cap_ = sub_cap_ = 0;
    const int spare = next_bank();
    bank_cap_[spare] = 0;
    bank_[spare].release();
    h.wide = wide_.get();
    h.cur = bank_[cur_].as<uint64_t>();
    h.cur_count = count_[cur_];
    h.prev = prev_ >= 0 ? bank_[prev_].as<uint64_t>() : nullptr;
    h.prev_count = prev_ >= 0 ? count_[prev_] : 0;
    h.km = layout_.km;
    h.tagbits = layout_.tagbits;
    h.layers = layers;
    update_bytes();
    h.held = device_bytes;
    return true;
  }

  void layer_keys(std::vector<uint64_t>& out) override { read_bank(cur_, count_[cur_], out); }

  void sample(uint32_t which, uint64_t limit, std::vector<int64_t>& rows, uint64_t& count) override {
    std::vector<uint64_t> keys;
    if (which == 0) read_bank(cur_, std::min(limit, count_[cur_]), keys);
    else if (prev_ >= 0) read_bank(prev_, std::min(limit, count_[prev_]), keys);
    rows.resize(keys.size() * n_);
    for (size_t k = 0; k < keys.size(); ++k)
      for (uint32_t i = 0; i < n_; ++i)
        rows[k * n_ + i] = wide_ ? wide_->value(keys[k], i) : static_cast<int64_t>((keys[k] >> (4u * i)) & 15u);
    count = keys.size();
  }

  const char* name() const override { return "SORTED_THREE_BANK_LDS_UNIQUE"; }
  uint64_t retry_count() const override { return retries; }

  void settle() override {
    if (!compacted_) return;
    MGBFS_HIP(hipSetDevice(device_));
    const uint64_t seq = seq_++;
    MGBFS_HIP(stamp_record(rec_, counters(), seq, stream_));
    end_compaction(await(rec_[0], seq));
  }

  void memory_returned(uint64_t bytes) override { budget_ += bytes; }

  double phase_seconds[kPhaseCount] = {};
  uint64_t phase_bytes[kPhaseCount] = {};
  uint64_t retries = 0;

  void fill_phases(double* seconds, uint64_t* bytes, uint32_t n) const override {
    for (uint32_t i = 0; i < n && i < kPhaseCount; ++i) {
      seconds[i] = phase_seconds[i];
      bytes[i] = phase_bytes[i];
    }
  }

 private:
  // Bank rows for the layers run ahead, so that they need no growth: what one
  // workgroup's table holds at the start; with the first owner layer as many
  // as the state space has, at most kAheadRows (a search that stays small
  // never pays for three 32 MB banks: rotations of 15 created and run 1.9 ms
  // with them from the start, 0.3 without).  Without the memory for it (an
  // eighth of the budget at most, so that larger layers find theirs) the
  // layers take the general path.
  void reserve_banks(uint64_t rows, uint64_t beside) {
    if (8 * (3 * rows + beside) > budget_ / 8) return;
    for (int b = 0; b < 3; ++b)
      if (!widen_bank(b, rows)) return;
  }
  uint64_t owner_rows() const {
    return std::max<uint64_t>(2 * kBlockParents, std::min({bound_ ? bound_ : kAheadRows, cap_limit_, kAheadRows}));
  }
  // grow_bank() with the layer in it kept.
  bool widen_bank(int b, uint64_t rows) {
    if (bank_cap_[b] >= rows) return true;
    if (!fits(rows * 8)) return false;
    DeviceBuffer fresh;
    fresh.allocate(rows * 8);
    if ((b == cur_ || b == prev_) && count_[b])
      MGBFS_HIP(hipMemcpyAsync(fresh.as<uint64_t>(), bank_[b].as<uint64_t>(), count_[b] * 8, hipMemcpyDeviceToDevice,
                               stream_));
    MGBFS_HIP(hipStreamSynchronize(stream_));
    bank_[b] = std::move(fresh);
    bank_cap_[b] = rows;
    update_bytes();
    return true;
  }
  // Entries of one slab array (with the routing dump area).
  static constexpr uint64_t owner_entries(uint32_t owners) { return owners * static_cast<uint64_t>(kSlabStride) + kRouteDump; }
  void start_bank() {
    if (!bank_cap_[0]) throw std::runtime_error("SORTED_VRAM_CAPACITY");  // lost to a growth that failed
    MGBFS_HIP(sorted_start(keymix(start_key_, layout_.km) << layout_.tagbits, bank_[0].as<uint64_t>(),
                           off_[0].as<uint32_t>(), control_.as<uint64_t>(), stream_));
  }
  uint64_t bank_room() const { return std::min({bank_cap_[0], bank_cap_[1], bank_cap_[2]}); }
  // Rows that a layer run ahead may have.
  uint64_t bank_rows() const { return std::min({bank_room(), cap_limit_, static_cast<uint64_t>(0xfffffff0u)}); }

  // Runs up to max_layers layers in the one-workgroup kernel or as owner
  // layers, whichever the current layer's size asks for; kAheadNone when it
  // is one for the general path (too large, or rejected on the device).
  int run_ahead(uint32_t max_layers) {
    if (general_only_) return kAheadNone;
    if (layers.size() == 1) reserve_banks(kBlockSlots, 0);
    const uint64_t F = count_[cur_], rows = bank_rows();
    const bool probe_prev = prev_ >= 0 && !layout_.prune;
    const uint64_t Fp = prev_ >= 0 ? count_[prev_] : 0;
    if (F <= kBlockParents && (!probe_prev || Fp <= kBlockParents) && bank_room() >= 2 * kBlockParents &&
        children_guess(F) <= kBlockChildren && block_rejected_ != layers.size()) {
      const int s = run_block(max_layers, static_cast<uint32_t>(rows));
      if (s != kAheadNone) return s;
    }
    if (F * gens_.count > 0x7fffffffull || owner_rejected_ == layers.size()) return kAheadNone;
    return run_owner(max_layers);
  }

  // Children expected of the current layer (see advance_general): the last
  // masked layer's children per parent plus 10%, else every child.
  uint64_t children_guess(uint64_t F) const {
    const uint32_t G = gens_.count;
    const bool masked = layout_.prune && layers.size() > 1;
    const uint64_t most = F * (masked && G > 1 ? G - 1 : G);
    if (!masked || last_ratio_ <= 0) return most;
    return std::min<uint64_t>(most, static_cast<uint64_t>(static_cast<double>(F) * last_ratio_ * 1.1));
  }

  int run_block(uint32_t max_layers, uint32_t rows) {
    BlockRun r{};
    for (int b = 0; b < 3; ++b) {
      r.bank[b] = bank_[b].as<uint64_t>();
      r.off[b] = off_[b].as<uint32_t>();
    }
    r.L = layout_;
    r.cur = static_cast<uint32_t>(cur_);
    r.prev = prev_ >= 0 ? static_cast<uint32_t>(prev_) : 3u;
    r.F = static_cast<uint32_t>(count_[cur_]);
    r.prev_count = prev_ >= 0 ? static_cast<uint32_t>(std::min<uint64_t>(count_[prev_], ~0u)) : 0u;
    r.depth = static_cast<uint32_t>(layers.size() - 1);
    r.max_layers = std::min(max_layers, kBlockLayers);
    r.rows = rows;
    r.rec = rec_;
    r.seq = seq_;
    r.counters = counters();
    seq_ += kBlockLayers + 2;
    MGBFS_HIP(sorted_block_run(r, action(), stream_));
    uint64_t first = 0;
    for (uint32_t i = 0;; ++i) {
      const LayerRecord& rec = await(rec_[i], r.seq + i);
      if (i == 0) {
        first = rec.stamps[0];
        end_compaction(rec);
      }
      const int s = take(rec, rec.children, rec.ticks - first);
      first = rec.ticks;
      if (s != kTakeNext) {
        if (i > 0 || rec.state == kLayerStop) {  // layers were accepted: the live banks have one fine bucket
          nbo_[cur_] = 1;
          if (prev_ >= 0) nbo_[prev_] = 1;
        }
        if (s == kTakeRejected) block_rejected_ = layers.size();
        return finish(s, i);
      }
    }
  }

  // A session of owner layers: each is one launch, which also reports the
  // layer before it; the host stays kOwnerAhead launches ahead.  256 owners
  // (one workgroup per CU) while the children fit their slabs, else 1,024.
  int run_owner(uint32_t max_layers) {
    const uint64_t F = count_[cur_], guess = children_guess(F);
    const uint32_t owners = guess <= kOwnersSmall * kOwnerMean / 2 ? kOwnersSmall : kOwnersMax;
    if (guess > static_cast<uint64_t>(owners) * kOwnerMean) return kAheadNone;
    reserve_banks(owner_rows(), kOwnerBuffers * owner_entries(kOwnersSmall));
    if (F > bank_rows()) return kAheadNone;
    const uint32_t rows = static_cast<uint32_t>(bank_rows());
    const uint64_t entries = owner_entries(owners);
    if (owner_.bytes() < kOwnerBuffers * entries * 8) {
      if (kOwnerBuffers * entries * 8 > budget_ / 8 || !fits(kOwnerBuffers * entries * 8 - owner_.bytes()))
        return kAheadNone;
      MGBFS_HIP(hipStreamSynchronize(stream_));
      owner_.release();
      owner_.allocate(kOwnerBuffers * entries * 8);
      update_bytes();
    }
    OwnerCtl* ctl = reinterpret_cast<OwnerCtl*>(control_.as<char>() + kCtlOffset);
    uint32_t* counts = reinterpret_cast<uint32_t*>(ctl + kOwnerRing);
    OwnerSlabs slab[kOwnerBuffers];  // candidates 0 and 1, layers 2 + bank index
    for (uint32_t k = 0; k < kOwnerBuffers; ++k)
      slab[k] = OwnerSlabs{owner_.as<uint64_t>() + k * entries, counts + k * kOwnersMax * kCountStride};
    const bool probe_prev = prev_ >= 0 && !layout_.prune;
    // 1,024 owners take 28 us where 256 take 18 (12,000 children, S_11 with
    // ten generators), so a shrinking search changes over; a new session
    // costs about 25 us.
    const uint32_t low = owners == kOwnersSmall ? kBlockChildren / 2 : 512 * kOwnersSmall;
    const OwnerRules rules{owners, rows, low, owners * kOwnerMean};
    const uint64_t seq = seq_;
    seq_ += kBlockLayers + 2;
    MGBFS_HIP(owner_begin(counts, kOwnerBuffers * kOwnersMax * kCountStride, ctl, static_cast<uint32_t>(F), stream_,
                          rec_, counters()));
    OwnerImport im{};
    im.cur = bank_[cur_].as<uint64_t>();
    im.F = static_cast<uint32_t>(F);
    im.own = slab[2 + cur_];
    if (probe_prev) {
      im.prev = bank_[prev_].as<uint64_t>();
      im.prev_count = static_cast<uint32_t>(count_[prev_]);
      im.own_prev = slab[2 + prev_];
    }
    im.masked = layout_.prune && layers.size() > 1;
    im.cand = slab[0];
    im.ctl = ctl;
    MGBFS_HIP(owner_import(im, action(), layout_, owners, stream_));
    int qcur = cur_, qprev = prev_;
    const uint32_t most = std::min(max_layers, kBlockLayers);
    uint32_t queued = 0, accepted = 0;
    uint64_t ticks = 0, children = 0;
    int s = kTakeNext;
    // Record r is layer r's (0: the imported one), written by launch r + 1.
    for (uint32_t r = 0;; ++r) {
      for (; queued < most && queued <= r + kOwnerAhead; ++queued) {
        const int nxt = free_bank(qcur, qprev);
        OwnerLayer a{};
        a.in = slab[queued & 1u];
        a.out = slab[(queued & 1u) ^ 1u];
        a.cur = slab[2 + qcur];
        if (qprev >= 0 && !layout_.prune) a.prev = slab[2 + qprev];
        a.next = slab[2 + nxt];
        a.before = ctl + queued % kOwnerRing;
        a.now = ctl + (queued + 1) % kOwnerRing;
        a.after = ctl + (queued + 2) % kOwnerRing;
        a.rules = rules;
        a.rec = rec_ + queued % kOwnerRing;
        a.seq = seq + queued;
        MGBFS_HIP(owner_layer(a, action(), layout_, stream_));
        qprev = qcur;
        qcur = nxt;
        if (queued + 1 == most)  // nothing follows the last layer to report it
          MGBFS_HIP(owner_report(ctl + most % kOwnerRing, rules, rec_ + most % kOwnerRing, seq + most, stream_));
      }
      const LayerRecord& rec = await(rec_[r % kOwnerRing], seq + r);
      if (r == 0) {
        end_compaction(rec);
        charge(0, rec.ticks - rec.stamps[0]);  // the import
        s = rec.state == kLayerNext ? kTakeNext : kTakeRejected;
      } else {
        s = take(rec, children, rec.ticks - ticks);
        accepted += s == kTakeNext || s == kTakeStop;
      }
      ticks = rec.ticks;
      children = rec.children;
      if (s != kTakeNext || r == most) break;
    }
    if (accepted) {
      MGBFS_HIP(owner_export(slab[2 + cur_], bank_[cur_].as<uint64_t>(), off_[cur_].as<uint32_t>(), slab[2 + prev_],
                             bank_[prev_].as<uint64_t>(), off_[prev_].as<uint32_t>(), owners, stream_));
      nbo_[cur_] = nbo_[prev_] = owners;
    }
    if (s == kTakeRejected) owner_rejected_ = layers.size();
    return finish(s, accepted);
  }

  enum Take { kTakeNext, kTakeStop, kTakeEmpty, kTakeRejected };
  // A layer's record into the engine's state and counters; C: children
  // generated for it.
  int take(const LayerRecord& rec, uint64_t C, uint64_t ticks) {
    charge(0, ticks);
    if (rec.state == kLayerRejected) return kTakeRejected;
    const uint64_t F = count_[cur_];
    const bool masked = layout_.prune && layers.size() > 1;
    candidates += C;
    unique_candidates += rec.unique;
    last_ratio_ = masked ? static_cast<double>(C) / static_cast<double>(F) : 0.0;
    const uint64_t bytes = 16 * F + 16 * C + 8 * rec.N;
    phase_bytes[0] += bytes;
    streamed_bytes += bytes;
    ++launches;
    if (rec.state == kLayerEmpty) return kTakeEmpty;
    const int nxt = next_bank();
    count_[nxt] = rec.N;
    prev_ = cur_;
    cur_ = nxt;
    layers.push_back(rec.N);
    return rec.state == kLayerStop ? kTakeStop : kTakeNext;
  }
  // Status of a finished run of layers, `accepted` of them before the last.
  int finish(int s, uint32_t accepted) {
    if (s == kTakeEmpty) {
      terminal = true;
      return MGBFS_COMPLETE;
    }
    if (s == kTakeRejected && accepted == 0) return kAheadNone;
    return MGBFS_LAYER;  // a rejected layer after accepted ones is met again by the next call
  }
  // Waits for a record in pinned memory: 6 us after its kernel against 16
  // for a copy and a stream wait.  The kernels always leave their records;
  // a stream that ends or fails without one is an error.
  const LayerRecord& await(const LayerRecord& rec, uint64_t seq) {
    auto there = [&] { return __atomic_load_n(&rec.seq, __ATOMIC_ACQUIRE) == seq; };
    while (true) {
      for (uint32_t spin = 0; spin < (1u << 18); ++spin)
        if (there()) return rec;
      const hipError_t e = hipStreamQuery(stream_);
      if (e == hipErrorNotReady) continue;
      MGBFS_HIP(e);
      if (!there()) throw std::runtime_error("SORTED_LAYER_RECORD");
    }
  }
  int free_bank(int cur, int prev) const {
    for (int b = 0; b < 3; ++b)
      if (b != cur && b != prev) return b;
    return -1;
  }
  uint32_t* error_word() { return reinterpret_cast<uint32_t*>(control_.as<uint64_t>() + 1); }
  // Back-edge masks of gens_ (tag bits 0..G-1; bit tagbits-1 is the in-bank
  // mark and bit tagbits-2 stays clear, so no entry is all ones), the
  // fine-bucket margin and the start state.
  void set_generators(const Graph& g) {
    bool pairs;  // every generator has its inverse in the set
    if (wide_) {
      std::memset(&gens_, 0, sizeof(gens_));
      gens_.count = g.generators;
      pairs = wide_->paired;
    } else {
      gens_ = g.packed_generators();
      pairs = fill_back_edge_masks(gens_);
      if (!pairs) throw std::runtime_error("SORTED_REQUIRES_INVERSE_CLOSED");
    }
    layout_.prune = pairs && gens_.count + 2 <= layout_.tagbits && !(flags_ & MGBFS_FLAG_TEST_NO_PRUNE);
    if (!layout_.prune)
      for (uint32_t a = 0; a < gens_.count; ++a) {
        gens_.child_mask[a] = 0;
        if (wide_) wide_->table.child_mask[a] = 0;
      }
    history_layers = layout_.prune ? 2 : 3;
    margin_ = fine_margin(gens_.count);
    start_key_ = wide_ ? wide_->start_key : g.start_key();
    if (wide_) {
      wide_dev_.allocate(sizeof(WideTable));
      MGBFS_HIP(hipMemcpy(wide_dev_.as<void>(), &wide_->table, sizeof(WideTable), hipMemcpyHostToDevice));
    }
  }
  ActionRef action() const { return ActionRef{&gens_, wide_ ? wide_dev_.as<WideTable>() : nullptr, gens_.count}; }
  // A layer this engine has no room or geometry for.  Wide keys go on in the
  // segmented backend, which made this engine.
  int out_of_room(uint32_t* fatal, uint32_t bits) {
    if (wide_) return kAdvanceHandover;
    *fatal = bits;
    terminal = true;
    return MGBFS_RESOURCE;
  }
  LayerCounters* counters() { return control_.as<LayerCounters>(); }
  void charge(uint32_t phase, uint64_t ticks) {
    const double s = static_cast<double>(ticks) * tick_seconds_;
    phase_seconds[phase] += s;
    kernel_seconds += s;
  }
  // A compaction runs unwaited; the next record tells when it ended.  (Not
  // when something else began: the host may have been away in between.)
  void compact(uint64_t* sub, uint32_t nsub, uint32_t fb, int nxt) {
    MGBFS_HIP(sorted_compact(sub, nsub, fb, off_[nxt].as<uint32_t>(), error_word(), bank_cap_[nxt],
                             bank_[nxt].as<uint64_t>(), stream_, &counters()->compacted));
  }
  void end_compaction(const LayerRecord& rec) {
    if (compacted_ && rec.compacted > compacted_) charge(3, rec.compacted - compacted_);
    compacted_ = 0;
  }
  // Routing output size as passed to the kernels; the test flag reports an
  // oversized output so they take their 64-bit addressing path.
  uint64_t routed(uint64_t entries) const {
    return (flags_ & MGBFS_FLAG_TEST_WIDE_ROUTING) ? ~0ull : entries;
  }
  int next_bank() const { return free_bank(cur_, prev_); }
  // Phase times (the kernels' start stamps) and modelled streaming bytes
  // (see the kernel file header).  Phase 2 is unique_diff alone; the fine
  // count scan is charged to phase 3 with the compaction it feeds.
  void account(const LayerRecord& rec, uint64_t F, uint64_t Fp, bool partitioned) {
    const uint64_t C = rec.children, N = rec.N;
    end_compaction(rec);
    const uint64_t routed = partitioned ? rec.stamps[1] : rec.stamps[2];
    const uint64_t ticks[4] = {routed - rec.stamps[0], rec.stamps[2] - routed, rec.stamps[3] - rec.stamps[2],
                               rec.ticks - rec.stamps[3]};
    for (int p = 0; p < 4; ++p) charge(p, ticks[p]);
    compacted_ = rec.ticks;
    const uint64_t be = 8 * F + 8 * C, bp = partitioned ? 16 * C : 0, bu = 8 * C + 8 * F + 8 * Fp + 8 * N;
    phase_bytes[0] += be;
    phase_bytes[1] += bp;
    phase_bytes[2] += bu;
    streamed_bytes += be + bp + bu;
    launches += partitioned ? 3 : 2;
  }
  void ensure_u32(DeviceBuffer& b, uint64_t words) {
    if (b.bytes() < words * 4) {
      MGBFS_HIP(hipStreamSynchronize(stream_));
      b.allocate(std::max<uint64_t>(words * 4, b.bytes() * 2));
    }
  }
  // Lane slabs (entries) and sub-bucket slabs (entries); grown, never shrunk.
  // A buffer goes before its successor is allocated, so its size is 0 until
  // that is there: a growth that throws leaves nothing to be used.
  bool ensure_slabs(uint64_t lane_entries, uint64_t sub_entries) {
    if (lane_cap_ >= lane_entries && sub_cap_ >= sub_entries) return true;
    uint64_t lane = std::max(lane_cap_, lane_entries), sub = std::max(sub_cap_, sub_entries);
    if (!fits((lane - lane_cap_ + sub - sub_cap_) * 8)) return false;
    MGBFS_HIP(hipStreamSynchronize(stream_));
    if (lane > lane_cap_) {
      lane_cap_ = 0;
      lane_.release();
      update_bytes();
      lane_.allocate(lane * 8);
      lane_cap_ = lane;
    }
    if (sub > sub_cap_) {
      sub_cap_ = 0;
      sub_.release();
      update_bytes();
      sub_.allocate(sub * 8);
      sub_cap_ = sub;
    }
    update_bytes();
    return true;
  }
  bool grow_bank(int b, uint64_t rows) {
    if (bank_cap_[b] >= rows) return true;
    uint64_t want = std::max<uint64_t>(rows, bank_cap_[b] + bank_cap_[b] / 4);
    if (!fits((want - bank_cap_[b]) * 8)) want = rows;
    if (!fits((want - bank_cap_[b]) * 8)) return false;
    MGBFS_HIP(hipStreamSynchronize(stream_));
    bank_cap_[b] = 0;
    bank_[b].release();
    update_bytes();
    bank_[b].allocate(want * 8);
    bank_cap_[b] = want;
    update_bytes();
    return true;
  }
  bool fits(uint64_t extra) const { return device_bytes + extra <= budget_; }
  void read_bank(int b, uint64_t count, std::vector<uint64_t>& out) {
    std::vector<uint64_t> raw(count);
    if (count) {
      MGBFS_HIP(hipMemcpyAsync(raw.data(), bank_[b].as<uint64_t>(), count * 8, hipMemcpyDeviceToHost, stream_));
      MGBFS_HIP(hipStreamSynchronize(stream_));
    }
    out.resize(count);
    for (uint64_t i = 0; i < count; ++i) out[i] = keyunmix(raw[i] >> layout_.tagbits, layout_.km);
  }
  void update_bytes() {
    device_bytes = control_.bytes() + fine_counts_.bytes() + lane_.bytes() + sub_.bytes() + lcount_.bytes() +
                   scount_.bytes() + scan_ws_.bytes() + owner_.bytes() + wide_dev_.bytes();
    for (int b = 0; b < 3; ++b) device_bytes += bank_[b].bytes() + off_[b].bytes();
  }

  PackedGenerators gens_;            // wide keys: only the count and empty masks
  std::unique_ptr<WideCode> wide_;   // set: keys are wide, their table in wide_dev_
  DeviceBuffer wide_dev_;
  SortedLayout layout_{};
  uint32_t n_, margin_ = 0, flags_ = 0, unique_grid_ = 2048, slack_ = 1;
  double last_ratio_ = 0.0;  // children per parent of the last masked layer
  uint64_t start_key_ = 0, budget_ = 0, cap_limit_ = 0, lane_cap_ = 0, sub_cap_ = 0;
  DeviceBuffer bank_[3], off_[3], lane_, sub_, lcount_, scount_, scan_ws_, fine_counts_, control_;
  uint64_t bank_cap_[3] = {0, 0, 0}, count_[3] = {0, 0, 0};
  uint32_t nbo_[3] = {0, 0, 0};  // fine buckets of each bank
  int cur_ = 0, prev_ = -1;
  DeviceBuffer owner_;               // owner layers' slab arrays
  LayerRecord* rec_ = nullptr;       // pinned: what the kernels report of their layers
  uint64_t seq_ = 1, bound_ = 0;     // next unused record number; state-space bound (0 = unknown)
  double tick_seconds_ = 0.0;        // one wall_clock64() tick
  size_t block_rejected_ = 0;        // layers.size() when the one-workgroup kernel last refused a layer
  size_t owner_rejected_ = 0;        // the same of the owner layers
  bool general_only_ = false;
  uint64_t compacted_ = 0;           // ticks of the record before a compaction not yet timed
};

Engine* make_sorted_engine(const Graph& g, const mgbfs_engine_options& o, const WideCode* wide) {
  return new SortedEngine(g, o, wide);
}

}  // namespace mgbfs
