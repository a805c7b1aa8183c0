// One permutation search by owners of the bitmap (rank_engine.hip), in memory
// that its owner lays out.
#pragma once
#include <vector>
#include "engine.hpp"
#include "kernels.hpp"

namespace mgbfs {

// Pinned records that searches run one after the other share.
struct RankRecords {
  static constexpr uint32_t kRing = 64;  // records, and control blocks of a search
  RankRecords();
  ~RankRecords();
  RankRecords(const RankRecords&) = delete;
  RankRecords& operator=(const RankRecords&) = delete;
  LayerRecord* rec = nullptr;
  static constexpr uint64_t kKeys = 1024;
  uint64_t* keys = nullptr;   // kKeys, of a small sample
  uint32_t* sizes = nullptr;  // kRankBlockLayers, of a run in one launch
  uint64_t base = 0;  // number of a run's layer 0
};

struct RankMemory {
  uint32_t* bitmap;       // owners x slice_words
  uint32_t* list;         // owners x list_cap
  uint32_t* words;        // RankRun::words_bytes
  uint32_t* messages[2];  // owners x cap, + kRouteDump
  uint32_t cap;           // messages per owner (a multiple of 4)
};

class RankRun {
 public:
  static constexpr int kSendAgain = -1;
  explicit RankRun(const Graph& g) : plan(rank_plan(g.elements, owners_for(g))) {}
  // 1: one workgroup runs the search.  0: the owners of its degree.
  static uint32_t owners_for(const Graph& g);
  static uint64_t words_bytes(const RankPlan& p);
  // Messages per owner (one owner: none): at first a fifth of all children there can be (the
  // widest LRX layer sends 15% of them), two fifths up to degree 10, where
  // memory is small (random sets' layers: engines created, run and dropped
  // for sets of degree 9 and 10 1.85 -> 1.22 ms each, without the growing);
  // at most all of them (a state is a child of `generators` states).
  static uint32_t first_cap(const RankPlan& p, uint32_t generators);
  static uint32_t last_cap(const RankPlan& p, uint32_t generators);

  void set_graph(const Graph& g);
  void start(hipStream_t stream);
  // The message buffers go: children sent to them are sent again.
  void drop_messages() {
    memory.cap = 0;
    memory.messages[0] = memory.messages[1] = nullptr;
    sent_ = false;
  }
  // Layers up to depth `target`: MGBFS_LAYER there, MGBFS_COMPLETE after the
  // last, kSendAgain when the children of the last layer did not fit the
  // messages (they are sent anew by the next run).  Launches queued past the
  // end may still be on the stream; they do nothing.
  int run(uint64_t target, RankRecords& records, hipStream_t stream);
  // States of the current layer (back = 0) or the one before, as packed keys.
  void export_layer(uint64_t back, uint64_t limit, uint64_t* keys, hipStream_t stream);
  // The message buffer that holds nothing between runs, as room for keys.
  uint64_t* spare(uint64_t* keys) const {
    *keys = memory.cap ? (static_cast<uint64_t>(plan.owners) * memory.cap + kRouteDump) / 2 : 0;
    return reinterpret_cast<uint64_t*>(memory.messages[parity_ ^ 1u]);
  }
  uint32_t generators() const { return gens_.count; }

  RankPlan plan;
  RankMemory memory{};
  std::vector<uint64_t> layers;
  double seconds = 0.0, tick_seconds = 0.0;  // between the records of layers run

 private:
  static constexpr uint32_t kAheadLayers = 4;
  static constexpr uint32_t kEnds = 4;  // list ends kept: of the last layers
  uint32_t* counts(uint32_t parity) { return memory.words + parity * plan.count_stride * plan.owners; }
  uint32_t* ends(uint64_t layer) { return memory.words + (2 * plan.count_stride + layer % kEnds) * plan.owners; }
  OwnerCtl* ctl(uint64_t layer);
  int run_block(uint64_t target, RankRecords& records, hipStream_t stream);
  void send(uint64_t d, hipStream_t stream);
  RankLayer layer_args(uint64_t d, LayerRecord* rec, uint64_t seq);
  const LayerRecord& await(const LayerRecord& rec, uint64_t seq, hipStream_t stream);

  RankGenerators gens_{};
  uint64_t start_key_ = 0;
  uint32_t parity_ = 0;  // the buffer holding the current layer's children
  bool sent_ = false;    // ... which are complete
};

}  // namespace mgbfs
