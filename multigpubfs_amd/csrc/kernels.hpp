// Internal launch wrappers shared by the engine and the C ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include "common.hpp"

namespace mgbfs {

hipError_t bitmap_seed(uint32_t degree, uint64_t start_key, uint32_t* bitmap, uint64_t bitmap_bits,
                       uint64_t* frontier, uint32_t* error, hipStream_t stream);
// New children go to next[*next_count - count_base + ...]: the counter may
// keep running across layers, count_base being its value at the layer start.
hipError_t bitmap_expand(const uint64_t* frontier, uint64_t count, const PackedGenerators& gens, uint32_t* bitmap,
                         uint64_t bitmap_bits, uint64_t* next, unsigned long long* next_count, uint64_t count_base,
                         uint64_t next_cap, uint32_t* error, hipStream_t stream);
// The same layer with its size read from the device (counts[0]); counts[1],
// zero before, receives the next layer's size.
hipError_t bitmap_expand_queued(const uint64_t* frontier, unsigned long long* counts, const PackedGenerators& gens,
                                uint32_t* bitmap, uint64_t bitmap_bits, uint64_t* next, uint64_t next_cap,
                                uint32_t* error, hipStream_t stream);
// Sorted-bank backend limits.
constexpr uint32_t kMaxPassBits = 10;     // buckets per routing pass (LDS counters)
constexpr uint32_t kMaxBucketBits = 20;   // sub-buckets per layer: 2^20
constexpr uint32_t kMaxFineBits = 10;     // bank partition bits beyond the layer's K
constexpr uint32_t kUniqueSlots = 8192;   // LDS hash slots per sub-bucket
constexpr uint32_t kUniqueCap = 5120;     // candidates per sub-bucket (table load factor <= 0.625)
constexpr uint32_t kSlabStride = 5120;    // entries between sub-bucket slab starts (>= kUniqueCap)

// Stored-value layout of the sorted backend: (keymix(key) << tagbits) | tag,
// keymix on b = max(32, 4n) bits (at least 32, so keymix's mask leaves the
// low word whole) and tagbits = 64 - b.
inline uint32_t sorted_key_bits(uint32_t degree) { return degree >= 8 ? 4 * degree : 32u; }
// Dump-area index for 32-bit destination indexing, or ~0 when the output
// (entries, plus the dump area) does not fit 32-bit indices.
inline uint32_t route_dump_index(uint64_t out_entries, uint64_t dump) {
  return out_entries + dump < ~0u ? static_cast<uint32_t>(out_entries) : ~0u;
}

struct SortedLayout {
  KeyMix km;
  uint32_t tagbits;  // 64 - sorted_key_bits(n)
  uint32_t prune;    // back-edge masks in use: tag bit i = skip generator i
  uint64_t tagmask;  // (1 << tagbits) - 1
};

// How a layer's children are made: nibble-packed permutations (generators by
// value) or wide keys (wide.hpp; the table in device memory).
struct WideTable;
struct ActionRef {
  const PackedGenerators* nibble;
  const WideTable* wide;  // device; null: nibble
  uint32_t count;         // generators
};

// Layers run ahead of the host (sorted_queue.hip).
// What the host learns of a layer, in pinned memory; seq is written last.
enum LayerState : uint32_t {
  kLayerNext = 0,      // accepted, the next layer runs
  kLayerStop = 1,      // accepted, no further layer runs
  kLayerEmpty = 2,     // no new states: the search is complete
  kLayerRejected = 3,  // not accepted (an overflow, or too many rows): the host redoes it
};
struct LayerRecord {
  uint64_t N, unique, ticks;  // ticks: wall_clock64() when the layer was counted
  uint64_t children;          // block_run: generated for this layer; owner layers: from it
  uint32_t state, pad;        // general path: the error word
  uint64_t seq;
  uint64_t stamps[4];         // general path: LayerCounters.stamps; else [0]: when the launch (the session) began
  uint64_t compacted;         // LayerCounters.compacted
};

// Device words of a layer on the general path.
struct LayerCounters {
  unsigned long long unique;    // distinct children
  uint32_t error, pad;
  unsigned long long children;  // generated
  unsigned long long compacted;  // wall_clock64() at the end of the last compaction
  unsigned long long stamps[4];  // wall_clock64() at the start of the layer, its partition, unique_diff and scan
};
static_assert(sizeof(LayerCounters) == 64, "one 64-byte line");

// One-workgroup layers: everything fits one LDS table.
constexpr uint32_t kBlockSlots = 16384;
constexpr uint32_t kBlockFill = 14336;     // entries accepted (plus one per lane in flight)
constexpr uint32_t kBlockParents = 4096;   // parents of such a layer at most
// A layer of more children than this is quicker with one owner per
// workgroup: on S_8 and S_10 LRX one workgroup takes 8 us for 1,200
// children, 15 for 2,600, 24 for 4,700 and 34 for 5,700 (10 generators: 44
// for 12,000, 300 for 28,000, as the table fills).
constexpr uint32_t kBlockChildren = 4096;

struct BlockRun {
  uint64_t* bank[3];
  uint32_t* off[3];
  SortedLayout L;
  uint32_t cur, prev;        // bank indices; prev 3: none
  uint32_t F, prev_count, depth;
  uint32_t generators, max_layers;
  uint32_t rows;             // rows every bank holds (and the caller's layer capacity)
  LayerRecord* rec;          // pinned: one record per layer run
  uint64_t seq;              // rec[i].seq = seq + i
  const LayerCounters* counters;
};

// Owner layers: `owners` sub-buckets (equal ranges of the top 32 bits), one
// workgroup each; the layers' states and the candidates live in slabs of
// kSlabStride entries per owner.
constexpr uint32_t kOwnersMax = 1024;
constexpr uint32_t kOwnersSmall = 256;
// Words from one owner's counter to the next (side by side,
// the reservations of all owners queue on a few cache lines: S_10 sorted 747,
// 723, 654, 641 us at 1, 8, 16, 32 words).
constexpr uint32_t kCountStride = 16;
constexpr uint32_t kOwnerMean = 4600;  // children per owner at most (a slab holds kUniqueCap)

// Totals of one owner layer; zeroed two launches before its own.
struct OwnerCtl {
  unsigned long long counts;  // states of the layer, + children made from it << 32
  unsigned long long unique;  // distinct children the layer was selected from
  uint32_t error;             // the layer is not usable
  uint32_t spill;             // the children made from it are incomplete (a slab was full)
  uint32_t halt;              // no layer: an earlier one was the last
  uint32_t imported;          // the session's first: goes on however few its children
};

struct OwnerRules {
  uint32_t owners;
  uint32_t rows;       // states a layer may have (bank rows, the caller's capacity)
  uint32_t low, high;  // children outside [low, high] end the session
};

struct OwnerSlabs {
  uint64_t* data;   // owners x kSlabStride entries
  uint32_t* count;  // entries per owner, kCountStride words apart
};

struct OwnerImport {
  const uint64_t* cur;   // dense banks
  const uint64_t* prev;  // null unless both retained layers are probed
  uint32_t F, prev_count, masked;
  OwnerSlabs own, own_prev, cand;
  OwnerCtl* ctl;  // the imported layer's
};

struct OwnerLayer {
  OwnerSlabs in, out;          // candidates of this layer; of the next one
  OwnerSlabs cur, prev, next;  // retained layers (prev.data null: masked) and the new one
  const OwnerCtl* before;
  OwnerCtl *now, *after;
  OwnerRules rules;
  LayerRecord* rec;  // record of the layer before
  uint64_t seq;
};

// Permutation bitmap by owners (rank_owner.hip).
constexpr uint32_t kRankDegree = 12;

struct RankPlan {
  uint32_t degree, owners, magic;  // magic: floor(2^32 / owners)
  uint32_t slice_words, list_cap;  // per owner: bitmap words (a multiple of 4), states
  uint32_t count_stride;           // words from one owner's message counter to the next
};

// Generators over byte permutations (rank_owner.hip: child_of), each with
// the tag of the children it makes (0: no inverse among the generators).
struct RankGenerator {
  uint32_t low[3], high[3], tag, pad;
};
struct RankGenerators {
  uint32_t count, tagged;  // tagged: how many have a tag
  RankGenerator of[kMaxGenerators];
};

struct RankLayer {
  RankPlan plan;
  uint32_t slots;        // children per state: generators, or one less when each state has a tag
  uint32_t claim;        // 0: send only (the layer is in the list already)
  const uint32_t* in;    // messages of this layer: owners x in_cap
  uint32_t* in_count;    // cleared (count_stride words apart)
  uint32_t in_cap;
  uint32_t* out;         // messages of the next layer
  uint32_t* out_count;
  uint32_t out_cap, out_dump;  // out_dump: set by rank_layer
  uint32_t* bitmap;      // owners x slice_words
  uint32_t* list;        // owners x list_cap: states in discovery order
  const uint32_t* ends_before;  // list ends per owner after the layer before
  uint32_t* ends_now;           // and after this one
  const OwnerCtl* before;
  OwnerCtl *now, *after;
  OwnerRules rules;
  LayerRecord* rec;      // record of the layer before
  uint64_t seq;
};

// One owner (degrees up to kRankBlockDegree): layers [depth, target)
// expanded in one launch by one workgroup.  sizes[i] (pinned, kRankBlockLayers)
// is the size of layer depth + 1 + i, the last of them 0 when the search ended;
// the record has their number in N and the start time in stamps[0].
constexpr uint32_t kRankBlockDegree = 8;
constexpr uint32_t kRankBlockLayers = 4096;

struct RankBlock {
  RankPlan plan;
  uint32_t tagged;  // every state but the start has a tag
  uint32_t* bitmap;
  uint32_t* list;
  uint32_t* ends;   // list end after layer d at ends[d % 4], 0 before layer 0
  uint32_t depth, target;
  uint32_t* sizes;
  LayerRecord* rec;
  uint64_t seq;
};

RankPlan rank_plan(uint32_t degree, uint32_t owners = 0);  // owners 0: those of a large search alone
hipError_t rank_seed(const RankPlan& p, uint64_t start_key, uint32_t* bitmap, uint32_t* list, uint32_t* ends,
                     hipStream_t stream);
// tags: of the children each generator makes.
RankGenerators rank_generators(const PackedGenerators& gens, const uint8_t* tags);
hipError_t rank_layer(const RankLayer& a, const RankGenerators& gens, hipStream_t stream);
hipError_t rank_block(const RankBlock& a, const RankGenerators& gens, hipStream_t stream);
// Up to `limit` states of the layer [lo, hi) as packed keys.
hipError_t rank_export(const RankPlan& p, const uint32_t* list, const uint32_t* lo, const uint32_t* hi, uint64_t limit,
                       uint64_t* keys, hipStream_t stream);
hipError_t rank_report(const OwnerCtl* ctl, const OwnerRules& rules, LayerRecord* rec, uint64_t seq,
                       hipStream_t stream);

hipError_t sorted_start(uint64_t stored, uint64_t* bank, uint32_t* off, uint64_t* control, hipStream_t stream);
hipError_t sorted_block_run(const BlockRun& run, const ActionRef& act, hipStream_t stream);
// Zeroes the owners' counts (`words` of them from `counts`) and the first
// control blocks; ctl[0] becomes the imported layer's, of F states.  rec: the
// record that the first layer will leave gets the time.
hipError_t owner_begin(uint32_t* counts, uint32_t words, OwnerCtl* ctl, uint32_t F, hipStream_t stream,
                       LayerRecord* rec = nullptr, const LayerCounters* counters = nullptr);
hipError_t owner_import(const OwnerImport& im, const ActionRef& act, const SortedLayout& L, uint32_t owners,
                        hipStream_t stream);
hipError_t owner_layer(const OwnerLayer& a, const ActionRef& act, const SortedLayout& L, hipStream_t stream);
// Reports the last layer queued (a layer launch reports the one before it).
hipError_t owner_report(const OwnerCtl* ctl, const OwnerRules& rules, LayerRecord* rec, uint64_t seq,
                        hipStream_t stream);
// Owner slabs -> dense bank and offset table of `owners` fine buckets, for
// the current layer and the one before.
hipError_t owner_export(const OwnerSlabs& cur, uint64_t* bank, uint32_t* off, const OwnerSlabs& prev,
                        uint64_t* prev_bank, uint32_t* prev_off, uint32_t owners, hipStream_t stream);

uint64_t scan_workspace_words(uint64_t n);
// rec: report the layer of `counters` with the scan's total (see scan.hip).
hipError_t exclusive_scan_u32(const uint32_t* in, uint64_t n, uint32_t* out, uint32_t* workspace, hipStream_t stream,
                              LayerCounters* counters = nullptr, LayerRecord* rec = nullptr, uint64_t seq = 0);
// A record of nothing but the counters' `compacted`.
hipError_t stamp_record(LayerRecord* rec, const LayerCounters* counters, uint64_t seq, hipStream_t stream);
hipError_t sorted_seed(uint64_t start_key, const SortedLayout& L, uint64_t* bank, uint32_t* off, uint32_t Ko,
                       hipStream_t stream);
// Children of bank[0..F) routed by lane (sub-bucket >> K2) into slabs: slab
// (lane * P + blockIdx % P) of `cap` entries, `stride` entries apart,
// cursors[] counts per slab
// (zeroed by the caller); a run beyond `cap` is dropped and sets err_bit.
// Routing outputs: `out` holds out_entries slab entries followed by a dump
// area of kRouteDump entries (a slab overflow is written there; the layer
// is then redone).
constexpr uint64_t kRouteDump = 8192;
// Sub-bucket of a stored value: floor(top32 * nsub / 2^32) (any nsub, a
// multiple of 2^K2); lane = sub-bucket >> K2 (K2 = 0: lanes are sub-buckets).
hipError_t sorted_expand_route(const uint64_t* bank, uint64_t F, const PackedGenerators& gens, const SortedLayout& L,
                               bool masked, uint32_t nsub, uint32_t K2, uint32_t NB, uint32_t P, uint32_t cap,
                               uint32_t stride,
                               uint32_t err_bit, uint32_t* cursors, uint32_t* error, uint64_t* out,
                               uint64_t out_entries, hipStream_t stream);
// The same for wide keys: `act` has its table in device memory.
hipError_t sorted_expand_route_wide(const uint64_t* bank, uint64_t F, const ActionRef& act, const SortedLayout& L,
                                    bool masked, uint32_t nsub, uint32_t K2, uint32_t NB, uint32_t P, uint32_t cap,
                                    uint32_t stride, uint32_t err_bit, uint32_t* cursors, uint32_t* error,
                                    uint64_t* out, uint64_t out_entries, hipStream_t stream);
// Lane slabs (lcount per slab, capacity and stride lcap) -> sub-bucket
// slabs of kUniqueCap entries, kSlabStride apart (scount per sub-bucket,
// zeroed by the caller).
hipError_t sorted_partition(const uint64_t* in, const uint32_t* lcount, uint32_t lcap, uint32_t P, uint32_t nsub,
                            uint32_t K2, uint32_t* scount, uint32_t* error, uint64_t* out, uint64_t out_entries,
                            hipStream_t stream, unsigned long long* stamp = nullptr);
// In-layer dedup of the sub-bucket slabs and difference against the
// current bank and, when given, the previous one (banks partitioned into
// nbo_c / nbo_p fine buckets); survivors are written back grouped by the
// layer's nsub << fb fine buckets.  merge: OR duplicates' back-edge masks.
hipError_t sorted_unique_diff(uint64_t* cand, const uint32_t* scount, uint32_t nsub, const uint64_t* cur,
                              const uint32_t* cur_off, uint32_t nbo_c, const uint64_t* prev, const uint32_t* prev_off,
                              uint32_t nbo_p, uint32_t fb, uint32_t* fine_counts, uint32_t* error,
                              unsigned long long* unique_total, unsigned long long* cand_total, uint32_t tagbits,
                              bool merge, uint32_t grid_limit, hipStream_t stream,
                              unsigned long long* stamp = nullptr);
// Writes nothing unless *error == 0 and the layer total off[nsub << fb]
// fits bank_rows, so it may be queued before the host has read either.  done
// (null: none) is raised to the time of its end.
hipError_t sorted_compact(const uint64_t* cand, uint32_t nsub, uint32_t fb, const uint32_t* off, const uint32_t* error,
                          uint64_t bank_rows, uint64_t* bank, hipStream_t stream, unsigned long long* done = nullptr);

// Sets kErrFutureCap in *error when off[n] > rows.
hipError_t sorted_capacity_check(const uint32_t* off, uint64_t n, uint64_t rows, uint32_t* error,
                                 hipStream_t stream);

hipError_t fill_u64(uint64_t* dst, uint64_t value, uint64_t count, hipStream_t stream);
hipError_t fill_u32(uint32_t* dst, uint32_t value, uint64_t count, hipStream_t stream);
hipError_t zero_u32x3(uint32_t* a, uint64_t na, uint32_t* b, uint64_t nb, uint32_t* c, uint64_t nc,
                      hipStream_t stream, unsigned long long* stamp = nullptr);

}  // namespace mgbfs
