// Host check of the sorted engine's buffers (sorted_engine.hip) on a HIP
// runtime in host memory.  The kernels only look at their arguments and
// report layers of given sizes; every allocation of a search fails in turn,
// and neither a repeated call nor a reset may hand the kernels memory that is
// not the engine's.
#include <vector>
#include "fake_hip.hpp"
#include "device_cache.hip"
#include "engine.hip"
#include "sorted_engine.hip"

using fake::holds;
using fake::require;

static std::vector<uint64_t> script;  // layer sizes of the search, the last one 0
static std::unique_ptr<mgbfs::Engine> engine;
static uint32_t queued;  // owner layers since the session began
static uint64_t next_size() { return script[engine->layers.size()]; }

namespace mgbfs {

hipError_t zero_u32x3(uint32_t* a, uint64_t na, uint32_t* b, uint64_t nb, uint32_t* c, uint64_t nc, hipStream_t s,
                      unsigned long long*) {
  require(holds(a, 4 * na) && (!nb || holds(b, 4 * nb)) && (!nc || holds(c, 4 * nc)), "counters");
  return fake::launch(s);
}
hipError_t sorted_start(uint64_t, uint64_t* bank, uint32_t* off, uint64_t* control, hipStream_t s) {
  require(holds(bank, 8) && holds(off, 8) && holds(control, 64), "the start bank");
  return fake::launch(s);
}
hipError_t sorted_block_run(const BlockRun& r, const ActionRef&, hipStream_t s) {
  for (int b = 0; b < 3; ++b) require(holds(r.bank[b], 8ull * r.rows) && holds(r.off[b], 8), "one workgroup's banks");
  r.rec->N = next_size();
  r.rec->children = 2 * r.F;
  r.rec->state = r.rec->N == 0 ? kLayerEmpty : (r.rec->N > r.rows ? kLayerRejected : kLayerStop);
  r.rec->seq = r.seq;
  return fake::launch(s);
}
hipError_t owner_begin(uint32_t* counts, uint32_t words, OwnerCtl* ctl, uint32_t, hipStream_t s, LayerRecord*,
                       const LayerCounters*) {
  require(holds(counts, 4ull * words) && holds(ctl, sizeof *ctl), "owners' counts");
  queued = 0;
  return fake::launch(s);
}
hipError_t owner_import(const OwnerImport& im, const ActionRef&, const SortedLayout&, uint32_t owners, hipStream_t s) {
  require(holds(im.cur, 8ull * im.F) && holds(im.own.data, 8ull * owners * kSlabStride) &&
              holds(im.cand.data, 8 * (owners * static_cast<uint64_t>(kSlabStride) + kRouteDump)),
          "an import");
  return fake::launch(s);
}
static void owner_record(LayerRecord* rec, uint64_t seq, uint32_t rows) {
  if (queued > 1) return;
  rec->N = queued == 0 ? engine->layers.back() : next_size();
  rec->state = rec->N == 0 ? kLayerEmpty : (rec->N > rows ? kLayerRejected : (queued == 0 ? kLayerNext : kLayerStop));
  rec->seq = seq;
  ++queued;
}
hipError_t owner_layer(const OwnerLayer& a, const ActionRef&, const SortedLayout&, hipStream_t s) {
  const uint64_t bytes = 8 * (a.rules.owners * static_cast<uint64_t>(kSlabStride) + kRouteDump);
  require(holds(a.in.data, bytes) && holds(a.out.data, bytes) && holds(a.cur.data, bytes) && holds(a.next.data, bytes),
          "owner slabs");
  owner_record(a.rec, a.seq, a.rules.rows);
  return fake::launch(s);
}
hipError_t owner_report(const OwnerCtl*, const OwnerRules& rules, LayerRecord* rec, uint64_t seq, hipStream_t s) {
  owner_record(rec, seq, rules.rows);
  return fake::launch(s);
}
hipError_t owner_export(const OwnerSlabs&, uint64_t* bank, uint32_t* off, const OwnerSlabs&, uint64_t* prev_bank,
                        uint32_t* prev_off, uint32_t owners, hipStream_t s) {
  require(holds(bank, 8 * engine->layers.back()) && holds(off, 4 * (owners + 1)) &&
              holds(prev_bank, 8 * engine->layers[engine->layers.size() - 2]) && holds(prev_off, 4 * (owners + 1)),
          "an export");
  return fake::launch(s);
}
hipError_t sorted_expand_route(const uint64_t* bank, uint64_t F, const PackedGenerators&, const SortedLayout&, bool,
                               uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t* cursors,
                               uint32_t*, uint64_t* out, uint64_t entries, hipStream_t s) {
  require(holds(bank, 8 * F) && holds(cursors, 4) && holds(out, 8 * (entries + kRouteDump)), "an expansion");
  return fake::launch(s);
}
hipError_t sorted_partition(const uint64_t* in, const uint32_t*, uint32_t, uint32_t, uint32_t nsub, uint32_t,
                            uint32_t* scount, uint32_t*, uint64_t* out, uint64_t entries, hipStream_t s,
                            unsigned long long*) {
  require(holds(in, 8) && holds(scount, 4ull * nsub) && holds(out, 8 * (entries + kRouteDump)), "a partition");
  return fake::launch(s);
}
hipError_t sorted_unique_diff(uint64_t* cand, const uint32_t* scount, uint32_t nsub, const uint64_t* cur, const uint32_t*,
                              uint32_t, const uint64_t*, const uint32_t*, uint32_t, uint32_t, uint32_t*, uint32_t*,
                              unsigned long long*, unsigned long long*, uint32_t, bool, uint32_t, hipStream_t s,
                              unsigned long long*) {
  require(holds(cand, 8ull * nsub * kSlabStride) && holds(scount, 4ull * nsub) &&
              holds(cur, 8 * engine->layers.back()),
          "a difference");
  return fake::launch(s);
}
uint64_t scan_workspace_words(uint64_t n) { return n / 1024 + 2; }
hipError_t exclusive_scan_u32(const uint32_t*, uint64_t n, uint32_t* out, uint32_t* workspace, hipStream_t s,
                              LayerCounters*, LayerRecord* rec, uint64_t seq) {
  require(holds(out, 4 * (n + 1)) && holds(workspace, 4 * scan_workspace_words(n)), "a scan");
  rec->N = next_size();
  rec->children = 2 * engine->layers.back();
  rec->ticks = 1;
  rec->state = 0;
  rec->seq = seq;
  return fake::launch(s);
}
hipError_t sorted_compact(const uint64_t* cand, uint32_t nsub, uint32_t, const uint32_t*, const uint32_t*,
                          uint64_t bank_rows, uint64_t* bank, hipStream_t s, unsigned long long*) {
  require(holds(cand, 8ull * nsub * kSlabStride) && holds(bank, 8 * bank_rows), "a compaction");
  return fake::launch(s);
}
hipError_t stamp_record(LayerRecord* rec, const LayerCounters*, uint64_t seq, hipStream_t s) {
  rec->seq = seq;
  return fake::launch(s);
}

}  // namespace mgbfs

using namespace mgbfs;

static Graph rotations_and_swap(uint32_t n) {
  Graph g;
  g.elements = n;
  g.generators = 3;
  g.inverse_closed = true;
  for (uint32_t i = 0; i < n; ++i) g.perms.push_back((i + 1) % n);
  for (uint32_t i = 0; i < n; ++i) g.perms.push_back((i + n - 1) % n);
  for (uint32_t i = 0; i < n; ++i) g.perms.push_back(i < 2 ? 1 - i : i);
  for (uint32_t i = 0; i < n; ++i) g.start.push_back(i);
  return g;
}

int main() {
  fake::Device& d = fake::dev();
  const Graph g = rotations_and_swap(13);
  mgbfs_engine_options o{};
  o.vram_budget = 2ull << 30;
  const std::vector<uint64_t> sizes{1, 3, 4000, 6000, 900000, 1200000, 5000, 20, 0};
  const std::vector<uint64_t> want(sizes.begin(), sizes.end() - 1);
  // Layers run ahead of the host, then the general path alone.
  for (uint32_t flags : {0u, static_cast<uint32_t>(MGBFS_FLAG_TEST_TIGHT_SLABS)})
    for (int stepwise = 0; stepwise < 2; ++stepwise)
      for (int after = 0; after < 3; ++after) {  // again at once, again with room, or reset with room
        long k = 0;
        for (bool failed = true; failed; ++k) {
          script = sizes;
          o.flags = flags;
          engine.reset();
          engine.reset(make_sorted_engine(g, o));
          auto search = [&] {
            uint64_t n = 0;
            uint32_t fatal = 0;
            int s = MGBFS_LAYER;
            if (!stepwise) return engine->run_to_end();
            while (s == MGBFS_LAYER) s = engine->advance(&n, &fatal);
            return s;
          };
          auto fails = [&] {
            try {
              return search() != MGBFS_COMPLETE;
            } catch (const std::exception&) {
              return true;
            }
          };
          d.room = k;
          failed = fails();
          if (failed && after == 0) require(fails(), "no memory, no search");
          d.room = -1;
          if (failed && after == 2) engine->reset();
          if (failed && !engine->terminal) require(search() == MGBFS_COMPLETE, "the search completes when there is room");
          if (!engine->terminal || engine->layers.size() == want.size()) require(engine->layers == want, "the layers");
          else require(std::equal(engine->layers.begin(), engine->layers.end(), want.begin()), "the layers so far");
        }
        require(k > 4, "allocations to fail");
      }
  // A search that stays within one workgroup keeps small banks.
  script = {1, 2, 2, 2, 1, 0};
  o.flags = 0;
  engine.reset(make_sorted_engine(g, o));
  const uint64_t made = engine->device_bytes;
  require(engine->run_to_end() == MGBFS_COMPLETE && engine->device_bytes - made < (1u << 20), "small banks");
  // Calls from a thread whose current device is another.
  for (uint32_t flags : {0u, static_cast<uint32_t>(MGBFS_FLAG_TEST_TIGHT_SLABS)}) {
    script = sizes;
    o.flags = flags;
    o.device = 1;
    engine.reset(make_sorted_engine(g, o));
    while (!engine->terminal) {
      uint64_t n = 0;
      uint32_t fatal = 0;
      d.current = 0;
      engine->advance(&n, &fatal);
      d.current = 0;
      engine->settle();
      std::vector<int64_t> rows;
      d.current = 0;
      engine->sample(0, 1, rows, n);
    }
    require(engine->layers == want && fake::all_on(1), "memory on the engine's device");
    d.current = 0;
  }
  engine.reset();
  std::printf("sorted memory ok\n");
  return 0;
}
