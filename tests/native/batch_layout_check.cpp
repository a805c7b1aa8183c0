// Host check of the batch engine's layouts (batch_engine.hip) on a HIP
// runtime in host memory: where an instance's parts lie, alone and after the
// restart that follows a full message slab, under every choice of history,
// layer share and bitmap bias.  The kernels only set what the check asks for.
#include <vector>
#include "rank_on_host.hpp"
#include "batch_engine.hip"

using fake::holds;
using namespace mgbfs;

static BatchInstance* inst;  // the device's
static uint32_t overflow;    // owned instances' next step ends in this error
static uint32_t slots;
static uint32_t exports;                    // samples of instances by owners
static uint32_t owned_nodes, shared_nodes;  // expansion kernels in the graphs built

extern "C" hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) {
  for (uint32_t i = 0; i < slots; ++i)
    if (inst[i].status & kInstActive) {
      inst[i].error = inst[i].rank.owners ? overflow : 0;
      inst[i].status = kInstDone;
    }
  return fake::launch(s);
}

namespace mgbfs {
hipError_t batch_reset_flag(uint32_t*, GraphChain&) { return hipSuccess; }
hipError_t batch_tiles(BatchInstance*, uint32_t, uint32_t, uint32_t*, uint32_t, GraphChain&) { return hipSuccess; }
hipError_t batch_clear(const BatchInstance*, uint32_t, const uint32_t*, uint32_t, GraphChain&) { return hipSuccess; }
hipError_t batch_expand(BatchInstance*, uint32_t, const uint32_t*, uint32_t, uint32_t, uint32_t, GraphChain&) {
  ++shared_nodes;
  return hipSuccess;
}
hipError_t batch_owned(BatchInstance*, uint32_t, uint32_t*, uint32_t, GraphChain&) {
  ++owned_nodes;
  return hipSuccess;
}
hipError_t batch_finish(BatchInstance*, uint32_t, uint32_t*, GraphChain&) { return hipSuccess; }
hipError_t batch_clear_visited(const BatchInstance*, const BatchInstall*, uint32_t, uint64_t, hipStream_t s) {
  return fake::launch(s);
}
hipError_t batch_install(BatchInstance* to, const BatchInstance* staged, const BatchInstall* req, uint32_t n,
                         hipStream_t s) {
  inst = to;
  for (uint32_t q = 0; q < n; ++q) {
    to[req[q].slot] = staged[q];
    if (req[q].seed) to[req[q].slot].status = kInstActive;
  }
  return fake::launch(s);
}
hipError_t batch_owned_export(const BatchInstance&, uint64_t, uint64_t* keys, hipStream_t s) {
  ++exports;
  keys[0] = 0;
  return fake::launch(s);
}
hipError_t batch_gather_sizes(const BatchInstance*, const uint32_t*, uint32_t, uint64_t*, hipStream_t s) {
  return fake::launch(s);
}
}  // namespace mgbfs

struct Range {
  char *from, *to;
};
static Range range(const void* p, uint64_t bytes) {
  char* at = static_cast<char*>(const_cast<void*>(p));
  return Range{at, at + bytes};
}

// Everything the kernels may touch of an instance.
static std::vector<Range> parts(const BatchInstance& d) {
  std::vector<Range> r{range(d.layer_sizes, 8ull * d.max_layers)};
  if (d.rank.owners) {
    const RankPlan& p = d.rank;
    r.push_back(range(d.bitmap, 4ull * p.owners * p.slice_words));
    r.push_back(range(d.words, 4 * OwnedWords::words(p)));
    r.push_back(range(d.list, 4ull * p.owners * p.list_cap));
    for (uint32_t* m : d.messages) r.push_back(range(m, 4 * (static_cast<uint64_t>(p.owners) * d.message_cap + kRouteDump)));
    return r;
  }
  r.push_back(range(d.front, 8 * d.cap));
  r.push_back(range(d.next, 8 * d.cap));
  if (d.visited == kVisBitmap) r.push_back(range(d.bitmap, (d.bitmap_bits + 31) / 32 * 4));
  else r.push_back(range(d.table, (d.rolling ? 3 : 1) * 8ull * d.table_slots));
  return r;
}

// Which degrees of a step's instances go by owners.
static bool takes(uint32_t degree, uint32_t large, uint32_t tens, uint32_t nines, uint32_t others) {
  OwnedChoice c;
  c.large = large;
  c.tens = tens;
  c.nines = nines;
  c.others = others;
  return c.takes(degree);
}

int main() {
  require(takes(12, 1, 0, 0, 5) && takes(11, 1, 1, 9, 9), "degree 11 and 12 always");
  require(takes(10, 0, 1, 0, 0) && takes(10, 0, 7, 0, 0) && takes(10, 1, 1, 0, 9) && takes(10, 0, 8, 99, 9) &&
              takes(10, 0, 4, 8, 4),
          "degree 10 alone, beside larger ones or many together");
  require(!takes(10, 0, 1, 0, 1) && !takes(10, 0, 3, 1, 0) && !takes(10, 0, 4, 9, 0) && !takes(10, 0, 7, 0, 8) &&
              !takes(10, 0, 3, 0, 1),
          "not few of degree 10 beside others");
  require(takes(9, 0, 4, 8, 0) && takes(9, 0, 8, 16, 9) && takes(9, 1, 0, 4, 9) && !takes(9, 0, 8, 17, 0) &&
              !takes(9, 0, 0, 200, 0) && !takes(9, 0, 0, 1, 0) && !takes(9, 1, 0, 5, 0) && !takes(9, 0, 3, 1, 0),
          "degree 9 beside enough larger ones");
  // Steps take the kernels that their instances need: degree 8, then 11, then
  // both.
  {
    auto rotations = [](uint32_t n) {
      Graph g;
      g.elements = n;
      g.generators = 2;
      for (uint32_t i = 0; i < n; ++i) g.perms.push_back((i + 1) % n);
      for (uint32_t i = 0; i < n; ++i) g.perms.push_back(i < 2 ? 1 - i : i);
      for (uint32_t i = 0; i < n; ++i) g.start.push_back(i);
      return g;
    };
    mgbfs_batch_options o{};
    slots = o.max_slots = 2;
    o.vram_budget = 4ull << 30;
    o.layers_per_graph = 4;
    BatchEngine b(o);
    int32_t s = 0;
    b.admit(rotations(8), 1, 0, &s);
    b.step(1);
    require(shared_nodes == 4 && owned_nodes == 0, "a step without instances by owners");
    b.admit(rotations(11), 1, 0, &s);
    b.step(1);
    require(shared_nodes == 4 && owned_nodes == 4, "a step of instances by owners alone");
    b.release(0);
    b.release(1);
    b.admit(rotations(8), 1, 0, &s);
    b.admit(rotations(11), 1, 0, &s);
    b.step(1);
    require(shared_nodes == 8 && owned_nodes == 8, "a step of both");
    b.release(0);
    b.release(1);
    b.admit(rotations(11), 1, 0, &s);
    b.step(1);
    require(shared_nodes == 8 && owned_nodes == 8, "graphs are built once");
  }
  // Calls from a thread whose current device is another.
  {
    Graph g;
    g.elements = 11;
    g.generators = 2;
    for (uint32_t i = 0; i < 11; ++i) g.perms.push_back((i + 1) % 11);
    for (uint32_t i = 0; i < 11; ++i) g.perms.push_back(i < 2 ? 1 - i : i);
    for (uint32_t i = 0; i < 11; ++i) g.start.push_back(i);
    mgbfs_release_cached_memory(0);
    mgbfs_batch_options o{};
    slots = o.max_slots = 2;
    o.vram_budget = 4ull << 30;
    o.device = 1;
    fake::Device& d = fake::dev();
    {
      BatchEngine b(o);
      int32_t s = 0;
      d.current = 0;
      b.admit(g, 1, 0, &s);
      d.current = 0;
      b.step(1);
      require(inst[s].rank.owners != 0, "an instance by owners");
      inst[s].count = 1;
      b.step(1);
      std::vector<int64_t> rows;
      uint64_t n = 0;
      d.current = 0;
      const size_t held = d.used;
      d.limit = held;  // small samples need no device memory
      b.sample(s, 1, rows, n);
      d.limit = ~static_cast<size_t>(0);
      d.current = 0;
      require(exports == 1 && n == 1 && b.poll(2).size() == 1, "a sample and the end");
      d.current = 0;
      b.release(s);
      require(fake::all_on(1), "memory on the engine's device");
    }
    mgbfs_release_cached_memory(1);
    d.current = 0;
  }
  uint32_t owned = 0, restarted = 0;
  for (uint32_t n : {9u, 10u, 11u})
    for (uint32_t history : {0u, 1u, 2u})
      for (uint32_t pct : {1u, 30u, 100u})
        for (uint32_t bias : {1u, 3u, 5u, 8u, 20u, 1000u})
          for (uint64_t expected : {0ull, 20000ull, 120000ull, 200000ull}) {
            Graph g;
            g.elements = n;
            g.generators = 3;
            g.inverse_closed = true;
            g.expected_states = expected;
            for (uint32_t i = 0; i < n; ++i) g.perms.push_back((i + 1) % n);
            for (uint32_t i = 0; i < n; ++i) g.perms.push_back((i + n - 1) % n);
            for (uint32_t i = 0; i < n; ++i) g.perms.push_back(i < 2 ? 1 - i : i);
            for (uint32_t i = 0; i < n; ++i) g.start.push_back(i);
            mgbfs_batch_options o{};
            slots = o.max_slots = 3;
            o.vram_budget = 24ull << 30;
            o.history = history;
            o.layer_pct = pct;
            o.bitmap_bias_permille = bias;
            BatchEngine b(o);
            int32_t s[3];
            for (int32_t& k : s) require(b.admit(g, 0, 40, &k) == 0, "three instances admitted");
            auto apart = [&] {
              std::vector<Range> all;
              for (uint32_t i = 0; i < 3; ++i)
                for (const Range& r : parts(inst[i])) all.push_back(r);
              std::sort(all.begin(), all.end(), [](const Range& x, const Range& y) { return x.from < y.from; });
              for (size_t i = 0; i < all.size(); ++i) {
                require(holds(all[i].from, all[i].to - all[i].from), "a part inside the arena");
                require(i == 0 || all[i - 1].to <= all[i].from, "parts that do not overlap");
              }
            };
            overflow = kErrFutureCap;
            b.step(1);
            apart();
            const bool by_owners = inst[0].rank.owners != 0;
            owned += by_owners;
            overflow = 0;
            b.step(1);
            apart();
            uint32_t visited = 0, layers = 0, restarts = 0;
            uint64_t cap = 0;
            for (int32_t k : s) {
              b.instance_info(k, visited, layers, cap, restarts);
              require(!by_owners || (visited == 1 && !inst[k].rank.owners && !inst[k].error && restarts == 1),
                      "an overflow starts over on the shared bitmap");
              restarted += restarts;
            }
          }
  require(owned > 20 && restarted == 3 * owned, "instances by owners among them");
  mgbfs_release_cached_memory(0);
  std::printf("batch layout ok\n");
  return 0;
}
