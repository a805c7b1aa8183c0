// Host check of rebound and reset engines (engine.hip, rank_engine.hip) on a
// HIP runtime in host memory: which form a graph gets, with what the engine
// itself holds counted as free, and what is left when the other form cannot
// be made.
#include <algorithm>
#include <numeric>
#include <random>
#include "rank_on_host.hpp"

static int others, refuse_other, hand_over;  // engines made in place of the owners; fail to; the next layer

namespace mgbfs {

class Other final : public Engine {
 public:
  Other(uint32_t kind, const char* name) : name_(name) {
    ++others;
    backend = kind;
    layers.assign(1, 1);
  }
  int advance(uint64_t* n, uint32_t*) override {
    if (hand_over) return kAdvanceHandover;
    *n = 0;
    terminal = true;
    return MGBFS_COMPLETE;
  }
  void reset() override { terminal = false; }
  void rebind(const Graph&) override { reset(); }
  bool handover(PackedHandover&) override { return true; }
  void layer_keys(std::vector<uint64_t>&) override {}
  void sample(uint32_t, uint64_t, std::vector<int64_t>&, uint64_t&) override {}
  const char* name() const override { return name_; }

 private:
  const char* name_;
};
Engine* make_sorted_engine(const Graph&, const mgbfs_engine_options&, const WideCode*) {
  if (refuse_other) throw std::runtime_error("SORTED_VRAM_CAPACITY");
  return new Other(MGBFS_BACKEND_SORTED, "sorted");
}
Engine* make_segmented_from_packed(const Graph&, const mgbfs_engine_options&, uint64_t, const PackedHandover&) {
  hand_over = 0;
  return new Other(MGBFS_BACKEND_SEGMENTED, "segmented");
}
hipError_t bitmap_seed(uint32_t, uint64_t, uint32_t*, uint64_t, uint64_t*, uint32_t*, hipStream_t s) {
  return fake::launch(s);
}
hipError_t fill_u64(uint64_t*, uint64_t, uint64_t, hipStream_t s) { return fake::launch(s); }

}  // namespace mgbfs

static Graph graph_of(uint32_t n, std::vector<std::vector<uint32_t>> gens, bool closed) {
  Graph g;
  g.elements = n;
  g.generators = static_cast<uint32_t>(gens.size());
  g.inverse_closed = closed;
  for (const auto& p : gens) g.perms.insert(g.perms.end(), p.begin(), p.end());
  for (uint32_t i = 0; i < n; ++i) g.start.push_back(i);
  return g;
}
static std::vector<std::vector<uint32_t>> swaps(uint32_t n, uint32_t count) {
  std::vector<std::vector<uint32_t>> out;
  for (uint32_t k = 0; k < count; ++k) {
    std::vector<uint32_t> p(n);
    std::iota(p.begin(), p.end(), 0u);
    std::swap(p[k % n], p[(k + 1 + k / n) % n]);
    out.push_back(p);
  }
  return out;
}
template <typename F>
static bool throws(F f) {
  try {
    f();
  } catch (const std::exception&) {
    return true;
  }
  return false;
}

int main() {
  fake::Device& d = fake::dev();
  // Free memory for one degree 10 engine's worst case, not for that and the
  // engine itself.
  const Graph ten = graph_of(10, swaps(10, 9), true);
  mgbfs_engine_options o{};
  for (uint32_t named : {0u, static_cast<uint32_t>(MGBFS_BACKEND_BITMAP)}) {
    o.backend = named;
    const size_t reserve = 2ull << 30;
    {
      o.vram_budget = 1ull << 40;
      std::unique_ptr<Engine> e(create(ten, o));
      require(e->backend == MGBFS_BACKEND_BITMAP && e->device_bytes > (16u << 20), "an engine by owners");
      o.vram_budget = 0;
    }
    size_t low = 0, high = 4ull << 30;  // the least free memory that runs it by owners
    while (high - low > (1u << 20)) {
      const size_t mid = (low + high) / 2;
      d.limit = mid;
      (rank_bitmap_takes(ten, o) ? high : low) = mid;
    }
    require(high > reserve, "free memory beyond the reserve");
    d.limit = high;
    std::unique_ptr<Engine> e(create(ten, o));
    others = 0;
    e->rebind(ten);
    require(others == 0 && std::strcmp(e->name(), "PERMUTATION_BITMAP_LEHMER") == 0 && !rank_bitmap_takes(ten, o),
            "the same graph keeps its form");
    // Sixteen generators need more than there is: the other form.
    Graph more = graph_of(10, swaps(10, 16), true);
    if (!named) {
      refuse_other = 1;
      require(throws([&] { e->rebind(more); }), "the other form cannot be made");
      const std::vector<uint32_t> turn{1, 2, 3, 4, 5, 6, 7, 8, 9, 0};
      require(throws([&] { e->rebind(graph_of(10, {turn}, false)); }),
              "a directed set is refused as before");
      e->rebind(ten);
      require(others == 0, "the engine by owners still runs");
      refuse_other = 0;
    }
    e->rebind(more);
    require(named ? e->device_bytes < (16u << 20) : others == 1, "the other form");
    require(e->layers.size() == 1 && !e->terminal, "at its start");
    d.limit = ~static_cast<size_t>(0);
  }
  // AUTO takes directed sets to the bitmap too, rebound as by name.
  {
    const Graph one = graph_of(9, {{1, 2, 3, 4, 5, 6, 7, 8, 0}, swaps(9, 1)[0]}, false);
    o.backend = MGBFS_BACKEND_AUTO;
    std::unique_ptr<Engine> e(create(one, o));
    require(e->backend == MGBFS_BACKEND_BITMAP && e->run_to_end() == MGBFS_COMPLETE && e->layers == plain(one),
            "a directed set by owners");
    e->rebind(graph_of(9, swaps(9, 3), false));
    require(e->run_to_end() == MGBFS_COMPLETE && e->layers == plain(graph_of(9, swaps(9, 3), false)), "and rebound");
  }
  // The plan by name holds what its engine comes to take.
  for (uint32_t n : {3u, 7u, 8u, 9u})
    for (uint32_t count : {1u, 2u, 16u}) {
      o.backend = MGBFS_BACKEND_BITMAP;
      o.vram_budget = 0;
      const Graph g = graph_of(n, swaps(n, std::min(count, n == 3 ? 3u : 16u)), true);
      const mgbfs_engine_plan_info p = plan_engine(g, o);
      std::unique_ptr<Engine> e(create(g, o));
      e->run_to_end();
      require(p.backend == e->backend && e->device_bytes <= p.device_bytes, "no more than planned");
    }
  // A given budget bounds a rebound engine by name too.
  o.backend = MGBFS_BACKEND_BITMAP;
  o.vram_budget = 64ull << 20;
  {
    const Graph two = graph_of(9, swaps(9, 2), false), sixteen = graph_of(9, swaps(9, 16), false);
    o.vram_budget = 16ull << 20;
    require(rank_bitmap_takes(two, o) && !rank_bitmap_takes(sixteen, o), "a budget between the two");
    std::unique_ptr<Engine> e(create(two, o));
    e->rebind(sixteen);
    require(e->device_bytes <= o.vram_budget && d.used <= o.vram_budget, "within its budget");
    require(throws([&] {
              Graph labels = two;
              labels.start[0] = labels.start[1];
              e->rebind(labels);
            }),
            "repeated labels are refused as before");
  }
  // An engine's calls from a thread whose current device is another.
  for (uint32_t kind : {0u, static_cast<uint32_t>(MGBFS_BACKEND_BITMAP)}) {
    o = mgbfs_engine_options{};
    o.backend = kind;
    o.device = 1;
    const Graph two = graph_of(9, swaps(9, 8), true), more = graph_of(9, swaps(9, 16), true);
    std::unique_ptr<Engine> e(create(two, o));
    uint64_t n = 0;
    std::vector<int64_t> rows;
    d.current = 0;
    e->rebind(more);
    d.current = 0;
    require(e->run_to_end() == MGBFS_COMPLETE, "a run");
    d.current = 0;
    e->reset();
    for (uint32_t fatal, k = 0; k < 6; ++k) {
      d.current = 0;
      e->advance(&n, &fatal);
    }
    d.current = 0;
    e->settle();
    e->sample(0, 4000, rows, n);
    require(n > 1024 && fake::all_on(1), "memory on the engine's device");
    d.current = 0;
  }
  o = mgbfs_engine_options{};
  // One workgroup or many, by the rebound graph's children.
  o.vram_budget = 0;
  for (uint32_t kind : {0u, static_cast<uint32_t>(MGBFS_BACKEND_BITMAP)}) {
    o.backend = kind;
    const Graph few = graph_of(8, swaps(8, 2), true), many = graph_of(8, swaps(8, 16), true);
    std::unique_ptr<Engine> e(create(few, o));
    block_runs = 0;
    e->run_to_end();
    require(block_runs == 1, "two generators of degree 8 by one workgroup");
    e->rebind(many);
    require(e->run_to_end() == MGBFS_COMPLETE && block_runs == 1 && e->layers == plain(many), "sixteen by many");
    e->rebind(few);
    e->run_to_end();
    require(block_runs == 2, "and back");
  }
  // A reset that cannot make its engine refuses calls, and the next one tries
  // again.
  o.backend = MGBFS_BACKEND_SORTED;
  {
    const Graph g = graph_of(13, swaps(13, 12), true);
    std::unique_ptr<Engine> e(create(g, o));
    uint64_t n = 0;
    uint32_t fatal = 0;
    hand_over = 1;
    require(e->advance(&n, &fatal) == MGBFS_COMPLETE && e->backend == MGBFS_BACKEND_SEGMENTED, "a hand-over");
    refuse_other = 1;
    require(throws([&] { e->reset(); }) && throws([&] { e->advance(&n, &fatal); }), "calls are refused");
    std::vector<int64_t> rows;
    require(throws([&] { e->sample(0, 1, rows, n); }) && e->name() != nullptr, "samples too");
    mgbfs_engine_info info{};
    e->settle();
    e->fill_info(info);
    refuse_other = 0;
    e->reset();
    require(e->advance(&n, &fatal) == MGBFS_COMPLETE && e->backend == MGBFS_BACKEND_SORTED, "until one succeeds");
  }
  std::printf("rebind ok\n");
  return 0;
}
