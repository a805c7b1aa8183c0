// Host check of the owner bitmap engine's message buffers (rank_engine.hip)
// on a HIP runtime in host memory, the kernels restated on the host: growth
// that cannot be had leaves the layers found, never reaches freed memory,
// and the search goes on or starts anew once there is room.
#include <algorithm>
#include <numeric>
#include <random>
#include <vector>
#include "rank_on_host.hpp"

int main() {
  // Sixteen generators of S_9: the widest layers send more children than
  // the first buffers hold.
  constexpr uint32_t n = 9;
  Graph g;
  g.elements = n;
  std::mt19937 rng(3);
  for (uint32_t k = 0; k < 16; ++k) {
    std::vector<uint32_t> p(n);
    std::iota(p.begin(), p.end(), 0u);
    std::shuffle(p.begin(), p.end(), rng);
    g.perms.insert(g.perms.end(), p.begin(), p.end());
  }
  g.generators = 16;
  for (int64_t i = 0; i < n; ++i) g.start.push_back(i);
  const std::vector<uint64_t> want = plain(g);
  mgbfs_engine_options o{};
  o.vram_budget = 1ull << 32;
  fake::Device& d = fake::dev();
  for (int stepwise = 0; stepwise < 2; ++stepwise) {
    std::unique_ptr<Engine> e(make_rank_bitmap_engine(g, o));
    const size_t held = d.used;
    auto search = [&] {
      uint64_t n = 0;
      uint32_t fatal = 0;
      int s = MGBFS_LAYER;
      if (!stepwise) return e->run_to_end();
      while (s == MGBFS_LAYER) s = e->advance(&n, &fatal);
      return s;
    };
    auto fails = [&] {
      try {
        search();
      } catch (const HipError&) {
        return true;
      }
      return false;
    };
    auto prefix = [&] {
      return !e->terminal && e->layers.size() < want.size() && std::equal(e->layers.begin(), e->layers.end(), want.begin());
    };
    auto samples = [&] {
      std::vector<int64_t> rows;
      uint64_t count = 0;
      e->sample(0, 1000, rows, count);
      return count == std::min<uint64_t>(1000, e->layers.back());
    };
    d.limit = held;  // no room to grow
    require(fails() && prefix() && samples(), "the first failure keeps the layers found");
    const size_t reached = e->layers.size();
    d.limit = d.used;  // what was given back is taken by others
    for (int again = 0; again < 3; ++again)
      require(fails() && e->layers.size() == reached && prefix() && samples(), "later calls fail in the same place");
    e->reset();
    require(fails() && e->layers.size() == 1 && samples(), "a reset engine asks for its first buffers");
    d.limit = ~static_cast<size_t>(0);
    require(search() == MGBFS_COMPLETE && e->layers == want, "the search completes when there is room");
    d.limit = d.used;
    e->reset();
    // Whole layers are read back without more memory and without harm.
    for (uint64_t count = 0, k = 0; k < 5; ++k) {
      uint32_t fatal = 0;
      std::vector<uint64_t> keys;
      require(e->advance(&count, &fatal) == MGBFS_LAYER, "a layer");
      e->layer_keys(keys);
      std::sort(keys.begin(), keys.end());
      require(keys.size() == e->layers.back() && std::unique(keys.begin(), keys.end()) == keys.end(), "its states");
    }
    require(search() == MGBFS_COMPLETE && e->layers == want, "and again without more");
    // A rebind that needs larger buffers than there is room for leaves the
    // old graph in place.
    std::unique_ptr<Engine> two;
    Graph few = g;
    few.generators = 2;
    few.perms.resize(2 * n);
    d.limit = ~static_cast<size_t>(0);
    two.reset(make_rank_bitmap_engine(few, o));
    uint64_t count = 0;
    uint32_t fatal = 0;
    require(two->advance(&count, &fatal) == MGBFS_LAYER, "a layer before the rebind");
    d.limit = d.used;
    bool refused = false;
    try {
      two->rebind(g);
    } catch (const HipError&) {
      refused = true;
    }
    d.limit = ~static_cast<size_t>(0);
    require(refused && two->run_to_end() == MGBFS_COMPLETE && two->layers == plain(few), "the old graph runs on");
  }
  std::printf("rank memory ok\n");
  return 0;
}
