// Host check of reaches_whole_group (rank_engine.hip): against the orbits of
// arrangements at degree 9, against groups of known order, and that the sets
// that searches are made of are recognised.
#include <algorithm>
#include <numeric>
#include <random>
#include "rank_on_host.hpp"

using namespace mgbfs;
using Perm = std::vector<uint32_t>;

static Graph graph_of(const std::vector<Perm>& gens) {
  Graph g;
  g.elements = static_cast<uint32_t>(gens[0].size());
  g.generators = static_cast<uint32_t>(gens.size());
  for (const Perm& p : gens) g.perms.insert(g.perms.end(), p.begin(), p.end());
  for (uint32_t i = 0; i < g.elements; ++i) g.start.push_back(i);
  return g;
}
static Perm turn(uint32_t n) {
  Perm p(n);
  for (uint32_t i = 0; i < n; ++i) p[i] = (i + 1) % n;
  return p;
}
static Perm swap_of(uint32_t n, uint32_t a, uint32_t b) {
  Perm p(n);
  std::iota(p.begin(), p.end(), 0u);
  std::swap(p[a], p[b]);
  return p;
}
static Perm inverse(const Perm& p) {
  Perm q(p.size());
  for (uint32_t i = 0; i < p.size(); ++i) q[p[i]] = i;
  return q;
}
static Perm cycles(uint32_t n, const std::vector<std::vector<uint32_t>>& c) {  // points from 1
  Perm p(n);
  std::iota(p.begin(), p.end(), 0u);
  for (const auto& k : c)
    for (size_t i = 0; i < k.size(); ++i) p[k[i] - 1] = k[(i + 1) % k.size()] - 1;
  return p;
}

int main() {
  std::mt19937 rng(7);
  for (uint32_t n = 9; n <= 12; ++n) {
    require(reaches_whole_group(graph_of({turn(n), inverse(turn(n)), swap_of(n, 0, 1)})), "rotations and a swap");
    require(reaches_whole_group(graph_of({turn(n), swap_of(n, 0, 1)})), "a rotation and a swap");
    std::vector<Perm> c;
    for (uint32_t i = 0; i + 1 < n; ++i) c.push_back(swap_of(n, i, i + 1));
    require(reaches_whole_group(graph_of(c)), "adjacent swaps");
    c.pop_back();
    require(!reaches_whole_group(graph_of(c)), "a fixed point");
    std::vector<Perm> threes;
    for (uint32_t i = 0; i + 2 < n; ++i) threes.push_back(cycles(n, {{i + 1, i + 2, i + 3}}));
    require(reaches_whole_group(graph_of(threes)), "three-cycles: the alternating group");
    require(!reaches_whole_group(graph_of({turn(n)})) && !reaches_whole_group(graph_of({turn(n), inverse(turn(n))})),
            "rotations");
    Perm mirror(n);
    for (uint32_t i = 0; i < n; ++i) mirror[i] = n - 1 - i;
    require(!reaches_whole_group(graph_of({turn(n), mirror})), "rotations and mirrors");
    uint32_t seen = 0, whole = 0;
    for (int k = 0; k < 300; ++k) {
      std::vector<Perm> g;
      for (int j = 0; j < 2 + k % 3; ++j) {
        Perm p(n);
        std::iota(p.begin(), p.end(), 0u);
        std::shuffle(p.begin(), p.end(), rng);
        g.push_back(p);
      }
      Perm root(n);  // orbits of points
      std::iota(root.begin(), root.end(), 0u);
      for (int pass = 0; pass < 12; ++pass)
        for (const Perm& p : g)
          for (uint32_t i = 0; i < n; ++i) root[i] = root[p[i]] = std::min(root[i], root[p[i]]);
      uint32_t parts = 0;
      for (uint32_t i = 0; i < n; ++i) parts += root[i] == i;
      const bool got = reaches_whole_group(graph_of(g));
      require(!got || parts == 1, "a whole group moves every point to every other");
      whole += parts == 1;
      seen += got;
      if (n == 9 && k < 40) {
        uint64_t total = 0;
        for (uint64_t s : plain(graph_of(g))) total += s;
        require(got == (total >= factorial_u64(9) / 2), "the orbit of an arrangement");
      }
    }
    // Nearly all transitive random sets generate the whole group.
    require(whole > 200 && seen + 8 >= whole && seen <= whole, "random sets");
  }
  // Blocks that are kept together: S_5 wr S_2, S_2 wr S_5, S_6 wr S_2, S_3 wr S_4.
  auto wreath = [](uint32_t inner, uint32_t outer) {
    const uint32_t n = inner * outer;
    Perm a(n), b(n), c(n), d(n);
    std::iota(a.begin(), a.end(), 0u);
    b = c = d = a;
    for (uint32_t i = 0; i < inner; ++i) a[i] = (i + 1) % inner;
    std::swap(b[0], b[1]);
    for (uint32_t i = 0; i < n; ++i) c[i] = (i + inner) % n;
    for (uint32_t i = 0; i < inner; ++i) std::swap(d[i], d[inner + i]);
    return graph_of({a, b, c, d});
  };
  require(!reaches_whole_group(wreath(5, 2)) && !reaches_whole_group(wreath(2, 5)) && !reaches_whole_group(wreath(6, 2)) &&
              !reaches_whole_group(wreath(3, 4)) && !reaches_whole_group(wreath(3, 3)),
          "blocks");
  // Primitive and small: the Mathieu groups of degree 11 (7,920 elements) and
  // 12 (95,040).
  const std::vector<std::vector<uint32_t>> a{{1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11}}, b{{3, 7, 11, 8}, {4, 10, 5, 6}},
      c{{1, 12}, {2, 11}, {3, 6}, {4, 8}, {5, 9}, {7, 10}};
  require(!reaches_whole_group(graph_of({cycles(11, a), cycles(11, b)})), "M_11");
  require(!reaches_whole_group(graph_of({cycles(12, a), cycles(12, b), cycles(12, c)})), "M_12");
  std::printf("groups ok\n");
  return 0;
}
