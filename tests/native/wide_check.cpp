// Host check of the packed keys of wide states (multigpubfs_amd/csrc/wide.hpp):
// child by child along random walks against the plain actions (permuted
// entries; int64 products wrapped mod 2^64, then rem_euclid), over the forms
// the code accepts, and the forms it must refuse.  Also the inverse masks.
#include <cstdio>
#include <numeric>
#include <random>
#include "wide.hpp"

using namespace mgbfs;

static std::mt19937_64 rng(11);

static std::vector<int64_t> plain_child(const Graph& g, const std::vector<int64_t>& s, uint32_t k) {
  std::vector<int64_t> out(g.elements);
  if (g.kind == 0) {
    for (uint32_t i = 0; i < g.elements; ++i) out[i] = s[g.perms[k * g.elements + i]];
    return out;
  }
  for (uint32_t r = 0; r < g.rows; ++r)
    for (uint32_t c = 0; c < g.cols; ++c) {
      uint64_t acc = 0;
      for (uint32_t j = 0; j < g.rows; ++j)
        acc += static_cast<uint64_t>(g.matrices[(k * g.rows + r) * g.rows + j]) * static_cast<uint64_t>(s[j * g.cols + c]);
      int64_t v = static_cast<int64_t>(acc);
      const uint32_t m = g.moduli[k];
      if (m) {
        v %= static_cast<int64_t>(m);
        if (v < 0) v += m;
      }
      out[r * g.cols + c] = v;
    }
  return out;
}

static bool walk(const Graph& g, const char* what) {
  WideCode w;
  if (!make_wide(g, w, 60)) {
    std::printf("%s: refused\n", what);
    return false;
  }
  uint64_t key = w.start_key;
  std::vector<int64_t> s = g.start;
  for (int step = 0; step < 400; ++step) {
    for (uint32_t e = 0; e < g.elements; ++e)
      if (w.value(key, e) != s[e]) {
        std::printf("%s: step %d entry %u\n", what, step, e);
        return false;
      }
    if (w.key_bits() < 64 && key >> w.key_bits()) return false;
    const uint32_t k = static_cast<uint32_t>(rng() % g.generators);
    const uint64_t child = wide_child(&w.table, key, k);
    for (uint32_t b = 0; b < g.generators; ++b)
      if ((w.table.child_mask[k] >> b) & 1u)
        if (wide_child(&w.table, child, b) != key) {
          std::printf("%s: generator %u does not lead back from %u\n", what, b, k);
          return false;
        }
    key = child;
    s = plain_child(g, s, k);
  }
  return true;
}

static Graph permutation_graph(uint32_t n, uint32_t labels, uint32_t gens, bool inverses) {
  Graph g;
  g.kind = 0;
  g.elements = n;
  for (uint32_t i = 0; i < n; ++i) g.start.push_back(static_cast<int64_t>(i % labels) * 1000003 - 7);
  std::shuffle(g.start.begin(), g.start.end(), rng);
  for (uint32_t k = 0; k < gens; ++k) {
    std::vector<uint32_t> p(n);
    std::iota(p.begin(), p.end(), 0u);
    if (k % 3 == 0) std::rotate(p.begin(), p.begin() + 1 % n, p.end());
    else std::shuffle(p.begin(), p.end(), rng);
    g.perms.insert(g.perms.end(), p.begin(), p.end());
    ++g.generators;
    if (inverses) {
      std::vector<uint32_t> q(n);
      for (uint32_t i = 0; i < n; ++i) q[p[i]] = i;
      g.perms.insert(g.perms.end(), q.begin(), q.end());
      ++g.generators;
    }
  }
  return g;
}

static Graph matrix_graph(uint32_t rows, uint32_t cols, uint32_t m, uint32_t gens, int64_t range) {
  Graph g;
  g.kind = 1;
  g.rows = rows;
  g.cols = cols;
  g.elements = rows * cols;
  g.generators = gens;
  for (uint32_t i = 0; i < g.elements; ++i) g.start.push_back(static_cast<int64_t>(rng() % m));
  for (uint32_t k = 0; k < gens; ++k) {
    for (uint32_t i = 0; i < rows * rows; ++i) g.matrices.push_back(static_cast<int64_t>(rng() % (2 * range + 1)) - range);
    g.moduli.push_back(m);
  }
  return g;
}

int main() {
  for (uint32_t n : {1u, 2u, 3u, 7u, 15u, 16u, 17u, 20u, 24u, 30u, 31u, 48u, 60u})
    for (uint32_t labels : {1u, 2u, 3u, 4u, 5u, 8u, 16u}) {
      if (labels > n || bits_for(labels) * n > 60) continue;
      for (bool inverses : {false, true}) {
        const Graph g = permutation_graph(n, labels, 4, inverses);
        if (!walk(g, "permutation")) return 1;
        WideCode w;
        make_wide(g, w, 60);
        if (inverses && !w.paired) return 1;
      }
    }
  for (uint32_t m : {2u, 3u, 4u, 5u, 101u, 211u, 256u, 257u, 521u, 4093u, 32749u, 32768u})
    for (uint32_t rows : {1u, 2u, 3u, 4u})
      for (uint32_t cols : {1u, 2u, 3u}) {
        if (bits_for(m) * rows * cols > 60) continue;
        if (!walk(matrix_graph(rows, cols, m, 5, 3), "matrix")) return 1;
        if (!walk(matrix_graph(rows, cols, m, 5, 1ll << 40), "matrix, large entries")) return 1;
      }
  for (uint32_t m : {(1u << 29) - 3, 1u << 30, (1u << 30) + 3})
    if (!walk(matrix_graph(1, 1, m, 3, 1ll << 32), "one large entry")) return 1;
  if (!walk(matrix_graph(2, 1, (1u << 30) - 35, 3, 5), "two large entries")) return 1;
  // Refused: too wide, a start outside the modulus, no or several moduli,
  // products that may wrap, too many generators.
  WideCode w;
  if (make_wide(permutation_graph(16, 16, 2, false), w, 60) || make_wide(permutation_graph(61, 2, 2, false), w, 64))
    return 2;
  Graph g = matrix_graph(2, 2, 257, 2, 3);
  g.start[1] = 257;
  if (make_wide(g, w, 60)) return 2;
  g.start[1] = -1;
  if (make_wide(g, w, 60)) return 2;
  g = matrix_graph(2, 2, 257, 2, 3);
  g.moduli[1] = 251;
  if (make_wide(g, w, 60)) return 2;
  g.moduli = {0, 0};
  if (make_wide(g, w, 60)) return 2;
  g = matrix_graph(2, 2, 257, 2, 3);
  g.matrices[3] = INT64_MIN;
  if (make_wide(g, w, 60)) return 2;
  if (make_wide(matrix_graph(2, 2, 257, 17, 3), w, 60)) return 2;
  // The modular reduction at its edges.
  for (uint32_t m : {2u, 3u, 5u, 65535u, 65536u, 65537u, (1u << 31) - 1, 1u << 31})
    for (int i = 0; i < 200000; ++i) {
      const uint64_t x = i < 4 ? ~0ull - i : rng();
      if (mod64(x, m, ~0ull / m) != x % m) return 3;
      const uint32_t y = i < 4 ? ~0u - i : static_cast<uint32_t>(rng());
      if (mod32(y, m, static_cast<uint32_t>((1ull << 32) / m)) != y % m) return 3;
    }
  std::printf("wide keys ok\n");
  return 0;
}
