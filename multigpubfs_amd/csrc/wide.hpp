// Packed keys for states outside the nibble encoding: permutations of up to
// 60 positions over few distinct labels, and small modular matrices.  A
// state of `elements` entries of `bits` bits each is one 64-bit key, so the
// sorted backend's layers (one word per state, equality of words) carry it
// instead of rows looked up through a hash table.
#pragma once
#include <algorithm>
#include <cstdint>
#include <cstring>
#include <vector>
#include "common.hpp"
#include "engine.hpp"

namespace mgbfs {

constexpr uint32_t kWideElements = 60;
constexpr uint32_t kWideRows = 8;

// The generators on packed keys.  Permutations are shift groups (see
// PackedGenerators): entry i of the child takes entry i + delta of the
// parent for every i in the group's mask, right shifts first.  Matrices
// have entries already reduced by the common modulus.
struct WideTable {
  uint32_t kind, count, elements, bits;  // kind 0 permutation, 1 matrix
  uint32_t rows, cols, modulus, narrow;  // narrow: row sums fit 32 bits
  uint64_t magic64;                      // floor(2^64 / modulus) or one less
  uint32_t magic32, pad;                 // floor(2^32 / modulus)
  uint32_t child_mask[kMaxGenerators];   // generators leading back from a child (see PackedGenerators)
  uint32_t groups[kMaxGenerators], right[kMaxGenerators];
  uint32_t shift[kMaxGenerators][kWideElements];
  uint64_t mask[kMaxGenerators][kWideElements];
  uint32_t mat[kMaxGenerators][kWideRows * kWideRows];
};

// x mod m from magic = floor(2^w / m): the estimated quotient is the exact
// one or one less (x e / 2^w < 1 for the magic's rounding error e <= 1), so
// one correction suffices.
__host__ __device__ __forceinline__ uint32_t mod32(uint32_t x, uint32_t m, uint32_t magic) {
  const uint32_t q = static_cast<uint32_t>((static_cast<uint64_t>(x) * magic) >> 32);
  const uint32_t r = x - q * m;
  return r >= m ? r - m : r;
}
__host__ __device__ __forceinline__ uint32_t mod64(uint64_t x, uint32_t m, uint64_t magic) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint64_t q = __umul64hi(x, magic);
#else
  const uint64_t q = static_cast<uint64_t>((static_cast<unsigned __int128>(x) * magic) >> 64);
#endif
  const uint64_t r = x - q * m;
  return static_cast<uint32_t>(r >= m ? r - m : r);
}

// Child of `key` under generator g; Table: a pointer to WideTable (on the
// device in the constant address space, so that a uniform g is read with
// scalar loads).
template <typename Table>
__host__ __device__ __forceinline__ uint64_t wide_child(Table t, uint64_t key, uint32_t g) {
  uint64_t child = 0;
  if (t->kind == 0) {
    const uint32_t right = t->right[g], groups = t->groups[g];
    uint32_t j = 0;
    for (; j < right; ++j) child |= (key >> t->shift[g][j]) & t->mask[g][j];
    for (; j < groups; ++j) child |= (key << t->shift[g][j]) & t->mask[g][j];
    return child;
  }
  const uint32_t rows = t->rows, cols = t->cols, bits = t->bits, m = t->modulus;
  const uint32_t low = (1u << bits) - 1u;
  for (uint32_t c = 0; c < cols; ++c)
    for (uint32_t r = 0; r < rows; ++r) {
      uint32_t v;
      if (t->narrow) {
        uint32_t acc = 0;
        for (uint32_t k = 0; k < rows; ++k)
          acc += t->mat[g][r * rows + k] * (static_cast<uint32_t>(key >> (bits * (k * cols + c))) & low);
        v = mod32(acc, m, t->magic32);
      } else {
        uint64_t acc = 0;
        for (uint32_t k = 0; k < rows; ++k)
          acc += static_cast<uint64_t>(t->mat[g][r * rows + k]) *
                 (static_cast<uint32_t>(key >> (bits * (k * cols + c))) & low);
        v = mod64(acc, m, t->magic64);
      }
      child |= static_cast<uint64_t>(v) << (bits * (r * cols + c));
    }
  return child;
}

// Wide keys: the table through the constant address space, so that a
// generator index that is uniform in the wave reads it with scalar loads.
struct WideAction {
  const WideTable* table;
  uint32_t generators;
  using ConstTable = const __attribute__((address_space(4))) WideTable*;
  __device__ __forceinline__ uint32_t count() const { return generators; }
  __device__ __forceinline__ uint64_t child(uint64_t key, uint32_t g) const {
    return wide_child((ConstTable)table, key, g);
  }
  __device__ __forceinline__ uint32_t mask(uint32_t g) const { return ((ConstTable)table)->child_mask[g]; }
};

// What a packed key stands for.
struct WideCode {
  WideTable table;
  std::vector<int64_t> labels;  // permutations: entry value -> label; matrices: empty (the value itself)
  uint64_t start_key = 0;
  bool paired = false;  // every generator has its inverse in the set (child_mask is complete)
  uint32_t key_bits() const { return table.bits * table.elements; }
  int64_t value(uint64_t key, uint32_t e) const {
    const uint64_t v = (key >> (table.bits * e)) & ((1ull << table.bits) - 1);
    return labels.empty() ? static_cast<int64_t>(v) : labels[v];
  }
};

inline uint32_t bits_for(uint64_t values) {
  uint32_t b = 1;
  while ((1ull << b) < values) ++b;
  return b;
}

inline bool wide_permutation(const Graph& g, WideCode& w, uint32_t max_bits) {
  WideTable& t = w.table;
  if (g.elements > kWideElements) return false;
  w.labels = g.start;
  std::sort(w.labels.begin(), w.labels.end());
  w.labels.erase(std::unique(w.labels.begin(), w.labels.end()), w.labels.end());
  t.bits = bits_for(w.labels.size());
  if (t.bits * g.elements > max_bits) return false;
  for (uint32_t i = 0; i < g.elements; ++i) {
    const uint64_t v = std::lower_bound(w.labels.begin(), w.labels.end(), g.start[i]) - w.labels.begin();
    w.start_key |= v << (t.bits * i);
  }
  const uint64_t entry = (1ull << t.bits) - 1;
  for (uint32_t k = 0; k < g.generators; ++k) {
    const uint32_t* p = &g.perms[static_cast<size_t>(k) * g.elements];
    for (int pass = 0; pass < 2; ++pass)  // right shifts (source at or above the destination) first
      for (uint32_t i = 0; i < g.elements; ++i) {
        if ((p[i] >= i) != (pass == 0)) continue;
        const uint32_t by = t.bits * (p[i] >= i ? p[i] - i : i - p[i]);
        uint32_t j = pass == 0 ? 0 : t.right[k];
        while (j < t.groups[k] && t.shift[k][j] != by) ++j;
        if (j == t.groups[k]) {
          t.shift[k][j] = by;
          ++t.groups[k];
          if (pass == 0) ++t.right[k];
        }
        t.mask[k][j] |= entry << (t.bits * i);
      }
  }
  w.paired = true;
  for (uint32_t a = 0; a < g.generators; ++a) {
    for (uint32_t b = 0; b < g.generators; ++b) {
      bool inverse = true;
      for (uint32_t i = 0; i < g.elements && inverse; ++i)
        inverse = g.perms[static_cast<size_t>(b) * g.elements + g.perms[static_cast<size_t>(a) * g.elements + i]] == i;
      if (inverse) t.child_mask[a] |= 1u << b;
    }
    w.paired &= t.child_mask[a] != 0;
  }
  return true;
}

// Matrices with one common modulus, canonical start entries, and products
// that cannot wrap in int64 (the wrapping action is then the modular one).
inline bool wide_matrix(const Graph& g, WideCode& w, uint32_t max_bits) {
  WideTable& t = w.table;
  const uint32_t n = g.rows;
  const uint64_t m = g.moduli[0];
  if (n > kWideRows || m < 2) return false;
  for (uint32_t x : g.moduli)
    if (x != m) return false;
  t.bits = bits_for(m);
  if (t.bits > 31 || t.bits * g.elements > max_bits) return false;
  for (int64_t v : g.start)
    if (v < 0 || v >= static_cast<int64_t>(m)) return false;
  const auto square = static_cast<unsigned __int128>(m - 1) * (m - 1) * n;
  if (square >> 64) return false;
  t.narrow = square < (1ull << 32);
  t.modulus = static_cast<uint32_t>(m);
  t.magic32 = static_cast<uint32_t>((1ull << 32) / m);
  t.magic64 = ~0ull / m;
  t.rows = n;
  t.cols = g.cols;
  for (uint32_t k = 0; k < g.generators; ++k)
    for (uint32_t r = 0; r < n; ++r) {
      unsigned __int128 sum = 0;
      for (uint32_t c = 0; c < n; ++c) {
        const int64_t v = g.matrices[(static_cast<size_t>(k) * n + r) * n + c];
        sum += static_cast<unsigned __int128>(v < 0 ? 0ull - static_cast<uint64_t>(v) : static_cast<uint64_t>(v)) * (m - 1);
        const int64_t rem = v % static_cast<int64_t>(m);
        t.mat[k][r * n + c] = static_cast<uint32_t>(rem < 0 ? rem + static_cast<int64_t>(m) : rem);
      }
      if (sum > static_cast<unsigned __int128>(INT64_MAX)) return false;
    }
  for (uint32_t e = 0; e < g.elements; ++e) w.start_key |= static_cast<uint64_t>(g.start[e]) << (t.bits * e);
  w.paired = true;
  for (uint32_t a = 0; a < g.generators; ++a) {
    for (uint32_t b = 0; b < g.generators; ++b) {
      bool inverse = true;
      for (uint32_t r = 0; r < n && inverse; ++r)
        for (uint32_t c = 0; c < n && inverse; ++c) {
          uint64_t acc = 0;
          for (uint32_t k = 0; k < n; ++k) acc += static_cast<uint64_t>(t.mat[b][r * n + k]) * t.mat[a][k * n + c];
          inverse = acc % m == (r == c ? 1u : 0u);
        }
      if (inverse) t.child_mask[a] |= 1u << b;
    }
    w.paired &= t.child_mask[a] != 0;
  }
  return true;
}

// The packed code of a graph in at most max_bits bits; false when it has
// none.  Only then is anything in `w` meaningful.
inline bool make_wide(const Graph& g, WideCode& w, uint32_t max_bits) {
  w = WideCode{};
  std::memset(&w.table, 0, sizeof(w.table));
  if (g.elements == 0 || g.generators == 0 || g.generators > kMaxGenerators) return false;
  w.table.kind = g.kind;
  w.table.count = g.generators;
  w.table.elements = g.elements;
  return g.kind == 0 ? wide_permutation(g, w, max_bits) : wide_matrix(g, w, max_bits);
}

}  // namespace mgbfs
