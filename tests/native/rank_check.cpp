// Host check of the owner bitmap's arithmetic: rank and unrank against each
// other and the digits they are made of, children by byte permutes, and the
// owner and position of a rank, for every degree it takes.
#include <algorithm>
#include <cstdio>
#include <numeric>
#include <random>
#include <vector>
#include "rank_owner.hip"

using namespace mgbfs;

static uint64_t pack(const std::vector<int>& p) {
  uint64_t k = 0;
  for (size_t i = 0; i < p.size(); ++i) k |= static_cast<uint64_t>(p[i]) << (4 * i);
  return k;
}

static uint64_t plain_rank(const std::vector<int>& p) {
  uint64_t r = 0;
  for (size_t i = 0; i < p.size(); ++i)
    r += factorial_u64(i) * std::count_if(p.begin(), p.begin() + i, [&](int s) { return s < p[i]; });
  return r;
}

template <uint32_t D>
static bool quotients(uint32_t below) {
  for (uint32_t x = 0; x < below; ++x)
    if (quotient<D>(x) != x / D || (D >= 9 ? (1u << 17) : (1u << 18)) / D + 1 >= (1u << 24)) return false;
  return true;
}

int main() {
  if (!quotients<2>(40320) || !quotients<3>(20160) || !quotients<4>(6720) || !quotients<5>(1680) ||
      !quotients<6>(336) || !quotients<7>(56) || !quotients<9>(11880) || !quotients<10>(1320) || !quotients<11>(132))
    return 6;
  std::mt19937 rng(5);
  for (uint32_t n = 3; n <= kRankDegree; ++n) {
    const RankPlan p = rank_plan(n);
    const uint64_t total = factorial_u64(n);
    if (static_cast<uint64_t>(p.owners) * p.list_cap < total || p.slice_words * 32ull < p.list_cap || p.slice_words % 4)
      return 1;
    std::vector<int> perm(n), child(n);
    PackedGenerators gens{};
    gens.count = kMaxGenerators;
    gens.degree = n;
    for (uint32_t g = 0; g < gens.count; ++g) {
      std::iota(perm.begin(), perm.end(), 0);
      std::shuffle(perm.begin(), perm.end(), rng);
      for (uint32_t i = 0; i < n; ++i) gens.src[g][i] = static_cast<uint8_t>(perm[i]);
      gens.child_tag[g] = static_cast<uint8_t>(g % 3);
    }
    const RankGenerators by = rank_generators(gens, gens.child_tag);
    if (by.count != gens.count || by.tagged != 10) return 7;
    for (uint32_t i = 0; i < 100000; ++i) {
      const uint32_t r = i < 50000 && i < total ? i : i == 60000 ? total - 1 : rng() % total;
      const Bytes b = unrank(r, n);
      if (rank_of(b) != r) return 3;
      const uint64_t key = key_of(b);
      for (uint32_t k = 0; k < n; ++k) perm[k] = static_cast<int>((key >> (4 * k)) & 15u);
      if (n < 12 && key >> (4 * n)) return 8;
      if (plain_rank(perm) != r || !std::is_permutation(perm.begin(), perm.end(), [&] {
            std::iota(child.begin(), child.end(), 0);
            return child.begin();
          }()))
        return 2;
      const uint32_t g = rng() % gens.count;
      for (uint32_t k = 0; k < n; ++k) child[k] = perm[gens.src[g][k]];
      if (key_of(child_of(bytes_of(key), by.of[g])) != pack(child) || rank_of(child_of(b, by.of[g])) != plain_rank(child))
        return 9;
      const Place at = place_of(r, p.owners, p.magic);
      if (at.owner != r % p.owners || at.position != r / p.owners || at.position >= p.list_cap) return 4;
      if (at.position * p.owners + at.owner != r) return 5;
    }
  }
  std::printf("rank ok\n");
  return 0;
}
