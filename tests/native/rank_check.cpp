// Host check of the owner bitmap's arithmetic: rank and unrank against
// lexicographic order, and the owner and position of a rank, for every
// degree it takes.
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

int main() {
  std::mt19937 rng(5);
  for (uint32_t n = 3; n <= kRankDegree; ++n) {
    const RankPlan p = rank_plan(n);
    const uint64_t total = factorial_u64(n);
    if (static_cast<uint64_t>(p.owners) * p.list_cap < total || p.slice_words * 32ull < p.list_cap || p.slice_words % 4)
      return 1;
    std::vector<int> perm(n);
    std::iota(perm.begin(), perm.end(), 0);
    const uint64_t in_order = std::min<uint64_t>(total, 50000);
    for (uint64_t r = 0; r < in_order; ++r) {
      if (rank_of(pack(perm), n) != r || unrank(static_cast<uint32_t>(r), n) != pack(perm)) return 2;
      std::next_permutation(perm.begin(), perm.end());
    }
    for (int i = 0; i < 100000; ++i) {
      const uint32_t r = i == 0 ? static_cast<uint32_t>(total - 1) : static_cast<uint32_t>(rng() % total);
      if (rank_of(unrank(r, n), n) != r) return 3;
      const Place at = place_of(r, p.owners, p.magic);
      if (at.owner != r % p.owners || at.position != r / p.owners || at.position >= p.list_cap) return 4;
      if (at.position * p.owners + at.owner != r) return 5;
    }
  }
  std::printf("rank ok\n");
  return 0;
}
