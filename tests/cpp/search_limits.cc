// Host model of the workgroup tier's ranges (dte_build.hip:
// rf_bound_team_body): every bucket that may be split again is pushed before
// the last one pushed is taken.  Prints the most ranges that wait at a time.
// With an argument: the words of the out-of-bag pass instead.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../datamininglibs_amd/csrc/dte_limits.h"

using namespace dte;

struct Entry {
  uint32_t key, weight;
};

int most_waiting(const std::vector<Entry>& node, int log_buckets) {
  uint32_t lo = 0xFFFFFFFFu, hi = 0, total = 0;
  for (const Entry& e : node) {
    lo = std::min(lo, e.key);
    hi = std::max(hi, e.key);
    total += e.weight;
  }
  if (total > (uint32_t)kBoundWeight) std::abort();
  struct Range {
    uint32_t k0;
    int bits;
  };
  auto bit_length = [](uint32_t v) {
    int b = 0;
    for (; v; v >>= 1) ++b;
    return b;
  };
  std::vector<Range> stack{{lo, bit_length(hi - lo)}};
  size_t most = 0;
  while (!stack.empty()) {
    const Range r = stack.back();
    stack.pop_back();
    const int shift = std::max(0, r.bits - log_buckets);
    const uint32_t n = 1u << (r.bits - shift);
    std::vector<uint32_t> weight(n, 0);
    for (const Entry& e : node)
      if (e.key >= r.k0 && (e.key - r.k0) >> shift < n) weight[(e.key - r.k0) >> shift] += e.weight;
    for (uint32_t b = 0; b < n; ++b)
      if (team_splits_again(weight[b], shift)) stack.push_back({r.k0 + (b << shift), shift});
    most = std::max(most, stack.size());
  }
  return (int)most;
}

// In-bag bits of the out-of-bag pass: whole words, no more than needed.
bool bag_words_fit() {
  for (int64_t rows : {1, 31, 32, 33, 40, 64, 1000, (1 << 19) - 1, 1 << 19, (1 << 19) + 1, 1 << 30}) {
    const int64_t held = std::min(rows, kBagRange), bytes = bag_lds_bytes(rows);
    if (bytes % 4 || bytes > 65536 || bytes * 8 < held || bytes * 8 >= held + 32) return false;
  }
  return true;
}

int main(int argc, char**) {
  if (argc > 1) return bag_words_fit() ? 0 : 1;
  std::mt19937 rng(1);
  int most = 0;
  for (int log_buckets : {7, 8}) {
    // bootstrapped rows with most keys in clusters, one per a few buckets
    for (int clusters = 30; clusters <= 52; ++clusters) {
      std::vector<Entry> node;
      while (node.size() < 2048) {
        int w = 0;  // Poisson(1), not 0
        while (!w) w = std::poisson_distribution<int>(1.0)(rng);
        node.push_back({(uint32_t)(node.size() % clusters * 997 + rng() % 40), (uint32_t)w});
      }
      most = std::max(most, most_waiting(node, log_buckets));
    }
    std::printf("bootstrap %d\n", most);
    // the heaviest node, its weight in clusters of the smallest weight that is
    // split again, all but the last few of a level in buckets of their own
    const uint32_t nb = 1u << log_buckets;
    std::vector<Entry> node;
    uint32_t left = kBoundWeight, k0 = 0;
    for (int bits = 28; bits > log_buckets && left > (uint32_t)kBoundRun; bits -= log_buckets) {
      const uint32_t width = 1u << (bits - log_buckets);
      for (uint32_t b = 0; b + 1 < nb && left > (uint32_t)kBoundRun; ++b, left -= kBoundRun + 1) {
        node.push_back({k0 + b * width, 32});
        node.push_back({k0 + b * width + width - 1, (uint32_t)kBoundRun + 1 - 32});
      }
      k0 += (nb - 1) * width;
    }
    node.push_back({0x0FFFFFFFu, left});
    const int heavy = most_waiting(node, log_buckets);
    std::printf("heavy %d entries %zu\n", heavy, node.size());
    most = std::max(most, heavy);
  }
  std::printf("most %d capacity %d\n", most, kTeamStack);
  return most <= kTeamStack ? 0 : 1;
}
