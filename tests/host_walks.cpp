// Index arithmetic of the kernels followed on the CPU (built and run by test_host_walks.py).
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include <algorithm>
#include <random>
#include <vector>

#include "group_walk.h"
#include "search.h"

using namespace mccnn;

#define EXPECT(cond, ...)                               \
  do {                                                  \
    if (!(cond)) {                                      \
      fprintf(stderr, "%s:%d: ", __FILE__, __LINE__);   \
      fprintf(stderr, __VA_ARGS__);                     \
      fprintf(stderr, "\n");                            \
      exit(1);                                          \
    }                                                   \
  } while (0)

// One block after the other walks its groups as both_grads_group_kernel does: a chunk is parked
// while the one before is in hand, and the rows of a group are sent after that.  Every pair is come
// to once, and the keys that a group is sent by are its own.
static void walk_groups(const std::vector<int> &counts, int group, int blocks) {
  constexpr int kChunk = 64;
  const int n = (int)counts.size(), groups = (n + group - 1) / group;
  std::vector<int> begins(n + 1, 0);
  for (int i = 0; i < n; ++i) begins[i + 1] = begins[i] + counts[i];
  std::vector<GroupCentre> listed(n, GroupCentre{-1, -1, -1, -1});
  for (int g = 0; g < groups; ++g) {
    std::vector<GroupCentre> own;
    for (int i = g * group; i < std::min(n, (g + 1) * group); ++i)
      if (counts[i] > 0) own.push_back({i, begins[i], counts[i], 4 * (g % 100)});
    if (own.empty()) own.push_back({g * group, begins[g * group], 0, 0});
    own.back().flags += 1;
    std::copy(own.begin(), own.end(), listed.begin() + (size_t)g * group);
  }
  std::vector<int> seen(begins[n], 0), sent(groups, 0);
  for (int block = 0; block < blocks; ++block) {
    GroupWalk<kChunk> walk(listed.data(), n, group, groups, blocks, block);
    int keys[2] = {-1, -1};
    auto park = [&](const GroupChunk &c) {
      if (c.first) keys[c.odd] = c.group;
    };
    auto read = [&]() {
      walk.fetch();
      return walk.read();
    };
    GroupChunk c = read();
    if (c.group < 0) continue;
    GroupChunk next = read(), ahead = read();
    park(c);
    while (true) {
      EXPECT(c.centre / group == c.group && c.group % blocks == block && c.rows == c.group % 100,
             "centre %d in group %d of block %d", c.centre, c.group, block);
      for (int m = c.begin; m < c.begin + std::min(c.left, kChunk); ++m) ++seen[m];
      if (next.group >= 0) park(next);
      if (c.last) {
        EXPECT(keys[c.odd] == c.group, "group %d sent by the keys of group %d", c.group, keys[c.odd]);
        ++sent[c.group];
      }
      if (next.group < 0) break;
      c = next;
      next = ahead;
      ahead = read();
    }
  }
  for (size_t m = 0; m < seen.size(); ++m) EXPECT(seen[m] == 1, "pair %zu: %d times", m, seen[m]);
  for (int g = 0; g < groups; ++g) {
    const int end = std::min(n, (g + 1) * group);
    EXPECT(sent[g] == (begins[end] > begins[g * group]), "group %d sent %d times", g, sent[g]);
  }
}

static void test_groups() {
  walk_groups({3, 70, 0, 0, 9, 1}, 2, 1);         // a group without pairs between two others
  walk_groups({3, 70, 0, 0, 0, 0, 9, 1}, 2, 1);   // two of them
  walk_groups({0, 0, 3, 0, 0, 0, 0, 0, 0, 0, 64, 65, 0}, 2, 1);
  walk_groups({0, 0, 0, 0}, 2, 1);
  std::mt19937 rng(7);
  for (int round = 0; round < 300; ++round) {
    const int group = 4 + (int)(rng() % 61), blocks = 1 << rng() % 9, longest = 1 + (int)(rng() % 200);
    const int empty = (int)(rng() % 4);           // of eight groups
    std::vector<int> counts(1 + rng() % 4000);
    for (size_t i = 0; i < counts.size(); ++i) {
      if (i % group == 0 && (int)(rng() % 8) < empty) {
        i += group - 1;                           // (stays without pairs)
        continue;
      }
      counts[i] = rng() % 5 ? (int)(rng() % (longest + 1)) : 0;
    }
    walk_groups(counts, group, blocks);
  }
}

// Slices of descending keys against the definition: of short tables for all pairs of bounds and spans,
// and of 2^31 - 1 keys, whose last positions a step must not run past.
static void test_slices() {
  auto expect = [](int x, int y, int64_t maxk, int64_t mink, const int64_t *keys, int first, int last) {
    KeyRange range{make_int2(x, y), maxk, mink};
    int2 got;
    find_slices<1>(&range, keys, &got);
    EXPECT(last > first ? got.x == first && got.y == last : got.x == 0 && got.y == 0,
           "keys %ld .. %ld of [%d, %d): [%d, %d), not [%d, %d)", (long)maxk, (long)mink, x, y, got.x,
           got.y, first, last);
  };
  const int64_t keys[] = {9, 9, 7, 7, 7, 6, 4, 3, 3, 1, 0};
  for (int x = 0; x <= 11; ++x)
    for (int y = x; y <= 11; ++y)
      for (int64_t mink = -1; mink <= 10; ++mink)
        for (int64_t maxk = mink; maxk <= 10; ++maxk) {
          int first = x, last = x;
          while (first < y && keys[first] > maxk) ++first;
          while (last < y && keys[last] >= mink) ++last;
          expect(x, y, maxk, mink, keys, first, last);
        }
  const int64_t n = ((int64_t)1 << 31) - 1;      // (pages that nothing is written to take no memory)
  int64_t *many = (int64_t *)mmap(nullptr, n * sizeof(int64_t), PROT_READ | PROT_WRITE,
                                  MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  EXPECT(many != MAP_FAILED, "no address space for 2^31 keys");
  for (int i = 0; i < 50; ++i) many[i] = 2, many[n - 1 - i] = -2;
  for (int begin : {0, 7, 50, 100, 1 << 30, (1 << 30) + 1, (int)n - 60, (int)n - 20})
    for (int end : {(int)n, (int)n - 1, (int)n - 3, (int)n - 9}) {
      const int zeros = begin < 50 ? 50 : begin, low = (int)n - 50;
      expect(begin, end, 0, 0, many, zeros, low);
      expect(begin, end, -1, -2, many, low > begin ? low : begin, end);
      expect(begin, end, 2, -2, many, begin, end);
      expect(begin, end, 2, 1, many, begin, zeros);
      expect(begin, end, -3, -4, many, end, end);
    }
  munmap(many, n * sizeof(int64_t));
}

int main(int argc, char **argv) {
  if (argc == 2 && !strcmp(argv[1], "groups")) test_groups();
  else if (argc == 2 && !strcmp(argv[1], "slices")) test_slices();
  else return 2;
  printf("ok\n");
  return 0;
}
