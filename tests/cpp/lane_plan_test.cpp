// The overlap plan of the wave kernels, on the host: both storages give the
// same tables, the lanes' sums are those of the lists, and the fixed storage
// takes nothing from the heap (sp_compute_step_noalloc builds its plan there).
#include <cstdio>
#include <cstdlib>
#include <new>
#include <random>

#include "lane_plan.h"

static long g_news = 0;
void *operator new(std::size_t n) {
  ++g_news;
  if (void *p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

using namespace frg;
constexpr int kItems = 200000, kElements = 1024, kOutputs = 32, kLanes = 64;
static LanePlanOf<FixedPlan<kItems, kElements, kOutputs>> fixed;
static unsigned ent[4 * kItems];
static int count[kLanes];

template <class P> void fill(P &p, const std::vector<std::vector<unsigned>> &lists) {
  p.begin(kElements, (int)lists.size());
  for (const auto &l : lists) {
    for (unsigned k : l) p.add(k);
    p.end_output();
  }
  p.deal(kLanes);
}

static int check(const std::vector<std::vector<unsigned>> &lists) {
  const long before = g_news;
  fill(fixed, lists);
  fixed.store(ent, count);
  if (g_news != before) { std::printf("the fixed plan used the heap\n"); return 1; }
  LanePlan heap;
  fill(heap, lists);
  std::vector<unsigned> e(heap.entries());
  std::vector<int> c(kLanes);
  heap.store(e.data(), c.data());
  if (heap.rows != fixed.rows || !std::equal(e.begin(), e.end(), ent) || !std::equal(c.begin(), c.end(), count) ||
      !std::equal(heap.lane_of.begin(), heap.lane_of.begin() + (long)lists.size() + 1, fixed.lane_of)) {
    std::printf("the storages differ\n");
    return 1;
  }
  if (fixed.lane_of[lists.size()] > kLanes) { std::printf("more than %d lanes\n", kLanes); return 1; }
  for (size_t k = 0; k < lists.size(); ++k) {
    std::vector<unsigned> want(kElements, 0), got(kElements, 0);
    for (unsigned x : lists[k]) ++want[x];
    for (int l = fixed.lane_of[k]; l < fixed.lane_of[k + 1]; ++l)
      for (int j = 0; j < count[l]; ++j) {
        const unsigned v = ent[((size_t)(j >> 2) * kLanes + l) * 4 + (j & 3)];
        got[v & 0xffff] += v >> 16;
      }
    if (want != got) { std::printf("output %d of %d\n", (int)k, (int)lists.size()); return 1; }
  }
  return 0;
}

int main() {
  std::mt19937 rng(5);
  for (int outputs : {1, 2, 9, 31, 32})
    for (int longest : {0, 1, 3, 60, 900}) {
      std::vector<std::vector<unsigned>> lists(outputs);
      for (auto &l : lists) {
        l.resize(longest ? rng() % (longest + 1) : 0);
        for (auto &k : l) k = rng() % (rng() % 2 ? 7 : kElements);
      }
      if (check(lists)) return 1;
    }
  // multiplicities that take several entries
  std::vector<std::vector<unsigned>> lists(3);
  lists[1].assign(150000, 1023);
  lists[2].assign(65536, 0);
  if (check({lists[0], lists[1]}) || check({lists[2]})) return 1;
  std::printf("ok\n");
  return 0;
}
