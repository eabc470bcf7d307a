// Host side of the sums over overlap lists in the wave kernels (no device code).
#pragma once
#include <algorithm>
#include <cstddef>
#include <vector>

namespace frg {

// Sums over lists of matrix elements, dealt to lanes: lanes lane_of[k] ..
// lane_of[k + 1] sum output k; entry j of lane l is element j % 4 of the
// quadruple at [(j / 4) * lanes + l] = index | multiplicity << 16, count[l]
// entries.  Repeated indices of an output are merged (simple cubic, range 6:
// 4095 overlap entries -> 1581), and a lane reads four entries per load.
//
// Use: begin, then per output add or add_list for its elements and end_output,
// then deal and store.  STORE holds item, mult, first and lane_of: HeapPlan in
// contexts, FixedPlan where nothing may be allocated.
template <class STORE> struct LanePlanOf : STORE {
  int rows = 0, lanes = 0, outputs = 0;
  size_t items = 0;

  int quads() const { return (rows + 3) / 4; }
  size_t entries() const { return (size_t)quads() * 4 * lanes; }
  void begin(size_t elements, int max_outputs) {
    this->shape(elements, max_outputs);
    items = 0;
    outputs = 0;
    this->first[0] = 0;
  }
  void add(unsigned k, unsigned times = 1) {
    add_list(1, [&](size_t) { return k; }, times);
  }
  // elements key(0) .. key(n - 1)
  template <class KEY> void add_list(size_t n, KEY key, unsigned times = 1) {
    this->room(items + n);
    unsigned *__restrict__ to = &this->item[0] + items, *__restrict__ m = &this->mult[0];
    for (size_t i = 0; i < n; ++i) {
      // (no branch: whether an element is new is not predictable)
      const unsigned k = key(i), had = m[k];
      *to = k;
      to += had == 0;
      m[k] = had + times;
    }
    items = to - &this->item[0];
  }
  void end_output() {
    // an entry holds multiplicities up to 0xffff; larger ones take several
    unsigned *list = &this->item[0], *m = &this->mult[0];
    for (size_t j = this->first[outputs], end = items; j < end; ++j) {
      const unsigned k = list[j];
      unsigned left = m[k];
      m[k] = 0;
      for (; left > 0xffffu; left -= 0xffffu) {
        this->room(items + 1);
        list = &this->item[0];
        list[items++] = k | 0xffff0000u;
      }
      list[j] = k | left << 16;
    }
    this->first[++outputs] = items;
  }
  // outputs <= nlanes
  void deal(int nlanes) {
    lanes = nlanes;
    auto need = [&](int k) { return std::max<int>(1, (int)((this->first[k + 1] - this->first[k] + rows - 1) / rows)); };
    for (rows = std::max(1, (int)((items + nlanes - 1) / nlanes));; ++rows) {
      int lane = 0;
      for (int k = 0; k < outputs; ++k) {
        this->lane_of[k] = lane;
        lane += need(k);
      }
      this->lane_of[outputs] = lane;
      if (lane <= nlanes) break;
    }
  }
  // ent: entries(), count: lanes
  void store(unsigned *ent, int *count) const {
    std::fill_n(ent, entries(), 0u);
    std::fill_n(count, lanes, 0);
    for (int k = 0; k < outputs; ++k) {
      size_t j = this->first[k];
      for (int l = this->lane_of[k]; l < this->lane_of[k + 1]; ++l) {
        const int n = (int)std::min<size_t>(rows, this->first[k + 1] - j);
        unsigned *to = ent + 4 * (size_t)l;
        const unsigned *from = &this->item[0] + j;
        for (int row = 0; row < n; row += 4, to += 4 * (size_t)lanes)
          for (int q = 0; q < 4 && row + q < n; ++q) to[q] = from[row + q];
        count[l] = n;
        j += n;
      }
    }
  }
};

struct HeapPlan {
  std::vector<unsigned> item, mult;
  std::vector<size_t> first;
  std::vector<int> lane_of;
  void shape(size_t elements, int max_outputs) {
    mult.assign(elements, 0);
    first.resize((size_t)max_outputs + 1);
    lane_of.resize((size_t)max_outputs + 1);
  }
  void room(size_t n) {  // (add_list writes one element ahead)
    if (item.size() < n + 1) item.resize(2 * n + 1);
  }
};
using LanePlan = LanePlanOf<HeapPlan>;

// the caller sees to it that the lists fit: at most ITEMS list elements
template <size_t ITEMS, size_t ELEMENTS, int OUTPUTS> struct FixedPlan {
  unsigned item[ITEMS + 1], mult[ELEMENTS];  // (add_list writes one element ahead)
  size_t first[OUTPUTS + 1];
  int lane_of[OUTPUTS + 1];
  void shape(size_t elements, int) { std::fill_n(mult, elements, 0u); }
  void room(size_t) {}
};

}  // namespace frg
