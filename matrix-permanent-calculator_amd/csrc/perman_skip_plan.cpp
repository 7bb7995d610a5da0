// perman_skip_plan.cpp -- host side of the search of the subsets without a zero row
// (ryser_skip_tree.hip): the order of its columns, its levels and records.
#include "skip_tree.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace perm {

void skip_order(int b, const uint64_t* sup, int* order) {
  uint64_t touched = 0, used = 0;
  for (int step = 0; step < b; ++step) {
    int best = -1, best_new = 0, best_nnz = 0;
    for (int k = 0; k < b; ++k) {
      if (used >> k & 1) continue;
      const int nz = __builtin_popcountll(sup[k]);
      const int nw = __builtin_popcountll(sup[k] & ~touched);
      if (best < 0 || nw < best_new || (nw == best_new && nz < best_nnz)) {
        best = k;
        best_new = nw;
        best_nnz = nz;
      }
    }
    used |= 1ull << best;
    order[step] = best;
    touched |= sup[best];
  }
}

namespace {

// Columns of the first level: enough of its prefixes survive to hold the
// chip's waves and to spread evenly over them, and the numbers themselves stay
// cheap; and the waves.  Kernel ms at 18, 20, 22, 23 columns with 8192 waves:
// grid 7x10 (n = 35) 0.177, 0.111, 0.109, 0.138; 8x9 0.132, 0.123, 0.123,
// 0.139; 8x10 0.76, 0.55, 0.48, 0.41; 8x8 with 4096 waves 0.033, 0.032, 0.046,
// 0.067.  The other levels: one column each 1.01, two 0.74, three 0.74 ms
// (8x10, an earlier form of the kernel).
int tree_top_bits(int b) { return std::min(b, std::max(18, std::min(23, b - 14))); }
uint32_t tree_waves(int top_bits) {
  return top_bits >= 20 ? 8192u : 1u << std::min(12, top_bits - 6);
}
int tree_level_bits(int left) { return left <= 20 ? 2 : 3; }

// Share of the subsets of the columns of values v[0, d) at which start + sum
// is 0 (start a half integer, v integers): a binomial, or by counting sums (0
// for rows of many values and a wide range).
double zero_share(double start, const double* v, int d) {
  if (start != std::nearbyint(start)) return 0.0;
  if (std::all_of(v, v + d, [&](double a) { return a == v[0]; })) {
    const double c = d ? -start / v[0] : start;
    if (c < 0.0 || c > d || c != std::nearbyint(c)) return 0.0;
    double share = std::ldexp(1.0, -d);
    for (int i = 1; i <= (int)c; ++i) share = share * (d + 1 - i) / i;
    return share;
  }
  constexpr int kRange = 256;
  double lo = 0.0, hi = 0.0;
  for (int i = 0; i < d; ++i) (v[i] < 0.0 ? lo : hi) += v[i];
  if (start + lo > 0.0 || start + hi < 0.0 || hi - lo >= kRange) return 0.0;
  double share[kRange] = {1.0};  // of sum = lo + index
  int top = 0;
  for (int i = 0; i < d; ++i) {
    const int a = (int)std::fabs(v[i]);
    top += a;
    for (int k = top; k >= 0; --k)
      share[k] = 0.5 * ((k <= top - a ? share[k] : 0.0) + (k >= a ? share[k - a] : 0.0));
  }
  return share[(int)(-start - lo)];
}

}  // namespace

double nonzero_share(int n, const double* x0, const double* cols, double* zero) {
  double share = 1.0;
  for (int j = 0; j < n; ++j) {
    double v[64];
    int d = 0;
    for (int k = 0; k < n - 1; ++k)
      if (const double a = cols[(size_t)k * n + j]; a != 0.0) v[d++] = a;
    zero[j] = zero_share(x0[j], v, d);
    share *= 1.0 - zero[j];
  }
  return share;
}

void plan_tree(int n, const double* x0, const double* cols, const int* order, const double* zero,
               TreePlan& tp) {
  const int B = n - 1;
  struct Row {
    int j, low;  // low: lowest column with an entry: x is known from there on
    double zero;
  };
  Row rows[64];
  for (int j = 0; j < n; ++j) {
    int low = 0;
    while (low < B && cols[(size_t)order[low] * n + j] == 0.0) ++low;
    rows[j] = {j, low, zero[j]};
  }
  std::stable_sort(rows, rows + n, [](const Row& a, const Row& b) { return a.low > b.low; });
  tp.top_bits = tree_top_bits(B);
  tp.waves = tree_waves(tp.top_bits);
  const int left = B - tp.top_bits, per = tree_level_bits(left);
  tp.levels.clear();
  tp.records.clear();
  tp.cost = 0.0;
  tp.single = true;
  double prefixes = 1.0;
  int at = 0;
  for (int base = B; base > 0;) {
    const int b = base == B ? tp.top_bits : base % per ? base % per : per;
    base -= b;
    SkipLevel lv{b, base, (uint32_t)tp.records.size(), 0};
    prefixes *= std::ldexp(1.0, b);
    tp.cost += 2.0 * prefixes;
    for (; at < n && rows[at].low >= base; ++at) {
      const int j = rows[at].j;
      const size_t first = tp.records.size();
      for (int c = B - 1; c >= rows[at].low; --c) {
        const double a = cols[(size_t)order[c] * n + j];
        if (a == 0.0) continue;
        size_t r = first;
        while (r < tp.records.size() && tp.records[r].value != a) ++r;
        if (r == tp.records.size()) tp.records.push_back({0, a, 0.0, 0});
        tp.records[r].mask |= 1ull << c;
      }
      if (tp.records.size() == first) tp.records.push_back({0, 0.0, 0.0, 0});
      tp.records[first].start = x0[j];
      tp.records.back().last = 1;
      tp.single = tp.single && tp.records.size() == first + 1;
      tp.cost += prefixes * (double)(tp.records.size() - first);
      prefixes *= 1.0 - rows[at].zero;
    }
    while (tp.records.size() % kSkipRecordStep) tp.records.push_back({0, 0.0, 1.0, 1});
    lv.end = (uint32_t)tp.records.size();
    tp.levels.push_back(lv);
  }
}

std::vector<uint64_t> pack_tree(const TreePlan& tp) {
  const size_t lev = tree_record_word(tp);
  std::vector<uint64_t> up(lev + tp.records.size() * sizeof(SkipRecord) / 8, 0);
  std::memcpy(up.data(), tp.levels.data(), tp.levels.size() * sizeof(SkipLevel));
  std::memcpy(up.data() + lev, tp.records.data(), tp.records.size() * sizeof(SkipRecord));
  return up;
}

SkipTreeLaunch tree_launch(const TreePlan& tp, const void* packed, int mode) {
  SkipTreeLaunch L{};
  L.levels = (const SkipLevel*)packed;
  L.records = (const SkipRecord*)((const uint64_t*)packed + tree_record_word(tp));
  L.n_levels = (int)tp.levels.size();
  L.top_bits = tp.top_bits;
  L.mode = mode;
  L.waves = tp.waves;
  L.single = tp.single;
  return L;
}

}  // namespace perm
