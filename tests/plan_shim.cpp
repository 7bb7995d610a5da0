// plan_shim.cpp -- C ABI over the host plans of the class walk
// (csrc/class_plan.cpp) and of the search (csrc/perman_skip_plan.cpp),
// compiled with them by tests/test_cpu_plans.py.  Test infrastructure only.
#include <cstring>

#include "../matrix-permanent-calculator_amd/csrc/class_plan.hpp"
#include "../matrix-permanent-calculator_amd/csrc/class_tree.hpp"
#include "../matrix-permanent-calculator_amd/csrc/nest_shape.hpp"
#include "../matrix-permanent-calculator_amd/csrc/ryser_host.hpp"
#include "../matrix-permanent-calculator_amd/csrc/skip_tree.hpp"

extern "C" {

int shim_class_bits() { return perm::kClassBits; }
int shim_root(int thin) { return perm::class_root(perm::kClassBits, thin); }
int shim_parent(int thin, int t) { return perm::class_parent(perm::kClassBits, thin, t); }
int shim_allowed(int thin, int t) { return perm::class_allowed(perm::kClassBits, thin, t); }
// The class walk's instructions per group of 32 subsets at which it is taken.
double shim_class_limit(int n) { return perm::kClassGain * (1 << perm::kClassBits) * (2 * n + 2); }

// out: cols[n-1], rows[n], classes[n], then live, thin, cost.
void shim_class_plan(int n, const uint64_t* sup, int* out) {
  perm::ClassPlan p;
  perm::plan_classes(n, sup, p);
  for (int k = 0; k < n - 1; ++k) *out++ = p.cols[k];
  for (int r = 0; r < n; ++r) *out++ = p.rows[r];
  for (int r = 0; r < n; ++r) *out++ = p.classes[r];
  *out++ = (int)p.live;
  *out++ = p.thin;
  *out++ = p.cost;
}

// Start vector (n, then n low parts) and its tables for the plan of `sup`;
// data: class_tables_bound(n) + class_split_doubles doubles; at: where the
// columns, the lane part and the walk offsets begin.  Returns the length.
long shim_class_tables(int n, const uint64_t* sup, const double* a, int walk_bits, double* x0,
                       double* data, long* at) {
  perm::ClassPlan p;
  perm::plan_classes(n, sup, p);
  perm::nw_start_vector(a, n, x0, x0 + n);
  std::vector<double> cols((size_t)(n - 1) * n);
  for (int k = 0; k < n - 1; ++k)
    for (int j = 0; j < n; ++j) cols[(size_t)k * n + j] = a[(size_t)j * n + k];
  perm::ClassTables t;
  perm::build_class_tables(p, x0, cols.data(), walk_bits, t);
  std::memcpy(data, t.data.data(), t.data.size() * sizeof(double));
  at[0] = (long)t.cols;
  at[1] = (long)t.lane;
  at[2] = (long)t.walk;
  return (long)t.data.size();
}
long shim_class_tables_room(int n, int walk_bits) {
  return (long)(perm::class_tables_bound(n) +
                (walk_bits < 0 ? 0 : perm::class_split_doubles(n, walk_bits)));
}

// The search's plan of a: order[n-1]; zero[n]; levels as rows of 4 (bits,
// base, begin, end) and records as masks and rows of 3 (value,
// start, last).  Returns the numbers of levels and records in counts.
double shim_tree_plan(int n, const double* a, double* x0, int* order, double* zero, int* levels,
                      uint64_t* masks, double* records, int* counts, double* cost) {
  perm::nw_start_vector(a, n, x0, x0 + n);
  std::vector<double> cols((size_t)(n - 1) * n);
  uint64_t sup[64] = {0};
  for (int k = 0; k < n - 1; ++k)
    for (int j = 0; j < n; ++j) {
      cols[(size_t)k * n + j] = a[(size_t)j * n + k];
      if (a[(size_t)j * n + k] != 0.0) sup[k] |= 1ull << j;
    }
  perm::skip_order(n - 1, sup, order);
  const double share = perm::nonzero_share(n, x0, cols.data(), zero);
  perm::TreePlan tp;
  perm::plan_tree(n, x0, cols.data(), order, zero, tp);
  for (size_t i = 0; i < tp.levels.size(); ++i) {
    levels[4 * i] = tp.levels[i].bits;
    levels[4 * i + 1] = tp.levels[i].base;
    levels[4 * i + 2] = (int)tp.levels[i].begin;
    levels[4 * i + 3] = (int)tp.levels[i].end;
  }
  for (size_t i = 0; i < tp.records.size(); ++i) {
    masks[i] = tp.records[i].mask;
    records[3 * i] = tp.records[i].value;
    records[3 * i + 1] = tp.records[i].start;
    records[3 * i + 2] = (double)tp.records[i].last;
  }
  counts[0] = (int)tp.levels.size();
  counts[1] = (int)tp.records.size();
  counts[2] = tp.top_bits;
  counts[3] = (int)tp.waves;
  counts[4] = tp.single;
  *cost = tp.cost;
  return share;
}
int shim_tree_limits(int which) {
  const int v[] = {perm::kSkipMaxLevels, perm::kSkipMaxLevelBits, perm::kSkipMaxTopBits,
                   (int)perm::kSkipRecordStep, perm::kSkipLevelRoom};
  return v[which];
}
}
