// skip_tree.hpp -- the skipping walk as a tree search (ryser_skip_tree.hip):
// what its host plan and its kernel share (no HIP headers).
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <vector>

namespace perm {

struct Partial;

// Columns of one value in one row.  A row is the records up to the one with
// `last`; x = start + sum over its records of value * popcount(S & mask).
struct SkipRecord {
  uint64_t mask;
  double value, start;  // start: x0 in a row's first record, 0 in the others
  uint64_t last;
};
// The subsets of columns [base, base + bits) below every prefix, and the
// records [begin, end) of the rows they complete.
struct SkipLevel {
  int32_t bits, base;
  uint32_t begin, end;
};
// Levels a wave's LDS holds prefixes of (the first one's prefixes are
// numbered, not stored), bits of a level after the first, and of the first.
constexpr int kSkipMaxLevels = 20;
constexpr int kSkipMaxLevelBits = 4;
constexpr int kSkipMaxTopBits = 26;
// Records per level: a multiple of this (rows of x = 1 fill up).
constexpr uint32_t kSkipRecordStep = 4;
// Stored prefixes per level: less than one full step, and one step's.
constexpr int kSkipLevelRoom = 32 + 64;

struct SkipTreeLaunch {
  const SkipRecord* records;  // device, 64-byte aligned
  const SkipLevel* levels;    // device: n_levels, columns from the top down to 0
  Partial* partials;          // device: `waves` records
  Partial* result;            // device: 1 record
  uint64_t* begin_tick;       // device
  int n_levels, top_bits, mode;  // mode 0 FP64, 1 double-double products
  uint32_t waves;
  bool single;  // every row is one record
};
// The search's plan (host; perman_skip_plan.cpp).
struct TreePlan {
  std::vector<SkipLevel> levels;
  std::vector<SkipRecord> records;
  int top_bits = 0;
  uint32_t waves = 0;
  bool single = true;
  double cost = 0.0;  // records expected to be met by all prefixes, and 2 per prefix
};
// Greedy order of b columns, the lowest first: next, the column adding the
// fewest rows not yet touched (ties by fewer nonzeros, then index).  sup[k]:
// rows with an entry in column k.
void skip_order(int b, const uint64_t* sup, int* order);
// x0: n start values; cols[k * n + j] = a[j][k], k < n - 1; an integer matrix.
// zero[j]: share of the subsets at which row j is zero.  Returns the share of
// the subsets at which no row is, the rows taken as independent.
double nonzero_share(int n, const double* x0, const double* cols, double* zero);
// order: of the walked columns (skip_order); n >= 7.
void plan_tree(int n, const double* x0, const double* cols, const int* order, const double* zero,
               TreePlan& tp);
// Levels and records as the device reads them (64-byte aligned there).
inline size_t tree_record_word(const TreePlan& tp) {
  return (tp.levels.size() * sizeof(SkipLevel) + 63) / 64 * 8;
}
std::vector<uint64_t> pack_tree(const TreePlan& tp);
// The launch's plan part; records, result and tick are the caller's.
SkipTreeLaunch tree_launch(const TreePlan& tp, const void* packed, int mode);

}  // namespace perm
