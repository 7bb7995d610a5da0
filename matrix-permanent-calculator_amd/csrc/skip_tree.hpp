// skip_tree.hpp -- the skipping walk as a tree search (ryser_skip_tree.hip):
// what its host plan and its kernel share.  No device code.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace perm {

struct Partial;
struct RunReport;

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
// Stored prefixes per level: less than one full step, and one step's.
constexpr int kSkipLevelRoom = 32 + 64;

struct SkipTreeLaunch {
  const SkipRecord* records;  // device
  const SkipLevel* levels;    // device: n_levels, columns from the top down to 0
  Partial* partials;          // device: `waves` records
  Partial* result;            // device: 1 record
  uint64_t* begin_tick;       // device
  int n_levels, top_bits, mode;  // mode 0 FP64, 1 double-double products
  uint32_t waves;
};
// Enqueue the search and the grid reduction, which reports.  pad of the sum:
// subsets of all columns formed (the rest was cut off).
hipError_t launch_skip_tree(const SkipTreeLaunch& L, hipStream_t stream, const RunReport& report);

}  // namespace perm
