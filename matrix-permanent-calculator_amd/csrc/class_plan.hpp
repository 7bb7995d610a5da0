// class_plan.hpp -- host side of the class walk (ryser_class_impl.hpp): which
// columns become class columns, which class every row is computed in, and
// the tables the kernel reads.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <vector>

namespace perm {

constexpr int kClassBits = 5;      // class columns: 2^5 subsets per group
constexpr int kClassLaneBits = 6;  // lane columns: the lanes of one wave
// Rows of classes of up to this many columns are visited in pairs.
constexpr int kClassPairBits = 2;

// The walk of one matrix: the walked columns k < n-1 in the order class |
// walk | lane | block, the rows in the order the kernel meets them, and the
// class each is computed in (its own or a superset).
struct ClassPlan {
  int n = 0;
  int cols[64];                    // original index of the i-th walked column
  int rows[64];                    // original index of the i-th row
  uint8_t classes[64];             // class of the i-th row
  uint8_t count[1 << kClassBits];  // rows in class T
  uint32_t live = 0;               // classes with rows
  bool thin = false;               // which tree (class_tree.hpp)
  int cost = 0;                    // FP64 instructions per lane and group
};

// sup[k]: rows with a nonzero in walked column k (k < n-1).  n - 1 >=
// kClassBits.
void plan_classes(int n, const uint64_t* sup, ClassPlan& p);

// What the kernel reads, as one array: the rows' records at 0; the columns
// after the class columns and the start vector (x0, then its low parts), n
// doubles each, rows in the plan's order; and, for a given split, the lane
// columns by row and the walk offsets (ClassMatrix in ryser_class.hpp).
struct ClassTables {
  std::vector<double> data;
  size_t cols = 0, lane = 0, walk = 0;  // where the parts begin
};

// x0: 2n doubles (start vector, its low parts); cols[k * n + j] = a[j][k] of
// the walked columns.  walk_bits >= 0: the last two parts for 2^walk_bits
// groups of 2^kClassBits subsets per lane (n - 1 >= kClassBits + walk_bits +
// kClassLaneBits); < 0: without them (the device expands them).
void build_class_tables(const ClassPlan& p, const double* x0, const double* cols, int walk_bits,
                        ClassTables& out);
// Doubles of the last two parts, and a bound of the first ones'.
inline size_t class_split_doubles(int n, int walk_bits) {
  return 8 * (size_t)n + ((size_t)n << walk_bits) + 2;
}
inline size_t class_tables_bound(int n) {
  return 32 * (size_t)n + 8 + (size_t)(n + 1) * n;
}

}  // namespace perm
