// class_tree.hpp -- the column-class tree of the class walk (host and device;
// no HIP headers).
//
// The first K walked columns ("class columns") split the rows into 2^K
// classes: row j's class T_j is the set of class columns with an entry in row
// j.  Over the 2^K subsets s of the class columns the row takes only
// 2^|T_j| values, one per s & T_j, so the product of the rows of class T is
// an array P_T of 2^|T| values.  The product over all rows at every s is
// formed bottom-up: P_T is multiplied into the array of its parent class,
// T plus one column, at 2^(|T|+1) multiplications.
//
// The tree: a prefix class {0..i} hangs below {0..i+1}; any other class
// below itself plus its lowest missing column.  (So the classes with largest
// column i form a subtree below {0..i}.)
//
// Thin tree: when no row is touched by both the first and the last class
// column, the classes of the last column are subsets of {1, .., K-1} and
// their subtree ends in that class instead of {0, .., K-1}: its array is half
// as long, and the final sum over the first and the last column is one factor
// each.  Nearly every matrix of density up to 0.35 has such columns, two of
// three at 0.4, one of thirty at 0.5 (n = 32).
#pragma once
#include <stdint.h>

namespace perm {

constexpr int class_popcount(int t) {
  int c = 0;
  for (; t; t &= t - 1) ++c;
  return c;
}

// The class whose array holds the product of all classes of the last column.
constexpr int class_root(int k, bool thin) { return (1 << k) - (thin ? 2 : 1); }
// Parent class of T (not the root).
constexpr int class_parent(int k, bool thin, int t) {
  int i = thin && (t >> (k - 1)) & 1 ? 1 : 0;
  while ((t >> i) & 1) ++i;  // lowest missing column
  return t | (1 << i);
}
// Classes that may hold rows.
constexpr bool class_allowed(int k, bool thin, int t) {
  return !thin || !((t & 1) && ((t >> (k - 1)) & 1));
}
// Index in P_C (C a subset of T) of entry s of P_T: the bits of s that
// belong to columns of C, packed.
constexpr int class_drop(int t, int c, int s) {
  int out = 0, o = 0, b = 0;
  for (int i = 0; i < 8; ++i) {
    if (!((t >> i) & 1)) continue;
    if ((c >> i) & 1) out |= ((s >> b) & 1) << o++;
    ++b;
  }
  return out;
}

}  // namespace perm
