// ryser_class.hpp -- launch descriptors of the class walk
// (ryser_class_impl.hpp).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "class_plan.hpp"
#include "ryser_device.hpp"

namespace perm {

// One matrix's tables (class_plan.hpp), on the device.
struct ClassMatrix {
  const double* records;    // per visit, 64 bytes (more for classes above 3 columns)
  const double* lanecols;   // n x 8: a row's entries in the lane columns, x0, x0's low part
  const double* blockcols;  // block_bits x n
  const double* walk;       // 2^walk_bits x n: offsets of the walk columns' subsets
  uint32_t live;            // classes with rows
  int32_t n;
  int32_t walk_bits;        // 2^walk_bits groups per lane
  int32_t block_bits;
};

// Workgroups [block_begin, block_end) of the walk (block b fixes the block
// columns by the bits of b), or the listed ones; the record of the i-th goes
// to partials[i].
struct ClassLaunch {
  ClassMatrix m;
  Partial* partials;
  uint64_t block_begin, block_end;
};
hipError_t launch_class(const ClassLaunch& L, hipStream_t stream);

}  // namespace perm
