// ryser_class.hpp -- launch descriptors of the class walk
// (ryser_class_impl.hpp).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "class_plan.hpp"
#include "ryser_device.hpp"
#include "ryser_kernels.hpp"

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
  int32_t thin;             // which tree: the kernel that walks it
};

// The descriptor of a matrix of order n split into 2^walk_bits groups per
// lane, from where its parts are on the device (ClassTables).
inline ClassMatrix class_matrix(int n, uint32_t live, bool thin, int walk_bits,
                                const double* records, const double* cols, const double* lane,
                                const double* walk) {
  const int before = walk_bits + kClassLaneBits;  // columns after the class ones
  return {records,   lane,      cols + (size_t)before * n,     walk, live,
          (int32_t)n, walk_bits, n - 1 - kClassBits - before, thin};
}

// Workgroups [block_begin, block_end) of the walk (block b fixes the block
// columns by the bits of b); the record of the i-th goes to partials[i].
struct ClassLaunch {
  ClassMatrix m;
  Partial* partials;
  uint64_t block_begin, block_end;
  uint64_t* begin_tick = nullptr;  // device: the launch's begin (RunReport)
};
hipError_t launch_class(const ClassLaunch& L, hipStream_t stream);

struct BatchItem;
// Fill the lane columns and walk offsets of mats[0, count) (entries with n =
// 0 are skipped) from their columns and start vectors.
hipError_t launch_class_expand(const ClassMatrix* mats, uint32_t count, hipStream_t stream);
// Persistent kernel over items [begin, end), each one workgroup's walk of
// one block (lane_base / 64) of its matrix; `counter` must be zero; the
// record of item i goes to partials[i].  max_n: largest order among them;
// thin: the tree of all of them.
hipError_t launch_class_batch(bool thin, const ClassMatrix* mats, const BatchItem* items,
                              uint32_t begin, uint32_t end, uint32_t* counter,
                              Partial* partials, int max_n, uint32_t grid, hipStream_t stream);

}  // namespace perm
