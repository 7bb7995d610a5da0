// perman_cached.hpp -- one call's kernels on the per-device cached stream and
// memory of the single-matrix calls.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

#include <functional>

#include "ryser_device.hpp"
#include "ryser_kernels.hpp"

namespace perm {

struct CachedRun {
  Partial sum;
  float ms = 0.f;  // from the first kernel's begin tick to the report
};
// Uploads `up` to the base of `bytes` of device memory, calls launch (which
// enqueues kernels on the stream, the last of which reports) and waits for
// the report.  One call at a time per device.
int run_cached(const void* up, size_t up_bytes, size_t bytes,
               const std::function<hipError_t(char* base, hipStream_t, const RunReport&)>& launch,
               CachedRun& out);

}  // namespace perm
