// ryser_class.hip -- kernel of the class walk (ryser_class_impl.hpp) for one
// matrix.
#include "ryser_class_impl.hpp"

namespace perm {

// Workgroup b of the launch walks block block_begin + b.
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(3)))
void ryser_class_kernel(ClassMatrix m, Partial* __restrict__ partials, uint64_t block_begin) {
  extern __shared__ double lds[];
  __shared__ Partial scratch[256 / kWave];
  // shader-clock and 100 MHz counters around the work (see ryser_dense_kernel)
  const uint64_t c0 = __builtin_amdgcn_s_memtime();
  const uint64_t r0 = __builtin_amdgcn_s_memrealtime();
  DD s;
  Moments mo;
  class_walk(m, block_begin + blockIdx.x, lds, s, mo);
  const uint64_t c1 = __builtin_amdgcn_s_memtime();
  const uint64_t r1 = __builtin_amdgcn_s_memrealtime();
  const double ratio = r1 > r0 ? (double)(c1 - c0) / (double)(r1 - r0) : 0.0;
  block_reduce_store(s, mo, scratch, partials + blockIdx.x, ratio);
}

hipError_t launch_class(const ClassLaunch& L, hipStream_t stream) {
  const ClassMatrix& m = L.m;
  if (m.n < 1 || m.n > 64 || m.walk_bits < 0 || m.block_bits < 0 || m.walk_bits > 24 ||
      kClassBits + m.walk_bits + kClassLaneBits + m.block_bits != m.n - 1 ||
      L.block_end <= L.block_begin || L.block_end > 1ull << m.block_bits ||
      L.block_end - L.block_begin > 0xffffffffull)
    return hipErrorInvalidValue;
  const size_t lds = (size_t)(m.n + 2) * kWave * sizeof(double);
  ryser_class_kernel<<<dim3((unsigned)(L.block_end - L.block_begin)), dim3(256), lds, stream>>>(
      m, L.partials, L.block_begin);
  return hipGetLastError();
}

}  // namespace perm
