// ryser_class.hip -- kernels of the class walk (ryser_class_impl.hpp): one
// matrix, and the items of a batch.
#include "ryser_batch.hpp"
#include "ryser_class_impl.hpp"

namespace perm {

// Waves per SIMD: the arrays of one path through the tree are 63 doubles per
// lane (150 registers), 47 in the thin tree (120).  The fourth wave is worth
// 8-9 % to a batch (512 matrices of n = 24, density 0.2..0.4: one kernel for
// both trees, at three waves, 2.21 ms; a kernel for each 2.03 ms).
template <bool THIN>
constexpr int kClassWaves = THIN ? 4 : 3;

// Workgroup b of the launch walks block block_begin + b.
template <bool THIN>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(kClassWaves<THIN>)))
void ryser_class_kernel(ClassMatrix m, Partial* __restrict__ partials, uint64_t block_begin,
                        uint64_t* __restrict__ begin_tick) {
  extern __shared__ double lds[];
  __shared__ Partial scratch[256 / kWave];
  // shader-clock and 100 MHz counters around the work (see ryser_dense_kernel)
  const uint64_t c0 = __builtin_amdgcn_s_memtime();
  const uint64_t r0 = __builtin_amdgcn_s_memrealtime();
  if (begin_tick && blockIdx.x == 0 && threadIdx.x == 0) *begin_tick = r0;
  DD s;
  Moments mo;
  class_walk<THIN>(m, block_begin + blockIdx.x, lds, s, mo);
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
  const auto kernel = m.thin ? ryser_class_kernel<true> : ryser_class_kernel<false>;
  kernel<<<dim3((unsigned)(L.block_end - L.block_begin)), dim3(256), lds, stream>>>(
      m, L.partials, L.block_begin, L.begin_tick);
  return hipGetLastError();
}

// Lane columns and walk offsets of one matrix per workgroup, the offsets as
// build_class_tables forms them (double-double sums in ascending column
// order).
__global__ __launch_bounds__(256) void class_expand_kernel(const ClassMatrix* __restrict__ mats) {
  const ClassMatrix m = mats[blockIdx.x];
  const int n = m.n;
  if (n == 0) return;
  const double* cols = m.blockcols - (size_t)(m.walk_bits + kClassLaneBits) * n;
  const double* x0 = m.blockcols + (size_t)m.block_bits * n;
  const double* lane0 = cols + (size_t)m.walk_bits * n;
  double* lane = const_cast<double*>(m.lanecols);
  for (int i = threadIdx.x; i < 8 * n; i += blockDim.x) {
    const int r = i >> 3, b = i & 7;
    lane[i] = b < kClassLaneBits ? lane0[(size_t)b * n + r] : x0[(b - kClassLaneBits) * n + r];
  }
  double* walk = const_cast<double*>(m.walk);
  const uint32_t entries = (uint32_t)n << m.walk_bits;
  for (uint32_t i = threadIdx.x; i < entries; i += blockDim.x) {
    const uint32_t t = i / (uint32_t)n, r = i - t * (uint32_t)n;
    double hi = 0.0, lo = 0.0;
    for (int b = 0; b < m.walk_bits; ++b) {
      if (!((t >> b) & 1)) continue;
      const DD e = two_sum(hi, cols[(size_t)b * n + r]);
      hi = e.hi;
      lo += e.lo;
    }
    walk[i] = hi + lo;
  }
}

hipError_t launch_class_expand(const ClassMatrix* mats, uint32_t count, hipStream_t stream) {
  if (count == 0) return hipSuccess;
  class_expand_kernel<<<count, 256, 0, stream>>>(mats);
  return hipGetLastError();
}

// Persistent: every workgroup takes items from the counter until they are
// drained.
template <bool THIN>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(kClassWaves<THIN>)))
void ryser_class_batch_kernel(const ClassMatrix* __restrict__ mats,
                              const BatchItem* __restrict__ items, uint32_t begin, uint32_t end,
                              uint32_t* __restrict__ counter, Partial* __restrict__ partials) {
  extern __shared__ double lds[];
  __shared__ Partial scratch[256 / kWave];
  __shared__ uint32_t ticket;
  for (;;) {
    if (threadIdx.x == 0) ticket = atomicAdd(counter, 1u);
    __syncthreads();
    const uint32_t it = (uint32_t)__builtin_amdgcn_readfirstlane((int)ticket) + begin;
    if (it >= end) break;
    const BatchItem d = items[it];
    const ClassMatrix m = mats[d.matrix];
    DD s;
    Moments mo;
    class_walk<THIN>(m, d.lane_base / kItemLanes, lds, s, mo);
    block_reduce_store(s, mo, scratch, partials + it);
    __syncthreads();  // (the tables, the records and the ticket are reused)
  }
}

hipError_t launch_class_batch(bool thin, const ClassMatrix* mats, const BatchItem* items,
                              uint32_t begin, uint32_t end, uint32_t* counter,
                              Partial* partials, int max_n, uint32_t grid, hipStream_t stream) {
  if (end <= begin || max_n < 1 || max_n > 64 || grid == 0) return hipErrorInvalidValue;
  const size_t lds = (size_t)(max_n + 2) * kWave * sizeof(double);
  const auto kernel = thin ? ryser_class_batch_kernel<true> : ryser_class_batch_kernel<false>;
  kernel<<<grid, 256, lds, stream>>>(mats, items, begin, end, counter, partials);
  return hipGetLastError();
}

}  // namespace perm
