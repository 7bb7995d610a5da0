// ryser_skip_tree.hip -- Ryser's sum over the subsets without a zero row, by
// a search from the last walked column down.
//
// For an integer matrix every x_j(S) is exact.  Deciding the columns from the
// highest to the lowest, row j's x is known once its lowest column is: a
// prefix of the subset at which some known x is zero contributes nothing,
// whatever the columns below.  The prefixes are grown a level (a few columns)
// at a time; what is left of 2^(n-1) subsets are those with a nonzero term
// and a few times as many prefixes (grid graph 8x10, n = 40: 3.1e6 terms of
// 5.5e11 subsets, 9e6 prefixes; the Gray walk with skips, whose waves skip
// only what all their 64 lanes can, walks 2.6e8).
//
// One wave searches its share depth first.  Per level it holds a stack of
// prefixes (subset, product of the rows known so far) in LDS; a step takes
// 64 >> bits prefixes of one level, gives each lane one prefix and one
// setting of the level's columns, completes the level's rows (x by the
// popcount of the subset in the row's mask: scalar operands, no per-lane
// table), and pushes the lanes without a zero onto the next level's stack,
// or, at column 0, adds their terms to the lane's sum.  The deepest level
// with a full step goes first, so a stack never holds more than a step's
// worth and 64; when the first level is used up, levels from the top down are
// emptied by part-filled steps.  The first level's prefixes are numbered:
// wave w takes the tiles of 64 numbers w, w + waves, ...; the numbers are
// scattered over the prefixes, since those that survive are alike in most of
// their bits (unscattered, 750 of 8192 waves hold all of the 8x10 grid's
// terms and the search takes 2.2 ms instead of 0.29).
//
// The order of all sums is fixed by the launch: the same result every time.
//
// Error: x is exact, a term is a product of n rounded factors and joins the
// lane's double-double sum at once, so its sq_sum is the sum of the squared
// terms, runs of one term each.  Prefixes share their rounded products with
// every term below them, whose signs alternate: against the double-double
// pass, the errors of 40 matrices of n = 29 to 33, 0/1 and signed, are 0.002
// to 0.43 of err_est, 0.18 on the quadratic mean (1/3 if err_est's model held
// exactly).
//
// Bound: the latency of a step (stack, then four records at a time as scalar
// loads) at eleven waves per compute unit (their stacks fill the LDS), 40 to
// 100 steps per wave; the first level's 2^18..2^23 numbers are 5 to 30 us of
// it.  Records one by one, with the level's description loaded in each step
// and a test of every row, took 1.4 times as long.  Kernel times, walk ->
// search: grid 8x10 (4 % of the bonds missing, n = 40) 6.05 -> 0.41 ms, 8x10
// 2.95 -> 0.20, 8x9 1.48 -> 0.12, 8x8 0.29 -> 0.032, 8x12 (n = 48, two passes)
// 233 -> 6.2; random 0/1 n = 30, density 0.1 0.28 -> 0.031, n = 33, 0.18 (two
// passes) 9.6 -> 0.33 ms.
#include "ryser_device.hpp"
#include "ryser_kernels.hpp"

namespace perm {

// Four records as two scalar loads.
typedef uint64_t Word8 __attribute__((ext_vector_type(8)));
typedef const Word8 __attribute__((address_space(4)))* RecordPtr;

template <bool DDP>
struct Prefix {
  uint64_t set;
  double prod, tail;  // (tail: double-double products only)
};

// A permutation of the numbers of `bits` bits without order: neighbours land
// anywhere.
__device__ __forceinline__ uint32_t scatter(uint32_t v, int bits) {
  const uint32_t mask = (1u << bits) - 1u;
  const int half = (bits + 1) / 2;
  v ^= v >> half;
  v = v * 0x9e3779b1u & mask;
  v ^= v >> half;
  v = v * 0x85ebca6bu & mask;
  return v ^ v >> half;
}

// Multiply the rows of records [begin, end) (a multiple of four) into p; false:
// one of them is zero (the product is: no x is below 1/2 otherwise, so 63 of
// them do not underflow).  Stops when that is so in every lane.  SINGLE: every
// row is one record.
template <bool DDP, bool SINGLE>
__device__ __forceinline__ bool complete_rows(Prefix<DDP>& p, RecordPtr records, uint32_t begin,
                                              uint32_t end) {
  static_assert(kSkipRecordStep == 4);
  double x = 0.0;
  for (uint32_t i = begin; i < end; i += 4) {
    const Word8 r[2] = {records[i / 2], records[i / 2 + 1]};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint64_t mask = r[k / 2][4 * (k % 2)];
      const double value = __builtin_bit_cast(double, (uint64_t)r[k / 2][4 * (k % 2) + 1]);
      const double start = __builtin_bit_cast(double, (uint64_t)r[k / 2][4 * (k % 2) + 2]);
      const uint64_t set = p.set & mask;
      const int count =
          __builtin_popcount((uint32_t)set) + __builtin_popcount((uint32_t)(set >> 32));
      if constexpr (SINGLE)
        x = __builtin_fma(value, (double)count, start);
      else
        x = __builtin_fma(value, (double)count, x + start);
      if (SINGLE || r[k / 2][4 * (k % 2) + 3]) {
        const double h = p.prod * x;
        if constexpr (DDP) {
          const double e = __builtin_fma(p.tail, x, __builtin_fma(p.prod, x, -h));
          const DD n = quick_two_sum(h, e);
          p.prod = n.hi;
          p.tail = n.lo;
        } else {
          p.prod = h;
        }
        x = 0.0;
      }
    }
    if (__builtin_amdgcn_ballot_w64(p.prod != 0.0) == 0) return false;
  }
  return p.prod != 0.0;
}

template <bool DDP, bool SINGLE>
__global__ __launch_bounds__(kWave)
void ryser_skip_tree_kernel(const SkipRecord* __restrict__ records_arg,
                            const SkipLevel* __restrict__ levels_arg, int n_levels, int top_bits,
                            uint32_t waves, Partial* __restrict__ partials,
                            uint64_t* __restrict__ begin_tick) {
  extern __shared__ uint64_t lds[];
  __shared__ Partial scratch[1];
  if (begin_tick && blockIdx.x == 0 && threadIdx.x == 0)
    *begin_tick = __builtin_amdgcn_s_memrealtime();
  const RecordPtr records = (RecordPtr)records_arg;
  const uint32_t lane = threadIdx.x;
  // lane l holds level l
  const SkipLevel mine = levels_arg[lane < (uint32_t)n_levels ? lane : 0u];
  auto of_level = [](int v, int l) { return __builtin_amdgcn_readlane(v, l); };
  constexpr uint32_t kWords = DDP ? 3 : 2;
  // stack of level l >= 1: sets, products(, tails), kSkipLevelRoom each
  auto stack = [&](int l) { return lds + (uint32_t)(l - 1) * kWords * kSkipLevelRoom; };
  uint32_t held = 0;  // lane l: prefixes on level l's stack
  uint64_t tile = blockIdx.x;
  const uint64_t tiles = 1ull << (top_bits - 6);
  int empty = 0;  // levels [0, empty) are used up
  int l = 0;
  DD s = {0.0, 0.0};
  Moments mo = {0.0, 0.0, 0.0};
  double formed = 0.0;
  double running = 0.0;  // sum of the |running sum| after each addition (double-double products)
  const int last = n_levels - 1;
  for (;;) {
    const SkipLevel lv = {of_level(mine.bits, l), of_level(mine.base, l),
                          (uint32_t)of_level((int)mine.begin, l),
                          (uint32_t)of_level((int)mine.end, l)};
    Prefix<DDP> p;
    if (l == 0) {
      if (tile >= tiles) {  // used up: on with what is held
        if (empty == 0) empty = 1;
        if (last == 0) break;
        l = 1;
        continue;
      }
      p.set = (uint64_t)scatter((uint32_t)tile * kWave + lane, top_bits) << lv.base;
      p.prod = 1.0;
      p.tail = 0.0;
      tile += waves;
      if (last == 0) formed += 1.0;
    } else {
      const uint32_t have = (uint32_t)__builtin_amdgcn_readlane((int)held, l);
      const uint32_t full = (uint32_t)kWave >> lv.bits;
      if (have < full && (l > empty || have == 0)) {
        // not a full step: back up, or, below used-up levels, down
        if (l > empty) {
          --l;
        } else {
          if (l == last) break;
          empty = ++l;
        }
        continue;
      }
      const uint32_t take = have < full ? have : full;
      const uint32_t at = have - take + (lane >> lv.bits);
      const uint64_t* st = stack(l);
      p.set = 0;
      p.prod = 0.0;
      p.tail = 0.0;
      if ((lane >> lv.bits) < take) {
        if (l == last) formed += 1.0;
        p.set = st[at] | (uint64_t)(lane & ((1u << lv.bits) - 1u)) << lv.base;
        p.prod = __builtin_bit_cast(double, st[kSkipLevelRoom + at]);
        if constexpr (DDP) p.tail = __builtin_bit_cast(double, st[2 * kSkipLevelRoom + at]);
      }
      held = lane == (uint32_t)l ? have - take : held;
    }
    const bool alive = complete_rows<DDP, SINGLE>(p, records, lv.begin, lv.end);
    if (l == last) {
      if (alive) {
        const bool odd = __builtin_popcountll(p.set) & 1;
        s = dd_add_d(s, odd ? -p.prod : p.prod);
        if constexpr (DDP) {
          running += __builtin_fabs(s.hi);
          s = dd_add_d(s, odd ? -p.tail : p.tail);
          running += __builtin_fabs(s.hi);
        }
        mo.a += __builtin_fabs(p.prod);
        mo.q = __builtin_fma(p.prod, p.prod, mo.q);
      }
      continue;
    }
    const uint64_t mask = __builtin_amdgcn_ballot_w64(alive);
    if (mask == 0) continue;
    ++l;
    const uint32_t have = (uint32_t)__builtin_amdgcn_readlane((int)held, l);
    if (alive) {
      const uint32_t at =
          have + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                           __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
      uint64_t* st = stack(l);
      st[at] = p.set;
      st[kSkipLevelRoom + at] = __builtin_bit_cast(uint64_t, p.prod);
      if constexpr (DDP) st[2 * kSkipLevelRoom + at] = __builtin_bit_cast(uint64_t, p.tail);
    }
    // the pushes are read by other lanes of this wave
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    held = lane == (uint32_t)l ? have + (uint32_t)__builtin_popcountll(mask) : held;
  }
  // `formed` rides through the reduction as the (unused) drift statistic
  mo.r = formed;
  if constexpr (DDP) running = wave_sum(running);
  block_reduce_store(s, mo, scratch, partials + blockIdx.x, running);
}

hipError_t launch_skip_tree(const SkipTreeLaunch& L, hipStream_t stream, const RunReport& report) {
  if (L.n_levels < 1 || L.n_levels > kSkipMaxLevels || L.top_bits < 6 ||
      L.top_bits > kSkipMaxTopBits || L.waves < 1 || L.waves > 1u << (L.top_bits - 6) ||
      (L.mode != 0 && L.mode != 1))
    return hipErrorInvalidValue;
  const size_t lds = (size_t)(L.n_levels - 1) * (L.mode ? 3 : 2) * kSkipLevelRoom * 8;
  const auto kernel =
      L.mode ? (L.single ? ryser_skip_tree_kernel<true, true> : ryser_skip_tree_kernel<true, false>)
             : (L.single ? ryser_skip_tree_kernel<false, true>
                         : ryser_skip_tree_kernel<false, false>);
  kernel<<<L.waves, kWave, lds, stream>>>(L.records, L.levels, L.n_levels, L.top_bits, L.waves,
                                          L.partials, L.begin_tick);
  if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  return launch_reduce(L.partials, L.waves, L.result, stream, report);
}

}  // namespace perm
