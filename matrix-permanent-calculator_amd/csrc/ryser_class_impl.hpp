// ryser_class_impl.hpp -- the Ryser walk by column classes (FP64).
//
// Same sum as ryser_dense_impl.hpp; what differs is how the products are
// formed.  The first K = 5 walked columns are chosen sparse and overlapping
// little; over their 2^5 subsets a row that m of them touch takes 2^m values
// only, so the rows are grouped by the set T of class columns touching them
// and the product of a class's rows is formed once per subset of T:
// sum_T r_T 2^|T| additions and multiplications per 32 subsets instead of
// 32 n each, plus the multiplications that join the classes' arrays
// (class_tree.hpp).  At n = 40 and density 0.5 that is 17.4 to 22.0 FP64
// instructions per subset (thirteen matrices) against 47.5 of the nested walk
// it replaces (80 of the plain one); a full matrix puts every row into the class of all five
// columns and costs what the plain walk does.
//
// One lane's 32 subsets are a group: x_j = L_j + U_j + O_j(s & T), where
//  * L_j (lane and block columns, x0) is a table in LDS, one row of 64
//    entries per matrix row, built once per workgroup and shared by its four
//    waves (lane l fixes the six lane columns by its bits, the workgroup the
//    block columns by the bits of its index, summed in double-double);
//  * U_j (walk columns) is the group's offset, the same in every lane: a
//    scalar load from a table of the 2^w walk subsets, whose entries are
//    correctly rounded sums; the four waves walk a quarter of the groups each;
//  * O_j(s) are the class columns' offsets, constant over the groups: scalar
//    loads from a stream of 64-byte records in the order the rows are met.
// Every x_j is thus at most nine roundings from exact (six lane columns),
// whatever the length of the walk; the nested walk's X drifts by one rounding
// per step.
//
// The matrix's class sizes are loop counts, not template parameters: one
// kernel serves every matrix of every order.  The loads of the next visit (a
// record, two U entries, two LDS rows) are issued between the additions and
// the multiplications of the current one.
//
// Bound: VALU issue (density 0.5: 84 to 87 % of the cycles at n = 40, 81 % at
// n = 36, 79 % at n = 32, and 61 % at n = 27, where a lane has four groups;
// thin tree 78 %).  FP64 instructions are nine tenths of it; the rest of the
// cycles wait for the visit's scalar loads, which three waves per SIMD -- 150
// VGPRs: the arrays of one path through the tree are 63 doubles -- do not
// quite cover; the thin tree's 120 allow four.  Thin against full tree, one
// pass: n = 27, density 0.2 35 against 43 us; n = 33, 0.3 1.44 against 1.98 ms;
// n = 36, 0.2 10.7 against 14.7 ms; n = 34, 0.4 3.6 against 4.4 ms.  Tried and
// dropped: K = 4 (86 VGPRs, five waves, 94 % busy) is 12 % slower, its 21.8
// instructions per subset at n = 36 outweighing the waves; visits of four rows of the small classes cost more scalar work than
// they hide; a second pair of chains in the final accumulation changes
// nothing.
#pragma once
#include <utility>

#include "class_tree.hpp"
#include "ryser_class.hpp"
#include "ryser_dense_impl.hpp"

namespace perm {

typedef double __attribute__((address_space(3)))* LdsPtr;

// Eight and two doubles as one scalar load each.
typedef double Double8 __attribute__((ext_vector_type(8), aligned(8)));
typedef double Double2 __attribute__((ext_vector_type(2), aligned(8)));
typedef uint32_t Word16 __attribute__((ext_vector_type(16)));
typedef const char __attribute__((address_space(4)))* ConstBytes;
typedef const Double8 __attribute__((address_space(4)))* Const8;
typedef const Double2 __attribute__((address_space(4)))* Const2;

// The row stream of one wave within a group, fetched one visit ahead: the
// next rows' table entries, the group's offsets of them and their record of
// class offsets.
struct RowFeed {
  ConstBytes records, walk;
  uint32_t record_off, row_off;  // byte offsets of the next record and row
  uint32_t lane_lds;    // this lane's entry of row 0 in LDS
  double xl[2];
  Double2 u;
  Double8 v;
  // The next two rows and their record.
  __device__ __forceinline__ void fetch() {
    asm volatile("" : "+s"(record_off), "+s"(row_off));
    uint32_t la = lane_lds + (row_off << 6);
    asm volatile("" : "+v"(la));
    const LdsPtr lp = (LdsPtr)(uintptr_t)la;
    u = *(Const2)(walk + row_off);
    v = *(Const8)(records + record_off);
    xl[0] = lp[0];
    xl[1] = lp[kWave];
  }
  __device__ __forceinline__ void advance(uint32_t rows) {
    record_off += 64;
    row_off += 8 * rows;
    fetch();
  }
  // (every fetched word is taken here, so the loads stay whole)
  __device__ __forceinline__ void take() { asm volatile("" : "+s"(u), "+s"(v)); }
  // control word of a class's first record (read as one of 16 words: the
  // compiler takes the wrong word of the vector of doubles)
  __device__ __forceinline__ uint32_t control() const {
    return __builtin_bit_cast(Word16, v)[14];
  }
};

// val[s] (FIRST) or val[s] *= : row value x + offset s of the row's 2^M.
template <int M, bool FIRST>
__device__ __forceinline__ void row_values(double (&val)[1 << M], double x, const Double8& v,
                                           int first) {
#pragma unroll
  for (int s = 0; s < (1 << M); ++s) {
    const double y = s ? x + v[first + s - 1] : x;
    if (FIRST) val[s] = y;
    else val[s] *= y;
  }
}

template <int V, bool FIRST>
__device__ __forceinline__ void multiply_in(double (&P)[V], const double (&val)[V]) {
#pragma unroll
  for (int s = 0; s < V; ++s) {
    if (FIRST) P[s] = val[s];
    else P[s] *= val[s];
  }
}

// A visit of one row (two when `two`) of a class of M <= 2 columns.
template <int M, bool FIRST>
__device__ __forceinline__ void visit_pair(double (&P)[1 << M], RowFeed& f, bool two) {
  double val[1 << M];
  row_values<M, true>(val, f.xl[0] + f.u[0], f.v, 0);
  if (two) {
    asm volatile("");  // a branch, not both sides and selects
    row_values<M, false>(val, f.xl[1] + f.u[1], f.v, (1 << M) - 1);
  }
  __builtin_amdgcn_sched_barrier(0);
  f.advance(two ? 2 : 1);
  multiply_in<1 << M, FIRST>(P, val);
  __builtin_amdgcn_sched_barrier(0);
}

// A visit of one row of a class of M >= 3 columns: 7 offsets from its first
// record, then 8 from each following one.
template <int M, bool FIRST>
__device__ __forceinline__ void visit_wide(double (&P)[1 << M], RowFeed& f) {
  constexpr int V = 1 << M;
  const double x = f.xl[0] + f.u[0];
  double val[8];
  row_values<3, true>(val, x, f.v, 0);
#pragma unroll
  for (int c = 1; c <= V / 8; ++c) {
    __builtin_amdgcn_sched_barrier(0);
    if (c < V / 8) {
      f.record_off += 64;
      asm volatile("" : "+s"(f.record_off));
      f.v = *(Const8)(f.records + f.record_off);
    } else {
      f.advance(1);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      if (FIRST) P[8 * (c - 1) + s] = val[s];
      else P[8 * (c - 1) + s] *= val[s];
    }
    __builtin_amdgcn_sched_barrier(0);
    if (c < V / 8) {
#pragma unroll
      for (int s = 0; s < 8; ++s) val[s] = x + f.v[s];
    }
  }
}

// The rows of one class into P.
template <int M>
__device__ __forceinline__ void class_rows(double (&P)[1 << M], RowFeed& f) {
  f.take();
  const uint32_t ctl = f.control();
  uint32_t more = ctl & 0xffu;
  if constexpr (M <= 2) {
    visit_pair<M, true>(P, f, ctl & 0x100u);
#pragma clang loop unroll(disable)
    for (; more > 0; --more) {
      f.take();
      visit_pair<M, false>(P, f, true);
    }
  } else {
    visit_wide<M, true>(P, f);
#pragma clang loop unroll(disable)
    for (; more > 0; --more) {
      f.take();
      visit_wide<M, false>(P, f);
    }
  }
}

// P_T: the product of the rows of class T and of its live children's arrays.
template <int K, bool THIN, int T>
__device__ __forceinline__ void class_eval(double (&P)[1 << class_popcount(T)], RowFeed& f,
                                           uint32_t live);

template <int K, bool THIN, int T, int C>
__device__ __forceinline__ void class_child(double (&P)[1 << class_popcount(T)], RowFeed& f,
                                            uint32_t live) {
  // (the classes without the last column meet it in the final sum only)
  constexpr bool kChild = C < T && class_allowed(K, THIN, C) &&
                          class_parent(K, THIN, C) == T &&
                          !(T == class_root(K, THIN) && C == (1 << (K - 1)) - 1);
  if constexpr (kChild) {
    if ((live >> C) & 1u) {
      double Q[1 << class_popcount(C)];
      class_eval<K, THIN, C>(Q, f, live);
#pragma unroll
      for (int s = 0; s < (1 << class_popcount(T)); ++s) P[s] *= Q[class_drop(T, C, s)];
    }
  }
}

template <int K, bool THIN, int T, int... C>
__device__ __forceinline__ void class_children(double (&P)[1 << class_popcount(T)], RowFeed& f,
                                               uint32_t live, std::integer_sequence<int, C...>) {
  (class_child<K, THIN, T, C>(P, f, live), ...);
}

template <int K, bool THIN, int T>
__device__ __forceinline__ void class_eval(double (&P)[1 << class_popcount(T)], RowFeed& f,
                                           uint32_t live) {
  class_rows<class_popcount(T)>(P, f);
  class_children<K, THIN, T>(P, f, live, std::make_integer_sequence<int, T>{});
}

// The walk of this workgroup's block `block` of one matrix: the calling
// wave's share of the groups, summed over its lanes' subsets (signs of the
// block and lane columns applied).  `lds` holds (n + 2) * 64 doubles (two
// rows are read ahead); every thread of the workgroup calls it.
template <bool THIN>
__device__ __forceinline__ void class_walk(const ClassMatrix& m, uint64_t block, double* lds,
                                           DD& s, Moments& mo) {
  constexpr int K = kClassBits;
  constexpr int kWaves = 256 / kWave;
  const int n = m.n;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  {
    // row j's start in lane j: x0 plus the block's columns, in double-double
    const int row = (int)lane < n ? (int)lane : 0;
    DD b = {m.lanecols[8 * row + kClassLaneBits], m.lanecols[8 * row + kClassLaneBits + 1]};
    for (int k = 0; k < m.block_bits; ++k)
      if ((block >> k) & 1) b = dd_add_d(b, m.blockcols[(size_t)k * n + row]);
    const double base = b.hi + b.lo;
    double sel[kClassLaneBits];
#pragma unroll
    for (int k = 0; k < kClassLaneBits; ++k) sel[k] = (lane >> k) & 1 ? 1.0 : 0.0;
    const ColPtr lanecols = (ColPtr)m.lanecols;
    for (int r = wave; r < n; r += kWaves) {
      double x = readlane_d(base, r);
#pragma unroll
      for (int k = 0; k < kClassLaneBits; ++k) x = __builtin_fma(sel[k], lanecols[8 * r + k], x);
      lds[r * kWave + lane] = x;
    }
  }
  __syncthreads();
  uint32_t live = m.live;
  const uint32_t groups = 1u << m.walk_bits;
  const uint32_t share = groups >= kWaves ? groups / kWaves : 1;
  s = {0.0, 0.0};
  mo = {0.0, 0.0, 0.0};
  if (wave * share >= groups) return;
  constexpr uint32_t kRun = 256 >> K;  // groups per run of 256 terms
  double p = 0.0, a_run = 0.0;
  for (uint32_t g = 0; g < share; ++g) {
    const uint32_t t = wave * share + g;
    // (the tests of its bits stay where they are, instead of 32 scalar
    // conditions kept over the loop)
    asm volatile("" : "+s"(live));
    RowFeed f;
    f.records = (ConstBytes)m.records;
    f.walk = (ConstBytes)(m.walk + (size_t)t * n);
    f.record_off = f.row_off = 0;
    f.lane_lds = (uint32_t)(uintptr_t)((LdsPtr)lds + lane);
    f.fetch();
    constexpr int kAll = (1 << K) - 1, kHalf = kAll / 2, kRoot = class_root(K, THIN);
    double P[1 << class_popcount(kRoot)];
    class_eval<K, THIN, kRoot>(P, f, live);
    double Q[1 << (K - 1)];
    if ((live >> kHalf) & 1u) {
      class_eval<K, THIN, kHalf>(Q, f, live);
    } else {
#pragma unroll
      for (int i = 0; i <= kHalf; ++i) Q[i] = 1.0;
    }
    double pg = 0.0;
    if constexpr (THIN) {
      // P over columns 1 .. K-1, Q over 0 .. K-2: the sums over the last and
      // over the first column are one factor each (6 instead of 8
      // instructions per four subsets)
      constexpr int kShared = 1 << (K - 2);
#pragma unroll
      for (int i = 0; i < kShared; ++i) {
        const double p0 = P[i], p1 = P[i + kShared], q0 = Q[2 * i], q1 = Q[2 * i + 1];
        const double dp = p0 - p1;
        pg = __builtin_fma(class_popcount(i) & 1 ? -dp : dp, q0 - q1, pg);
        mo.a = __builtin_fma(__builtin_fabs(p0) + __builtin_fabs(p1),
                             __builtin_fabs(q0) + __builtin_fabs(q1), mo.a);
      }
    } else {
#pragma unroll
      for (int i = 0; i <= kAll; ++i) {
        const double q = Q[i & kHalf];
        pg = __builtin_fma(class_popcount(i) & 1 ? -P[i] : P[i], q, pg);
        mo.a = __builtin_fma(__builtin_fabs(P[i]), __builtin_fabs(q), mo.a);
      }
    }
    p = __builtin_fma(__builtin_popcount(t) & 1 ? -1.0 : 1.0, pg, p);
    if ((g & (kRun - 1)) == kRun - 1 || g + 1 == share) {  // fold into double-double
      s = dd_add_d(s, p);
      mo.r = __builtin_fma(p, p, mo.r);
      p = 0.0;
      const double d = mo.a - a_run;
      mo.q = __builtin_fma(d, d, mo.q);
      a_run = mo.a;
    }
  }
  if ((__builtin_popcountll(block) ^ __builtin_popcount(lane)) & 1) {
    s.hi = -s.hi;
    s.lo = -s.lo;
  }
}

}  // namespace perm
