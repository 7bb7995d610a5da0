#include "class_plan.hpp"

#include <algorithm>
#include <cstring>

#include "class_tree.hpp"

namespace perm {

namespace {

constexpr int kClasses = 1 << kClassBits;
constexpr int kHalf = kClasses / 2 - 1;  // the classes without the last column end here
// Search effort: from kWideN on the walk takes a millisecond and more.
constexpr int kWideN = 32;
constexpr int kWidth = 6;

struct Beam {
  uint64_t used = 0;
  uint64_t level[kClassBits + 1] = {};  // rows touched by m of the chosen columns
  int cols[kClassBits];
  int weight = 0;  // sum over rows of 2^(columns touching it)
};

// Rows of every class for the class columns c[0..K).
void split_rows(int n, const uint64_t* sup, const int* c, uint64_t (&rows)[kClasses]) {
  const uint64_t all = n == 64 ? ~0ull : (1ull << n) - 1;
  rows[0] = all;
  for (int k = 0; k < kClassBits; ++k)
    for (int t = (1 << k) - 1; t >= 0; --t) {
      rows[t | 1 << k] = rows[t] & sup[c[k]];
      rows[t] &= ~sup[c[k]];
    }
}

bool has_live_child(const uint64_t (&rows)[kClasses], bool thin, int t) {
  for (int i = 0; i < kClassBits; ++i) {
    const int c = t & ~(1 << i);
    if (c != t && rows[c] && class_parent(kClassBits, thin, c) == t) return true;
  }
  return false;
}

// Move rows up until every class with rows has a parent with rows (the
// kernel starts an array from a row of its class).  A class may be computed
// in any superset: the row's entries in the extra columns are zeros.
// Returns false if the thin tree does not hold them.
bool settle(uint64_t (&rows)[kClasses], bool thin) {
  const int root = class_root(kClassBits, thin);
  auto count = [&](int t) { return __builtin_popcountll(rows[t]); };
  auto leaf = [&](int t) { return !has_live_child(rows, thin, t); };
  auto move_one = [&](int from, int to) {
    const uint64_t one = rows[from] & -rows[from];
    rows[from] &= ~one;
    rows[to] |= one;
  };
  for (int t = 0; t < kClasses; ++t)
    if (rows[t] && !class_allowed(kClassBits, thin, t)) return false;
  for (int m = 0; m < kClassBits; ++m)
    for (int t = 0; t < kClasses; ++t) {
      if (class_popcount(t) != m || !rows[t] || t == root || t == kHalf) continue;
      const int p = class_parent(kClassBits, thin, t);
      if (rows[p]) continue;
      int other = -1;
      for (int i = 0; i < kClassBits; ++i)
        if (!((t >> i) & 1) && rows[t | 1 << i]) other = t | 1 << i;
      if (other >= 0 && count(t) <= 2 && leaf(t)) {
        rows[other] |= rows[t];
        rows[t] = 0;
        continue;
      }
      // a row for the parent from a class inside it that can spare one
      int donor = -1;
      for (int c = 0; c < p; ++c)
        if ((c & ~p) == 0 && rows[c] && (count(c) > 1 || leaf(c)) &&
            (donor < 0 || class_popcount(c) >= class_popcount(donor)))
          donor = c;
      if (donor < 0) {  // no class can spare a row
        if (thin) return false;
        for (int c = 0; c < root; ++c) {  // all in the root
          rows[root] |= rows[c];
          rows[c] = 0;
        }
        return true;
      }
      move_one(donor, p);
    }
  for (int c = kClasses - 1; !rows[root] && c >= 0; --c)  // (no row of the last column)
    if ((c & ~root) == 0 && rows[c] && (count(c) > 1 || leaf(c))) move_one(c, root);
  return rows[root] != 0;
}

int plan_cost(const uint64_t (&rows)[kClasses], bool thin) {
  int cost = thin ? 3 * kClasses / 2 : 2 * kClasses;  // the final sum
  for (int t = 0; t < kClasses; ++t) {
    if (!rows[t]) continue;
    cost += (2 * __builtin_popcountll(rows[t]) - 1) << class_popcount(t);
    if (t != class_root(kClassBits, thin) && t != kHalf)
      cost += 1 << class_popcount(class_parent(kClassBits, thin, t));
  }
  return cost;
}

void order_rows(const uint64_t (&rows)[kClasses], int t, int& at, ClassPlan& p) {
  for (uint64_t r = rows[t]; r; r &= r - 1) {
    p.classes[at] = (uint8_t)t;
    p.rows[at++] = __builtin_ctzll(r);
  }
  for (int c = 0; c < t; ++c)
    if (rows[c] && class_parent(kClassBits, p.thin, c) == t &&
        !(t == class_root(kClassBits, p.thin) && c == kHalf))
      order_rows(rows, c, at, p);
}

}  // namespace

void plan_classes(int n, const uint64_t* sup, ClassPlan& p) {
  const int B = n - 1;
  // candidates: the sparsest columns (all of them where the search is small
  // against the walk)
  const bool wide = n >= kWideN;
  const int width = wide ? kWidth : 2, cands = wide ? B : std::min(B, 12);
  uint8_t cand[64];
  {
    // counting sort by rows touched
    uint8_t start[66] = {0}, touched[64];
    for (int c = 0; c < B; ++c) {
      touched[c] = (uint8_t)__builtin_popcountll(sup[c]);
      ++start[touched[c] + 1];
    }
    for (int k = 1; k < 66; ++k) start[k] = (uint8_t)(start[k] + start[k - 1]);
    for (int c = 0; c < B; ++c) cand[start[touched[c]]++] = (uint8_t)c;
  }
  Beam beam[kWidth], next[kWidth];
  int nb = 1;
  beam[0].level[0] = (1ull << n) - 1;
  beam[0].weight = n;
  for (int k = 0; k < kClassBits; ++k) {
    int nn = 0;
    struct Pick {
      int weight, from, col;
      uint64_t used;
    } pick[kWidth];
    for (int i = 0; i < nb; ++i)
      for (int ci = 0; ci < cands; ++ci) {
        const int c = cand[ci];
        if ((beam[i].used >> c) & 1) continue;
        int w = beam[i].weight;
        for (int m = 0; m <= k; ++m)
          w += __builtin_popcountll(beam[i].level[m] & sup[c]) << m;
        if (nn == width && w >= pick[nn - 1].weight) continue;
        const uint64_t used = beam[i].used | 1ull << c;
        bool dup = false;
        for (int j = 0; j < nn; ++j) dup |= pick[j].used == used;
        if (dup) continue;
        int at = nn < width ? nn++ : nn - 1;
        for (; at > 0 && pick[at - 1].weight > w; --at) pick[at] = pick[at - 1];
        pick[at] = {w, i, c, used};
      }
    for (int j = 0; j < nn; ++j) {
      Beam& b = next[j];
      b = beam[pick[j].from];
      const uint64_t s = sup[pick[j].col];
      b.used = pick[j].used;
      b.cols[k] = pick[j].col;
      b.weight = pick[j].weight;
      for (int m = k; m >= 0; --m) {
        b.level[m + 1] |= b.level[m] & s;
        b.level[m] &= ~s;
      }
    }
    nb = nn;
    std::copy(next, next + nn, beam);
  }
  uint64_t rows[kClasses], best[kClasses];
  int best_cols[kClassBits];
  p.cost = -1;
  p.thin = false;
  auto consider = [&](const int* c, bool thin) {
    split_rows(n, sup, c, rows);
    if (!settle(rows, thin)) return;
    const int cost = plan_cost(rows, thin);
    if (p.cost >= 0 && cost >= p.cost) return;
    p.cost = cost;
    p.thin = thin;
    std::memcpy(best, rows, sizeof(rows));
    std::copy(c, c + kClassBits, best_cols);
  };
  for (int i = 0; i < std::min(nb, wide ? 3 : 1); ++i) {
    int c[kClassBits];
    std::copy(beam[i].cols, beam[i].cols + kClassBits, c);
    std::sort(c, c + kClassBits, [&](int a, int b) {
      const int x = __builtin_popcountll(sup[a]), y = __builtin_popcountll(sup[b]);
      return x != y ? x < y : a < b;
    });
    consider(c, false);
    // the thin tree: two columns without a common row at its ends
    for (int a = 0; a < kClassBits; ++a)
      for (int b = a + 1; b < kClassBits; ++b) {
        if (sup[c[a]] & sup[c[b]]) continue;
        int d[kClassBits], at = 1;
        d[0] = c[a];
        d[kClassBits - 1] = c[b];
        for (int k = 0; k < kClassBits; ++k)
          if (k != a && k != b) d[at++] = c[k];
        consider(d, true);
        if (!wide) continue;
        std::swap(d[0], d[kClassBits - 1]);
        consider(d, true);
      }
    std::reverse(c, c + kClassBits);
    consider(c, false);
  }
  // Exchanges of two columns' places in the tree, while they help (2-3 % of
  // the walk for about 20 us here).
  for (int round = 0; wide && round < 4; ++round) {
    const int before = p.cost;
    int from[kClassBits];
    std::copy(best_cols, best_cols + kClassBits, from);
    const bool thin = p.thin;
    for (int i = 0; i < kClassBits; ++i)
      for (int j = i + 1; j < kClassBits; ++j) {
        std::swap(from[i], from[j]);
        consider(from, thin);
        std::swap(from[i], from[j]);
      }
    if (p.cost == before) break;
  }
  p.n = n;
  uint64_t used = 0;
  int at = 0;
  for (int k = 0; k < kClassBits; ++k) {
    p.cols[at++] = best_cols[k];
    used |= 1ull << best_cols[k];
  }
  for (int c = 0; c < B; ++c)
    if (!((used >> c) & 1)) p.cols[at++] = c;
  p.live = 0;
  for (int t = 0; t < kClasses; ++t) {
    p.count[t] = (uint8_t)__builtin_popcountll(best[t]);
    if (best[t]) p.live |= 1u << t;
  }
  at = 0;
  order_rows(best, class_root(kClassBits, p.thin), at, p);
  if (best[kHalf]) order_rows(best, kHalf, at, p);
}

void build_class_tables(const ClassPlan& p, const double* x0, const double* cols, int walk_bits,
                        ClassTables& out) {
  const int n = p.n, B = n - 1;
  auto entry = [&](int r, int i) { return cols[(size_t)p.cols[i] * n + p.rows[r]]; };
  std::vector<double>& d = out.data;
  d.clear();
  d.reserve(class_tables_bound(n) + (walk_bits < 0 ? 0 : class_split_doubles(n, walk_bits)));
  // records: 7 offsets and the control word, then 8 offsets each
  auto add_row = [&](int r, double* o) {  // the 2^m - 1 offsets of row r
    const int t = p.classes[r];
    double hi[kClasses] = {0.0}, lo[kClasses] = {0.0};
    int m = 0;
    for (int i = 0; i < kClassBits; ++i) {
      if (!((t >> i) & 1)) continue;
      const double c = entry(r, i);
      for (int s = 0; s < 1 << m; ++s) {
        const double v = hi[s] + c, bb = v - hi[s];
        lo[s | 1 << m] = lo[s] + ((hi[s] - (v - bb)) + (c - bb));
        hi[s | 1 << m] = v;
      }
      ++m;
    }
    for (int s = 1; s < 1 << m; ++s) o[s - 1] = hi[s] + lo[s];
  };
  for (int r = 0; r < n;) {
    const int t = p.classes[r], m = class_popcount(t), c = p.count[t];
    const int end = r + c;
    for (int visit = 0; r < end; ++visit) {
      const int rows = m > kClassPairBits ? 1 : visit == 0 ? (c & 1 ? 1 : 2) : 2;
      double o[2 * kClasses] = {0.0};
      for (int i = 0; i < rows; ++i) add_row(r + i, o + i * ((1 << m) - 1));
      uint64_t control = 0;
      if (visit == 0)
        control = (uint64_t)((c - rows) / (m > kClassPairBits ? 1 : 2)) | (rows == 2 ? 0x100u : 0u);
      double word;
      std::memcpy(&word, &control, sizeof(word));
      d.insert(d.end(), o, o + 7);
      d.push_back(word);
      if (m > 3) d.insert(d.end(), o + 7, o + (1 << m) - 1);
      r += rows;
    }
  }
  d.resize(d.size() + 8, 0.0);  // read ahead by one record
  out.cols = d.size();
  for (int b = kClassBits; b < B; ++b)
    for (int r = 0; r < n; ++r) d.push_back(entry(r, b));
  for (int part = 0; part < 2; ++part)
    for (int r = 0; r < n; ++r) d.push_back(x0[part * n + p.rows[r]]);
  if (walk_bits < 0) return;
  const int walk0 = kClassBits, lane0 = walk0 + walk_bits;
  out.lane = d.size();
  for (int r = 0; r < n; ++r) {
    for (int b = 0; b < kClassLaneBits; ++b) d.push_back(entry(r, lane0 + b));
    d.push_back(x0[p.rows[r]]);
    d.push_back(x0[n + p.rows[r]]);
  }
  // offsets of the walk columns' subsets, each the rounded double-double sum
  out.walk = d.size();
  const size_t subsets = (size_t)1 << walk_bits;
  d.resize(out.walk + subsets * n + 2, 0.0);  // (two entries read ahead)
  double* u = d.data() + out.walk;
  std::vector<double> lo(subsets * n, 0.0);
  for (int b = 0; b < walk_bits; ++b) {
    const size_t half = (size_t)1 << b;
    double c[64];
    for (int r = 0; r < n; ++r) c[r] = entry(r, walk0 + b);
    for (size_t t = 0; t < half; ++t)
      for (int r = 0; r < n; ++r) {
        const double h = u[t * n + r];
        const double v = h + c[r], bb = v - h;
        lo[(half + t) * n + r] = lo[t * n + r] + ((h - (v - bb)) + (c[r] - bb));
        u[(half + t) * n + r] = v;
      }
  }
  for (size_t i = 0; i < subsets * n; ++i) u[i] += lo[i];
}

}  // namespace perm
