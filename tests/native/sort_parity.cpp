// The canonical list's sort (beamtrace2007_amd/csrc/poly_order.h, compiled
// here for the host) with its two steps run as the kernels run them: blocks
// ranked by counting, then runs merged pairwise by binary search. Whatever the
// corners and areas hold - NaNs, infinities, zeros of both signs, equal
// polygons - every place must be taken once, and the list must be in order; a
// list without NaNs must equal std::stable_sort's by the plain comparison of
// values.
//
// Prints "ok <lists>".
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <numeric>
#include <vector>

#include "../../beamtrace2007_amd/csrc/poly_order.h"

namespace {

struct Rng {
  uint64_t s;
  uint32_t next() {
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    return uint32_t(s >> 11);
  }
  int below(int n) { return int(next() % uint32_t(n)); }
};

// The comparison of values, a strict order while no NaN is among them.
bool plainLess(const btg::OutPoly& a, const btg::OutPoly& b) {
  if (a.tri != b.tri) return a.tri < b.tri;
  if (a.n != b.n) return a.n < b.n;
  for (int k = 0; k < a.n; ++k) {
    if (a.x[k] != b.x[k]) return a.x[k] < b.x[k];
    if (a.y[k] != b.y[k]) return a.y[k] < b.y[k];
  }
  return a.area < b.area;
}

// The sort's steps; false if a place is out of range, taken twice or left.
bool sorted(const std::vector<btg::OutPoly>& v, int block, std::vector<int>& order) {
  const int n = int(v.size());
  order.assign(size_t(n), -1);
  auto put = [&](std::vector<int>& o, int64_t at, int k) {
    if (at < 0 || at >= n || o[size_t(at)] != -1) return false;
    o[size_t(at)] = k;
    return true;
  };
  for (int i = 0; i < n; ++i) {
    const int base = i / block * block, m = std::min(block, n - base);
    int rank = 0;
    for (int j = 0; j < m; ++j)
      if (base + j != i) rank += btg::goesBefore(v[size_t(base + j)], base + j, v[size_t(i)], i);
    if (!put(order, base + rank, i)) return false;
  }
  for (int64_t run = block; run < n; run *= 2) {
    std::vector<int> out(size_t(n), -1);
    for (int i = 0; i < n; ++i) {
      const int64_t mine = i / run, sib = (mine ^ 1) * run;
      int lo = 0;
      if (sib < n)
        lo = btg::mergeBefore(v[size_t(order[size_t(i)])], (mine & 1) != 0, int(std::min<int64_t>(run, n - sib)),
                              [&](int k) { return v[size_t(order[size_t(sib + k)])]; });
      if (!put(out, (mine & ~int64_t(1)) * run + (i - mine * run) + lo, order[size_t(i)])) return false;
    }
    order = out;
  }
  return true;
}

}  // namespace

int main(int argc, char** argv) {
  const int lists = argc > 1 ? std::atoi(argv[1]) : 1000;
  const float inf = std::numeric_limits<float>::infinity(), nan = std::nanf("");
  const float odd[] = {0.0f, -0.0f, 1.0f, -1.0f, inf, -inf, 2.0f, 1e-40f, nan, -nan};
  Rng r{0x2545F4914F6CDD1Dull};
  for (int l = 0; l < lists; ++l) {
    const bool nans = l % 2 == 0;
    const int n = 1 + r.below(300), tris = 1 + r.below(l % 3 ? 3 : 60);
    const int block = 1 << r.below(9);  // runs of one polygon up to one block for the whole list
    std::vector<btg::OutPoly> v(static_cast<size_t>(n));
    for (btg::OutPoly& p : v) {
      auto value = [&] { return r.below(3) ? odd[r.below(nans ? 10 : 8)] : float(r.below(4)); };
      for (int k = 0; k < 4; ++k) {
        p.x[k] = value();
        p.y[k] = value();
      }
      p.n = 3 + r.below(2);
      p.tri = r.below(tris);
      p.area = value();
    }
    if (l % 5 == 0) std::fill(v.begin(), v.end(), v[0]);  // equal polygons
    if (l == 0) {  // two numbers on either side of a NaN
      v.assign(3, btg::OutPoly{});
      const float x[3] = {2, nan, 1};
      for (int k = 0; k < 3; ++k) {
        v[size_t(k)].n = 3;
        v[size_t(k)].x[0] = x[k];
      }
    }
    std::vector<int> order;
    if (!sorted(v, block, order)) {
      std::printf("list %d (%d polygons, blocks of %d): a place is taken twice\n", l, int(v.size()), block);
      return 1;
    }
    for (size_t k = 1; k < order.size(); ++k)
      if (btg::polyLess(v[size_t(order[k])], v[size_t(order[k - 1])])) {
        std::printf("list %d: places %zu and %zu are not in order\n", l, k - 1, k);
        return 1;
      }
    bool plain = true;
    for (const btg::OutPoly& p : v) {
      plain = plain && p.area == p.area;
      for (int k = 0; k < p.n; ++k) plain = plain && p.x[k] == p.x[k] && p.y[k] == p.y[k];
    }
    if (plain) {
      std::vector<int> want(v.size());
      std::iota(want.begin(), want.end(), 0);
      std::stable_sort(want.begin(), want.end(), [&](int a, int b) { return plainLess(v[size_t(a)], v[size_t(b)]); });
      if (want != order) {
        std::printf("list %d: not std::stable_sort's order\n", l);
        return 1;
      }
    }
  }
  std::printf("ok %d\n", lists);
  return 0;
}
