// The order of a canonical polygon list and the places its sort gives to
// polygons (sortBlocks, mergeRuns). Host and device code, so that the places
// are checked on the CPU.
#pragma once

#include "engine.h"

namespace btg {

// -1, 0 or 1: a before, with or after b. NaNs come last and together: with
// a comparison that only asks a < b a NaN would equal every number, the order
// would not be transitive, two polygons could be given one place and another
// place none. Caller's polygons reach the lists as they are (receivers that face
// away from the light), NaN corners included.
BTG_HD int orderOf(float a, float b) {
  if (a == b) return 0;
  if (a < b) return -1;
  if (b < a) return 1;
  return int(a != a) - int(b != b);
}

// The reference's canonical order (polyLess): triangle, corner count, corners,
// area; -1, 0 or 1 as orderOf.
BTG_HD int polyOrder(const OutPoly& a, const OutPoly& b) {
  if (a.tri != b.tri) return a.tri < b.tri ? -1 : 1;
  if (a.n != b.n) return a.n < b.n ? -1 : 1;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (k >= a.n) break;
    if (const int o = orderOf(a.x[k], b.x[k])) return o;
    if (const int o = orderOf(a.y[k], b.y[k])) return o;
  }
  return orderOf(a.area, b.area);
}
BTG_HD bool polyLess(const OutPoly& a, const OutPoly& b) { return polyOrder(a, b) < 0; }

// Whether polygon a, at place ia, goes before polygon b, at place ib: equal
// polygons keep their order, so that no two share a place.
BTG_HD bool goesBefore(const OutPoly& a, int ia, const OutPoly& b, int ib) {
  const int o = polyOrder(a, b);
  return o < 0 || (o == 0 && ia < ib);
}

// How many of the sibling run's `count` polygons, at(0) to at(count - 1) in
// order, go before `own`, a polygon of the second or of the first run of the
// pair (elements of the first precede their equals).
template <class At>
BTG_HD int mergeBefore(const OutPoly& own, bool second, int count, At at) {
  int lo = 0, hi = count;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    const OutPoly other = at(mid);
    if (polyOrder(other, own) < int(second))
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

}  // namespace btg
