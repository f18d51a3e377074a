// The kd predicates of a beam: which children of an inner node it enters
// (decide) and whether it can meet a box (overlaps), src/beam/beam_core.h:139-195,
// in the reference's arithmetic and, for the trace kernel, in a few
// operations on nine per-beam bounds that give the same answers. Host and
// device code, so that the two forms are compared on the CPU.
#pragma once

#include "beam_dev.h"

namespace btg {

enum { kNear = 0, kFar = 1, kBoth = 2, kBand = 3 };

// The beam's |w| per axis and its far plane (CoreBeam's aw, farA, farC), for
// the exact kd predicates.
struct Dirs {
  C4 aw0, aw1, aw2, farA;
  float farC;
  bool hasFar;
};

// Per-axis fields picked by value (a select of loaded values, never of
// addresses, so the beam stays in registers).
BTG_HD C4 awOf(const Dirs& b, int a) {
  C4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x0 = b.aw0.v[i], x1 = b.aw1.v[i], x2 = b.aw2.v[i];
    r.v[i] = a == 0 ? x0 : (a == 1 ? x1 : x2);
  }
  return r;
}

// Signed distances from the apex to a box's slabs along each axis, in the
// rays' direction: nIn[k] to the face they enter by, nOut[k] to the face they
// leave by (the Nmin / Nmax of beam_core.h:146-149, 171-173). The descent
// carries them instead of the box: narrowing the box to a child moves one
// face of the split axis onto the split plane, whose distance is the
// descent's own Ns, so only that one value changes per kd step.
struct SlabDist {
  F3 nIn, nOut;
};
// decide (beam_core.h:139-164): near / far / both children of an inner node.
BTG_HD int decide(const Dirs& b, int a, float Ns, const SlabDist& sd) {
  const C4 awa = awOf(b, a);
#pragma unroll
  for (int k = 1; k <= 2; ++k) {
    const int cc = a + k >= 3 ? a + k - 3 : a + k;
    const C4 lhs = scaled(awOf(b, cc), Ns);
    if (allBelow(lhs, scaled(awa, comp(sd.nIn, cc)), kKdRel)) return kFar;
    if (allAbove(lhs, scaled(awa, comp(sd.nOut, cc)), kKdRel)) return kNear;
  }
  if (b.hasFar && allAbove(scaled(b.farA, Ns), scaled(awa, b.farC), kKdRel)) return kNear;
  return kBoth;
}

// overlaps (beam_core.h:166-195): false if the beam certainly misses the box
// whose slab distances are sd.
BTG_HD bool overlaps(const Dirs& b, const SlabDist& sd) {
  const float nmin[3] = {sd.nIn.x, sd.nIn.y, sd.nIn.z}, nmax[3] = {sd.nOut.x, sd.nOut.y, sd.nOut.z};
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (nmax[k] < 0) return false;
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      if (k == e) continue;
      if (allBelow(scaled(awOf(b, e), nmax[k]), scaled(awOf(b, k), nmin[e]), kKdRel)) return false;
    }
  if (b.hasFar) {
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (allAbove(scaled(b.farA, nmin[k]), scaled(awOf(b, k), b.farC), kKdRel)) return false;
  }
  return true;
}

// ------------------------------------------------- kd predicates in ratios
// Each comparison of decide and overlaps asks whether l = x[i] X lies below
// r = y[i] Y, by a relative margin of kKdRel, for all four corners i, with
// x, y >= 0 fixed for the beam and X, Y the node's slab distances: whether
// max_i (x[i] / y[i]) X < Y up to a factor 1 +- 2 kKdRel. So the trace keeps
// the beam's nine maxima (KdBounds) and decides a comparison with a multiply
// and two compares instead of four corners' products, sums and margins. The
// maxima carry a relative error below 4e-7 (a reciprocal, two products), far
// less than the margin: a product below Y kBelow holds in the reference's
// arithmetic, one at or above Y kNotBelow fails there (some l >= r; rounding is
// monotonic), and a beam whose product falls between the two, 2.4e-5 wide,
// takes the reference's own arithmetic (decide, overlaps). Bit for bit the
// same decisions; the band is met by fewer than 1 in 10^5
// ordinary decisions.
// A corner with y[i] = 0 has r = 0, which no l is below: its ratio is infinite,
// and infinity times X is infinite (not below) or, at X = 0, NaN, which
// compares false (not below). Denormal products never decide: `slow` marks
// beams with some 0 < x[i] < 1e-18 or x[i] > 1e18 (and NaNs), "below" asks for
// Y above 1e-12 (kTiny) and "not below" for a product of at least 1e-36 (kFloor).
// Why: the trace kernel is bound by VALU issue with a quarter of its lanes
// active, and the exact predicates took 24 to 216 operations each behind early
// exits that a divergent wave seldom takes. By the bounds a decision takes about
// 40 and a box test 30, and the beam's sixteen |w| and far-plane registers go.
// Measured: soft-shadow trace kernel 944 -> 750 ms over sixteen blob and atrium
// jobs (1.13 -> 0.92 s a batch), 112 -> 92 ms on the plant at 512 x 512 (137.5 ->
// 117.0 ms a frame), 16.7 -> 14.2 ms on the conference hall at 501 x 377.
constexpr float kBelow = 1.0f - 2.3e-5f, kNotBelow = 1.0f + 1e-6f, kTiny = 1e-12f, kFloor = 1e-36f;
constexpr float kSmallDir = 1e-18f, kLargeDir = 1e18f;
constexpr float kWide = 1e15f;  // coordinates up to here cannot overflow a product with a |w| of at most kLargeDir

struct KdBounds {
  float up[3];    // up[a] = max_i aw_a[i] / aw_{a+1}[i]   (axes mod 3)
  float down[3];  // down[a] = max_i aw_{a+1}[i] / aw_a[i]
  float far[3];   // max_i aw_a[i] farC / farA[i]; infinite without a far plane
  bool slow;
};

BTG_HD float max4(const C4& v) {
  return __builtin_fmaxf(__builtin_fmaxf(v.v[0], v.v[1]), __builtin_fmaxf(v.v[2], v.v[3]));
}
BTG_HD float min4(const C4& v) {
  return __builtin_fminf(__builtin_fminf(v.v[0], v.v[1]), __builtin_fminf(v.v[2], v.v[3]));
}
// max_i x[i] / y[i] given the reciprocals of y and its minimum.
BTG_HD float maxRatio(const C4& x, const C4& ry, float miny) {
  C4 q;
#pragma unroll
  for (int i = 0; i < 4; ++i) q.v[i] = x.v[i] * ry.v[i];
  return miny > 0 ? max4(q) : __builtin_inff();
}
BTG_HD C4 rcp4(const C4& v) {
  C4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#if defined(__HIP_DEVICE_COMPILE__)
    r.v[i] = __builtin_amdgcn_rcpf(v.v[i]);  // within 1 ulp
#else
    r.v[i] = 1.0f / v.v[i];
#endif
  }
  return r;
}
// True when every v[i] is 0 or within [kSmallDir, kLargeDir].
BTG_HD bool plainDirs(const C4& v) {
  bool ok = true;
#pragma unroll
  for (int i = 0; i < 4; ++i) ok = ok && (v.v[i] == 0 || (v.v[i] >= kSmallDir && v.v[i] <= kLargeDir));
  return ok;
}

// OneFar: farA[i] = farC for every corner (any-hit queries).
template <bool OneFar>
BTG_HD void farBounds(const Dirs& d, KdBounds& kb) {
  if (!d.hasFar) {
    kb.far[0] = kb.far[1] = kb.far[2] = __builtin_inff();
    return;
  }
  if (OneFar) {
    kb.far[0] = max4(d.aw0);
    kb.far[1] = max4(d.aw1);
    kb.far[2] = max4(d.aw2);
    kb.slow = kb.slow || !(d.farC >= kSmallDir && d.farC <= kLargeDir);
    return;
  }
  const C4 rf = scaled(rcp4(d.farA), d.farC);
  const float mf = min4(d.farA);
  kb.far[0] = maxRatio(d.aw0, rf, mf);
  kb.far[1] = maxRatio(d.aw1, rf, mf);
  kb.far[2] = maxRatio(d.aw2, rf, mf);
  kb.slow = kb.slow || !plainDirs(d.farA) || !(d.farC >= kSmallDir && d.farC <= kLargeDir);
}

template <bool OneFar>
BTG_HD KdBounds kdBounds(const Dirs& d) {
  KdBounds kb;
  const C4 r0 = rcp4(d.aw0), r1 = rcp4(d.aw1), r2 = rcp4(d.aw2);
  const float m0 = min4(d.aw0), m1 = min4(d.aw1), m2 = min4(d.aw2);
  kb.up[0] = maxRatio(d.aw0, r1, m1);
  kb.up[1] = maxRatio(d.aw1, r2, m2);
  kb.up[2] = maxRatio(d.aw2, r0, m0);
  kb.down[0] = maxRatio(d.aw1, r0, m0);
  kb.down[1] = maxRatio(d.aw2, r1, m1);
  kb.down[2] = maxRatio(d.aw0, r2, m2);
  kb.slow = !(plainDirs(d.aw0) && plainDirs(d.aw1) && plainDirs(d.aw2));
  farBounds<OneFar>(d, kb);
  return kb;
}

// The bounds as words at col[w * Stride], three per axis: up, down, far of
// axis a at words 3 a .. 3 a + 2. The trace keeps them in an LDS column: the
// axis is per lane and per node, so they are read by address rather than
// selected among registers.
constexpr int kBoundWords = 9;
template <int Stride>
BTG_HD void boundsStore(float* col, const KdBounds& kb) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    col[(3 * a) * Stride] = kb.up[a];
    col[(3 * a + 1) * Stride] = kb.down[a];
    col[(3 * a + 2) * Stride] = kb.far[a];
  }
}

// decide by the bounds: kNear, kFar, kBoth, or kBand where the reference's
// arithmetic has to say. Ns > 0.
template <int Stride>
BTG_HD int decideBounds(const float* col, bool slow, int a, float Ns, const SlabDist& sd) {
  const int c1 = a == 2 ? 0 : a + 1, c2 = a == 0 ? 2 : a - 1;
  const float* pa = col + 3 * a * Stride;
  const float* p2 = col + 3 * c2 * Stride;
  const float up = pa[0], down = pa[Stride], far = pa[2 * Stride], up2 = p2[0], down2 = p2[Stride];
  const float in1 = comp(sd.nIn, c1), in2 = comp(sd.nIn, c2);
  const float t1 = down * Ns, t2 = up * comp(sd.nOut, c1), t3 = up2 * Ns, t4 = down2 * comp(sd.nOut, c2);
  const float lo = __builtin_fmaf(Ns, kBelow, -kTiny), hi = __builtin_fmaf(Ns, kNotBelow, kFloor);
  const bool f1 = t1 < __builtin_fmaf(in1, kBelow, -kTiny), f2 = t3 < __builtin_fmaf(in2, kBelow, -kTiny);
  const bool n1 = t2 < lo, n2 = t4 < lo, n3 = far < lo;
  const bool band = slow | (!f1 & (t1 < __builtin_fmaf(in1, kNotBelow, kFloor))) | (!f2 & (t3 < __builtin_fmaf(in2, kNotBelow, kFloor))) | (!n1 & (t2 < hi)) |
                    (!n2 & (t4 < hi)) | (!n3 & (far < hi));
  if (band) return kBand;
  return f1 ? kFar : (n1 ? kNear : (f2 ? kFar : ((n2 | n3) ? kNear : kBoth)));
}

// overlaps by the bounds: 0, 1, or kBand.
template <int Stride>
BTG_HD int overlapsBounds(const float* col, bool slow, const SlabDist& sd) {
  const float nmin[3] = {sd.nIn.x, sd.nIn.y, sd.nIn.z}, nmax[3] = {sd.nOut.x, sd.nOut.y, sd.nOut.z};
  bool miss = (nmax[0] < 0) | (nmax[1] < 0) | (nmax[2] < 0);
  bool band = false;
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    const int k1 = (e + 1) % 3, k2 = (e + 2) % 3;
    // aw_e / aw_k1 = up[e], aw_e / aw_k2 = down[k2]
    const float t1 = col[(3 * e) * Stride] * nmax[k1], t2 = col[(3 * k2 + 1) * Stride] * nmax[k2];
    const float t = __builtin_fminf(__builtin_fminf(t1, t2), col[(3 * e + 2) * Stride]);
    miss |= t < __builtin_fmaf(nmin[e], kBelow, -kTiny);
    band |= t < __builtin_fmaf(nmin[e], kNotBelow, kFloor);
  }
  if (slow) return kBand;
  return miss ? 0 : (band ? int(kBand) : 1);
}

}  // namespace btg
