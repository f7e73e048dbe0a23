// The conservative child-box test of the traversal, on the compact boxes of a child group
// (dr_octree_build.h): which children a ray's walk may skip.  Host and device.  (Child boxes in the
// cells of a grid per group are known from compressed wide BVHs, Ylitie, Karras and Laine 2017; the error
// bound and the acceptance rule below are this tree's.)
//
// A leaf accepts a hit only at p = fl(o + fl(d * t)), t >= 0, inside its box, so a child may be
// skipped if no real point o + d * t with t >= 0 lies within a rounding error of the boxes
// below it.  The test runs on the scaled distance T = t * max|d.k|, per axis between
//   near = (min - o) * iv - er    and    far = (max - o) * iv + er,    iv = max|d.k| / d.k,
// and keeps the child if max(near, 0) <= far over the three axes.  A plane's distance is one fused
// product, plane * iv + c, with cn = -o * iv - er and cf = -o * iv + er formed once per ray.
//
// er covers every rounding on the way.  With u = 2^-24, M the largest magnitude of a box
// coordinate and O the largest of o: o + d t misses p by at most u (2 M + O) per axis; iv (one
// hardware reciprocal, one product) is off by 3 u relative; the roundings of cn or cf, of the
// grid's origin and cell and of the plane come to at most u (6 M + 4 O) |iv|.  Together less than
// u (11 M + 8 O) |iv|, and er = 16 u (M + O) |iv|.
// An axis the ray hardly moves along has its |iv| cut to kMaxIv.  Its interval then only has to
// hold the largest T that a hit can have, at most 1.01 (M + O): er's slack of 3 u (M + O) |iv| is
// above 190 (M + O) there.
//
// T is scaled by a power of two (t_unit) so that every T of interest lies in [0, 1]: the near distance
// of one axis, cut to [0, 1] by an output modifier, then needs no maximum with 0, 8 vector instructions
// of an expansion's 163 (1080p 16 spp 13.31 -> 13.21 ms, 512x512 adjoint 5.89 -> 5.84 ms).  A box further
// than 1 would be kept; there is none: its far distance on the axis with iv = 1 is below 1.
//
// Why: an expansion with the reference's own boxes read 200 B over three 128-B lines in 13 loads,
// and its octant and slab tests branched per child.  4M incoherent rays through 2.1 M triangles
// moved 10.8 GB through the fabric (5.3 TB/s, above the 4.7 TB/s that a large copy reaches on this
// card), and a 1080p frame kept the VALU 88% busy.  One line of byte-sized boxes needs 5 loads and
// 163 vector operations without a branch (200 or so for the 7 live children before).  Measured,
// before -> after: 4,194,304 incoherent rays 2.08 -> 1.33 ms, 1080p primary rays over the same
// triangles 1.38 -> 1.00 ms, path trace 1080p 16 spp 24.3 -> 21.4 ms, 512x512 adjoint 14.1 -> 12.2 ms.
#pragma once
#include <string.h>
#include "dr_geom.h"
#include "dr_octree_build.h"

namespace dr {

DR_HD int bits_of(float v) { int i; memcpy(&i, &v, 4); return i; }
DR_HD float float_of(int i) { float v; memcpy(&v, &i, 4); return v; }

constexpr float kMaxIv = 1073741824.0f;        // 2^30
constexpr float kBoxSlack = 9.5367431640625e-7f;   // 16 * 2^-24

// A ray prepared for the box test.
struct BoxRay {
  V3 iv, cn, cf;
  int canon;     // canonicalOrder (Octree.impl.cuh:181-183): the children are visited in the order canon ^ i
};

// A reciprocal within 1 ulp (inf for 0).
DR_HD float fast_rcp(float v) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_rcpf(v);
#else
  return 1.0f / v;
#endif
}
// v cut to [0, 1] (an output modifier of the instruction that forms v).
DR_HD float unit_clamp(float v) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_fmed3f(v, 0.0f, 1.0f);
#else
  return __builtin_fminf(__builtin_fmaxf(v, 0.0f), 1.0f);
#endif
}
DR_HD float max3(float a, float b, float c) { return __builtin_fmaxf(__builtin_fmaxf(a, b), c); }
DR_HD float min3(float a, float b, float c) { return __builtin_fminf(__builtin_fminf(a, b), c); }

// The power of two that scales T: 1/4 of s = M + O rounded down, so that a hit's T, at most 1.01 (M + O),
// and every box's far distance on the axis the ray moves along most stay below 1 (from 2^-60 up: the
// unit times kMaxIv stays finite).
DR_HD float t_unit(float s) { return float_of((252 << 23) - (bits_of(__builtin_fmaxf(s, 8.6736174e-19f)) & 0x7f800000)); }

// Prepares a ray; false if it cannot hit anything (a zero direction: dot(d, n) is 0 for every
// plane; a component that is not finite: t or the hit point is not a number, or t is not below FLT_MAX).
DR_HD bool box_ray(V3 o, V3 d, float reach, BoxRay &r) {
  const float ax = __builtin_fabsf(d.x), ay = __builtin_fabsf(d.y), az = __builtin_fabsf(d.z);
  const float dm = max3(ax, ay, az);
  const float om = max3(__builtin_fabsf(o.x), __builtin_fabsf(o.y), __builtin_fabsf(o.z));
  // (a sum, unlike a maximum, keeps a NaN; of eighths, so that six finite components stay below infinity)
  const float sum = __builtin_fmaf(ax, 0.125f, __builtin_fmaf(ay, 0.125f, __builtin_fmaf(az, 0.125f,
                    __builtin_fmaf(__builtin_fabsf(o.x), 0.125f, __builtin_fmaf(__builtin_fabsf(o.y), 0.125f,
                                   __builtin_fabsf(o.z) * 0.125f)))));
  const bool able = sum < __builtin_inff() && dm > 0.0f;
  int c = (d.z < 0) ? 1 : 0;
  if (d.y < 0) c += 2;
  if (d.x < 0) c += 4;
  r.canon = c;
  // the reciprocals of very short or long directions are taken of the direction scaled by a power of two
  const float sc = dm < 1e-30f ? 1.2676506e30f : (dm > 1e30f ? 7.8886091e-31f : 1.0f);
  const float ds = dm * sc;
  // coordinates whose products with iv could overflow: every box is kept
  const float s = om + reach;
  const float unit = t_unit(s);
  float ix = __builtin_fminf(ds * fast_rcp(ax * sc), kMaxIv) * unit, iy = __builtin_fminf(ds * fast_rcp(ay * sc), kMaxIv) * unit,
        iz = __builtin_fminf(ds * fast_rcp(az * sc), kMaxIv) * unit;
  if (!(s < 1e27f)) ix = iy = iz = 0.0f;
  const float e = s < 1e27f ? __builtin_fmaf(kBoxSlack, s, 1e-36f) : 0.0f;   // (1e-36: products that underflow)
  r.iv = v3(d.x < 0 ? -ix : ix, d.y < 0 ? -iy : iy, d.z < 0 ? -iz : iz);
  const V3 oi = v3(-o.x * r.iv.x, -o.y * r.iv.y, -o.z * r.iv.z);
  r.cn = v3(oi.x - e * ix, oi.y - e * iy, oi.z - e * iz);
  r.cf = v3(oi.x + e * ix, oi.y + e * iy, oi.z + e * iz);
  return able;
}

// The test on one box in full precision (the root's).
DR_HD bool box_kept(const Box &b, const BoxRay &r) {
  const bool px = r.iv.x < 0, py = r.iv.y < 0, pz = r.iv.z < 0;
  const float nx = __builtin_fmaf(px ? b.e.x : b.s.x, r.iv.x, r.cn.x), fx = __builtin_fmaf(px ? b.s.x : b.e.x, r.iv.x, r.cf.x);
  const float ny = __builtin_fmaf(py ? b.e.y : b.s.y, r.iv.y, r.cn.y), fy = __builtin_fmaf(py ? b.s.y : b.e.y, r.iv.y, r.cf.y);
  const float nz = __builtin_fmaf(pz ? b.e.z : b.s.z, r.iv.z, r.cn.z), fz = __builtin_fmaf(pz ? b.s.z : b.e.z, r.iv.z, r.cf.z);
  return !(__builtin_fmaxf(max3(nx, ny, nz), 0.0f) > min3(fx, fy, fz));
}

// Byte k of the 8 in words lo, hi as a float.
DR_HD float cell_of(uint32_t lo, uint32_t hi, int k) {
  return (float)(((k < 4 ? lo : hi) >> (8 * (k & 3))) & 0xffu);
}

// The test on the 8 child boxes of a group: bit k is set if child k is kept.  w: the group's 12
// words of boxes.  Without a branch: per child six byte conversions, six fused products, two
// three-way extrema and two operations that shift its decision (the sign of far - near) into
// the mask.
DR_HD uint32_t group_children(V3 origin, V3 cell, const uint32_t w[12], const BoxRay &r) {
  const bool px = r.iv.x < 0, py = r.iv.y < 0, pz = r.iv.z < 0;
  // words of the near and the far planes per axis: the min side is near if the ray moves up
  const uint32_t nx0 = px ? w[6] : w[0], nx1 = px ? w[7] : w[1], fx0 = px ? w[0] : w[6], fx1 = px ? w[1] : w[7];
  const uint32_t ny0 = py ? w[8] : w[2], ny1 = py ? w[9] : w[3], fy0 = py ? w[2] : w[8], fy1 = py ? w[3] : w[9];
  const uint32_t nz0 = pz ? w[10] : w[4], nz1 = pz ? w[11] : w[5], fz0 = pz ? w[4] : w[10], fz1 = pz ? w[5] : w[11];
  const float sx = cell.x * r.iv.x, sy = cell.y * r.iv.y, sz = cell.z * r.iv.z;
  const float bnx = __builtin_fmaf(origin.x, r.iv.x, r.cn.x), bfx = __builtin_fmaf(origin.x, r.iv.x, r.cf.x);
  const float bny = __builtin_fmaf(origin.y, r.iv.y, r.cn.y), bfy = __builtin_fmaf(origin.y, r.iv.y, r.cf.y);
  const float bnz = __builtin_fmaf(origin.z, r.iv.z, r.cn.z), bfz = __builtin_fmaf(origin.z, r.iv.z, r.cf.z);
  uint32_t skip = 0;
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
#endif
  for (int k = 7; k >= 0; --k) {
    const float n = max3(unit_clamp(__builtin_fmaf(cell_of(nx0, nx1, k), sx, bnx)), __builtin_fmaf(cell_of(ny0, ny1, k), sy, bny),
                         __builtin_fmaf(cell_of(nz0, nz1, k), sz, bnz));
    const float f = min3(__builtin_fmaf(cell_of(fx0, fx1, k), sx, bfx), __builtin_fmaf(cell_of(fy0, fy1, k), sy, bfy),
                         __builtin_fmaf(cell_of(fz0, fz1, k), sz, bfz));
    const float gap = f - n;
#ifdef __HIP_DEVICE_COMPILE__
    skip = __builtin_amdgcn_alignbit(skip, (uint32_t)__float_as_int(gap), 31);   // skip << 1 | sign bit of gap
#else
    skip = (skip << 1) | (gap < 0.0f ? 1u : 0u);
#endif
  }
  return ~skip & 0xffu;
}

// Given that the exact slab test of box `b` passes: whether it then passes for every box that b
// lies inside.  Each of the test's operations is monotonic in the plane it takes, so the outer
// box's interval holds b's, unless a NaN enters: an axis with an infinite 1/d and o on a plane.
// Such an axis is clear if o lies strictly between b's planes (an outer plane is further out).
DR_HD bool slab_nests(const Box &b, V3 o, V3 inv) {
  const bool x = __builtin_isfinite(inv.x) || (b.s.x < o.x && o.x < b.e.x);
  const bool y = __builtin_isfinite(inv.y) || (b.s.y < o.y && o.y < b.e.y);
  const bool z = __builtin_isfinite(inv.z) || (b.s.z < o.z && o.z < b.e.z);
  return x && y && z;
}

// The exact slab tests of node `node` and of the nodes above it, the root's box included.
DR_HD bool ancestors_hit(const float4 *nodes, const Box &root, int node, V3 o, V3 inv) {
  while (node >= 0) {
    const float4 a = nodes[kNodeF4 * (size_t)node], b = nodes[kNodeF4 * (size_t)node + 1];
    if (!slab_hit(a.x, a.y, a.z, a.w, b.x, b.y, o, inv)) return false;
    node = bits_of(b.z);
  }
  return slab_hit(root.s.x, root.s.y, root.s.z, root.e.x, root.e.y, root.e.z, o, inv);
}

// Whether leaf node `leaf` (-1: the tree is one leaf) accepts the hit at p of the ray (o, d):
// castInLeaf's box test (Octree.impl.cuh:607-611), and the slab tests on the way to the leaf, its
// own and its ancestors'.  One 32-B record decides unless the leaf pokes out of an ancestor.
//
// A hit further than m = 16 u (M + O) inside a nested leaf's box on every axis is accepted at once
// (11 operations instead of the slab test's 90 with its three divisions): with d.k > 0, p = fl(o + fl(d t))
// misses o + d t by at most u (2 M + O), so (min - o) / d <= t - (m - u (2 M + O)) / |d|, and the slab
// test's two roundings and its 1 / d add at most 3 u (M + O) / |d|; so its min side is <= t, and its max
// side >= t by the same steps, on every axis: it passes, and by the argument of slab_nests so do the
// ancestors'.  A zero d.k leaves o.k = p.k strictly inside (sides of -inf and +inf).  Directions so
// short that 1 / d could overflow on an axis that moves take the long way.
DR_HD bool leaf_accepts(const float4 *nodes, const Box &root, float reach, int leaf, V3 o, V3 d, V3 p) {
  if (leaf < 0) return contains(root, p);
  const float4 a = nodes[kNodeF4 * (size_t)leaf], b = nodes[kNodeF4 * (size_t)leaf + 1];
  Box lb;
  lb.s = v3(a.x, a.y, a.z);
  lb.e = v3(a.w, b.x, b.y);
  const V3 ad = v3(__builtin_fabsf(d.x), __builtin_fabsf(d.y), __builtin_fabsf(d.z));
  const float m = __builtin_fmaf(kBoxSlack, reach + max3(__builtin_fabsf(o.x), __builtin_fabsf(o.y), __builtin_fabsf(o.z)), 1e-36f);
  const float deep = __builtin_fminf(min3(p.x - lb.s.x, p.y - lb.s.y, p.z - lb.s.z), min3(lb.e.x - p.x, lb.e.y - p.y, lb.e.z - p.z));
  const bool shortest = min3(ad.x > 0 ? ad.x : 1.0f, ad.y > 0 ? ad.y : 1.0f, ad.z > 0 ? ad.z : 1.0f) > 1e-30f;
  if (deep > m && shortest && bits_of(b.w) != 0) return true;
  if (!contains(lb, p)) return false;
  const V3 inv = v3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
  if (!slab_hit(lb.s.x, lb.s.y, lb.s.z, lb.e.x, lb.e.y, lb.e.z, o, inv)) return false;
  if (bits_of(b.w) != 0 && slab_nests(lb, o, inv)) return true;
  return ancestors_hit(nodes, root, bits_of(b.z), o, inv);
}

}  // namespace dr
