// Device-side octree closest-hit traversal (Octree::cast, Octree.impl.cuh:174-212,
// castInLeaf :584-612, Triangle::cast Triangle.impl.h:334-348) over the
// structure-of-arrays group layout built by flatten_octree().
//
// Order of work is the reference's: children of an expanded node are visited
// in the order canonical ^ i (i = 0..7), a leaf that accepts a hit ends the
// cast, and inside a leaf the first triangle with the strictly smallest t wins.
// Which subtrees are skipped is decided by a conservative test on compact child
// boxes (dr_group.h): it never skips one that holds a leaf able to accept a hit.
// Whether the reference would have reached the leaf at all (its slab tests on the
// leaf's box and on those of its ancestors) is decided exactly when a hit is about to
// be accepted, so the walk visits a superset of the reference's leaves in the
// reference's order and accepts the same first hit.
#pragma once
#include "dr_geom.h"
#include "dr_group.h"
#include "dr_octree_build.h"

namespace dr {

struct DevTree {
  const float4 *__restrict__ groups;   // kGroupF4 float4 per group
  const float4 *__restrict__ nodes;    // kNodeF4 float4 per node below the root
  const float4 *__restrict__ recs;     // 4 float4 per triangle record, one per leaf entry
  const float4 *__restrict__ urecs;    // the same records once per distinct triangle
  const int *__restrict__ lref;        // leaf entry -> record in urecs
  float rsx, rsy, rsz, rex, rey, rez;  // root box
  int root_is_leaf, root_start, root_count;
  float reach;                         // largest magnitude of a box coordinate
};

__device__ __forceinline__ Box root_box(const DevTree &T) {
  Box b;
  b.s = v3(T.rsx, T.rsy, T.rsz);
  b.e = v3(T.rex, T.rey, T.rez);
  return b;
}

struct Hit {
  int id;        // -1 miss
  float t;
  V3 p;
};

// Work counters of one cast (measurement launches only; nullptr elsewhere).
struct CastCounters {
  int expand;    // groups expanded (80-B reads: grid, head and 8 child boxes)
  int leaves;    // leaves whose triangles were tested (+ the 8-B read of their entries)
  int plane;     // triangle records whose plane test ran (first 32 B)
  int inside;    // records that reached the inside test (second 32 B)
  int live;      // children of expanded groups with a non-empty leaf below
  int slab;      // children that the box test kept
};

// One edge of Triangle::containsVertex (Triangle.impl.h:299-301): fl(fl(D / fl(sqrt(S))) + tol) >= thr
// with D = dot(edge, p - vertex), S = dot(p - vertex, p - vertex), correctly rounded division
// and square root.
__device__ __forceinline__ bool edge_exact(float D, float S, float thr) {
  return D / __builtin_sqrtf(S) + kInsideTol >= thr;
}
// The same decision from the hardware reciprocal square root where it is certain.
// q = D * rsq(S) is within about 2 ulp of the correctly
// rounded quotient (rsq within 1 ulp, one product rounding, the quotient's two roundings), and
// the sum with tol adds at most one ulp more.  An edge is decided only when q + tol lies more
// than kEdgeMargin * (|q| + tol), about 34 ulp, from thr; S outside [1e-30, 1e30] (where
// denormals or overflow could enter) is left to the exact form.
// hi and lo are the left side's upper and lower bound less thr (a difference of fp32 values has
// the sign of the comparison): lo >= 0 passes, hi < 0 fails.
constexpr float kEdgeMargin = 4e-6f;
__device__ __forceinline__ void edge_bounds(float D, float S, float thr, float &lo, float &hi) {
  const float q = D * __builtin_amdgcn_rsqf(S);
  const float r = q + kInsideTol;
  const float m = kEdgeMargin * (__builtin_fabsf(q) + kInsideTol);
  lo = (r - m) - thr;
  hi = (r + m) - thr;
}

// Triangle::containsVertex minus the degenerate test (degenerate triangles have no record).
// The three edge conditions are ANDed; they are decided by edge_bounds where it is certain and by
// the exact form otherwise, so the result is the reference's bit for bit.  p equals a vertex
// (inside by definition) only if that vertex's S is 0, which the range of S leaves to the exact form.
__device__ __forceinline__ bool inside(V3 p, V3 a, V3 b, V3 c, float thr0, float thr1, float thr2) {
  const V3 ab = b - a, bc = c - b, ca = a - c;
  const V3 ax = p - a, bx = p - b, cx = p - c;
  const float D0 = dot(ab, ax), S0 = dot(ax, ax), D1 = dot(bc, bx), S1 = dot(bx, bx), D2 = dot(ca, cx),
              S2 = dot(cx, cx);
  float l0, l1, l2, h0, h1, h2;
  edge_bounds(D0, S0, thr0, l0, h0);
  edge_bounds(D1, S1, thr1, l1, h1);
  edge_bounds(D2, S2, thr2, l2, h2);
  if (min3(S0, S1, S2) >= 1e-30f && max3(S0, S1, S2) <= 1e30f) {
    if (min3(h0, h1, h2) < 0.0f) return false;
    if (l0 >= 0.0f && l1 >= 0.0f && l2 >= 0.0f) return true;   // (three tests: a NaN must not pass)
  } else if (eq(p, a) || eq(p, b) || eq(p, c)) {
    return true;
  }
  return edge_exact(D0, S0, thr0) && edge_exact(D1, S1, thr1) && edge_exact(D2, S2, thr2);
}

// Traversal stack: per level and lane two words, read and written together,
//   x = group << 8 | mask of children still to visit (bit i = child canon ^ i)
//   y = first interior child's group << 8 | interior mask (bit k = child k)
// so popping an interior child needs no memory read.  A level is on the stack only while it has
// children to visit: the last child's pop takes it off, and a group with none is not pushed, so a
// step never searches for work and a walk ends in the step that runs out of it.  (With empty
// levels left on the stack, each pop looped over LDS reads with part of the wave: 1080p 16 spp
// 19.9 -> 18.4 ms, 99,991 bounce rays 280 -> 245 us, the 256x256 frame 503 -> 462 us with the
// fused planes of dr_group.h.)
constexpr int kStackWordsPerLevel = 2;

// The children of group g to visit -> stack entry: those with a non-empty leaf below them that
// the box test keeps, in visiting order.
__device__ __forceinline__ void group_entry(const float4 *__restrict__ G, int g, const BoxRay &r, uint32_t &lo,
                                            uint32_t &hi, CastCounters *cc = nullptr) {
  const float4 *q = G + kGroupF4 * (size_t)g;
  const float4 grid = q[0], cell = q[1], b0 = q[2], b1 = q[3], b2 = q[4];
  const uint32_t head = (uint32_t)__float_as_int(grid.w), base = (uint32_t)__float_as_int(cell.w);
  const uint32_t w[12] = {(uint32_t)__float_as_int(b0.x), (uint32_t)__float_as_int(b0.y), (uint32_t)__float_as_int(b0.z),
                          (uint32_t)__float_as_int(b0.w), (uint32_t)__float_as_int(b1.x), (uint32_t)__float_as_int(b1.y),
                          (uint32_t)__float_as_int(b1.z), (uint32_t)__float_as_int(b1.w), (uint32_t)__float_as_int(b2.x),
                          (uint32_t)__float_as_int(b2.y), (uint32_t)__float_as_int(b2.z), (uint32_t)__float_as_int(b2.w)};
  uint32_t m = group_children(v3(grid.x, grid.y, grid.z), v3(cell.x, cell.y, cell.z), w, r) & head & 0xffu;
  if (cc) { cc->live += __builtin_popcount(head & 0xffu); cc->slab += __builtin_popcount(m); }
  // bit k to bit k ^ canon: per set bit of canon the pairs that far apart trade places (a shift of 0
  // trades nothing)
  const uint32_t c1 = r.canon & 1, c2 = r.canon & 2, c4 = r.canon & 4;
  uint32_t t = (m ^ (m >> c1)) & 0x55u;
  m ^= t ^ (t << c1);
  t = (m ^ (m >> c2)) & 0x33u;
  m ^= t ^ (t << c2);
  t = (m ^ (m >> c4)) & 0x0fu;
  m ^= t ^ (t << c4);
  lo = ((uint32_t)g << 8) | m;
  hi = (base << 8) | ((head >> 8) & 0xffu);
}

// One lane's closest-hit query, advanced in bounded steps so that a kernel can
// interleave many of them (and batch their leaf tests) across a wave.  kWalkIdle is the kernel's: a lane
// without work.  With it in the state, a ballot over lanes to trace, to test, to finish or to refill is
// one comparison; of two conditions it was three instructions, in five places of every iteration.
enum : int { kWalkIdle = 0, kWalkTrace = 1, kWalkLeaf = 2, kWalkDone = 3 };
constexpr int kNoLeaf = -2;
struct Walk {
  V3 o, d;
  BoxRay box;
  int ex;              // validateNotSameAsObject's object, or -1
  int sp, state;
  int leaf, llink, lend;   // held leaf: its node (-1: the root, kNoLeaf: none held), first leaf entry and their end
  bool hit;            // result once state == kWalkDone
  Hit h;
};

__device__ __forceinline__ void walk_begin(const DevTree &T, Walk &w, V3 o, V3 d, int exclude, uint2 *stk) {
  w.o = o;
  w.d = d;
  w.ex = exclude;
  w.hit = false;
  w.sp = -1;
  w.leaf = kNoLeaf;
  if (T.root_is_leaf) {
    w.leaf = -1;
    w.llink = T.root_start;
    w.lend = T.root_start + T.root_count;
    w.state = kWalkLeaf;
    return;
  }
  const bool alive = box_ray(o, d, T.reach, w.box) && box_kept(root_box(T), w.box);
  w.state = alive ? kWalkTrace : kWalkDone;
  // a level whose one child is group 0: the root's group is expanded by the walk's first step, with
  // the expansions of the other lanes, rather than in the divergent code that hands out work
  w.sp = 0;
  stk[0] = make_uint2(1u, 1u << w.box.canon);
}

// Pops one child: expands an interior child, or holds a leaf child until the wave's next leaf batch.
// A lane that holds a leaf walks on: the children after it are expanded as if the leaf held no hit,
// and the lane waits (kWalkLeaf) only at its next leaf, which stays on the stack, or at the walk's end.
// Lanes waiting for a batch were idle in the expansions, most of the work; a batch's leaves are those of
// the waiting and of the walking lanes.  The next child is popped in the same step: a lane that only took
// its leaf sat out the expansion (that form: 1080p 16 spp 16.2 ms against 15.9 without walking on).
// Measured, before -> after: 1080p 16 spp 14.00 -> 13.28 ms, 512x512 adjoint 6.10 -> 5.87 ms, 99,991
// bounce rays 184 -> 174 us, 1080p primary rays 743 -> 731 us, batch of 24 5.78 -> 5.50 ms; 4M
// incoherent rays, whose waves wait for memory, 1.218 -> 1.215 ms.
__device__ __forceinline__ void walk_step(const DevTree &T, Walk &w, uint2 *stk, int stride, CastCounters *cc) {
  uint2 f = stk[w.sp * stride];
  int k = w.box.canon ^ __builtin_ctz(f.x);
  if (!((f.y >> k) & 1u) && w.leaf == kNoLeaf) {
    const int *E = (const int *)T.groups + kGroupWords * (size_t)(f.x >> 8) + kGroupEntry + k;
    w.leaf = (int)(f.x >> 8) * 8 + k;
    w.llink = E[0];
    w.lend = E[1];
    const uint32_t rest = f.x & (f.x - 1);
    stk[w.sp * stride].x = rest;
    w.sp -= (rest & 0xffu) ? 0 : 1;
    // (a measurement launch counts the work of a walk that waits at every leaf)
    if (cc || w.sp < 0) { w.state = kWalkLeaf; return; }
    f = stk[w.sp * stride];
    k = w.box.canon ^ __builtin_ctz(f.x);
  }
  const uint32_t im = f.y & 0xffu;
  if (!((im >> k) & 1u)) { w.state = kWalkLeaf; return; }
  const uint32_t rest = f.x & (f.x - 1);
  stk[w.sp * stride].x = rest;
  w.sp -= (rest & 0xffu) ? 0 : 1;
  const int child = (int)(f.y >> 8) + __builtin_popcount(im & ((1u << k) - 1u));
  uint2 e;
  group_entry(T.groups, child, w.box, e.x, e.y, cc);
  if (cc) cc->expand++;
  // Stored whether it has children or not (there is a level for it: the group's own depth).  With a
  // branch around the store the compiler moved the load of the group's second word into it, a second
  // round trip to memory in every step (with the ballots over states: 1080p 16 spp 15.14 -> 14.00 ms,
  // 1080p primary rays 785 -> 743 us, 512x512 adjoint 6.40 -> 6.10 ms).
  stk[(w.sp + 1) * stride] = e;
  w.sp += (e.x & 0xffu) ? 1 : 0;
  if (w.sp < 0) w.state = w.leaf != kNoLeaf ? kWalkLeaf : kWalkDone;
}

// Inclusive prefix sum and maximum over the 64 lanes of the wave (every lane active): DPP row
// shifts by 1, 2, 4 and 8 scan each row of 16 lanes, then lane 15 of rows 0 and 2 is added to
// the row after it and lane 31 to the upper half (a lane without a source takes 0).
template <int kCtrl, int kRows = 0xf>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t v) {   // (the compiler folds it into the sum or maximum)
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, kRows, 0xf, kRows == 0xf);
}
__device__ __forceinline__ int wave_incl_scan(int count, int &total) {
  uint32_t v = (uint32_t)count;
  v += dpp_or_zero<0x111>(v);        // row_shr:1
  v += dpp_or_zero<0x112>(v);        // row_shr:2
  v += dpp_or_zero<0x114>(v);        // row_shr:4
  v += dpp_or_zero<0x118>(v);        // row_shr:8
  v += dpp_or_zero<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
  v += dpp_or_zero<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
  total = __builtin_amdgcn_readlane((int)v, 63);
  return (int)v;
}
__device__ __forceinline__ int wave_incl_max(int x) {   // x >= 0
  uint32_t v = (uint32_t)x;
  v = max(v, dpp_or_zero<0x111>(v));
  v = max(v, dpp_or_zero<0x112>(v));
  v = max(v, dpp_or_zero<0x114>(v));
  v = max(v, dpp_or_zero<0x118>(v));
  v = max(v, dpp_or_zero<0x142, 0xa>(v));
  v = max(v, dpp_or_zero<0x143, 0xc>(v));
  return (int)v;
}

// One wave's LDS for walk_leaf_wave.
struct LeafLds {
  unsigned long long best[64];   // per lane: the smallest key of its leaf
  unsigned char first[64];       // per record of a round: the lane whose leaf starts there; 0 between calls
};
__device__ __forceinline__ void leaf_lds_init(LeafLds &L) { L.first[__lane_id()] = 0; }

// castInLeaf for every pending lane of the wave at once, with all 64 lanes sharing
// the records.  Must be called by every lane of the wave (wave-uniform control flow);
// `pending` marks the lanes whose leaf is tested; `lds` is the wave's own
// (and `ins`, counting the records that reach the inside test, for measurement launches).
//   * The records of the pending leaves are numbered 0..total-1 in lane order (wave
//     prefix sum of the counts); lane j tests records j, j + 64, ...
//   * A record's owner is the last lane whose first record number is <= the record's: the
//     lanes whose leaf starts in a round leave their number at that place in LDS, and a
//     prefix maximum spreads it; its ray, exclusion and first record come from the owner
//     with __shfl.  (Renders are bound by vector instructions: counting the prefix sums <=
//     the record's in two levels took 45 vector and 7 LDS instructions of a round's 330,
//     this takes 12 and 3.  With the shorter inside() above, 1080p 16 spp 21.2 -> 19.7 ms, the
//     256x256 frame 586 -> 501 us, 4M incoherent rays 1.30 -> 1.28 ms.)
//   * A record that passes Triangle::cast with t < FLT_MAX offers the 64-bit key
//     (t bits << 32 | leaf entry) to the owner's slot in `best`
//     (LDS, one uint64 per lane) with an atomic min.  t > 0, so the keys order by t
//     first and by position second: the owner gets the first record with the smallest
//     t, which is what the sequential strict '<' scan keeps (Octree.impl.cuh:595-606).
//   * The owner then applies the leaf-box acceptance.
// kIndexed: read the records through lref from urecs (a third of the footprint on
// scenes whose triangles sit in several leaves; one more dependent load per record, issued
// one round ahead).
// The next round's owners and record indices are found during the current round (incoherent
// cast 2.31 -> 2.12 ms with the lref read ahead; 1080p render 25.6 -> 24.1 ms and the
// 64-request batch 247 -> 228 ms with the owner search ahead).
template <bool kIndexed = false>
__device__ __forceinline__ void walk_leaf_wave(const DevTree &T, Walk &w, bool pending, bool clip, LeafLds &lds,
                                               int *ins, CastCounters *cc) {
  const int lane = (int)__lane_id();
  const int cnt = pending ? w.lend - w.llink : 0;
  int total;
  const int incl = wave_incl_scan(cnt, total);
  const int start = incl - cnt;
  auto put = [](auto *p, auto v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT); };
  auto get = [](auto *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT); };
  if (pending) put(&lds.best[lane], ~0ull);
  if (cc && pending) put(&ins[lane], 0);
  const int link = (pending ? w.llink : 0) - start;      // leaf entry of record j: link + j
  // owner of record base + lane (wave-uniform call; one call per round, in order)
  int last = 0;                                          // the previous round's last owner
  auto owner_of = [&](int base) {
    const bool here = cnt > 0 && (unsigned)(start - base) < 64u;
    if (here) put(&lds.first[start - base], (unsigned char)lane);
    const int v = max(wave_incl_max((int)get(&lds.first[lane])), last);
    if (here) put(&lds.first[start - base], (unsigned char)0);
    last = __builtin_amdgcn_readlane(v, 63);
    return v;
  };
  // tests record j (of owner `owner`; its 64 B in r0..r3) for its owner; every lane takes part
  auto test_record = [&](int j, int owner, int entry, float4 r0, float4 r1, float4 r2, float4 r3) {
    const V3 o = v3(__shfl(w.o.x, owner), __shfl(w.o.y, owner), __shfl(w.o.z, owner));
    const V3 d = v3(__shfl(w.d.x, owner), __shfl(w.d.y, owner), __shfl(w.d.z, owner));
    const int ex = __shfl(w.ex, owner);
    if (j < total) {
      const V3 a = v3(r0.x, r0.y, r0.z), n = v3(r0.w, r1.x, r1.y);
      const float dp = dot(a - o, n);
      const float dd = dot(d, n);
      const float t = dp / dd;
      if (!(clip && (dp < -kVecEps)) && !(dp * dd <= 0) && (t < FLT_MAX)) {
        if (cc) __hip_atomic_fetch_add(&ins[owner], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        if (__float_as_int(r3.w) != ex) {
          const V3 p = o + d * t;
          const V3 b = v3(r1.z, r1.w, r2.x), c = v3(r2.y, r2.z, r2.w);
          if (inside(p, a, b, c, r3.x, r3.y, r3.z)) {
            const unsigned long long key =
                ((unsigned long long)__float_as_uint(t) << 32) | (unsigned long long)(unsigned)entry;
            __hip_atomic_fetch_min(&lds.best[owner], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
          }
        }
      }
    }
  };
  // The index of a lane's record in the next round (its owner, and with kIndexed the lref entry)
  // is found while the current round's records are fetched and tested, so a round's record
  // loads start at once.
  const float4 *R = kIndexed ? T.urecs : T.recs;
  int own = owner_of(0);
  int el = __shfl(link, own) + lane;                     // every lane takes part
  int kn = 0;
  if (lane < total) kn = kIndexed ? T.lref[el] : el;
  for (int base = 0; base < total; base += 64) {
    const int j = base + lane;
    const int owner = own, entry = el;
    const int k = j < total ? kn : 0;      // (lanes past the last record read record 0)
    const float4 r0 = R[4 * k + 0], r1 = R[4 * k + 1], r2 = R[4 * k + 2], r3 = R[4 * k + 3];
    if (base + 64 < total) {
      own = owner_of(base + 64);
      el = __shfl(link, own) + j + 64;
      if (j + 64 < total) kn = kIndexed ? T.lref[el] : el;
    }
    test_record(j, owner, entry, r0, r1, r2, r3);
  }
  if (!pending) return;
  if (cc) {
    cc->leaves++;
    cc->plane += cnt;
    cc->inside += __hip_atomic_load(&ins[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  }
  const unsigned long long key = get(&lds.best[lane]);
  bool hit = false;
  if (key != ~0ull) {
    const float t = __uint_as_float((unsigned)(key >> 32));
    const int k = (int)(key & 0xffffffffu);
    const V3 p = w.o + w.d * t;
    // the record's id is read beside the leaf box, before the box test that decides whether
    // it is needed
    const int rid = kIndexed ? __float_as_int(T.urecs[4 * T.lref[k] + 3].w) : __float_as_int(T.recs[4 * k + 3].w);
    if (leaf_accepts(T.nodes, root_box(T), T.reach, w.leaf, w.o, w.d, p)) {
      hit = true;
      w.h.id = rid;
      w.h.t = t;
      w.h.p = p;
    }
  }
  w.hit = hit;
  w.leaf = kNoLeaf;
  w.state = (hit || w.sp < 0) ? kWalkDone : kWalkTrace;
}

}  // namespace dr
