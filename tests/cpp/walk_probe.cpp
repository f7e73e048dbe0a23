// The traversal's skip and accept rules (dr_group.h) on the host, against the reference's walk.
// tests/test_walk_host.py builds it with the host octree builder and runs every mode.
//
// Both walks share the triangle test.  `reference` visits the nodes of the built octree as
// Octree::cast does (exact slab test of every child on the way); `compact` walks the flattened
// groups with group_children and decides acceptance with leaf_accepts, as the kernels do.  They
// must agree on the triangle and on every bit of t for every ray.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>
#include "dr_group.h"

using namespace dr;

namespace {

struct Result { int id = -1; float t = FLT_MAX; };

bool edge_ok(V3 e, V3 x, float thr) { return dot(e, x) / mag(x) + kInsideTol >= thr; }

// Triangle::cast without backface clipping; t >= 0 or false
bool tri_hit(const Tri &t, V3 o, V3 d, float &dist, V3 &p) {
  if (eq(t.a, t.b) || eq(t.b, t.c) || eq(t.c, t.a)) return false;
  const TriPre pre = tri_pre(t);
  const float dp = dot(t.a - o, pre.n), dd = dot(d, pre.n);
  if (dp * dd <= 0) return false;
  dist = dp / dd;
  if (!(dist < FLT_MAX)) return false;
  p = o + d * dist;
  if (eq(p, t.a) || eq(p, t.b) || eq(p, t.c)) return true;
  return edge_ok(t.b - t.a, p - t.a, pre.thr0) && edge_ok(t.c - t.b, p - t.b, pre.thr1) &&
         edge_ok(t.a - t.c, p - t.c, pre.thr2);
}

int canonical(V3 d) { return (d.z < 0 ? 1 : 0) + (d.y < 0 ? 2 : 0) + (d.x < 0 ? 4 : 0); }

bool reference(const OctreeHost &h, int node, V3 o, V3 d, V3 inv, Result &r, bool is_root) {
  const Box &b = h.bounds[node];
  if (h.children[node] < 0) {
    float best = FLT_MAX;
    int id = -1;
    V3 bp = v3(0, 0, 0);
    for (int k = h.list_off[node]; k < h.list_off[node + 1]; k++) {
      float t;
      V3 p;
      if (tri_hit(h.tris[h.list[k]], o, d, t, p) && t < best) { best = t; id = h.list[k]; bp = p; }
    }
    if (id < 0 || !contains(b, bp)) return false;
    r.id = id;
    r.t = best;
    return true;
  }
  if (is_root && !slab_hit(b.s.x, b.s.y, b.s.z, b.e.x, b.e.y, b.e.z, o, inv)) return false;
  for (int i = 0; i < 8; i++) {
    const int c = h.children[node] + (canonical(d) ^ i);
    const Box &q = h.bounds[c];
    if (!slab_hit(q.s.x, q.s.y, q.s.z, q.e.x, q.e.y, q.e.z, o, inv)) continue;
    if (reference(h, c, o, d, inv, r, false)) return true;
  }
  return false;
}

struct Counts { long long groups = 0, chains = 0; };

bool compact(const OctreeFlat &f, const std::vector<Tri> &tris, int g, V3 o, V3 d, const BoxRay &ray, Result &r, Counts &n) {
  const float *G = &f.groups[(size_t)g * kGroupWords];
  uint32_t w[12];
  memcpy(w, G + kGroupBoxes, sizeof(w));
  const uint32_t head = (uint32_t)bits_of(G[kGroupHead]), interior = (head >> 8) & 0xffu;
  const uint32_t kept = group_children(v3(G[0], G[1], G[2]), v3(G[4], G[5], G[6]), w, ray) & head & 0xffu;
  n.groups++;
  for (int i = 0; i < 8; i++) {
    const int k = ray.canon ^ i;
    if (!((kept >> k) & 1u)) continue;
    if ((interior >> k) & 1u) {
      if (compact(f, tris, bits_of(G[kGroupBase]) + __builtin_popcount(interior & ((1u << k) - 1u)), o, d, ray, r, n)) return true;
      continue;
    }
    float best = FLT_MAX;
    int id = -1;
    V3 bp = v3(0, 0, 0);
    for (int e = bits_of(G[kGroupEntry + k]); e < bits_of(G[kGroupEntry + k + 1]); e++) {
      const int tri = bits_of(f.recs[(size_t)e * kRecWords + 15]);
      float t;
      V3 p;
      if (tri_hit(tris[tri], o, d, t, p) && t < best) { best = t; id = tri; bp = p; }
    }
    const float4 *nodes = (const float4 *)f.nodes.data();
    if (id >= 0 && leaf_accepts(nodes, f.root, f.reach, 8 * g + k, o, d, bp)) {
      if (bits_of(f.nodes[(size_t)(8 * g + k) * kNodeWords + 7]) == 0) n.chains++;
      r.id = id;
      r.t = best;
      return true;
    }
  }
  return false;
}

}  // namespace

// walk_probe TRIS.bin RAYS.bin SPLIT DEPTH: prints "ok rays hits groups chains", or the first rays that differ
int main(int argc, char **argv) {
  if (argc != 5) return 2;
  auto load = [](const char *path, std::vector<float> &v) {
    FILE *f = std::fopen(path, "rb");
    if (!f) return false;
    std::fseek(f, 0, SEEK_END);
    v.resize((size_t)std::ftell(f) / 4);
    std::fseek(f, 0, SEEK_SET);
    const bool ok = std::fread(v.data(), 4, v.size(), f) == v.size();
    std::fclose(f);
    return ok;
  };
  std::vector<float> t, rays;
  if (!load(argv[1], t) || !load(argv[2], rays)) return 2;
  OctreeHost h;
  OctreeFlat f;
  if (build_octree(t.data(), (int)(t.size() / 9), std::atoi(argv[3]), std::atoi(argv[4]), 4, h) != 0) return 2;
  if (flatten_octree(h, f) != 0 || f.root_is_leaf) return 2;
  Counts n;
  int bad = 0;
  long long hits = 0;
  for (size_t i = 0; i + 6 <= rays.size(); i += 6) {
    const V3 o = v3(rays[i], rays[i + 1], rays[i + 2]), d = v3(rays[i + 3], rays[i + 4], rays[i + 5]);
    Result a, b;
    reference(h, 0, o, d, v3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z), a, true);
    BoxRay r;
    if (box_ray(o, d, f.reach, r) && box_kept(f.root, r)) compact(f, h.tris, 0, o, d, r, b, n);
    hits += a.id >= 0;
    if (a.id != b.id || memcmp(&a.t, &b.t, 4) != 0) {
      if (bad++ < 5)
        std::printf("ray %zu (%a %a %a) (%a %a %a): reference %d %a, compact %d %a\n", i / 6, o.x, o.y, o.z, d.x, d.y,
                    d.z, a.id, a.t, b.id, b.t);
    }
  }
  if (bad) { std::printf("%d rays differ\n", bad); return 1; }
  std::printf("ok %zu %lld %lld %lld\n", rays.size() / 6, hits, n.groups, n.chains);
  return 0;
}
