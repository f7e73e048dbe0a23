// Path tracing: DumbRenderer::renderBlocksGPU and Renderer::backward on gfx950.
//
// The work of a render is a list of path jobs (pixel, sample) per 8x16 framebuffer
// block; idle lanes take the next jobs with a wave64 ballot + mbcnt prefix and one LDS
// atomic per wave, so lanes whose path ended early are regenerated instead of idling.
// Each lane's current ray (camera/bounce ray or light photon) is a Walk advanced by one
// node pop per loop iteration; leaf tests and the path updates of finished casts run
// once enough lanes of the wave need them, which keeps the wave's lanes in step.
// Finished sample colours are staged in LDS and summed per pixel in the reference's
// subpixel order before the pixel is written (set, or blended with 1/iteration).
// k_render_stream runs the jobs of many blocks as one stream per persistent workgroup;
// render_block (k_render, k_batch) runs one block per workgroup at a time.
#include "dr_common.h"
#include "dr_plugins.h"
#include "dr_shade.h"

#include <algorithm>
#include <cmath>
#include <new>
#include <type_traits>
#include <vector>

namespace dr {

constexpr int kRB = 256;               // lanes per workgroup
constexpr int kLdsBytes = 160 * 1024;  // LDS of a CU
constexpr int kRoundSamples = 16;      // samples per pixel staged in LDS per round
constexpr int kBlockPixels = 128;      // BlockBasedFrameBuffer<8,16>
constexpr int kLeafMin = 16;           // pending leaves that trigger the (wave-shared) leaf tests
constexpr int kShadeMin = 32;          // finished casts of a busy wave that trigger the adjoint's path updates
constexpr int kAdjointRefillMin = 4;   // idle lanes that pop the adjoint's queue
// Waves per SIMD the render kernels are compiled for.  The register cap this sets (168 VGPRs) costs
// k_render_stream<BenchPath> and k_backward no vector register, k_render_stream<RefPath> 12 B of scratch a
// lane and k_batch_stream 12 and 28 B; 2 waves a SIMD were slower by a third (46.4 / 34.9 ms on an
// earlier 1080p frame).
constexpr int kRenderWaves = 3;

// Per-lane path state.
struct Path {
  uint32_t pix = 0, samp = 0;
  int layer = 0, phase = 0, light = 0;  // phase 0: geometry ray, 1: light photon
  V3 o, d;
  int restrict_tri = -1;
  float beta[3], L[3];
  int h = -1, kind = 0, mid = 0;
  V3 p, nu;
  bool has_sample = false;
  V3 sdir;
  float sweight = 0.0f;
  float contrib[3];                     // photon contribution if lit
  float gl_k = 0.0f;                    // (adjoint) cos_i/pi * cos_l*A/d^2 of the pending photon
};

// A value that is the same in every lane (a function of the kernel's parameters), moved to
// a scalar register.  Call with every lane that holds it agreeing on it.
__device__ __forceinline__ float uni(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ UDiv uni(UDiv D) { return {uni(D.d), uni(D.m)}; }
__device__ __forceinline__ UDiv udiv_uniform(uint32_t d) { return uni(make_udiv(d)); }

// The first ray of a path: sample `samp` of pixel `pix`, kNoPixel for a pixel outside the image.
constexpr uint32_t kNoPixel = 0xffffffffu;
struct PathStart {
  uint32_t pix, samp;
  V3 o, d;
};

// Job start: camera ray of sample `s` of pixel `lp` of block `block`.
__device__ __forceinline__ PathStart path_start(const dr_render_params &P, const FrameK &K, int block, int lp, int s,
                                                uint32_t samp0) {
  PathStart ps;
  int x, y;
  ps.pix = kNoPixel;
  ps.samp = samp0 + (uint32_t)s;
  ps.o = ps.d = v3(0.0f, 0.0f, 0.0f);
  if (!block_pixel(K, P.width, P.height, block, lp, x, y)) return ps;
  ps.pix = (uint32_t)y * (uint32_t)P.width + (uint32_t)x;
  const int i = (int)udiv((uint32_t)s, K.fy), j = s - i * P.fsaa_y;
  float u[4];
  rng4(P, ps.pix, ps.samp, 0, 0, u);
  camera_ray(P, K, x, y, i, j, u[0], u[1], u[2], u[3], ps.o, ps.d);
  return ps;
}
__device__ __forceinline__ void begin_path(Path &st, const PathStart &s) {
  st.pix = s.pix;
  st.samp = s.samp;
  st.o = s.o;
  st.d = s.d;
  st.layer = 0;
  st.phase = 0;
  st.restrict_tri = -1;
  for (int c = 0; c < 3; c++) { st.beta[c] = 1.0f; st.L[c] = 0.0f; }
}
// Starts the job's path, or returns false (and leaves the lane idle) for a pixel outside the image.
__device__ __forceinline__ bool start_path(const dr_render_params &P, const FrameK &K, int block, int lp, int s,
                                           uint32_t samp0, Path &st) {
  const PathStart ps = path_start(P, K, block, lp, s, samp0);
  if (ps.pix == kNoPixel) return false;
  begin_path(st, ps);
  return true;
}

// Sets up the next light photon of the current vertex (phase 1), or returns false.
__device__ __forceinline__ bool next_photon(const dr_render_params &P, Path &st, float *cinfo = nullptr) {
  for (int l = st.light + 1; l < P.nlights; l++) {
    const dr_light Lt = P.lights[l];
    V3 q, w;
    float cos_i, gl;
    if (!light_photon(P, Lt, l, st.pix, st.samp, st.layer, st.p, st.nu, q, w, cos_i, gl)) continue;
    const dr_material M = P.materials[st.mid];
    const float k = cos_i * kInvPi;
    for (int c = 0; c < 3; c++) st.contrib[c] = st.beta[c] * ((M.albedo[c] * k) * (Lt.emission[c] * gl));
    st.gl_k = k * gl;
    st.light = l;
    st.phase = 1;
    st.o = q;
    st.d = w;
    st.restrict_tri = -1;
    return true;
  }
  return false;
}

// Vertex setup after a geometry hit of the ray with direction `dir`.
__device__ __forceinline__ void setup_vertex(const dr_render_params &P, const FrameK &K, const float4 *__restrict__ shade,
                                             const Hit &hh, V3 dir, Path &st) {
  st.h = hh.id;
  st.p = hh.p;
  const float4 sh = shade[hh.id];
  st.mid = __float_as_int(sh.w);
  st.kind = P.materials[st.mid].kind;
  const V3 du = normalized(dir);
  st.nu = facing_normal(v3(sh.x, sh.y, sh.z), du);
  st.has_sample = next_sample(P, K, st.kind, st.pix, st.samp, st.layer, st.nu, du, st.sdir, st.sweight);
  st.light = -1;
}

// Reflection factor A of the current vertex for its sampled direction.
__device__ __forceinline__ void reflect_factor(const dr_render_params &P, const Path &st, float A[3]) {
  const dr_material M = P.materials[st.mid];
  if (st.kind == DR_METAL) {
    const float f5 = schlick5(st.nu, st.sdir);
    for (int c = 0; c < 3; c++) A[c] = M.albedo[c] + (1.0f - M.albedo[c]) * f5;
  } else {
    for (int c = 0; c < 3; c++) A[c] = M.albedo[c];
  }
}

// Shading tables of one scene.
struct Tables {
  const float4 *shade;   // per triangle: (unit normal, material id bits)
  const float *faces;    // per triangle: kFaceWords floats (vertices, vertex normals)
};

// What a stream reads throughout, where it lies in constant memory: the first argument of
// k_render_stream, part of a batch's request.
struct RenderArgs {
  DevTree T;
  Tables tb;
  dr_render_params P;
  FrameK K;
};
typedef const __attribute__((address_space(4))) RenderArgs *ConstArgs;
// The arguments, to be read anew by what follows.  Kernel arguments are loaded once and kept in scalar
// registers; these are more than there are, and what does not fit went to lanes of vector registers:
// 559 of the 2,791 vector instructions of k_render_stream<BenchPath> moved scalars back, 15 do now
// (1080p 16 spp 15.60 -> 15.14 ms, reference plugins 1080p 3.11 -> 2.96 ms).
__device__ __forceinline__ const RenderArgs &again(ConstArgs A) {
  asm volatile("" : "+s"(A));
  return *(const RenderArgs *)A;
}

// Path updates of the benchmark plugins (DR_PLUGINS_BENCHMARK).
struct BenchPath {
  // render_block: finished casts that trigger the path updates, idle lanes that trigger new path
  // jobs.  k_render_stream: finished casts of a wave with all lanes busy that trigger the path
  // updates (in proportion with fewer lanes; 1080p 16 spp 16.4 / 15.9 / 15.8 ms at 16 / 24 / 32),
  // idle lanes that pop the queue (1, 4, 10: 16.2, 15.9, 15.9 ms), lanes that wait at a leaf for the
  // leaf tests (8, 12, 16, 20: 13.50, 13.33, 13.29, 13.32 ms)
  static constexpr int kShadeMin = 32, kRefillMin = 8, kStreamShadeMin = 32, kStreamRefillMin = 4,
                       kStreamLeafMin = 16;
  Path st;
  __device__ __forceinline__ bool start(const dr_render_params &P, const FrameK &K, int block, int lp, int s,
                                        uint32_t samp0) {
    return start_path(P, K, block, lp, s, samp0, st);
  }
  __device__ __forceinline__ void begin(const PathStart &s) { begin_path(st, s); }
  __device__ __forceinline__ uint32_t pixel() const { return st.pix; }
  __device__ __forceinline__ uint32_t sample() const { return st.samp; }
  __device__ __forceinline__ V3 ray_o() const { return st.o; }
  __device__ __forceinline__ V3 ray_d() const { return st.d; }
  __device__ __forceinline__ int ray_excl() const { return st.restrict_tri; }
  __device__ __forceinline__ const float *color() const { return st.L; }
  __device__ __forceinline__ bool photon() const { return st.phase == 1; }
  // Next bounce after the last photon of a vertex; false when the path ends.
  __device__ __forceinline__ bool advance(const dr_render_params &P) {
    if (!st.has_sample) return false;
    float A[3];
    reflect_factor(P, st, A);
    for (int c = 0; c < 3; c++) st.beta[c] = st.beta[c] * (A[c] * st.sweight);
    st.o = st.p;
    st.d = st.sdir;
    st.restrict_tri = st.h;
    st.layer++;
    st.phase = 0;
    return true;
  }
  // After the lane's cast ended.  A geometry hit sets up the vertex, then photons
  // (Lambert) or the next bounce; a photon adds its contribution if it reached the
  // vertex, then the next photon.  Returns true when the path is done.
  __device__ __forceinline__ bool shade(const dr_render_params &P, const FrameK &K, const Tables &tb, const Walk &w) {
    bool photons = false;
    if (st.phase == 0) {
      if (!w.hit) return true;
      setup_vertex(P, K, tb.shade, w.h, w.d, st);
      photons = st.kind == DR_LAMBERT;
    } else {
      const V3 e = w.h.p - st.p;
      const bool lit = w.hit && (w.h.id == st.h || (e.x * e.x + e.y * e.y + e.z * e.z) <= (8.0f * kVecEps));
      if (lit) for (int c = 0; c < 3; c++) st.L[c] += st.contrib[c];
      photons = true;
    }
    if (photons && next_photon(P, st)) return false;
    return !advance(P);
  }
};

// Path updates of the reference estimator (DR_PLUGINS_REFERENCE), DumbRenderer.cu:256-443:
// every layer casts each light's photons (one, or a spotlight's samples); a photon that first reaches another surface
// continues through it with that surface's getReflectedColor (observer = the photon
// direction) as its colour when that colour is not black (:396-413).  Colours are
// carried forward: L += beta * (getReflectedColor of each direct photon), and the
// child layer's throughput is beta * getReflectedColor(indirect photon) * sampleWeight.
//
// Only what the shadow casts need stays live across them: the vertex (triangle, point,
// incoming direction, material) and the photon.  The shading record and the indirect
// sample are computed again where they are used; both are functions of the vertex and
// of counter-based random numbers, so the order of evaluation does not change them.
struct RefPath {
  // the same thresholds (reference plugins at 1080p, 1 spp: 3.23 / 3.12 / 3.26 ms at 32 / 44 / 52; leaf
  // tests 2.78 / 2.76 / 2.75 / 2.84 ms at 4 / 6 / 8 / 16)
  static constexpr int kShadeMin = 32, kRefillMin = 8, kStreamShadeMin = 44, kStreamRefillMin = 4,
                       kStreamLeafMin = 8;
  uint32_t pix, samp;
  int layer, phase, light, lk, excl, trans;   // lk: photons of the current light still to send
  V3 o, d;                          // the next ray to cast
  float beta[3], L[3];
  int h, mid;                       // current vertex: triangle, material
  V3 hp, din;                       //   hit point, incoming ray direction
  V3 pd;                            // current photon: direction, colour, unit direction?
  float pc[3];
  bool unit;

  __device__ __forceinline__ bool start(const dr_render_params &P, const FrameK &K, int block, int lp, int s,
                                        uint32_t samp0) {
    const PathStart ps = path_start(P, K, block, lp, s, samp0);
    if (ps.pix == kNoPixel) return false;
    begin(ps);
    return true;
  }
  __device__ __forceinline__ void begin(const PathStart &s) {
    pix = s.pix;
    samp = s.samp;
    o = s.o;
    d = s.d;
    layer = 0;
    phase = 0;
    excl = -1;
    for (int c = 0; c < 3; c++) { beta[c] = 1.0f; L[c] = 0.0f; }
  }
  __device__ __forceinline__ uint32_t pixel() const { return pix; }
  __device__ __forceinline__ uint32_t sample() const { return samp; }
  __device__ __forceinline__ V3 ray_o() const { return o; }
  __device__ __forceinline__ V3 ray_d() const { return d; }
  __device__ __forceinline__ int ray_excl() const { return excl; }
  __device__ __forceinline__ const float *color() const { return L; }
  __device__ __forceinline__ bool photon() const { return phase == 1; }

  // The vertex's shading record (reference shaders; only the point for the others).
  __device__ __forceinline__ RefHit hit_record(const dr_render_params &P, const Tables &tb,
                                               const dr_material &M) const {
    RefHit H;
    H.p = hp;
    if (is_reference_kind(M.kind)) {
      const TexCtx T = tex_ctx(P);
      H = ref_hit(tb.faces, h, hp, T, material_maps(T, M));
    }
    return H;
  }
  __device__ __forceinline__ V3 facing(const Tables &tb) const {
    const float4 sh = tb.shade[h];
    return facing_normal(v3(sh.x, sh.y, sh.z), normalized(din));
  }
  // Direct light of the current photon at the vertex.
  __device__ __forceinline__ void add_direct(const dr_render_params &P, const Tables &tb) {
    const dr_material M = P.materials[mid];
    if (M.kind == DR_LAMBERT) {
      const V3 wn = unit ? pd : normalized(pd);
      const float cos_i = -dot(facing(tb), wn);
      if (cos_i > 0.0f) {
        const float k = cos_i * kInvPi;
        for (int c = 0; c < 3; c++) L[c] += beta[c] * ((M.albedo[c] * k) * pc[c]);
      }
    } else {
      const RefHit H = hit_record(P, tb, M);
      float f[3];
      reflect_ref(M, H, pd, pc, neg(din), true, 0, tex_ctx(P), f);
      for (int c = 0; c < 3; c++) L[c] += beta[c] * f[c];
    }
  }
  // The indirect sample of the vertex and the child layer's ray and throughput; false when
  // the path ends here.
  __device__ __forceinline__ bool next_layer(const dr_render_params &P, const FrameK &K, const Tables &tb) {
    if (layer >= P.max_bounces) return false;
    const dr_material M = P.materials[mid];
    float u[4];
    rng4(P, pix, samp, (uint32_t)layer, 1, u);
    float sw = 1.0f;
    if (layer >= P.rr_start) {
      if (u[2] >= P.rr_survive) return false;
      sw = K.inv_rr;
    }
    const RefHit H = hit_record(P, tb, M);
    V3 sdir;
    int stype = 0;
    float F[3];
    if (M.kind == DR_LAMBERT) {
      sdir = cosine_dir(facing(tb), u[0], u[1]);
      for (int c = 0; c < 3; c++) F[c] = M.albedo[c];
    } else if (M.kind == DR_MIRROR || M.kind == DR_METAL) {
      const V3 nu = facing(tb);
      sdir = reflect_unit(normalized(din), nu);
      if (M.kind == DR_METAL) {
        const float f5 = schlick5(nu, sdir);
        for (int c = 0; c < 3; c++) F[c] = M.albedo[c] + (1.0f - M.albedo[c]) * f5;
      } else {
        for (int c = 0; c < 3; c++) F[c] = M.albedo[c];
      }
    } else {
      if (!sample_ref(P, M, H, din, pix, samp, layer, u, sdir, stype)) return false;
      const float white[3] = {1.0f, 1.0f, 1.0f};
      reflect_ref(M, H, neg(sdir), white, neg(din), false, stype, tex_ctx(P), F);
    }
    for (int c = 0; c < 3; c++) beta[c] = beta[c] * (F[c] * sw);
    o = hp;
    d = sdir;
    excl = h;
    layer++;
    phase = 0;
    return true;
  }
  // After the lane's cast ended; true when the path is done.
  __device__ __forceinline__ bool shade(const dr_render_params &P, const FrameK &K, const Tables &tb, const Walk &w) {
    if (phase == 0) {
      if (!w.hit) return true;                        // the layer ray missed (:418-421)
      h = w.h.id;
      hp = w.h.p;
      din = w.d;
      mid = __float_as_int(tb.shade[h].w);
      const int kind = P.materials[mid].kind;
      light = (kind == DR_MIRROR || kind == DR_METAL) ? P.nlights : -1;   // delta BSDFs take no direct light
      lk = 0;
    } else if (w.hit) {
      const V3 e = w.h.p - hp;
      if (w.h.id == h || (e.x * e.x + e.y * e.y + e.z * e.z) <= (8.0f * kVecEps)) {
        add_direct(P, tb);
      } else {
        const int hb = w.h.id;
        const dr_material Mb = P.materials[__float_as_int(tb.shade[hb].w)];
        if (is_reference_kind(Mb.kind) && trans < kMaxTransmit) {
          const TexCtx T = tex_ctx(P);
          const RefHit B = ref_hit(tb.faces, hb, w.h.p, T, material_maps(T, Mb));
          float tc[3];
          reflect_ref(Mb, B, pd, pc, pd, true, 0, T, tc);
          if (((tc[0] + tc[1]) + tc[2]) > kVecEps) {
            for (int c = 0; c < 3; c++) pc[c] = tc[c];
            o = w.h.p + normalized(pd) * (64.0f * kVecEps);
            d = pd;
            excl = hb;
            trans++;
            return false;
          }
        }
      }
    }
    // next photon: the current light's remaining samples (last first, DumbRenderer.cu:290-293),
    // then the following lights; a light that casts no shadows illuminates at once (:306-315)
    while (true) {
      if (lk == 0) {
        if (++light >= P.nlights) break;
        lk = light_samples(P.lights[light]);
        if (lk == 0) continue;
      }
      lk--;
      V3 q, wv;
      bool u1;
      float c3[3];
      if (!photon_ref(P, P.lights[light], light, lk, pix, samp, layer, hp, q, wv, c3, u1)) continue;
      pd = wv;
      unit = u1;
      for (int c = 0; c < 3; c++) pc[c] = c3[c];
      if (!light_casts_shadows(P.lights[light])) {
        add_direct(P, tb);
        continue;
      }
      o = q;
      d = wv;
      excl = -1;
      trans = 0;
      phase = 1;
      return false;
    }
    return !next_layer(P, K, tb);
  }
};

// ------------------------------------------------------------------ forward
// LDS used by one block render.
struct BlockLds {
  uint2 *stk;           // this lane's first stack level ([level][lane])
  float *samp_col;      // kBlockPixels * kRoundSamples * 3 sample colours
  float *acc;           // kBlockPixels * 3 pixel sums
  int *next_job;
  LeafLds *leaf;        // this wave's (walk_leaf_wave)
  int *ins;             // this wave's inside-test counts (measurement launches only)
};

// Work counters of a render (measurement launches only), summed over the launch.
enum : int {
  kRcSegments = 0,      // casts: camera and bounce rays and light photons
  kRcPhotons,           //   of which light photons (shadow rays)
  kRcExpand,            // group expansions (8 child box tests)
  kRcLeaves,            // leaves tested
  kRcPlane,             // triangle plane tests
  kRcInside,            // triangle inside tests
  kRcPaths,             // path jobs (pixel samples) started
  kRcLive,              // children of expanded groups with a non-empty leaf below (box tests)
  kRcSlab,              // children that the box test kept
  kRcCount
};
struct RenderCounters {
  CastCounters cast = {0, 0, 0, 0, 0, 0};
  int segments = 0, photons = 0, paths = 0;
};
// Adds one lane's counters to the launch's totals (every lane of the wave calls it).
__device__ __forceinline__ void flush_counters(const RenderCounters &c, unsigned long long *out) {
  const int v[kRcCount] = {c.segments, c.photons,     c.cast.expand, c.cast.leaves, c.cast.plane,
                           c.cast.inside, c.paths, c.cast.live, c.cast.slab};
#pragma unroll
  for (int k = 0; k < kRcCount; k++) {
    unsigned long long x = (unsigned long long)v[k];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off);
    if (__lane_id() == 0) atomicAdd(&out[k], x);
  }
}

// Framebuffer pixel `lp` of block `block` (inside the image): the colour of this iteration, set
// (iteration 1) or blended with weight 1/iteration (DumbRenderer.cu:64, BlockBasedFrameBuffer.impl.cuh:125-156).
__device__ __forceinline__ void store_pixel(const FrameK &K, float *__restrict__ frame, int block, int lp,
                                            const float a[3]) {
  float4 *f = (float4 *)frame + (size_t)kBlockPixels * block + lp;
  const float4 col = make_float4(a[0], a[1], a[2], 1.0f);
  const float amount = K.amount;
  if (amount >= 1.0f) *f = col;
  else {
    const float4 old = *f;
    const float ia = K.keep;
    *f = make_float4((col.x * amount) + (old.x * ia), (col.y * amount) + (old.y * ia),
                     (col.z * amount) + (old.z * ia), (col.w * amount) + (old.w * ia));
  }
}

// Renders framebuffer block `block` of one request (all lanes of the workgroup call it),
// in rounds of kRoundSamples samples per pixel.  K = frame_k(P).
// refill_min: an idle lane takes a new job once at least this many lanes of its wave
// are idle (or the whole wave is).
template <class PathT, bool kStats = false>
__device__ __forceinline__ void render_block(const DevTree &T, const Tables &tb, const dr_render_params &P,
                                             const FrameK &K, float *__restrict__ frame, int block,
                                             const BlockLds &lds, int refill_min, RenderCounters *rc = nullptr) {
  CastCounters *cc = kStats ? &rc->cast : nullptr;
  const int spp = P.fsaa_x * P.fsaa_y;
  const uint32_t samp0 = (uint32_t)(P.iteration > 1 ? P.iteration - 1 : 0) * (uint32_t)spp;
  const float spw = uni(1.0f / (((float)P.fsaa_x) * ((float)P.fsaa_y)));
  const bool clip = P.cull_backfaces != 0;
  const int lane = (int)__lane_id();
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  float *samp_col = lds.samp_col;
  for (int t = threadIdx.x; t < kBlockPixels * 3; t += kRB) lds.acc[t] = 0.0f;

  for (int s_base = 0; s_base < spp; s_base += kRoundSamples) {
    const int ns = min(kRoundSamples, spp - s_base);
    const UDiv Dns = udiv_uniform((uint32_t)ns);
    const int njobs = kBlockPixels * ns;   // job j: pixel j / ns, sample s_base + j % ns
    if (threadIdx.x == 0) *lds.next_job = 0;
    __syncthreads();
    PathT ps;
    int job = -1;
    Walk w;
    w.state = kWalkDone;
    bool exhausted = false;
    auto finish = [&](const float *L) {
      // getPixelColor: the layer colour (SimpleStochasticLense, DefaultPerspectiveLense) or the
      // colour times the lens filter (SphericalSegmentLense.impl.cuh:31-34)
      if (P.lens == DR_SPHERICAL_SEGMENT_LENS)
        for (int c = 0; c < 3; c++) samp_col[3 * job + c] = L[c] * P.lens_p[4 + c];
      else
        for (int c = 0; c < 3; c++) samp_col[3 * job + c] = L[c];
      job = -1;
    };
    for (;;) {
      const bool want = (job < 0) && !exhausted;
      const uint64_t wmask = __ballot(want);
      const uint64_t busy = __ballot(job >= 0);
      if (wmask && (__popcll(wmask) >= refill_min || busy == 0)) {
        const int leader = __ffsll((unsigned long long)wmask) - 1;
        int base = 0;
        if (lane == leader) base = atomicAdd(lds.next_job, __popcll(wmask));
        base = __shfl(base, leader);
        if (want) {
          const int slot = base + __popcll(wmask & below);
          if (slot < njobs) {
            job = slot;
            const int rp = (int)udiv((uint32_t)slot, Dns), s = s_base + (slot - rp * ns);
            if (!ps.start(P, K, block, rp, s, samp0)) {
              const float zero[3] = {0.0f, 0.0f, 0.0f};
              finish(zero);
            } else {
              walk_begin(T, w, ps.ray_o(), ps.ray_d(), ps.ray_excl(), lds.stk);
              if (kStats) { rc->paths++; rc->segments++; }
            }
          } else {
            exhausted = true;
          }
        }
      }
      if (__ballot(job >= 0) == 0) {
        if (__ballot(!exhausted) == 0) break;
        continue;
      }
      // ---- one traversal step of every ray in flight
      if (job >= 0 && w.state == kWalkTrace) walk_step(T, w, lds.stk, kRB, cc);
      // ---- leaf tests, batched
      const bool pend = job >= 0 && w.leaf != kNoLeaf;
      const uint64_t pm = __ballot(pend && w.state == kWalkLeaf);
      if (pm && (__popcll(pm) >= kLeafMin || __ballot(job >= 0 && w.state == kWalkTrace) == 0))
        walk_leaf_wave(T, w, pend, clip, *lds.leaf, kStats ? lds.ins : nullptr, cc);
      // ---- path updates of the finished casts, batched
      const uint64_t dm = __ballot(job >= 0 && w.state == kWalkDone);
      if (dm && (__popcll(dm) >= PathT::kShadeMin || __ballot(job >= 0 && w.state != kWalkDone) == 0)) {
        if (job >= 0 && w.state == kWalkDone) {
          if (ps.shade(P, K, tb, w)) {
            finish(ps.color());
          } else {
            walk_begin(T, w, ps.ray_o(), ps.ray_d(), ps.ray_excl(), lds.stk);
            if (kStats) { rc->segments++; rc->photons += ps.photon() ? 1 : 0; }
          }
        }
      }
    }
    __syncthreads();
    if (threadIdx.x < kBlockPixels) {
      for (int s = 0; s < ns; s++)
        for (int c = 0; c < 3; c++) lds.acc[3 * threadIdx.x + c] += samp_col[3 * (threadIdx.x * ns + s) + c] * spw;
    }
    __syncthreads();
  }
  int x, y;
  if (threadIdx.x < kBlockPixels && block_pixel(K, P.width, P.height, block, threadIdx.x, x, y))
    store_pixel(K, frame, block, threadIdx.x, lds.acc + 3 * threadIdx.x);
  __syncthreads();
}

// One framebuffer block per workgroup (sample counts above the streamed kernel's limit).
template <class PathT, bool kStats = false>
__global__ __launch_bounds__(kRB, kRenderWaves) void k_render(DevTree T, Tables tb, dr_render_params P, FrameK K,
                                                               float *__restrict__ frame, int start_block, int levels,
                                                               unsigned long long *__restrict__ counts = nullptr) {
  extern __shared__ __align__(16) uint32_t lds[];
  __shared__ float acc[kBlockPixels * 3];
  __shared__ int next_job;
  __shared__ LeafLds leaf[kRB / 64];
  __shared__ int ins[kStats ? kRB : 1];
  const BlockLds L = {(uint2 *)lds + threadIdx.x, (float *)(lds + levels * kStackWordsPerLevel * kRB), acc, &next_job,
                      leaf + (threadIdx.x >> 6), kStats ? ins + (threadIdx.x & ~63u) : nullptr};
  leaf_lds_init(*L.leaf);
  RenderCounters rc;
  render_block<PathT, kStats>(T, tb, P, K, frame, start_block + (int)blockIdx.x, L, PathT::kRefillMin, &rc);
  if (kStats) flush_counters(rc, counts);
}

// ------------------------------------------------------------------ streamed blocks
// k_render_stream: the same path loop with no barrier between framebuffer blocks.  A
// workgroup is persistent and takes tiles (2^tile_shift pixels of a block, 128 at most) from a
// counter in global memory; its waves take path jobs from one stream that runs through those
// tiles in turn (job q: pixel q / spp of the stream, sample q % spp; stream pixel u is pixel
// u % 2^tile_shift of the workgroup's tile number u >> tile_shift), so lanes whose paths end near
// the end of a tile start the next tile's paths instead of waiting for the tile's longest path.
//   * A wave takes `chunk` jobs at a time (64 at most, all of one tile) and forms their camera rays
//     with as many lanes, into a queue in LDS; lanes that become idle pop the next entry.
//   * With one sample per pixel a finished path writes its pixel.
//   * With more, sample colours are staged in a ring of nslots = 2^slot_shift pixel slots of spp
//     samples.  Stream pixel u uses slot u % nslots and may start once that is in its turn u / nslots,
//     i.e. once pixel u - nslots has been written out.  A slot's word holds its turn << 9 | samples to
//     come.  The lane that finishes a pixel's last sample sums its spp staged colours in sample
//     order, as render_block does, writes the pixel, and begins the slot's next turn.
//     Frames are therefore bit-identical to render_block's.
//   * Tile number k of the workgroup is fetched by the wave that forms its first jobs, and
//     only once tile k - 1 has been fetched, so tile ids rise with k and the tiles past
//     the launch's range form a suffix of the stream.  The ids sit in a ring of
//     kStreamRing entries; a job of tile number k is formed only once every pixel of tile
//     number k - kStreamRing has been written (pixels written per ring entry are
//     counted cumulatively), so no job still needs an entry when it is reused.
//   * Progress: jobs are formed and popped in order within a wave.  Every job before the oldest one
//     not yet started is held by a lane, and a lane's path always ends; so its tile's ring entry
//     and its pixel's slot become free, the entries before it in its queue have been popped, and
//     its wave pops it once lanes of the wave are idle.
constexpr int kStreamSamples = 2048;      // staged sample colours per workgroup
constexpr int kStreamRing = 64;
constexpr int kStreamMaxSpp = 256;        // higher sample counts take render_block's rounds

// log2 of the pixel slots for `samples` staged colours, -1 for no staging
constexpr int stream_slot_shift(int spp, int samples) {
  int n = 0;
  while ((2 << n) * spp <= samples) n++;
  return spp == 1 ? -1 : n;
}
// LDS words of one wave's queue of path starts: direction, pixel, stream
// pixel, and the origin for lenses that sample it.
__host__ __device__ constexpr int stream_queue_words(bool origins) { return 64 * (origins ? 8 : 5); }
constexpr size_t stream_lds(int levels, int spp, int slot_shift, bool origins) {
  const size_t nslots = slot_shift < 0 ? 0 : (size_t)1 << slot_shift;
  return ((size_t)levels * kStackWordsPerLevel * kRB + nslots * (3 * spp + 1) +
          (kRB / 64) * (size_t)stream_queue_words(origins)) * 4;
}

// Words of LDS that other waves change (an atomic access stays an LDS instruction; a volatile one
// would go through a flat address).
__device__ __forceinline__ int lds_get(const int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
__device__ __forceinline__ void lds_put(int *p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }

// LDS of a workgroup's stream beside the dynamic part (stream_lds).
struct StreamLds {
  int tiles[kStreamRing];          // (tile id + 1) << 8 | tile number & 255
  int px_done[kStreamRing];        // pixels written, cumulative per ring entry
  unsigned next_job;
  int end_k;                       // first tile number past the range
  LeafLds leaf[kRB / 64];
};
// The tiles of a stream and its launch shape.
struct StreamShape {
  int ntiles, tile_shift, chunk, slot_shift;
};

// One stream (every lane of the workgroup calls it): tiles from the counter `next_tile` until they run out.
// ins: this wave's inside-test counts (measurement launches only).
template <class PathT, bool kStats>
__device__ __forceinline__ void stream_paths(ConstArgs args,
                                             float *__restrict__ frame, int start_block, const StreamShape &S, int levels,
                                             unsigned *next_tile, int refill_min, uint32_t *lds, StreamLds &sh, int *ins,
                                             RenderCounters &rc) {
  const DevTree T = again(args).T;
  const dr_render_params &P = again(args).P;
  const int ntiles = S.ntiles, tile_shift = S.tile_shift, chunk = S.chunk, slot_shift = S.slot_shift;
  const int spp = P.fsaa_x * P.fsaa_y;
  const int nslots = slot_shift < 0 ? 0 : 1 << slot_shift;
  const bool origins = P.lens == DR_SPHERICAL_SEGMENT_LENS;
  uint2 *stk = (uint2 *)lds + threadIdx.x;
  float *samp = (float *)(lds + levels * kStackWordsPerLevel * kRB);   // nslots * spp * 3
  int *turn = (int *)(samp + (size_t)nslots * spp * 3);              // nslots
  float *queue = (float *)(turn + nslots) + (threadIdx.x >> 6) * stream_queue_words(origins);   // [word][entry]
  LeafLds &leaf = sh.leaf[threadIdx.x >> 6];
  leaf_lds_init(leaf);
  for (int t = threadIdx.x; t < nslots; t += kRB) turn[t] = spp;
  for (int t = threadIdx.x; t < kStreamRing; t += kRB) { sh.tiles[t] = 0; sh.px_done[t] = 0; }
  if (threadIdx.x == 0) { sh.next_job = 0; sh.end_k = 0x7fffffff; }
  __syncthreads();

  CastCounters *cc = kStats ? &rc.cast : nullptr;
  const uint32_t samp0 = (uint32_t)(P.iteration > 1 ? P.iteration - 1 : 0) * (uint32_t)spp;
  const float spw = uni(1.0f / (((float)P.fsaa_x) * ((float)P.fsaa_y)));
  const UDiv Dspp = udiv_uniform((uint32_t)spp);
  const bool clip = P.cull_backfaces != 0;
  const int lane = (int)__lane_id();
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  PathT ps;
  Walk w;                 // (kWalkIdle: the lane has no path)
  w.state = kWalkIdle;
  w.leaf = kNoLeaf;
  int u = 0;              // stream pixel of this lane's path
  // the wave's queue (wave-uniform): entries [qpos, qlen) of the jobs from qbase on
  unsigned qbase = 0;
  int qpos = 0, qlen = 0;
  bool taken = false;     // the jobs from qbase on are this wave's and not formed yet
  bool ended = false;     // the stream has no more jobs for this wave
  // pixel p of tile e of the ring: its block and place in it
  auto tile_block = [&](int e) { return start_block + (((e >> 8) - 1) >> (7 - tile_shift)); };
  auto tile_pixel = [&](int e, int p) {
    return ((((e >> 8) - 1) & ((1 << (7 - tile_shift)) - 1)) << tile_shift) + (p & ((1 << tile_shift) - 1));
  };
  auto pixel_written = [&](const FrameK &K, const float a[3]) {
    const int kk = (u >> tile_shift) & (kStreamRing - 1);
    // (the tile's ring entry stays until every pixel of the tile is written)
    const int e = lds_get(&sh.tiles[kk]);
    if (ps.pixel() != kNoPixel) store_pixel(K, frame, tile_block(e), tile_pixel(e, u), a);
    atomicAdd(&sh.px_done[kk], 1);
  };
  for (;;) {
    // ---- path updates of the finished casts, batched.  The thresholds here and of the leaf tests are
    // shares of the lanes that have a path: a wave near the end of the frame, with few, would otherwise
    // hold each finished cast until its slowest ray (517x389 at 1 spp: 1067 -> 968 us)
    const uint64_t dm = __ballot(w.state == kWalkDone);
    bool fresh = false;   // the lane has a new ray
    const uint64_t lm = __ballot(w.state != kWalkIdle);
    if (dm && __popcll(dm) * 64 >= __popcll(lm) * PathT::kStreamShadeMin) {
      const RenderArgs &A = again(args);
      if (w.state == kWalkDone) {
        const bool outside = ps.pixel() == kNoPixel;
        if (outside || ps.shade(A.P, A.K, A.tb, w)) {
          // stages the sample's colour (the lens filter applied: getPixelColor, see render_block; a job
          // outside the image stages black); the lane that completes the pixel writes it out
          const float *col = ps.color();
          float c[3] = {col[0], col[1], col[2]};
          if (origins)
            for (int k = 0; k < 3; k++) c[k] = c[k] * A.P.lens_p[4 + k];
          if (outside) c[0] = c[1] = c[2] = 0.0f;
          if (nslots == 0) {
            const float a[3] = {0.0f + c[0] * spw, 0.0f + c[1] * spw, 0.0f + c[2] * spw};
            pixel_written(A.K, a);
          } else {
            const int slot = u & (nslots - 1);
            float *src = samp + 3 * (size_t)slot * spp;
            float *dst = src + 3 * (int)(ps.sample() - samp0);
            dst[0] = c[0];
            dst[1] = c[1];
            dst[2] = c[2];
            __threadfence_block();
            const int left = atomicSub(&turn[slot], 1);
            if ((left & 511) == 1) {
              __threadfence_block();   // the other samples' colours, staged before their lanes' subtractions
              float a[3] = {0.0f, 0.0f, 0.0f};
              for (int k = 0; k < spp; k++)
                for (int j = 0; j < 3; j++) a[j] += src[3 * k + j] * spw;
              pixel_written(A.K, a);
              __threadfence_block();
              lds_put(&turn[slot], (((left >> 9) + 1) << 9) | spp);
            }
          }
          w.state = kWalkIdle;
        } else {
          fresh = true;
          if (kStats) { rc.segments++; rc.photons += ps.photon() ? 1 : 0; }
        }
      }
    }
    // ---- the queue is empty: the next jobs of the stream, and their camera rays
    if (qpos == qlen && !ended) {
      if (!taken) {
        unsigned q = 0;
        if (lane == 0) q = atomicAdd(&sh.next_job, (unsigned)chunk);
        qbase = (unsigned)__builtin_amdgcn_readfirstlane((int)q);
        taken = true;
      }
      // the tile of these jobs (wave-uniform); its first jobs' wave fetches its id once the tile before has one
      const int k = uni((int)udiv(qbase, Dspp)) >> tile_shift;
      const int kk = k & (kStreamRing - 1);
      bool past = k >= uni(lds_get(&sh.end_k));
      int e = 0;
      if (!past && uni(lds_get(&sh.px_done[kk])) >= (k / kStreamRing) << tile_shift) {   // the ring entry is tile k's
        e = uni(lds_get(&sh.tiles[kk]));
        if ((e & 0xff) != (k & 0xff)) e = 0;
        if (e == 0 && qbase == (unsigned)((k << tile_shift) * spp)) {
          const int prev = k > 0 ? uni(lds_get(&sh.tiles[(k - 1) & (kStreamRing - 1)])) : 0;
          if (k == 0 || (prev != 0 && (prev & 0xff) == ((k - 1) & 0xff))) {
            int id = 0;
            if (lane == 0) id = (int)atomicAdd(next_tile, 1u);
            id = __builtin_amdgcn_readfirstlane(id);
            if (id >= ntiles) {
              if (lane == 0) atomicMin(&sh.end_k, k);
              past = true;
            } else {
              e = ((id + 1) << 8) | (k & 0xff);
              if (lane == 0) lds_put(&sh.tiles[kk], e);
            }
          }
        }
      }
      ended = past;
      if (e != 0) {
        taken = false;
        qpos = 0;
        qlen = chunk;
        if (lane < chunk) {
          const int q = (int)qbase + lane;
          const int uq = (int)udiv((uint32_t)q, Dspp), s = q - uq * spp;
          const RenderArgs &A = again(args);
          const PathStart st = path_start(A.P, A.K, tile_block(e), tile_pixel(e, uq), s, samp0);
          queue[0 * 64 + lane] = st.d.x;
          queue[1 * 64 + lane] = st.d.y;
          queue[2 * 64 + lane] = st.d.z;
          queue[3 * 64 + lane] = __int_as_float((int)st.pix);
          queue[4 * 64 + lane] = __int_as_float(uq);
          if (origins) {
            queue[5 * 64 + lane] = st.o.x;
            queue[6 * 64 + lane] = st.o.y;
            queue[7 * 64 + lane] = st.o.z;
          }
        }
        __threadfence_block();
      }
    }
    // ---- idle lanes pop the next entries whose pixel slot is free
    const uint64_t idle = __ballot(w.state == kWalkIdle);
    if (qpos < qlen && idle && (__popcll(idle) >= refill_min || idle == ~0ull)) {
      const int entry = qpos + __popcll(idle & below);
      const bool some = w.state == kWalkIdle && entry < qlen;
      int uq = 0;
      bool free = false;
      if (some) {
        uq = __float_as_int(queue[4 * 64 + entry]);
        // (turns are compared in the 23 bits a slot's word keeps)
        free = nslots == 0 || (((lds_get(&turn[uq & (nslots - 1)]) >> 9) ^ (uq >> slot_shift)) & 0x7fffff) == 0;
      }
      const uint64_t stuck = __ballot(some && !free);
      const bool take = some && (stuck == 0 || lane < __ffsll((unsigned long long)stuck) - 1);
      qpos += __popcll(__ballot(take));
      if (take) {
        PathStart st;
        st.d = v3(queue[0 * 64 + entry], queue[1 * 64 + entry], queue[2 * 64 + entry]);
        st.pix = (uint32_t)__float_as_int(queue[3 * 64 + entry]);
        st.samp = samp0 + (qbase + (uint32_t)entry - (uint32_t)uq * (uint32_t)spp);
        const RenderArgs &A = again(args);
        st.o = v3(A.P.cam[0], A.P.cam[1], A.P.cam[2]);
        if (origins) st.o = v3(queue[5 * 64 + entry], queue[6 * 64 + entry], queue[7 * 64 + entry]);
        u = uq;
        w.state = kWalkTrace;
        ps.begin(st);
        fresh = true;
        if (kStats && st.pix != kNoPixel) { rc.paths++; rc.segments++; }
      }
    }
    if (__ballot(w.state != kWalkIdle) == 0) {
      if (qpos == qlen && ended) break;
      __builtin_amdgcn_s_sleep(1);   // the next jobs wait for a slot or a tile id
      continue;
    }
    if (fresh) {
      walk_begin(again(args).T, w, ps.ray_o(), ps.ray_d(), ps.ray_excl(), stk);
      if (ps.pixel() == kNoPixel) {
        w.state = kWalkDone;
        w.leaf = kNoLeaf;
      }
    }
    // ---- one traversal step of every ray in flight
    if (w.state == kWalkTrace) walk_step(T, w, stk, kRB, cc);
    // ---- leaf tests, batched
    const uint64_t pm = __ballot(w.state == kWalkLeaf);
    if (pm && (__popcll(pm) * 64 >= __popcll(__ballot(w.state != kWalkIdle)) * PathT::kStreamLeafMin ||
               __ballot(w.state == kWalkTrace) == 0))
      walk_leaf_wave(T, w, w.leaf != kNoLeaf, clip, leaf, ins, cc);
  }
}

template <class PathT, bool kStats>
__global__ __launch_bounds__(kRB, kRenderWaves) void k_render_stream(RenderArgs by_value,
                                                                      float *__restrict__ frame, int start_block,
                                                                      StreamShape S, int levels,
                                                                      unsigned *__restrict__ work,
                                                                      unsigned long long *__restrict__ counts) {
  extern __shared__ __align__(16) uint32_t lds[];
  __shared__ StreamLds sh;
  __shared__ int ins_all[kStats ? kRB : 1];
  RenderCounters rc;
  // (by_value is the kernel's first argument)
  stream_paths<PathT, kStats>((ConstArgs)__builtin_amdgcn_kernarg_segment_ptr(), frame, start_block, S, levels, work, PathT::kStreamRefillMin, lds, sh,
                              kStats ? ins_all + (threadIdx.x & ~63u) : nullptr, rc);
  if (kStats) flush_counters(rc, counts);
  // ---- the last wave out resets the block counter for the next launch
  if (__lane_id() == 0) {
    __threadfence();
    const unsigned total = gridDim.x * (kRB / 64);
    if (atomicAdd(work + 1, 1u) == total - 1) {
      atomicExch(work, 0u);
      atomicExch(work + 1, 0u);
    }
  }
}

// ------------------------------------------------------------------ adjoint
// Vertex records of each lane's current path ([vertex][word][lane] in the
// workgroup's slice of a scratch buffer): material id, reflection factor A (3),
// direct sum d (3) with L_k = A (d + s L_{k+1}), the sample weight s, and dA/dalbedo
// (1, or 1 - f5 for a Schlick metal, whose A = F0 + (1 - F0) f5).
// The path is replayed from its Philox key; after it ends S_k = d_k + s_k L_{k+1}
// is formed backwards and dL/dalbedo += w dL/dI beta_k dA_k S_k.  dL/demission is
// added during the replay: w dL/dI beta_k A_k (cos_i/pi)(cos_l A/d^2).
// Rays are step-wise walks as in render_block.  The grid is persistent (one vertex-record
// slice per workgroup).  Paths are independent, so there is no barrier in the loop: each wave takes
// `chunk` jobs of one framebuffer block at a time from a counter in global memory, forms their
// camera rays and loss gradients with as many lanes into a queue in LDS, and its idle lanes pop the
// next entry, as in k_render_stream.  (With one block per workgroup at a time the lanes waited for
// each block's longest path: 512x512 16 spp 10.6 -> 7.3 ms.)
// Reductions: the lanes of a wave that add to the same parameter in the same path
// update are summed across the wave first (one LDS atomic per distinct material or
// light and channel), and the workgroup's LDS sums go to the FP64 outputs with one global atomic
// per parameter.  Three forms, by the materials and lights and by the stacks beside the sums:
//   kSumsFp64   the LDS sums are FP64 and go out once, at the end.  Taken unless FP32 sums leave room for
//               more workgroups a CU (10 levels: from 857 materials and lights on): 512x512 at
//               16 spp 6.2 ms in FP64 with three a CU (600 materials), and 7.7 ms with two against 6.9 ms in
//               FP32 with three (1,500), 13.8 ms with one against 8.6 ms with two (2,500).
//   kSumsFp32   FP32 sums.  A wave moves all of them out whenever flush_paths(spp) of its paths have ended,
//               so that what adds up in FP32 is the paths of one framebuffer block (128 spp), and no more
//               than 2,048.
//   kSumsTight  LDS holds the stacks and as many FP32 sums as fit (the lights' always): the queues lie
//               beside the vertex records, and the few parameters left over (sizes a whisker below the
//               limit) are added to the outputs.  (All terms added to the outputs, with FP64 atomics on
//               few addresses: 80 ms against 15.6 ms, 12,620 materials.)
constexpr int kVtxWords = 9;
// Samples a pixel of one launch: the jobs of a block are counted in 31 bits.  A call with more takes several
// launches.
constexpr int kLaunchSamples = 1 << 23;
enum : int { kSumsTight, kSumsFp32, kSumsFp64 };
__device__ __forceinline__ int flush_paths(int spp) { return min(spp, 16) * (kBlockPixels / (kRB / 64)); }
constexpr int kAdjointQueueWords = 64 * 11;   // direction, pixel, sample, loss gradient, origin

// Sum of v over the 64 lanes of the wave, returned to every lane: an inclusive scan within
// each row of 16 lanes with DPP row shifts (1, 2, 4, 8; a lane without a source adds 0)
// leaves the row totals in lanes 15, 31, 47 and 63, which are read out and added.
template <int kCtrl>
__device__ __forceinline__ float dpp_f_or_zero(float v) {   // the DPP source's bits, 0 where it has none
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp_f_or_zero<0x111>(v);   // row_shr:1
  v += dpp_f_or_zero<0x112>(v);   // row_shr:2
  v += dpp_f_or_zero<0x114>(v);   // row_shr:4
  v += dpp_f_or_zero<0x118>(v);   // row_shr:8
  return (lane_value(v, 15) + lane_value(v, 31)) + (lane_value(v, 47) + lane_value(v, 63));
}

// Lanes that must share a parameter before their terms are summed across the wave: a sum
// costs six cross-lane steps per channel, a lane's own LDS atomic one contended add.
// (512x512 16-spp adjoint of 64 materials and 4 lights: 6.21, 5.92, 5.87, 5.88 and 6.36 ms at 1, 8, 16,
// 32 and 65, the last of which never sums)
constexpr int kWaveSumMin = 16;

// Adds v[0..2] of every lane with `has` to sum 3 * key + c (add(index, value)), one key at a time: the lanes
// sharing a key are summed across the wave first (one atomic per channel) when there are at
// least kWaveSumMin of them, and add their own terms otherwise.  Wave-uniform call.
template <class Add>
__device__ __forceinline__ void wave_add3(Add add, bool has, int key, const float v[3]) {
  const int lane = (int)__lane_id();
  uint64_t act = __ballot(has);
  if (__popcll(act) < kWaveSumMin) {          // too few terms for any sum across the wave to pay
    if (has) {
      add(3 * key + 0, v[0]);
      add(3 * key + 1, v[1]);
      add(3 * key + 2, v[2]);
    }
    return;
  }
  while (act) {
    const int leader = __ffsll((unsigned long long)act) - 1;
    const int k = __builtin_amdgcn_readlane(key, leader);
    const bool sel = has && key == k;
    if (__popcll(__ballot(sel)) >= kWaveSumMin) {
      const float s0 = wave_sum(sel ? v[0] : 0.0f), s1 = wave_sum(sel ? v[1] : 0.0f), s2 = wave_sum(sel ? v[2] : 0.0f);
      if (lane == leader) {
        add(3 * k + 0, s0);
        add(3 * k + 1, s1);
        add(3 * k + 2, s2);
      }
    } else if (sel) {
      add(3 * k + 0, v[0]);
      add(3 * k + 1, v[1]);
      add(3 * k + 2, v[2]);
    }
    has = has && !sel;
    act = __ballot(has);
  }
}

template <int kSums>
__global__ __launch_bounds__(kRB, kRenderWaves) void k_backward(DevTree T, const float4 *__restrict__ shade,
                                                                 dr_render_params P, FrameK FK,
                                                                 const float *__restrict__ dl,
                                                                 double *__restrict__ g_albedo,
                                                                 double *__restrict__ g_emission,
                                                                 float *__restrict__ vtx_all,
                                                                 int *__restrict__ next_unit, int nblocks, int chunk,
                                                                 int unit_chunks, int levels, int maxv, int tight,
                                                                 int s0) {
  extern __shared__ __align__(16) uint32_t lds[];
  __shared__ LeafLds leaf_all[kRB / 64];
  LeafLds &leaf = leaf_all[threadIdx.x >> 6];
  leaf_lds_init(leaf);
  uint2 *stk = (uint2 *)lds + threadIdx.x;
  // this workgroup's slice of the scratch buffer: vertex records (and kSumsTight's queues)
  constexpr int kQueues = (kRB / 64) * kAdjointQueueWords;
  float *vtx = vtx_all + (size_t)blockIdx.x * ((size_t)maxv * kVtxWords * kRB + (kSums == kSumsTight ? kQueues : 0));
  uint32_t *beside = lds + levels * kStackWordsPerLevel * kRB;
  float *queues;
  if constexpr (kSums == kSumsTight) queues = vtx + (size_t)maxv * kVtxWords * kRB;
  else queues = (float *)beside;
  float *queue = queues + (threadIdx.x >> 6) * kAdjointQueueWords;   // [word][entry]
  // sums of nmat*3 albedo, then nlights*3 emission
  using Acc = std::conditional_t<kSums == kSumsFp64, double, float>;
  Acc *gacc = (Acc *)(kSums == kSumsTight ? beside : beside + kQueues);
  // (kSumsTight: of the last `tight` of them)
  const int ngrad = 3 * (P.nmat + P.nlights), nlds = kSums == kSumsTight ? tight : ngrad, first = ngrad - nlds;
  const int spp = P.fsaa_x * P.fsaa_y;
  const uint32_t samp0 = (uint32_t)(P.iteration > 1 ? P.iteration - 1 : 0) * (uint32_t)spp;
  const float spw = uni(1.0f / (((float)P.fsaa_x) * ((float)P.fsaa_y)));
  const int ns = min(spp - s0, kLaunchSamples);   // this launch's samples of a pixel, from s0 on
  const UDiv Dns = udiv_uniform((uint32_t)ns);
  const bool clip = P.cull_backfaces != 0;
  const bool origins = P.lens == DR_SPHERICAL_SEGMENT_LENS;
  const int lane = (int)__lane_id();
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (int t = threadIdx.x; t < nlds; t += kRB) gacc[t] = (Acc)0;
  __syncthreads();
  auto add = [&](int i, float v) {
    if (kSums != kSumsTight || i >= first) atomicAdd(&gacc[kSums == kSumsTight ? i - first : i], (Acc)v);
    else atomicAdd(i < 3 * P.nmat ? &g_albedo[i] : &g_emission[i - 3 * P.nmat], (double)v);
  };
  // units of unit_chunks chunks, numbered block by block
  const int nchunks = kBlockPixels * ns / chunk, parts = (nchunks + unit_chunks - 1) / unit_chunks;
  auto V_ = [&](int k, int w) -> float & { return vtx[((size_t)k * kVtxWords + w) * kRB + threadIdx.x]; };
  // sums t, t + step, ... into the FP64 gradients
  auto flush = [&](int t0, int step) {
    for (int t = t0; t < nlds; t += step) {
      Acc v;
      if constexpr (kSums != kSumsFp64) v = atomicExch(&gacc[t], (Acc)0);
      else v = gacc[t];
      if (v != (Acc)0) {
        const int i = first + t;
        if (i < 3 * P.nmat) atomicAdd(&g_albedo[i], (double)v);
        else atomicAdd(&g_emission[i - 3 * P.nmat], (double)v);
      }
    }
  };

  Path st;
  Walk w;
  w.state = kWalkIdle;            // the lane has no path
  w.leaf = kNoLeaf;
  int K = 0;                      // vertices recorded for the current path
  bool fin = false;               // the current path has ended; its albedo terms are pending
  float wdl[3] = {0, 0, 0};       // spw * dL/dI (* lens filter) of the current pixel
  // the wave's queue (wave-uniform): entries [qpos, qlen); the unit's next chunks [cnext, cend) of block `block`
  int qpos = 0, qlen = 0, block = 0, cnext = 0, cend = 0;
  int paths = 0;                  // ended since the wave last moved the FP32 sums out
  bool ended = false;
  // the vertex's reflection factor and dA/dalbedo, then the next bounce (or the path's end)
  auto advance = [&]() {
    const dr_material M = P.materials[st.mid];
    float f5 = 0.0f;
    const bool metal = st.kind == DR_METAL && st.has_sample;
    if (metal) f5 = schlick5(st.nu, st.sdir);
    for (int c = 0; c < 3; c++) V_(K - 1, 1 + c) = metal ? M.albedo[c] + (1.0f - M.albedo[c]) * f5 : M.albedo[c];
    V_(K - 1, 8) = metal ? 1.0f - f5 : 1.0f;
    V_(K - 1, 7) = st.has_sample ? st.sweight : 0.0f;
    if (!st.has_sample) { fin = true; return; }
    for (int c = 0; c < 3; c++) st.beta[c] = st.beta[c] * (V_(K - 1, 1 + c) * st.sweight);
    st.o = st.p;
    st.d = st.sdir;
    st.restrict_tri = st.h;
    st.layer++;
    st.phase = 0;
  };
  for (;;) {
    // ---- path updates of the finished casts, batched (the threshold in proportion to the busy
    // lanes, as in k_render_stream)
    bool fresh = false;           // the lane has a new ray
    const uint64_t dm = __ballot(w.state == kWalkDone);
    if (dm && __popcll(dm) * 64 >= __popcll(__ballot(w.state != kWalkIdle)) * kShadeMin) {
      bool lit = false;
      float ev[3] = {0.0f, 0.0f, 0.0f};
      int lkey = 0;
      if (w.state == kWalkDone) {
        bool photons = false;
        if (st.phase == 0) {
          if (!w.hit) fin = true;
          else {
            setup_vertex(P, FK, shade, w.h, w.d, st);
            V_(K, 0) = __int_as_float(st.mid);
            for (int c = 0; c < 4; c++) V_(K, 4 + c) = 0.0f;
            K++;
            photons = st.kind == DR_LAMBERT;
            if (!photons) advance();
          }
        } else {
          const V3 e = w.h.p - st.p;
          lit = w.hit && (w.h.id == st.h || (e.x * e.x + e.y * e.y + e.z * e.z) <= (8.0f * kVecEps));
          if (lit) {
            const dr_material M = P.materials[st.mid];
            const float *E = P.lights[st.light].emission;
            for (int c = 0; c < 3; c++) {
              V_(K - 1, 4 + c) += st.gl_k * E[c];
              ev[c] = wdl[c] * st.beta[c] * M.albedo[c] * st.gl_k;
            }
            lkey = P.nmat + st.light;
          }
          photons = true;
        }
        if (photons && !next_photon(P, st)) advance();
        fresh = !fin;
      }
      // dL/demission of this update's lit photons
      wave_add3(add, lit, lkey, ev);
      // dL/dalbedo of the paths that ended: S_k backwards, then beta_k forwards
      const uint64_t fm = __ballot(fin);
      if (fm) {
        if (fin) {
          float Ln[3] = {0, 0, 0};
          for (int k = K - 1; k >= 0; k--)
            for (int c = 0; c < 3; c++) {
              const float S = V_(k, 4 + c) + V_(k, 7) * Ln[c];
              Ln[c] = V_(k, 1 + c) * S;
              V_(k, 4 + c) = S;
            }
        }
        float beta[3] = {1, 1, 1};
        int kmax = fin ? K : 0;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) kmax = max(kmax, __shfl_xor(kmax, off));
        for (int k = 0; k < kmax; k++) {
          const bool has = fin && k < K;
          float av[3] = {0.0f, 0.0f, 0.0f};
          int m = 0;
          if (has) {
            m = __float_as_int(V_(k, 0));
            const float dA = V_(k, 8);
            for (int c = 0; c < 3; c++) {
              av[c] = wdl[c] * beta[c] * dA * V_(k, 4 + c);
              beta[c] = beta[c] * (V_(k, 1 + c) * V_(k, 7));
            }
          }
          wave_add3(add, has, m, av);
        }
        if (fin) { w.state = kWalkIdle; fin = false; }
        if (kSums != kSumsFp64 && (paths += __popcll(fm)) >= flush_paths(ns)) {
          flush(lane, 64);
          paths = 0;
        }
      }
    }
    // ---- the queue is empty: the next chunk of the unit, or the next unit
    if (qpos == qlen && !ended) {
      if (cnext == cend) {
        int unit = 0;
        if (lane == 0) unit = atomicAdd(next_unit, 1);
        unit = uni(unit);
        block = unit / parts;
        cnext = (unit - block * parts) * unit_chunks;
        cend = min(cnext + unit_chunks, nchunks);
        ended = block >= nblocks;
      }
      if (!ended) {
        if (lane < chunk) {
          const int q = cnext * chunk + lane;
          const int lp = (int)udiv((uint32_t)q, Dns);
          const PathStart ps = path_start(P, FK, block, lp, s0 + (q - lp * ns), samp0);
          const float *g = dl + 4 * ((size_t)kBlockPixels * block + lp);
          queue[0 * 64 + lane] = ps.d.x;
          queue[1 * 64 + lane] = ps.d.y;
          queue[2 * 64 + lane] = ps.d.z;
          queue[3 * 64 + lane] = __int_as_float((int)ps.pix);
          queue[4 * 64 + lane] = __int_as_float((int)ps.samp);
          // SphericalSegmentLense::getPixelColor scales the sample colour by its filter
          for (int c = 0; c < 3; c++) queue[(5 + c) * 64 + lane] = spw * g[c] * (origins ? P.lens_p[4 + c] : 1.0f);
          if (origins) {
            queue[8 * 64 + lane] = ps.o.x;
            queue[9 * 64 + lane] = ps.o.y;
            queue[10 * 64 + lane] = ps.o.z;
          }
        }
        __threadfence_block();
        qpos = 0;
        qlen = chunk;
        cnext++;
      }
    }
    // ---- idle lanes pop the next entries
    const uint64_t idle = __ballot(w.state == kWalkIdle);
    if (qpos < qlen && idle && (__popcll(idle) >= kAdjointRefillMin || idle == ~0ull)) {
      const int entry = qpos + __popcll(idle & below);
      const bool take = w.state == kWalkIdle && entry < qlen;
      qpos += __popcll(__ballot(take));
      if (take) {
        PathStart ps;
        ps.d = v3(queue[0 * 64 + entry], queue[1 * 64 + entry], queue[2 * 64 + entry]);
        ps.pix = (uint32_t)__float_as_int(queue[3 * 64 + entry]);
        ps.samp = (uint32_t)__float_as_int(queue[4 * 64 + entry]);
        for (int c = 0; c < 3; c++) wdl[c] = queue[(5 + c) * 64 + entry];
        ps.o = v3(P.cam[0], P.cam[1], P.cam[2]);
        if (origins) ps.o = v3(queue[8 * 64 + entry], queue[9 * 64 + entry], queue[10 * 64 + entry]);
        fresh = ps.pix != kNoPixel;            // (a pixel outside the image has no paths)
        if (fresh) w.state = kWalkTrace;
        begin_path(st, ps);
        K = 0;
      }
    }
    if (__ballot(w.state != kWalkIdle) == 0) {
      if (qpos == qlen && ended) break;
      continue;
    }
    if (fresh) walk_begin(T, w, st.o, st.d, st.restrict_tri, stk);
    if (w.state == kWalkTrace) walk_step(T, w, stk, kRB, nullptr);
    const uint64_t pm = __ballot(w.state == kWalkLeaf);
    if (pm && (__popcll(pm) * 64 >= __popcll(__ballot(w.state != kWalkIdle)) * kLeafMin ||
               __ballot(w.state == kWalkTrace) == 0))
      walk_leaf_wave(T, w, w.leaf != kNoLeaf, clip, leaf, nullptr, nullptr);
  }
  __syncthreads();
  flush(threadIdx.x, kRB);
}

// ------------------------------------------------------------------ batched requests
struct DevRequest {
  RenderArgs A;
  float *frame;
};

__global__ void k_zero(int *counter, int n) {
  for (int i = (int)threadIdx.x; i < n; i += (int)blockDim.x) counter[i] = 0;
}

// A request of a batch as a stream; `weight`: the relative cost of a tile.
struct StreamRequest {
  int req;
  float weight;
  StreamShape S;
};

// The streamed requests of one plugin set: persistent workgroups, spread over the requests by cost
// (first[workgroup]), each run one request's stream until its tiles are gone and then join the one
// with the most work left.  A workgroup waits for its longest path once per request it works on.
// (One block at a time from a queue of (request, blocks) items it did so for every block: 24 requests
// of 128^2 to 512^2 at 1 to 16 spp 8.5 -> 6.5 ms.)
template <class PathT>
__global__ __launch_bounds__(kRB, kRenderWaves) void k_batch_stream(const DevRequest *__restrict__ reqs,
                                                                    const StreamRequest *__restrict__ list, int n,
                                                                    const int *__restrict__ first,
                                                                    unsigned *__restrict__ next_tile, int levels,
                                                                    int refill_min) {
  extern __shared__ __align__(16) uint32_t lds[];
  __shared__ StreamLds sh;
  __shared__ int pick;
  int i = first[blockIdx.x];
  RenderCounters rc;
  for (;;) {
    i = uni(i);
    // the requests are read-only while the kernel runs: the constant address space keeps their loads scalar
    typedef const __attribute__((address_space(4))) DevRequest *ConstRequest;
    const StreamRequest E = list[i];
    const ConstRequest R = (ConstRequest)(uintptr_t)&reqs[uni(E.req)];
    const StreamShape S = {uni(E.S.ntiles), uni(E.S.tile_shift), uni(E.S.chunk), uni(E.S.slot_shift)};
    stream_paths<PathT, false>(&R->A, R->frame, 0, S, levels, next_tile + i, refill_min, lds, sh, nullptr, rc);
    // the request with the most work left
    if (threadIdx.x < 64) {
      int best = 0, at = -1;
      for (int j = (int)threadIdx.x; j < n; j += 64) {
        const int left = list[j].S.ntiles - (int)__hip_atomic_load(&next_tile[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int key = left > 0 ? __float_as_int((float)left * list[j].weight) : 0;   // (positive floats order as ints)
        if (key > best) { best = key; at = j; }
      }
      const int top = __builtin_amdgcn_readlane(wave_incl_max(best), 63);
      const uint64_t who = __ballot(top > 0 && best == top);
      if (threadIdx.x == 0) pick = -1;
      if (who && (int)threadIdx.x == __ffsll((unsigned long long)who) - 1) pick = at;
    }
    __syncthreads();
    i = pick;
    if (i < 0) break;
    __syncthreads();
  }
}

// Requests of more than kStreamMaxSpp samples a pixel: persistent workgroups drain a queue of (request,
// first block, block count) items, one block at a time.
template <class PathT>
__global__ __launch_bounds__(kRB, kRenderWaves) void k_batch(const DevRequest *__restrict__ reqs, const int4 *__restrict__ items,
                                                int nitems, int *__restrict__ counter, int levels, int refill_min) {
  extern __shared__ __align__(16) uint32_t lds[];
  __shared__ float acc[kBlockPixels * 3];
  __shared__ int next_job;
  __shared__ int item;
  __shared__ LeafLds leaf[kRB / 64];
  const BlockLds L = {(uint2 *)lds + threadIdx.x, (float *)(lds + levels * kStackWordsPerLevel * kRB), acc, &next_job,
                      leaf + (threadIdx.x >> 6), nullptr};
  leaf_lds_init(*L.leaf);
  for (;;) {
    if (threadIdx.x == 0) item = atomicAdd(counter, 1);
    __syncthreads();
    const int it = __builtin_amdgcn_readfirstlane(item);   // the same in every lane: scalar loads below
    __syncthreads();
    if (it >= nitems) break;
    const int4 w = items[it];
    const DevRequest &R = reqs[w.x];
    for (int b = w.y; b < w.y + w.z; b++) render_block<PathT>(R.A.T, R.A.tb, R.A.P, R.A.K, R.frame, b, L, refill_min);
  }
}

static int check_params(dr_scene s, const dr_render_params *p) {
  if (!s || !p) return fail(DR_ERR_ARG, "render: null scene or parameters");
  if (p->shading && p->shading->scene != s) return fail(DR_ERR_ARG, "render: shading tables of another scene");
  if (!p->shading && !s->has_materials)
    return fail(DR_ERR_ARG, "render: no material ids (dr_scene_set_materials or dr_render_params.shading)");
  const int max_mat = p->shading ? p->shading->max_mat : s->max_mat;
  if (p->width < 1 || p->height < 1 || p->fsaa_x < 1 || p->fsaa_y < 1 || p->max_bounces < 0 || p->max_bounces > 64)
    return fail(DR_ERR_ARG, "render: bad image size, subpixel grid or max_bounces");
  if ((int64_t)p->fsaa_x * p->fsaa_y > INT32_MAX) return fail(DR_ERR_ARG, "render: more than 2^31 - 1 samples a pixel");
  if (p->nlights < 0 || p->nlights > kMaxLights || (p->nlights > 0 && !p->lights))
    return fail(DR_ERR_ARG, "render: 0 <= nlights <= 16 with a light table required");
  if (!p->materials || p->nmat <= max_mat) return fail(DR_ERR_ARG, "render: material table smaller than the ids in use");
  if (!(p->rr_survive > 0.0f && p->rr_survive <= 1.0f)) return fail(DR_ERR_ARG, "render: rr_survive must be in (0, 1]");
  if (s->max_depth > kMaxTreeDepth) return fail(DR_ERR_ARG, "render: octree deeper than the traversal stack");
  if (p->lens != DR_STOCHASTIC_LENS && p->lens != DR_PERSPECTIVE_LENS && p->lens != DR_SPHERICAL_SEGMENT_LENS)
    return fail(DR_ERR_ARG, "render: unknown lens");
  if (p->plugins != DR_PLUGINS_BENCHMARK && p->plugins != DR_PLUGINS_REFERENCE)
    return fail(DR_ERR_ARG, "render: unknown plugin set");
  if (p->nmaps < 0 || p->ntextures < 0 || (p->nmaps > 0 && !p->maps) || (p->ntextures > 0 && (!p->textures || !p->texels)))
    return fail(DR_ERR_ARG, "render: texture tables missing");
  return DR_OK;
}

static int block_count(const dr_render_params *p) { return ((p->width + 7) / 8) * ((p->height + 15) / 16); }

// The shading tables a render reads: its dr_shading handle's, or the scene's own.
static Tables tables_of(dr_scene s, const dr_render_params *p) {
  if (p->shading) return {(const float4 *)p->shading->shade.p, (const float *)p->shading->faces.p};
  return {(const float4 *)s->shade.p, (const float *)s->faces.p};
}

}  // namespace dr

namespace dr {
// Allows launches of `kern` with `bytes` of dynamic LDS.  The limit belongs to the kernel, not to a launch:
// it is always set to all that the kernel's own arrays leave, never to one caller's size, which a launch
// from another thread, or a batch's launch for its largest request, could exceed.
static int allow_lds(const void *kern, size_t bytes) {
  if (bytes <= 64 * 1024) return DR_OK;
  hipFuncAttributes a;
  DR_HIP_CHECK(hipFuncGetAttributes(&a, kern));
  DR_HIP_CHECK(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes - (int)a.sharedSizeBytes));
  return DR_OK;
}

// Pixel slots of a stream, and the workgroups per CU of kernel `kern` with them.  Deep trees, whose
// stacks leave no room for all the slots beside the registers' three workgroups a CU, get half the
// slots if that gives a workgroup more (1080p 16 spp: 15.8 ms with 2,048 samples staged and three,
// 17.6 ms with 1,024 and three, 22.4 ms with 2,048 and two).
static int stream_slots(const void *kern, int levels, int spp, bool origins, int &slot_shift, int &per_cu) {
  slot_shift = stream_slot_shift(spp, kStreamSamples);
  const size_t all = stream_lds(levels, spp, slot_shift, origins);
  const int rc = allow_lds(kern, all);
  if (rc != DR_OK) return rc;
  DR_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kRB, all));
  if (per_cu < kRenderWaves && slot_shift > 3) {
    int more = 0;
    DR_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&more, kern, kRB,
                                                              stream_lds(levels, spp, slot_shift - 1, origins)));
    if (more > per_cu) {
      per_cu = more;
      slot_shift--;
    }
  }
  return DR_OK;
}

// The stream of `nblocks` blocks over `resident` workgroups.
// Tiles: 32 a workgroup, so that the last ones even out over the chip, but of at least 64 jobs: a
// tile costs an atomic on one address and its waves wait for its id.  (Whole blocks: 517x389 at
// 1 spp 968 us, 256x256 at 4 spp 461 us in one block per workgroup, 1080p at 16 spp 17.7 ms; so:
// 720 us, 308 us, 15.8 ms.  Tiles of 32 jobs: 910 us, 345 us; 8 a workgroup: 17.1 ms at 1080p.)
// Jobs a wave takes at a time: 1/32 of its share, between 8 and 64 (a wave's queue is its own: at
// the end of a small frame its entries wait while other waves are idle; 517x389 at 1 spp 784 us
// with 16, 715 us with 8), and a divisor of a tile's.
static StreamShape stream_shape(long long nblocks, int spp, int slot_shift, double resident) {
  StreamShape S;
  S.slot_shift = slot_shift;
  S.tile_shift = 7;
  while (S.tile_shift > 3 && (spp << S.tile_shift) >= 128 && (double)(nblocks << (7 - S.tile_shift)) < 32 * resident)
    S.tile_shift--;
  S.ntiles = (int)(nblocks << (7 - S.tile_shift));
  const double groups = std::min((double)S.ntiles, resident);
  const double per_wave = (double)nblocks * kBlockPixels * spp / (groups * (kRB / 64));
  S.chunk = 64;
  while (S.chunk > 8 && (S.chunk > per_wave / 32 || (spp << S.tile_shift) % S.chunk != 0)) S.chunk /= 2;
  return S;
}
// Whether a render of `nblocks` blocks up to block `end_block` takes the streamed kernels.
static bool streams(long long nblocks, int end_block, int spp) {
  return spp <= kStreamMaxSpp && (nblocks + 4) * kBlockPixels * spp < (1ll << 31) && end_block < (1 << 23);
}

static int launch_render(dr_scene s, const dr_render_params *p, float *frame, int start_block, int end_block,
                         unsigned long long *counts, void *stream) {
  int rc = check_params(s, p);
  if (rc != DR_OK) return rc;
  if (!frame || start_block < 0 || end_block > block_count(p) || start_block > end_block)
    return fail(DR_ERR_ARG, "dr_render_blocks: bad frame or block range");
  if (start_block == end_block) return DR_OK;
  const int levels = s->max_depth > 0 ? s->max_depth : 1;
  const Tables tb = tables_of(s, p);
  const bool ref = p->plugins == DR_PLUGINS_REFERENCE;
  const int spp = p->fsaa_x * p->fsaa_y;
  // streamed tiles (k_render_stream) unless the sample count or the stream length is too large or no
  // work counters are left for a captured launch; one block per workgroup otherwise
  const long long nrange = end_block - start_block;
  unsigned *work = nullptr;
  if (streams(nrange, end_block, spp) && (work = scene_work(s, (hipStream_t)stream)) != nullptr) {
    const bool origins = p->lens == DR_SPHERICAL_SEGMENT_LENS;
    auto kern = counts ? (ref ? k_render_stream<RefPath, true> : k_render_stream<BenchPath, true>)
                       : (ref ? k_render_stream<RefPath, false> : k_render_stream<BenchPath, false>);
    int slot_shift, per_cu;
    if ((rc = stream_slots((const void *)kern, levels, spp, origins, slot_shift, per_cu)) != DR_OK) return rc;
    const size_t lds_s = stream_lds(levels, spp, slot_shift, origins);
    const long long resident = (long long)s->num_cu * std::max(per_cu, 1);
    const StreamShape S = stream_shape(nrange, spp, slot_shift, (double)resident);
    const long long groups = std::min<long long>(S.ntiles, resident);
    hipLaunchKernelGGL(kern, dim3((unsigned)groups), dim3(kRB), lds_s, (hipStream_t)stream,
                       RenderArgs{s->tree, tb, *p, frame_k(*p)}, frame, start_block, S, levels, work, counts);
    DR_HIP_CHECK(hipGetLastError());
    return DR_OK;
  }
  const size_t lds = ((size_t)levels * kStackWordsPerLevel * kRB + (size_t)kBlockPixels * kRoundSamples * 3) * 4;
  auto kernel = counts ? (ref ? k_render<RefPath, true> : k_render<BenchPath, true>)
                       : (ref ? k_render<RefPath, false> : k_render<BenchPath, false>);
  if ((rc = allow_lds((const void *)kernel, lds)) != DR_OK) return rc;
  hipLaunchKernelGGL(kernel, dim3(end_block - start_block), dim3(kRB), lds, (hipStream_t)stream, s->tree, tb, *p,
                     frame_k(*p), frame, start_block, levels, counts);
  DR_HIP_CHECK(hipGetLastError());
  return DR_OK;
}
}  // namespace dr

extern "C" int dr_render_blocks(dr_scene s, const dr_render_params *p, float *frame, int start_block, int end_block,
                                void *stream) {
  return dr::launch_render(s, p, frame, start_block, end_block, nullptr, stream);
}

extern "C" int dr_render_stats(dr_scene s, const dr_render_params *p, float *frame, int start_block, int end_block,
                               uint64_t *counts, void *stream) {
  if (!counts) return dr::fail(DR_ERR_ARG, "dr_render_stats: null counters");
  return dr::launch_render(s, p, frame, start_block, end_block, (unsigned long long *)counts, stream);
}

namespace dr {

static decltype(&k_backward<kSumsFp64>) backward_kernel(int sums) {
  return sums == kSumsFp64 ? k_backward<kSumsFp64> : (sums == kSumsFp32 ? k_backward<kSumsFp32> : k_backward<kSumsTight>);
}
// Launch shape of the adjoint.
struct BackwardShape {
  int sums, nlds;         // kSums* of k_backward, and the sums it holds in LDS
  int levels, maxv;
  size_t lds, slice;      // LDS bytes, and bytes of one workgroup's slice of the scratch buffer
  int nblocks, groups, chunk, unit_chunks;
};
// Workgroups of the persistent grid: one per resident slot, at most one per 256 paths, and at
// most as many as `vtx_bytes` of vertex records hold.
static int backward_shape(dr_scene s, const dr_render_params *p, size_t vtx_bytes, BackwardShape &B) {
  B.levels = s->max_depth > 0 ? s->max_depth : 1;
  B.maxv = p->max_bounces + 1;
  B.nblocks = block_count(p);
  B.slice = (size_t)B.maxv * kVtxWords * kRB * sizeof(float);
  const size_t stacks = (size_t)B.levels * kStackWordsPerLevel * kRB * 4, queues = (kRB / 64) * (size_t)kAdjointQueueWords * 4;
  const size_t ngrad = 3 * (size_t)(p->nmat + p->nlights);
  if (stacks + 4 * ngrad > kLdsBytes) return fail(DR_ERR_ARG, "dr_backward: too many materials and lights for LDS");
  const size_t leaf = (kRB / 64) * sizeof(LeafLds), fixed = stacks + queues + leaf;
  auto per_cu_with = [&](size_t sums) { return std::min<size_t>(kRenderWaves, kLdsBytes / (fixed + sums)); };
  if (per_cu_with(8 * ngrad) > 0 && per_cu_with(8 * ngrad) >= per_cu_with(4 * ngrad)) B.sums = kSumsFp64;
  else B.sums = per_cu_with(4 * ngrad) > 0 ? kSumsFp32 : kSumsTight;
  B.nlds = (int)ngrad;
  B.lds = stacks + queues + (B.sums == kSumsFp64 ? 8 : 4) * ngrad;
  if (B.sums == kSumsTight) {
    B.nlds = (int)std::min(ngrad, (kLdsBytes - stacks - leaf) / 4);
    B.lds = stacks + 4 * (size_t)B.nlds;
    B.slice += queues;
  }
  const void *kern = (const void *)backward_kernel(B.sums);
  const int rc = allow_lds(kern, B.lds);
  if (rc != DR_OK) return rc;
  int per_cu = 0;
  DR_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kRB, B.lds));
  const long long resident = (long long)s->num_cu * std::max(per_cu, 1);
  const long long jobs = (long long)B.nblocks * kBlockPixels * std::min(kLaunchSamples, p->fsaa_x * p->fsaa_y);
  B.groups = (int)std::min<long long>({(jobs + kRB - 1) / kRB, resident, (long long)(vtx_bytes / B.slice)});
  // jobs a wave takes at a time: 1/32 of its share, between 8 and 64
  const long long per_wave = jobs / ((long long)std::max(B.groups, 1) * (kRB / 64));
  B.chunk = 64;
  while (B.chunk > 8 && B.chunk > per_wave / 32) B.chunk /= 2;
  B.unit_chunks = 1;
  while (jobs / B.chunk / B.unit_chunks + B.nblocks >= (1 << 30)) B.unit_chunks *= 2;
  return DR_OK;
}

static int check_backward(dr_scene s, const dr_render_params *p, const float *dl_dframe, const double *g_albedo,
                          const double *g_emission) {
  int rc = check_params(s, p);
  if (rc != DR_OK) return rc;
  if (!dl_dframe || !g_albedo || (p->nlights > 0 && !g_emission)) return fail(DR_ERR_ARG, "dr_backward: null buffers");
  if (p->plugins != DR_PLUGINS_BENCHMARK) return fail(DR_ERR_ARG, "dr_backward: only the benchmark plugin set has an adjoint");
  return DR_OK;
}

// Scratch of one adjoint launch: the unit counter, then `groups` vertex-record slices.
constexpr size_t kCounterBytes = 256;

static void launch_backward(dr_scene s, const dr_render_params *p, const float *dl, double *ga, double *ge,
                            void *scratch_mem, const BackwardShape &B, hipStream_t stream) {
  int *counter = (int *)scratch_mem;
  float *vtx = (float *)((char *)scratch_mem + kCounterBytes);
  const int spp = p->fsaa_x * p->fsaa_y;
  for (int s0 = 0; s0 < spp; s0 += std::min(spp - s0, kLaunchSamples)) {
    hipLaunchKernelGGL(k_zero, dim3(1), dim3(64), 0, stream, counter, 1);
    hipLaunchKernelGGL(backward_kernel(B.sums), dim3(B.groups), dim3(kRB), B.lds, stream, s->tree, tables_of(s, p).shade,
                       *p, frame_k(*p), dl, ga, ge, vtx, counter, B.nblocks, B.chunk, B.unit_chunks, B.levels, B.maxv,
                       B.nlds, s0);
  }
}

}  // namespace dr

namespace dr {

// Unit counter and vertex records of dr_backward_noalloc: a file-scope device array
// (kNoAllocBytes on every device the library runs on, held until the process ends).  Host
// code never passes `scratch` itself (its host-side name is not a device address): it
// passes the address hipGetSymbolAddress gives for the current device, resolved once per
// device.
constexpr size_t kNoAllocBytes = 40u << 20;
static __device__ __align__(256) float scratch[kNoAllocBytes / sizeof(float)];
constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static float *g_scratch_ptr[kMaxDevices] = {};

int noalloc_scratch_init(int device, float **out) {
  if (device < 0 || device >= kMaxDevices) return fail(DR_ERR_ARG, "dr_backward_noalloc: device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      return fail(DR_ERR_HIP, std::string("dr_backward_noalloc: scratch address: ") + hipGetErrorString(e));
    g_scratch_ptr[device] = (float *)ptr;
  }
  if (out) *out = g_scratch_ptr[device];
  return DR_OK;
}

}  // namespace dr

extern "C" int dr_backward_noalloc(dr_scene s, const dr_render_params *p, const float *dl_dframe, double *g_albedo,
                                   double *g_emission, void *stream) {
  int rc = dr::check_backward(s, p, dl_dframe, g_albedo, g_emission);
  if (rc != DR_OK) return rc;
  int device = 0;
  // as many persistent workgroups as the array holds vertex records for (after the unit counter)
  dr::BackwardShape B;
  if ((rc = dr::backward_shape(s, p, dr::kNoAllocBytes - dr::kCounterBytes, B)) != DR_OK) return rc;
  if (B.slice > dr::kNoAllocBytes - dr::kCounterBytes)
    return dr::fail(DR_ERR_ARG, "dr_backward_noalloc: one workgroup's vertex records exceed the 40 MiB scratch array");
  DR_HIP_CHECK(hipGetDevice(&device));
  float *mem = nullptr;
  if ((rc = dr::noalloc_scratch_init(device, &mem)) != DR_OK) return rc;
  dr::launch_backward(s, p, dl_dframe, g_albedo, g_emission, mem, B, (hipStream_t)stream);
  DR_HIP_CHECK(hipGetLastError());
  return DR_OK;
}

extern "C" int dr_backward(dr_scene s, const dr_render_params *p, const float *dl_dframe, double *g_albedo,
                           double *g_emission, void *stream) {
  int rc = dr::check_backward(s, p, dl_dframe, g_albedo, g_emission);
  if (rc != DR_OK) return rc;
  dr::BackwardShape B;
  if ((rc = dr::backward_shape(s, p, SIZE_MAX, B)) != DR_OK) return rc;
  // unit counter and vertex records: the scene's buffer for this stream, grown when a call needs more
  void *mem = nullptr;
  if ((rc = dr::scene_scratch(s, (hipStream_t)stream, dr::kCounterBytes + (size_t)B.groups * B.slice, &mem)) != DR_OK)
    return rc;
  dr::launch_backward(s, p, dl_dframe, g_albedo, g_emission, mem, B, (hipStream_t)stream);
  DR_HIP_CHECK(hipGetLastError());
  return DR_OK;
}

// ------------------------------------------------------------------ batch host side
struct dr_batch_s {
  int num_cu = 1;
  int levels = 1;                  // of the deepest tree
  dr_batch_tuning tuning{1, 1, 1};
  dr::DevBuf reqs, counters;       // counters: one per streamed request and plugin set, then one per item queue
  struct Streams {                 // the streamed requests of a plugin set
    int n = 0;
    size_t lds = 0;
    dr::DevBuf list, first;
  } streams[2];
  struct Items {                   // work items of the others
    int n = 0;
    dr::DevBuf list;
  } items[2];
  std::vector<dr::DevRequest> host_reqs;
  std::vector<char> streamed;        // per request: takes the streamed kernels
  std::vector<dr_scene> scenes;      // references held until dr_batch_destroy
  std::vector<dr_shading> shadings;
  hipStream_t cap_stream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

namespace dr {

static size_t batch_lds(int levels) {
  return ((size_t)levels * kStackWordsPerLevel * kRB + (size_t)kBlockPixels * kRoundSamples * 3) * 4;
}
static bool request_streams(const dr_render_params &P) {
  const int nb = block_count(&P);
  return streams(nb, nb, P.fsaa_x * P.fsaa_y);
}
// Relative cost of a pixel of a request.
static double pixel_cost(const dr_render_params &P) {
  return (double)P.fsaa_x * P.fsaa_y * (1.0 + P.max_bounces) * (1.0 + P.nlights);
}

// Queue of (request, first block, count) of the requests of plugin set `set` (0 =
// benchmark, 1 = reference) that are not streamed, heaviest per-block cost first.
static std::vector<int4> make_items(dr_batch b, int tile, int set) {
  const std::vector<DevRequest> &R = b->host_reqs;
  std::vector<std::pair<double, int4>> v;
  for (int r = 0; r < (int)R.size(); r++) {
    const dr_render_params &P = R[r].A.P;
    if ((P.plugins == DR_PLUGINS_REFERENCE) != (set == 1) || b->streamed[r]) continue;
    const int nb = block_count(&P);
    for (int b = 0; b < nb; b += tile)
      v.push_back({pixel_cost(P) * std::min(tile, nb - b), make_int4(r, b, std::min(tile, nb - b), 0)});
  }
  std::stable_sort(v.begin(), v.end(), [](const std::pair<double, int4> &a, const std::pair<double, int4> &b) {
    return a.first > b.first;
  });
  std::vector<int4> out;
  out.reserve(v.size());
  for (auto &e : v) out.push_back(e.second);
  return out;
}

// The streamed requests of plugin set `set`: their shapes, and the request each workgroup starts with.
static int make_streams(dr_batch b, int set) {
  dr_batch_s::Streams &st = b->streams[set];
  const void *kern = set == 0 ? (const void *)k_batch_stream<BenchPath> : (const void *)k_batch_stream<RefPath>;
  std::vector<int> ids;
  double total = 0.0;
  for (int r = 0; r < (int)b->host_reqs.size(); r++) {
    const dr_render_params &P = b->host_reqs[r].A.P;
    if ((P.plugins == DR_PLUGINS_REFERENCE) != (set == 1) || !b->streamed[r]) continue;
    ids.push_back(r);
    total += pixel_cost(P) * block_count(&P);
  }
  st.n = (int)ids.size();
  if (st.n == 0) return DR_OK;
  const int grid = b->num_cu * b->tuning.groups_per_cu;
  std::vector<StreamRequest> list(st.n);
  std::vector<int> first(grid);
  double before = 0.0;
  for (int i = 0, g = 0; i < st.n; i++) {
    const dr_render_params &P = b->host_reqs[ids[i]].A.P;
    const int spp = P.fsaa_x * P.fsaa_y;
    const bool origins = P.lens == DR_SPHERICAL_SEGMENT_LENS;
    int slot_shift, per_cu;
    const int rc = stream_slots(kern, b->levels, spp, origins, slot_shift, per_cu);
    if (rc != DR_OK) return rc;
    st.lds = std::max(st.lds, stream_lds(b->levels, spp, slot_shift, origins));
    const double cost = pixel_cost(P) * block_count(&P);
    list[i].req = ids[i];
    list[i].S = stream_shape(block_count(&P), spp, slot_shift, std::max(1.0, grid * cost / total));
    list[i].weight = (float)(pixel_cost(P) * (1 << list[i].S.tile_shift));
    before += cost;
    // workgroup g starts with the request that holds the share (g + 1/2) / grid of the cost
    for (; g < grid && (i == st.n - 1 || (g + 0.5) * total < before * grid); g++) first[g] = i;
  }
  int rc = dev_upload(st.list, list.data(), list.size() * sizeof(StreamRequest));
  if (rc == DR_OK) rc = dev_upload(st.first, first.data(), first.size() * sizeof(int));
  return rc;
}

// Counter resets, then the persistent kernels of the plugin sets that have requests (one after the
// other on the stream).
static int launch_batch(dr_batch b, hipStream_t stream) {
  int *counters = (int *)b->counters.p;
  const int n0 = b->streams[0].n, ncounters = n0 + b->streams[1].n + 2;
  const DevRequest *reqs = (const DevRequest *)b->reqs.p;
  hipLaunchKernelGGL(k_zero, dim3(1), dim3(256), 0, stream, counters, ncounters);
  const dim3 grid(b->num_cu * b->tuning.groups_per_cu);
  for (int set = 0; set < 2; set++) {
    const dr_batch_s::Streams &st = b->streams[set];
    if (st.n == 0) continue;
    hipLaunchKernelGGL(set == 0 ? k_batch_stream<BenchPath> : k_batch_stream<RefPath>, grid, dim3(kRB), st.lds, stream, reqs,
                       (const StreamRequest *)st.list.p, st.n, (const int *)st.first.p,
                       (unsigned *)counters + (set == 0 ? 0 : n0), b->levels, b->tuning.refill_min);
  }
  for (int set = 0; set < 2; set++) {
    const dr_batch_s::Items &it = b->items[set];
    if (it.n == 0) continue;
    const int rc = allow_lds(set == 0 ? (const void *)k_batch<BenchPath> : (const void *)k_batch<RefPath>, batch_lds(b->levels));
    if (rc != DR_OK) return rc;
    hipLaunchKernelGGL(set == 0 ? k_batch<BenchPath> : k_batch<RefPath>, grid, dim3(kRB), batch_lds(b->levels), stream, reqs,
                       (const int4 *)it.list.p, it.n, counters + ncounters - 2 + set, b->levels, b->tuning.refill_min);
  }
  DR_HIP_CHECK(hipGetLastError());
  return DR_OK;
}

static void free_lists(dr_batch b) {
  dev_free(b->reqs);
  for (int set = 0; set < 2; set++) {
    dev_free(b->items[set].list);
    dev_free(b->streams[set].list);
    dev_free(b->streams[set].first);
  }
  dev_free(b->counters);
}

// Uploads what a launch with b->tuning reads.
static int upload_lists(dr_batch b) {
  int rc = dev_upload(b->reqs, b->host_reqs.data(), b->host_reqs.size() * sizeof(DevRequest));
  for (int set = 0; set < 2 && rc == DR_OK; set++) {
    const std::vector<int4> items = make_items(b, b->tuning.tile_blocks, set);
    b->items[set].n = (int)items.size();
    rc = dev_upload(b->items[set].list, items.data(), items.size() * sizeof(int4));
    if (rc == DR_OK) rc = make_streams(b, set);
  }
  const std::vector<int> zeros(b->streams[0].n + b->streams[1].n + 2, 0);
  return rc == DR_OK ? dev_upload(b->counters, zeros.data(), zeros.size() * sizeof(int)) : rc;
}

// The shorter of two launches with the tuning t, in ms.
static int time_tuning(dr_batch b, const dr_batch_tuning &t, hipStream_t stream, float &ms) {
  b->tuning = t;
  hipEvent_t e[3] = {nullptr, nullptr, nullptr};
  int rc = upload_lists(b);
  for (int k = 0; k < 3 && rc == DR_OK; k++)
    if (hipEventCreate(&e[k]) != hipSuccess) rc = fail(DR_ERR_HIP, "dr_batch_create: event");
  for (int k = 0; k < 3 && rc == DR_OK; k++) {
    if (hipEventRecord(e[k], stream) != hipSuccess) rc = fail(DR_ERR_HIP, "dr_batch_create: event");
    else if (k < 2) rc = launch_batch(b, stream);
  }
  if (hipStreamSynchronize(stream) != hipSuccess && rc == DR_OK) rc = fail(DR_ERR_HIP, "dr_batch_create: timing");
  float a = 0.0f, c = 0.0f;
  if (rc == DR_OK && (hipEventElapsedTime(&a, e[0], e[1]) != hipSuccess || hipEventElapsedTime(&c, e[1], e[2]) != hipSuccess))
    rc = fail(DR_ERR_HIP, "dr_batch_create: timing");
  ms = std::min(a, c);
  for (hipEvent_t x : e)
    if (x) (void)hipEventDestroy(x);
  free_lists(b);
  return rc;
}

// Chooses the launch shape of `b` by timed launches of a proxy: its requests into scratch frames, with fewer
// samples a pixel (about kProxySamples in all, but one a pixel) where they have more.  From as many workgroups as the registers allow
// and the streamed kernels' refill, one step at a time: workgroups a CU, idle lanes before a refill, and
// the blocks of a queue item where there is a queue.  A change has to give kTuneGain on the proxy, which
// cannot rank closer ones: 3 workgroups a CU are the best of 1, 2, 3, 4, 6 or within 2% of it on batches of
// 24 requests (5.18 ms) to one 1024x1024 frame (0.48 ms), and 16 requests of 32 to 128 pixels take
// 0.397 ms with 3, 0.378 ms with 2.
constexpr double kProxySamples = 1e6, kTuneGain = 0.95;
static int autotune(dr_batch b) {
  dr_batch_s proxy;
  proxy.num_cu = b->num_cu;
  proxy.levels = b->levels;
  proxy.host_reqs = b->host_reqs;
  proxy.streamed = b->streamed;                 // each request in the kernel it takes uncut
  double samples = 0.0;
  for (const DevRequest &r : b->host_reqs) samples += (double)r.A.P.width * r.A.P.height * r.A.P.fsaa_x * r.A.P.fsaa_y;
  const double cut = std::sqrt(std::min(1.0, kProxySamples / samples));
  size_t bytes = 0;
  for (DevRequest &r : proxy.host_reqs) {
    dr_render_params &P = r.A.P;
    P.fsaa_x = std::max(1, (int)(P.fsaa_x * cut));
    P.fsaa_y = std::max(1, (int)(P.fsaa_y * cut));
    P.iteration = 1;
    r.A.K = frame_k(P);
    bytes += (size_t)block_count(&P) * kBlockPixels * 16;
  }
  dr_batch_tuning best{1, kRenderWaves, BenchPath::kStreamRefillMin};
  DevBuf frames;
  if (hipMalloc(&frames.p, bytes) != hipSuccess) {   // no room to try others
    (void)hipGetLastError();
    b->tuning = best;
    return DR_OK;
  }
  char *at = (char *)frames.p;
  for (DevRequest &r : proxy.host_reqs) {
    r.frame = (float *)at;
    at += (size_t)block_count(&r.A.P) * kBlockPixels * 16;
  }
  // the proxy reads the requests' tables, which a stream of the caller may still be filling
  if (hipDeviceSynchronize() != hipSuccess) {
    dev_free(frames);
    return fail(DR_ERR_HIP, "dr_batch_create: synchronize");
  }
  float best_ms = 0.0f;
  int rc = time_tuning(&proxy, best, b->cap_stream, best_ms);
  const struct { int32_t dr_batch_tuning::*field; int values[2]; } axes[] = {
      {&dr_batch_tuning::groups_per_cu, {2, 4}}, {&dr_batch_tuning::refill_min, {1, 8}}, {&dr_batch_tuning::tile_blocks, {2, 4}}};
  for (const auto &axis : axes) {
    if (axis.field == &dr_batch_tuning::tile_blocks && std::count(b->streamed.begin(), b->streamed.end(), 0) == 0) continue;
    const dr_batch_tuning base = best;
    for (int v : axis.values) {
      if (rc != DR_OK) break;
      dr_batch_tuning t = base;
      t.*axis.field = v;
      float ms = 0.0f;
      rc = time_tuning(&proxy, t, b->cap_stream, ms);
      if (rc == DR_OK && ms < kTuneGain * best_ms) { best_ms = ms; best = t; }
    }
  }
  dev_free(frames);
  b->tuning = best;
  return rc;
}

}  // namespace dr

extern "C" int dr_batch_create(const dr_request *reqs, int n, const dr_batch_tuning *tuning, dr_batch *out) {
  if (!reqs || n < 1 || !out) return dr::fail(DR_ERR_ARG, "dr_batch_create: bad arguments");
  *out = nullptr;
  dr_batch b = new (std::nothrow) dr_batch_s();
  if (!b) return dr::fail(DR_ERR_ALLOC, "dr_batch_create: out of host memory");
  int rc = DR_OK;
  for (int r = 0; r < n && rc == DR_OK; r++) {
    rc = dr::check_params(reqs[r].scene, &reqs[r].params);
    if (rc == DR_OK && !reqs[r].frame) rc = dr::fail(DR_ERR_ARG, "dr_batch_create: null frame");
    if (rc != DR_OK) break;
    dr::DevRequest d;
    d.A = {reqs[r].scene->tree, dr::tables_of(reqs[r].scene, &reqs[r].params), reqs[r].params, dr::frame_k(reqs[r].params)};
    dr::scene_retain(reqs[r].scene);
    b->scenes.push_back(reqs[r].scene);
    if (reqs[r].params.shading) {
      dr::shading_retain(reqs[r].params.shading);
      b->shadings.push_back(reqs[r].params.shading);
    }
    d.frame = reqs[r].frame;
    b->host_reqs.push_back(d);
    b->streamed.push_back(dr::request_streams(d.A.P));
    b->levels = std::max(b->levels, reqs[r].scene->max_depth);
  }
  if (rc == DR_OK) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&b->num_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) b->num_cu = 1;
    if (hipStreamCreate(&b->cap_stream) != hipSuccess) rc = dr::fail(DR_ERR_HIP, "dr_batch_create: stream");
  }
  if (rc == DR_OK) {
    if (tuning) b->tuning = *tuning;
    else rc = dr::autotune(b);
    if (rc == DR_OK && (b->tuning.tile_blocks < 1 || b->tuning.groups_per_cu < 1 || b->tuning.refill_min < 1))
      rc = dr::fail(DR_ERR_ARG, "dr_batch_create: tuning values must be >= 1");
  }
  if (rc == DR_OK) rc = dr::upload_lists(b);
  if (rc == DR_OK) {
    hipError_t e = hipStreamBeginCapture(b->cap_stream, hipStreamCaptureModeThreadLocal);
    if (e == hipSuccess) {
      rc = dr::launch_batch(b, b->cap_stream);
      hipError_t e2 = hipStreamEndCapture(b->cap_stream, &b->graph);
      if (rc == DR_OK && e2 != hipSuccess) rc = dr::fail(DR_ERR_HIP, "dr_batch_create: graph capture");
      if (rc == DR_OK && hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0) != hipSuccess)
        rc = dr::fail(DR_ERR_HIP, "dr_batch_create: graph instantiation");
    } else {
      rc = dr::fail(DR_ERR_HIP, std::string("dr_batch_create: capture: ") + hipGetErrorString(e));
    }
  }
  if (rc != DR_OK) { dr_batch_destroy(b); return rc; }
  *out = b;
  return DR_OK;
}

extern "C" int dr_batch_run(dr_batch b, void *stream) {
  if (!b || !b->exec) return dr::fail(DR_ERR_ARG, "dr_batch_run: bad batch");
  DR_HIP_CHECK(hipGraphLaunch(b->exec, (hipStream_t)stream));
  return DR_OK;
}

extern "C" int dr_batch_get_tuning(dr_batch b, dr_batch_tuning *out) {
  if (!b || !out) return dr::fail(DR_ERR_ARG, "dr_batch_get_tuning: bad arguments");
  *out = b->tuning;
  return DR_OK;
}

extern "C" void dr_batch_destroy(dr_batch b) {
  if (!b) return;
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  if (b->cap_stream) (void)hipStreamDestroy(b->cap_stream);
  dr::free_lists(b);
  for (dr_shading h : b->shadings) dr::shading_release(h);
  for (dr_scene sc : b->scenes) dr::scene_release(sc);
  delete b;
}
