// Batch closest-hit ray cast (Octree::cast over a ray batch, Octree.impl.cuh:174-212).
//
// A persistent grid of 256-lane blocks; each lane carries one ray and its own
// DFS stack in LDS.  The loop advances every traversing lane by one bounded step
// per iteration and batches the rarer, divergent work (leaf tests, taking new
// rays) until enough lanes need it; a leaf batch spreads the records of all
// pending leaves over the whole wave (walk_leaf_wave).
#include <algorithm>
#include "dr_common.h"

namespace dr {

constexpr int kCastBlock = 256;
constexpr int kWavesPerBlock = kCastBlock / 64;
constexpr int kWaveChunk = 128;       // most rays a wave takes from the global counter at a time
// idle lanes that trigger a refill (12, 16, 20, 24, 32: 4M incoherent rays 1225, 1222, 1217, 1217, 1217 us;
// 1080p primary rays 736, 746, 751, 727, 728 us)
constexpr int kRefillMin = 24;
// lanes waiting at a leaf that trigger the (wave-shared) leaf tests (1080p primary rays 731, 721, 718,
// 729 us with 4, 8, 10, 16; 4M incoherent rays 1215, 1227, 1231, 1238 us)
constexpr int kLeafMin = 4;
// ... and fewer in a wave with few rays left, which would otherwise hold each leaf until its slowest ray
__device__ __forceinline__ int leaf_min(int rays) { return min(kLeafMin, (5 * rays + 15) >> 4); }

constexpr double kManyRecords = 2048; // records a ray meets from which small batches go out over more waves

// One bounded step per loop iteration.  A lane that is traversing pops one child:
// an interior child is expanded and pushed, a leaf child is held and the walk goes on to
// the next leaf.  Held leaves are tested together once at least kLeafMin lanes wait at
// their next one (or no lane is still traversing), and idle lanes take new rays once kRefillMin of
// them are idle (or no lane is busy), so the node expansions, which dominate the
// work, run with most lanes of the wave active.
//
// Rays are handed out dynamically: a wave owns a range of `chunk` rays (kWaveChunk for a large
// batch, see launch_cast) taken from the global counter work[0]; lanes that need a ray take the next ones of the
// range, and the wave takes a new range when it runs out.  The last wave to exit
// (counted in work[1]) sets both counters back to zero for the next launch.
//
// Results are staged per range in LDS (kSlots ranges per wave) and written out as
// whole lines once no ray of the range is still being traced: rays end at scattered
// times, and 4-B stores issued as they end would leave L2 as partial sectors.  When a
// wave needs a slot for a new range while both hold unfinished ranges, the older one
// is written out as far as it is done, and its remaining rays store their results
// directly.
constexpr int kCastCounters = 6;     // per-ray counters of dr_cast_stats
constexpr int kSlots = 2;
constexpr int kPendingId = -2;        // staged entry of a ray still being traced

template <bool kStats>
__global__ __launch_bounds__(kCastBlock, 4) void k_cast(DevTree T, const float *__restrict__ rays, int n, int clip,
                                                      const int *__restrict__ exclude, int *__restrict__ out_id,
                                                      float *__restrict__ out_t, float *__restrict__ out_p,
                                                      int *__restrict__ stats, unsigned *__restrict__ work, int chunk) {
  extern __shared__ __align__(16) uint2 stk_base[];
  __shared__ LeafLds leaf_all[kWavesPerBlock];
  __shared__ int ins_all[kStats ? kCastBlock : 1];      // per lane: inside tests of its leaf (measurement)
  __shared__ int res_id_all[kWavesPerBlock][kSlots][kWaveChunk];
  __shared__ float res_t_all[kWavesPerBlock][kSlots][kWaveChunk];
  uint2 *stk = stk_base + threadIdx.x;
  LeafLds &leaf = leaf_all[threadIdx.x >> 6];
  leaf_lds_init(leaf);
  int *ins = kStats ? ins_all + (threadIdx.x & ~63u) : nullptr;
  int *res_id = &res_id_all[threadIdx.x >> 6][0][0];
  float *res_t = &res_t_all[threadIdx.x >> 6][0][0];
  constexpr int S = kCastBlock;

  const int lane = (int)__lane_id();
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  unsigned wcur = 0, wend = 0;          // the wave's current range of rays (wave-uniform)
  // staging slots (wave-uniform): slot k holds the results of range [base_k, base_k + len_k)
  // while len_k > 0; `cur` is the slot of the current range
  unsigned base0 = 0, base1 = 0;
  int len0 = 0, len1 = 0, cur = 0;
  int r = -1;
  bool exhausted = false;
  Walk w;
  w.state = kWalkIdle;          // the lane has no ray
  w.leaf = kNoLeaf;
  CastCounters cnt_local = {0, 0, 0, 0, 0, 0};
  CastCounters *cc = kStats ? &cnt_local : nullptr;
  auto finish = [&]() {
    const int id = w.hit ? w.h.id : -1;
    const float t = w.hit ? w.h.t : FLT_MAX;
    const unsigned u = (unsigned)r;
    if (len0 > 0 && u - base0 < (unsigned)len0) {
      res_id[u - base0] = id;
      res_t[u - base0] = t;
    } else if (len1 > 0 && u - base1 < (unsigned)len1) {
      res_id[kWaveChunk + (u - base1)] = id;
      res_t[kWaveChunk + (u - base1)] = t;
    } else {
      out_id[r] = id;
      out_t[r] = t;
    }
    if (out_p) {
      out_p[3 * (size_t)r + 0] = w.hit ? w.h.p.x : 0.0f;
      out_p[3 * (size_t)r + 1] = w.hit ? w.h.p.y : 0.0f;
      out_p[3 * (size_t)r + 2] = w.hit ? w.h.p.z : 0.0f;
    }
    if (kStats) {
      int *o = stats + kCastCounters * (size_t)r;
      o[0] = cnt_local.expand;
      o[1] = cnt_local.leaves;
      o[2] = cnt_local.plane;
      o[3] = cnt_local.inside;
      o[4] = cnt_local.live;
      o[5] = cnt_local.slab;
      cnt_local = {0, 0, 0, 0, 0, 0};
    }
    r = -1;
    w.state = kWalkIdle;
  };
  // writes the finished entries of slot k (range base, len) as whole lines (wave-uniform)
  auto flush = [&](int k, unsigned base, int len) {
    __builtin_amdgcn_wave_barrier();
    for (int j = lane; j < len; j += 64) {
      const int id = res_id[k * kWaveChunk + j];
      if (id != kPendingId) {
        out_id[base + j] = id;
        out_t[base + j] = res_t[k * kWaveChunk + j];
      }
    }
  };
  // a range whose rays have all been handed out and finished leaves its slot
  auto retire = [&](int k, unsigned base, int &len) {
    if (len > 0 && (k != cur || wcur == wend) &&
        __ballot(r >= 0 && (unsigned)r - base < (unsigned)len) == 0) {
      flush(k, base, len);
      len = 0;
    }
  };

  // The results, the staged ranges and the refill are looked at only after a ray has ended (or while
  // idle lanes wait for a range): most iterations end none.  Looked at in every one they were a sixth
  // of the loop's cycles, and three copies of finish() took registers (1M rays 502 -> 452 us, 99,991
  // bounce rays 186 -> 177 us, 4M incoherent rays 1.26 -> 1.24 ms).  Smaller ranges near the end of the
  // batch, to let the waves end together, cost more than they gave (1M rays 452 -> 499 us).
  bool look = true;
  // Lanes that take rays: of a short range no more than it holds.  (With all lanes taking, the waves that
  // start first found idle lanes and took the ranges of those still to start: 1,000 bounce rays 79 ->
  // 69 us, 16,000 111 -> 99 us, 1,000 rays of a view 46.4 -> 42 us.)
  const int width = min(chunk, 64);
  const uint64_t wide = ~0ull >> (64 - width);
  const unsigned refill_min = (unsigned)min(kRefillMin, max(1, (3 * width) >> 3));
  for (;;) {
    const bool done = w.state == kWalkDone;
    if (look || __ballot(done) != 0) {
      if (done) finish();
      retire(0, base0, len0);
      retire(1, base1, len1);
      // ---- refill idle lanes
      const uint64_t wmask = __ballot(w.state == kWalkIdle) & wide;
      const unsigned need = (unsigned)__popcll(wmask);
      const unsigned rem = wend - wcur;
      look = false;
      if (rem > 0 || !exhausted) {
        if (need >= refill_min) {
          const unsigned idx = (unsigned)__popcll(wmask & below);
          int slot = idx < rem ? (int)(wcur + idx) : -1;
          if (rem >= need) {
            wcur += need;
          } else if (exhausted) {
            wcur = wend;
          } else {
            unsigned nb = 0;
            if (lane == 0) nb = atomicAdd(work, (unsigned)chunk);
            nb = (unsigned)__builtin_amdgcn_readfirstlane((int)nb);   // wave-uniform: kept in scalar registers
            const unsigned top = min(nb + (unsigned)chunk, (unsigned)n);
            const unsigned len = nb < top ? top - nb : 0u;
            exhausted = nb + (unsigned)chunk >= (unsigned)n;
            if (idx >= rem && idx - rem < len) slot = (int)(nb + idx - rem);
            wcur = nb + min(need - rem, len);
            wend = nb + len;
            if (len > 0) {
              // the new range takes the slot the current range does not hold; an unfinished
              // range still there is written out as far as it is done
              const int k = (cur == 0 ? len0 : len1) > 0 ? 1 - cur : cur;
              if (k == 0 && len0 > 0) flush(0, base0, len0);
              if (k == 1 && len1 > 0) flush(1, base1, len1);
              __builtin_amdgcn_wave_barrier();
              for (int j = lane; j < (int)len; j += 64) res_id[k * kWaveChunk + j] = kPendingId;
              if (k == 0) { base0 = nb; len0 = (int)len; }
              else { base1 = nb; len1 = (int)len; }
              cur = k;
            }
          }
          if (w.state == kWalkIdle && lane < width && slot >= 0) {
            r = slot;
            const float2 *R = (const float2 *)(rays + 6 * (size_t)r);
            const float2 q0 = R[0], q1 = R[1], q2 = R[2];
            walk_begin(T, w, v3(q0.x, q0.y, q1.x), v3(q1.y, q2.x, q2.y), exclude ? exclude[r] : -1, stk);
          }
          look = (unsigned)__popcll(__ballot(w.state == kWalkIdle) & wide) >= refill_min;
        }
      }
      if (__ballot(w.state != kWalkIdle) == 0) {
        if (exhausted && wcur == wend) break;
        look = true;
        continue;
      }
    }
    // ---- one traversal step
    if (w.state == kWalkTrace) walk_step(T, w, stk, S, cc);

    // ---- castInLeaf for the pending leaves, the whole wave sharing their records
    const uint64_t pm = __ballot(w.state == kWalkLeaf);
    if (pm && (__popcll(pm) >= leaf_min(__popcll(__ballot(w.state != kWalkIdle))) || __ballot(w.state == kWalkTrace) == 0))
      walk_leaf_wave<true>(T, w, w.leaf != kNoLeaf, clip != 0, leaf, ins, cc);
  }
  // every ray of the wave has ended: the ranges still staged go out
  if (len0 > 0) flush(0, base0, len0);
  if (len1 > 0) flush(1, base1, len1);
  // ---- the last wave out resets the counters
  if (lane == 0) {
    __threadfence();
    const unsigned total = gridDim.x * (kCastBlock / 64);
    if (atomicAdd(work + 1, 1u) == total - 1) {
      atomicExch(work, 0u);
      atomicExch(work + 1, 0u);
    }
  }
}

static int launch_cast(dr_scene s, const float *rays, int n, unsigned flags, const int32_t *exclude, int32_t *out_id,
                       float *out_t, float *out_point, int32_t *stats, void *stream) {
  if (s->max_depth > kMaxTreeDepth) return fail(DR_ERR_ARG, "dr_cast: octree deeper than the traversal stack");
  if (n == 0) return DR_OK;
  const int levels = s->max_depth > 0 ? s->max_depth : 1;
  const int clip = (int)(flags & DR_CAST_CLIP_BACKFACES);
  const size_t lds = (size_t)levels * kStackWordsPerLevel * kCastBlock * sizeof(uint32_t);
  int per_cu = 0;
  DR_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_cast<false>, kCastBlock, lds));
  // (the registers would allow five, which share the caches worse: 4M incoherent rays 1.29 against
  // 1.24 ms, 400,000 bounce rays 935 against 893 us)
  per_cu = std::min(per_cu, 4);
  // Rays a wave takes at a time.  A batch that the chip can hold at once is bound by its longest ray:
  // it goes one ray a lane over as many waves as give every SIMD one, then over lanes (99,991 bounce
  // rays 246 us with 128 a wave, 228 us with 32, 191 us with 64; 4,096 rays 101 us with 128, 183 us
  // with 1 on four waves a SIMD, 81 us with 4 on one; 64 rays 46 -> 24 us; two or four waves a SIMD, with
  // as many lanes of each as the range holds: 4,096 bounce rays 112 and 177 us).  A larger one takes
  // whole ranges, with two of them staged.
  // Where a ray meets thousands of records (the reference's build stops at some grids), a wave spends its
  // time in their rounds, each a trip to memory that other waves of the SIMD hide: four waves a SIMD.
  // What counts is how many a ray can expect, not the longest leaf, which may be out of most rays' way.
  // Rays over a sphere mesh with one leaf of many records, and over a heightfield of 524,288 triangles;
  // one against four waves a SIMD:
  //   records met, in the longest leaf     4,096 rays      16,384         65,536
  //       8,    2,000                       68  /  166 us    66 /  182     101 /  208 us
  //      24,    8,084                      139  /  227      208 /  323     316 /  427
  //     147,   30,167                      639  /  739     1269 / 1383    1000 / 1123
  //     267,    2,285                      152  /  252      227 /  333     377 /  405
  //    2618,    9,237                      472  /  502      991 /  884    2407 / 1226
  //   10228,   35,491                     2353  / 1941     3884 / 3069    9938 / 5589
  //   63983,   87,368                     7366  / 2900    17736 / 9637   51498 / 26950
  const int waves = s->ray_records >= kManyRecords ? 16 : 4;
  int chunk = 1;
  while (chunk < 64 && (long long)chunk * s->num_cu * waves < n) chunk *= 2;
  if ((long long)n > 2LL * 64 * kWavesPerBlock * s->num_cu * std::max(per_cu, 1)) chunk = kWaveChunk;
  // persistent grid: at most one block per resident slot, fewer for small batches
  const long long need = ((long long)n + kWavesPerBlock * chunk - 1) / (kWavesPerBlock * chunk);
  const int blocks = (int)std::max(1LL, std::min<long long>(need, (long long)s->num_cu * std::max(per_cu, 1)));
  unsigned *work = scene_work(s, (hipStream_t)stream);
  if (!work) work = (unsigned *)s->work.p + 2 * s->work_slots.eager();   // (casts have no kernel without counters)
  if (stats)
    hipLaunchKernelGGL(k_cast<true>, dim3(blocks), dim3(kCastBlock), lds, (hipStream_t)stream, s->tree, rays, n, clip,
                       (const int *)exclude, (int *)out_id, out_t, out_point, (int *)stats, work, chunk);
  else
    hipLaunchKernelGGL(k_cast<false>, dim3(blocks), dim3(kCastBlock), lds, (hipStream_t)stream, s->tree, rays, n,
                       clip, (const int *)exclude, (int *)out_id, out_t, out_point, (int *)nullptr, work, chunk);
  DR_HIP_CHECK(hipGetLastError());
  return DR_OK;
}

}  // namespace dr

extern "C" int dr_cast(dr_scene s, const float *rays, int n, unsigned flags, const int32_t *exclude, int32_t *out_id,
                       float *out_t, float *out_point, void *stream) {
  if (!s || n < 0 || (n > 0 && (!rays || !out_id || !out_t))) return dr::fail(DR_ERR_ARG, "dr_cast: bad arguments");
  return dr::launch_cast(s, rays, n, flags, exclude, out_id, out_t, out_point, nullptr, stream);
}

extern "C" int dr_cast_stats(dr_scene s, const float *rays, int n, unsigned flags, const int32_t *exclude,
                             int32_t *out_id, float *out_t, int32_t *out_counts, void *stream) {
  if (!s || n < 0 || (n > 0 && (!rays || !out_id || !out_t || !out_counts)))
    return dr::fail(DR_ERR_ARG, "dr_cast_stats: bad arguments");
  return dr::launch_cast(s, rays, n, flags, exclude, out_id, out_t, nullptr, out_counts, stream);
}
