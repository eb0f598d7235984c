// render_common.h -- ray state, compositing and host helpers shared by the
// full renderer (render.hip) and the cache renderers (cache.hip).
#pragma once
#include "fvc_internal.h"
#include "march.h"
#include "wave.h"

namespace fvc {

// BaseRayInitInfo + SegmentedRayPayload of the reference
// (renderer_common.h:65-88) in one 48-byte record: origin, direction, far,
// next bin start t, and the bin position in the step table (start index m,
// bins advanced j, so t == T[m][j]).
struct RayState {
  float ox, oy, oz, dx, dy, dz, far_, t;
  int m, j;
  int scene;  // scene of the ray's view (mixed-scene batches; else 0)
  int pad;
};
// Where a ray stands between sub-iterations: next bin start t == T[m][j].
// The alive list compacts this and the pixel index; the rest of the ray
// (RayState, written once per frame at its pixel) stays in place.
struct RayDyn {
  float t;
  int j;
};

// Ray of pixel (x, y) clipped to the scene AABB, its start snapped by
// valid_t_from_t with the bin index kept: t = t_from_step(m + near_i)
// (initRayPayloads_split_kernel, renderer.cu:86-134, deterministic branch).
// Returns false when the ray misses the AABB.
__device__ __forceinline__ bool init_ray_state(const fvc_raymarch_info& rm, V3 aabb_from, V3 aabb_to, int x, int y,
                                               RayState& st) {
  const Ray r = gen_ray(rm.cam_info, (float)x + 0.5f, (float)y + 0.5f);
  float t0, t1;
  const bool hit = ray_aabb(r, aabb_from, aabb_to, t0, t1);
  const fvc_stepsize_info& s = rm.stepsize_info;
  st.ox = r.o.x; st.oy = r.o.y; st.oz = r.o.z;
  st.dx = r.d.x; st.dy = r.d.y; st.dz = r.d.z;
  st.far_ = hit ? fminf_(t1, s.far_) : s.far_;
  const float mf = hit ? roundf(step_from_t(s, fmaxf_(t0, s.near_)) - s.near_i) : 0.0f;
  st.t = hit ? t_from_step(s, mf + s.near_i) : s.near_;
  st.m = (int)mf;
  st.j = 0;
  st.scene = st.pad = 0;
  return hit;
}

__device__ __forceinline__ MarchRay march_ray(const RayState& s, const StepTableView& tab) {
  MarchRay r;
  r.row = step_row(tab, s.m);
  r.o = V3{s.ox, s.oy, s.oz};
  r.d = V3{s.dx, s.dy, s.dz};
  r.slab = ray_slab(r.o, r.d);
  r.far_ = s.far_;
  r.m = s.m;
  r.j = s.j;
  r.t1 = s.t;
  r.sk = no_skip();
  return r;
}

// samples a compositing lane loads ahead
static const int COMPOSITE_BATCH = 16;

// slots of Renderer::counters
enum { CNT_ALIVE = 0, CNT_SAMPLES = 1, CNT_CACHE = 2, CNT_STEPS = 3, CNT_TILES = 4, CNT_OVERFLOW = 6,
       CNT_SLOTS = 8 /* and 9 */ };

// Device control block of a frame's sub-iteration loop (also in
// Renderer::counters): one record per iteration, all zero when the frame
// starts.  Iteration it's marcher reads its alive count, plans the samples per
// ray from it and counts the samples and bins; its composite counts the rays
// left into the next record.  The host launches iterations in bursts, reads
// the alive count once per burst and the records at the end.
// (A kernel of its own that planned each iteration took 4 us and a launch gap:
// 256x256 1580 -> 1533 us a frame, 1279x717 1355 -> 1330, 1920x1080 11735 ->
// 11675.)
enum { CTL_LOG = 32 };
enum { LOG_ALIVE = 0, LOG_STEPS = 1, LOG_R = 2, LOG_C = 3, LOG_BINS = 4 };
static const int CTL_LOG_FIELDS = 5;
static const int MAX_SUBITER = 1000;        // PerformanceRenderer::MAX_SUBITER
static const int CTL_WORDS = CTL_LOG + CTL_LOG_FIELDS * (MAX_SUBITER + 1);
inline int ctl_at(int it, int field) { return CTL_LOG + CTL_LOG_FIELDS * it + field; }

// Samples per ray of an iteration: TARGET_BATCH_SIZE / n_alive clamped to
// [1, max_steps] and to the stream capacity (performance_renderer.cu:249-250).
struct StepPlan { int target, max_steps, cap; };
inline StepPlan step_plan(int64_t target, int max_steps, int64_t cap) {
  const int64_t top = 0x7fffffff;
  return StepPlan{(int)std::min(target, top), max_steps, (int)std::min(cap, top)};
}
FVC_HD int plan_steps(const StepPlan& p, int n) {
  int k = p.target / (n > 1 ? n : 1);
  k = k < 1 ? 1 : (k > p.max_steps ? p.max_steps : k);
  if (n > 0 && (int64_t)n * k > p.cap) k = p.cap / n > 1 ? p.cap / n : 1;
  return k;
}

inline CacheView cache_view(const CacheStore& C) {
  CacheView cv;
  cv.cam = C.rm.cam_info;
  cv.st = C.rm.stepsize_info;
  cv.fx = C.fx; cv.fy = C.fy; cv.fz = C.fz; cv.bx = C.bx; cv.by = C.by;
  cv.table = C.table.as<int>();
  cv.known = C.known.as<float>();
  cv.pool = C.pool.as<Voxel>();
  cv.pool8 = C.pool.as<Voxel8>();
  cv.scales = C.scales.as<float>();
  cv.lat8 = C.lat8 ? 1 : 0;
  cv.interp_fn = FVC_FN_LINEAR;
  cv.inter_brick = 1;
  return cv;
}

// Class of an occupied sample [t0, t0 + dt) of a ray whose origin / direction
// in the cache camera's frame are oc / dc (sample_cache_performance_kernel,
// cache_performance_renderer.cu:96-160): SAMPLE_RESAMPLE outside the cache
// frustum or outside [near, known_to] of its pixel, SAMPLE_CACHE when the
// nearest voxel's brick is set and its density is > 0, else SAMPLE_SKIP.
enum { SAMPLE_SKIP = 0, SAMPLE_RESAMPLE = 1, SAMPLE_CACHE = 2 };
__device__ __forceinline__ int classify_sample(const CacheView& cv, V3 oc, V3 dc, float t0, float dt) {
  const float t1 = t0 + dt;
  const float tm = (t0 + t1) * 0.5f;
  float tf;
  const V3 f = cam2froxel(oc + tm * dc, cv.cam, cv.st, tf);
  const bool in_fov = f.x >= 0.0f && f.x < (float)cv.fx && f.y >= 0.0f && f.y < (float)cv.fy;
  const bool inside = in_fov && f.z >= 0.0f && f.z < (float)cv.fz;
  bool unsampled = true;
  if (in_fov) {
    const float known = cv.known[(int64_t)(int)f.y * cv.fx + (int)f.x];
    unsampled = tf < cv.st.near_ || tf > known;
  }
  if (!inside || unsampled) return SAMPLE_RESAMPLE;
  const int vx = (int)floorf(f.x), vy = (int)floorf(f.y), vz = (int)floorf(f.z);
  const int slot = cv.table[((int64_t)(vz >> 3) * cv.by + (vy >> 3)) * cv.bx + (vx >> 3)];
  if (slot >= 0 && vox_density(cv, (int64_t)slot * BRICK_VOXELS + brick_voxel(vx, vy, vz)) > 0.0f)
    return SAMPLE_CACHE;
  return SAMPLE_SKIP;
}

__device__ __forceinline__ float h2f(uint32_t bits16) { return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16); }

// Lanes per ray of the marchers and composites for n alive rays.  Where few
// rays are alive a lane per ray leaves most of the chip idle and the kernel
// is as long as one ray's chain of loads (row entries, bitfield word, jump),
// one chain per sample; a group spends one chain per G bins.  With many rays
// the lanes that test bins of an empty box are work done for nothing, so the
// group shrinks as the rays grow.  Measured on whole frames (us), G in the
// order 1 / 4 / 8 / 16 over the whole frame: 256x256 of the small scene 4040
// / 2570 / 2320 / 2170, reprojected 320x180 1285 / 815 / 715 / 730, 640x360
// 1725 / 1350 / 1410 / 1690, 1279x717 (its later launches) 3580 / 3270 / 3480 / 3490.
static const int GROUP16_RAYS = 1 << 15, GROUP4_RAYS = 1 << 19;
FVC_HD int group_lanes(int n_alive) { return n_alive <= GROUP16_RAYS ? 16 : (n_alive <= GROUP4_RAYS ? 4 : 1); }
// blocks of 256 threads that take any count of alive rays up to n
inline unsigned ray_blocks(int64_t n) {
  int64_t t = n;
  for (int64_t k : {std::min<int64_t>(n, GROUP16_RAYS), std::min<int64_t>(n, GROUP4_RAYS)})
    t = std::max(t, k * group_lanes((int)k));
  return (unsigned)((t + 255) / 256);
}
// LDS of a marcher block: the coarse tables of nlvl cascades, then the t0 of
// the samples of a block's rays (groups)
inline size_t march_lds(int nlvl) {
  return (size_t)nlvl * COARSE_WORDS * 4 + (size_t)(256 / 4) * MAX_STEPS_PER_LAUNCH * 4;
}

// march_trip's loop by a group of G lanes, up to n_steps samples of the ray.
// Every step calls step(samples, cnt, t0) on all lanes of the group: bit k of
// samples marks lane k's bin, of start t0 on that lane, as a sample; cnt
// samples came before.  Returns false when the ray ended.  Lanes of a group
// stay together; groups of a wave need not.
template <int G, class Step>
__device__ __forceinline__ bool march_group_steps(const MarchGrid& g, const uint32_t* coarse, MarchRay& r, int n_steps,
                                                  int& cnt, int& bins, Step&& step) {
  const int lane = lane_id(), sub = lane & (G - 1), sh = lane & ~(G - 1);
  const uint32_t all = (1u << G) - 1u;
  bool alive = true;
  while (cnt < n_steps) {
    float t0, hi;
    const int res = march_probe(g, coarse, r, r.j + sub, t0, hi);
    const uint32_t occ = (uint32_t)(__ballot(res == PROBE_SAMPLE) >> sh) & all;
    const uint32_t past = (uint32_t)(__ballot(res == PROBE_PAST) >> sh) & all;
    const GroupPlan p = group_plan(G, occ, past, n_steps - cnt);
    step(p.samples, cnt, t0);
    cnt += __popc(p.samples);
    bins += p.bins;
    r.j += p.bins;
    if (p.ended) {
      alive = false;
      bins++;
      break;
    }
    if (p.full) break;
#pragma unroll
    for (int d = 1; d < G; d <<= 1) hi = fmaxf(hi, __shfl_xor(hi, d, G));
    if (hi > 0.0f) bins += table_jump(g.tab, r.row, r.m, r.j, r.t1, hi);
  }
  r.t1 = g.tab.t[r.row.base + r.j];
  return alive;
}
// ... with the samples' t0 at t0s[0..cnt) (in LDS; the caller orders the reads)
template <int G>
__device__ __forceinline__ bool march_group(const MarchGrid& g, const uint32_t* coarse, MarchRay& r, int n_steps,
                                            float* t0s, int& cnt, int& bins) {
  const int sub = lane_id() & (G - 1);
  return march_group_steps<G>(g, coarse, r, n_steps, cnt, bins, [&](uint32_t samples, int before, float t0) {
    if ((samples >> sub) & 1u) t0s[before + __popc(samples & ((1u << sub) - 1u))] = t0;
  });
}

// One step of front-to-back compositing (accumulate_performance_kernel,
// performance_renderer.cu:93-120): v = half4 (r, g, b raw, log sigma).
// composite_alpha: the sample's opacity; composite_add: its colour and the
// transmittance after it; false once T < 1e-4.
__device__ __forceinline__ float composite_alpha(uint2 v, float t0, const fvc_stepsize_info& st) {
  const float ls = h2f(v.y >> 16);
  const float density = expf(ls);
  const float dt = step_dt(st, t0);
  const float alpha = 1.0f - expf(-density * dt);
  return fminf_(fmaxf_(alpha, 0.0f), 1.0f);
}
__device__ __forceinline__ V3 composite_colour(uint2 v) {
  const float cr = h2f(v.x & 0xffffu), cg = h2f(v.x >> 16), cb = h2f(v.y & 0xffffu);
  return V3{1.0f / (1.0f + expf(-cr)), 1.0f / (1.0f + expf(-cg)), 1.0f / (1.0f + expf(-cb))};
}
__device__ __forceinline__ bool composite_add(float4& res, float alpha, V3 c, float alpha_thre) {
  if (alpha > alpha_thre) {
    const float w = alpha * res.w;
    res.x = res.x + w * c.x;
    res.y = res.y + w * c.y;
    res.z = res.z + w * c.z;
    res.w = res.w * (1.0f - alpha);
  }
  return !(res.w < 1e-4f);
}
__device__ __forceinline__ bool composite_sample(float4& res, uint2 v, float t0, const fvc_stepsize_info& st,
                                                 float alpha_thre) {
  const float alpha = composite_alpha(v, t0, st);
  if (!(alpha > alpha_thre)) return !(res.w < 1e-4f);
  return composite_add(res, alpha, composite_colour(v), alpha_thre);
}
// Compositing of up to G samples by a lane group, lane k holding sample k.
// The lanes form opacities, colours and weights in parallel; what a lane by
// itself adds and multiplies one after the other stays in that order, on every
// lane of the group, so results are the same bit for bit.
// group_transmittance: T after all G samples, from each lane's factor
// (1 - alpha, or 1 for a sample that does not count); returns T before the
// lane's own.  group_add: acc + x of lane 0 + x of lane 1 ...
// Measured with the broadcasts by LDS permutes (4 a sample) and each sample's
// weight formed on every lane, then so, the next samples loaded ahead: a
// launch of the full composite of 256x256 10.5 -> 8.3 us, of the reprojected
// one of 640x360 25.0 -> 20.8 us; whole frames 1640 -> 1575 and 1160 -> 1150.
template <int G>
__device__ __forceinline__ float group_transmittance(float factor, float& T) {
  const int sub = lane_id() & (G - 1);
  float before = T;
  each<G>([&](auto u) {
    before = sub == u ? T : before;
    T = T * group_lane<G, u>(factor);
  });
  return before;
}
template <int G>
__device__ __forceinline__ float group_add(float acc, float x) {
  each<G>([&](auto u) { acc = acc + group_lane<G, u>(x); });
  return acc;
}
// Up to G samples of a ray, n of them in the stream: returns whether the ray
// stays visible; n_done counts the samples composited.
template <int G>
__device__ __forceinline__ bool composite_group(float4& res, uint2 v, float t0, int n, const fvc_stepsize_info& st,
                                                float alpha_thre, int& n_done) {
  const int lane = lane_id(), sub = lane & (G - 1);
  const float alpha = composite_alpha(v, t0, st);
  const bool counts = sub < n && alpha > alpha_thre;
  const float factor = counts ? 1.0f - alpha : 1.0f;
  float T = res.w;
  const float before = group_transmittance<G>(factor, T);
  const float after = before * factor;
  // the sample that ends the ray, if any: those after it do not count
  const uint32_t ends = (uint32_t)(__ballot(sub < n && after < 1e-4f) >> (lane & ~(G - 1))) & ((1u << G) - 1u);
  const int last = ends ? __ffs(ends) - 1 : G - 1;
  const V3 c = composite_colour(v);
  const bool adds = counts && sub <= last;
  const float w = alpha * before;
  res.x = group_add<G>(res.x, adds ? w * c.x : 0.0f);
  res.y = group_add<G>(res.y, adds ? w * c.y : 0.0f);
  res.z = group_add<G>(res.z, adds ? w * c.z : 0.0f);
  res.w = ends ? __shfl(after, last, G) : T;
  n_done += min(n, last + 1);
  return ends == 0;
}
// to_8bit (raymarch_common.h:554-557)
FVC_HD int to_8bit(float f) {
  const int v = (int)(f * 256.0f);
  return v < 0 ? 0 : (v > 255 ? 255 : v);
}

// host helpers (render.hip)
StepTableView step_table(Renderer& r, const fvc_raymarch_info* rms, int n_views);
MarchGrid march_grid(Renderer& r, const fvc_raymarch_info* rms, int n_views);
void upload_scene_refs(Renderer& r, const Views& vs);
int read_counter(Renderer& r, int idx, hipStream_t s);
void zero_counters(Renderer& r, hipStream_t s);
int launch_init_rays(Renderer& r, const Views& vs, hipStream_t s);
void launch_init_rays_async(Renderer& r, const Views& vs, hipStream_t s);
void prepare_views(Renderer& r, const Views& vs);
// per-iteration log entries {alive, n_steps, resample, cache, bins} of a frame
struct IterLog { int alive, n_steps, n_r, n_c, bins; };
std::vector<IterLog> read_iter_log(Renderer& r, int n_it, hipStream_t s);
void launch_write_image(Renderer& r, const Views& vs, hipStream_t s);
int next_burst(const Renderer& r, int it);

}  // namespace fvc
