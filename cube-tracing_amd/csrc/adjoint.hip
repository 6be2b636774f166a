// adjoint.hip -- differentiable voxel path tracer and its path-replay
// adjoint (radiance with respect to per-voxel albedo and emission).
//
// One thread per pixel of the batch of views; each loops over its
// samples in order, so the forward image is deterministic.  Path segments
// use intersect() semantics (closest voxel, traverse_mode<kTraceBounce>),
// scattering is cosine-weighted (weight = albedo).  The adjoint re-traces
// every path from its seed and keeps the path's vertices in registers
// while it walks them backwards:
//   S_{K+1} = 0,  S_k = e_k + a_k * S_{k+1}
//   dL/de_k = beta_k,  dL/da_k = beta_k * S_{k+1}.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "ct_device.h"
#include "ct_internal.h"

namespace ct {
using namespace dev;

namespace {

constexpr int kBlockA = 256;
constexpr float kFar = 1e9f;  // MAX_DISTANCE, defines.glsl:30
// Lanes that wait before a wave shades (walk_stream).  Forward and backward
// at 512^2, 16 samples: 16.2 ms with 32, 15.9 with 40, 15.8 with 48 to 56, and
// more below 32; path tracing at 1080p 520, 505, 508, 520 us.
constexpr int kAdjWait = 48;

struct AView {
  uint32_t width, height, base;  // base: global index of the view's first pixel
  uint32_t pad;
  float inv_view[16], inv_proj[16];
};

struct AArgs {
  DScene S;
  const ct_aabb *aabbs;
  const AView *views;
  const uint2 *blocks;  // per block: (view, first pixel of the view)
  uint32_t per_lane;    // pixels per lane of a block
  uint32_t spp, max_depth, seed;
  const float *albedo;
  const float *emission;
};

struct alignas(16) Vertex {
  uint32_t g;  // primitive slot
  F3 beta;     // throughput arriving at the vertex
};

// Camera ray through (x + u, y + v) (get_ray_from_current_pixel,
// rgen.glsl:18-42, with the jitter drawn from the sample's stream).
CT_D void view_ray(const AView &V, uint32_t x, uint32_t y, uint32_t &seed, F3 &o, F3 &d) {
  const float jx = rnd(seed);
  const float jy = rnd(seed);
  const float pcx = (float)x + jx, pcy = (float)y + jy;
  const float ux = pcx / (float)V.width, uy = pcy / (float)V.height;
  const float dx = ux * 2.0f - 1.0f, dy = uy * 2.0f - 1.0f;
  float ov[4], t4[4], d4[4];
  mat4_vec(V.inv_view, 0.0f, 0.0f, 0.0f, 1.0f, ov);
  mat4_vec(V.inv_proj, dx, dy, 1.0f, 1.0f, t4);
  const F3 nt = normalize(f3(t4[0], t4[1], t4[2]));
  mat4_vec(V.inv_view, nt.x, nt.y, nt.z, 0.0f, d4);
  o = f3(ov[0], ov[1], ov[2]);
  d = f3(d4[0], d4[1], d4[2]);
}

// transpose(world2obj) * vec4(n, 0) for the 3-row packing.
CT_D F3 world_normal(const float *w, F3 n) {
  return f3(((w[0] * n.x + w[1] * n.y) + w[2] * n.z) + 0.0f * 0.0f,
            ((w[3] * n.x + w[4] * n.y) + w[5] * n.z) + 0.0f * 0.0f,
            ((w[6] * n.x + w[7] * n.y) + w[8] * n.z) + 0.0f * 0.0f);
}
// The slot and the world hit position and normal of the segment's closest
// voxel (bi, bp); the segment is tested from ro = compute_ray_origin(origin,
// dir), as intersect() does.
CT_D void segment_hit(const AArgs &A, F3 ro, F3 dir, uint32_t bi, uint32_t bp, uint32_t &g, F3 &pos, F3 &nrm) {
  const DInst &I = A.S.inst[bi];
  float w[12];
#pragma unroll
  for (int k = 0; k < 12; ++k) w[k] = I.w2o[k];
  const F3 oo = xform3(w, ro, 1.0f), od = xform3(w, dir, 0.0f);
  const F3 sinv = f3(safe_inverse(od.x), safe_inverse(od.y), safe_inverse(od.z));
  const F3 sg = f3(-gsign(od.x), -gsign(od.y), -gsign(od.z));
  g = I.first + bp;
  const ct_aabb &bb = A.aabbs[g];
  const F3 c = muls(add(f3(bb.minimum[0], bb.minimum[1], bb.minimum[2]), f3(bb.maximum[0], bb.maximum[1], bb.maximum[2])),
                    0.5f);
  float t;
  F3 on;
  intersect_box<true, false>(c, oo, od, sg, sinv, t, &on);
  pos = add(ro, muls(dir, t));
  nrm = world_normal(w, on);
}

CT_D F3 albedo_of(const AArgs &A, uint32_t g) {
  return f3(A.albedo[3 * (size_t)g], A.albedo[3 * (size_t)g + 1], A.albedo[3 * (size_t)g + 2]);
}

// A lane's path: its pixel, the sample of the pixel, and the segment to trace
// next (from `o` along `d`, the k-th of the sample).
struct Path {
  uint32_t p, gpix, pixel_seed, s, k, seed;
  F3 o, d, beta, L, sum;  // throughput and radiance of the sample, sum over samples
  bool more;              // the sample goes on
};

CT_D void start_sample(const AArgs &A, const AView &V, Path &P) {
  P.seed = tea(P.pixel_seed, P.s);
  view_ray(V, P.p % V.width, P.p / V.width, P.seed, P.o, P.d);
  P.beta = f3(1.0f, 1.0f, 1.0f);
  P.L = f3(0.0f, 0.0f, 0.0f);
  P.k = 0u;
  P.more = true;
}
// Closest voxel of the path's segment: its slot, world hit position and
// normal.
template <int kWalk>
CT_D bool segment(const AArgs &A, const Path &P, uint32_t *stk, uint32_t &g, F3 &pos, F3 &nrm) {
  const F3 ro = compute_ray_origin(P.o, P.d);
  if constexpr (kWalk == kWalkGrid) {
    GridWalk<kTraceBounce> w{A.S.grid};
    w.start(A.S, ro, P.d, kFar, kInvalid, kInvalid);
    w.run();
    if (w.best == kInvalid) return false;
    // the walk's box test is segment_hit's
    g = gld(A.S.grid.slots + w.best);
    pos = add(ro, muls(P.d, w.best_t));
    nrm = world_normal(A.S.grid.w2o, w.best_n);
    return true;
  } else {
    float bt = kFar;
    uint32_t bi = kInvalid, bp = kInvalid;
    bool ovf = false;
    TraceCnt cnt;
    traverse_mode<kTraceBounce, kWalk>(A.S, ro, P.d, kFar, kInvalid, kInvalid, bt, bi, bp, stk, kBlockA, cnt, ovf);
    if (bi == kInvalid) return false;
    segment_hit(A, ro, P.d, bi, bp, g, pos, nrm);
    return true;
  }
}

// Traces every path of the wave's A.per_lane * 64 pixels.  A lane that has
// ended its path starts the next sample of its pixel, or takes the next pixel
// of the wave, at once: paths of a wave have 1 to max_depth + 1 segments, each
// of a few steps or many, and a wave that waits for its longest runs at 31% of
// its lanes (with this 44%).  The samples of a pixel stay in order on one lane, so the
// image is the same whatever the schedule.  hit(path, g, pos, nrm) shades a
// vertex and returns whether the path goes on from path.o along path.d;
// end(path) takes a finished sample (path.s, from 1 up to spp).
//
// Measured with the walk's new step loop: forward of 8 views at 512^2 with 16
// samples 8.9 -> 6.3 ms, path tracing at 1080p with 1 sample 448 -> 400 us.
template <int kWalk, class Hit, class End>
CT_D void trace_paths(const AArgs &A, Hit hit, End end) {
  __shared__ uint32_t stk[kWalk == kWalkGrid ? 1 : (kStackLds > 0 ? kStackLds : 1) * kBlockA];
  __shared__ uint32_t taken[kBlockA / 64];
  if (threadIdx.x < kBlockA / 64) taken[threadIdx.x] = 0u;
  __syncthreads();
  const uint2 b = A.blocks[blockIdx.x];
  const AView &V = *as_constant(A.views + b.x);
  const uint32_t wave = threadIdx.x >> 6, first = b.y + wave * (64u * A.per_lane),
                 last = min(first + 64u * A.per_lane, V.width * V.height);
  Path P;
  P.s = A.spp;
  P.more = false;
  F3 ro;
  auto next = [&]() -> bool {
    if (!P.more) {
      if (P.s == A.spp) {
        P.p = first + atomicAdd(&taken[wave], 1u);
        if (P.p >= last) return false;
        P.gpix = V.base + P.p;
        P.pixel_seed = tea(P.gpix, A.seed);
        P.s = 0u;
        P.sum = f3(0, 0, 0);
      }
      start_sample(A, V, P);
    }
    ro = compute_ray_origin(P.o, P.d);
    return true;
  };
  auto done = [&](bool found, uint32_t g, F3 pos, F3 nrm) {
    P.more = found && hit(P, g, pos, nrm);
    if (!P.more) {
      P.sum = add(P.sum, P.L);
      ++P.s;
      end(P);
    }
  };
  if constexpr (kWalk == kWalkGrid) {
    GridWalk<kTraceBounce> w{A.S.grid};
    walk_stream<kTraceBounce, kAdjWait>(
        w,
        [&]() -> bool {
          if (!next()) return false;
          w.start(A.S, ro, P.d, kFar, kInvalid, kInvalid);
          return true;
        },
        [&]() {
          // the walk's box test is segment_hit's
          const bool found = w.best != kInvalid;
          done(found, found ? gld(A.S.grid.slots + w.best) : 0u, add(ro, muls(P.d, w.best_t)),
               world_normal(A.S.grid.w2o, w.best_n));
        });
  } else {
    while (next()) {
      uint32_t g = 0u;
      F3 pos = f3(0, 0, 0), nrm = f3(0, 0, 0);
      const bool found = segment<kWalk>(A, P, stk + threadIdx.x, g, pos, nrm);
      done(found, g, pos, nrm);
    }
  }
}

// Lambertian scatter of a path at a vertex.
CT_D void scatter(Path &P, F3 pos, F3 nrm) {
  F3 sd = random_cosine_direction(P.seed, nrm);
  if (normal_near_zero(sd)) sd = nrm;
  P.d = sd;
  P.o = compute_ray_origin(compute_ray_origin(pos, nrm), nrm);
  ++P.k;
}

CT_D void store_pixel(const AArgs &A, const Path &P, float *image) {
  const F3 I = divs(P.sum, (float)A.spp);
  image[3 * (size_t)P.gpix] = I.x;
  image[3 * (size_t)P.gpix + 1] = I.y;
  image[3 * (size_t)P.gpix + 2] = I.z;
}

template <int kWalk>
__global__ void __launch_bounds__(kBlockA) k_adj_forward(AArgs A, float *image) {
  trace_paths<kWalk>(
      A,
      [&](Path &P, uint32_t g, F3 pos, F3 nrm) -> bool {
        P.L = add(P.L, muls(P.beta, A.emission[g]));
        if (P.k == A.max_depth) return false;
        P.beta = mulv(P.beta, albedo_of(A, g));
        scatter(P, pos, nrm);
        return true;
      },
      [&](Path &P) {
        if (P.s == A.spp) store_pixel(A, P, image);
      });
}

constexpr uint32_t kBvhLdsDepth = 5;
// kLds: the path's vertices, max_depth + 1 per lane, lie in LDS vertex by
// vertex, else in private memory.  Beside the BVH's stack (28 KB a block)
// they leave a CU fewer blocks than the 5 of the stack alone: 3 up to depth 5,
// 2 from 6 on.  4 views of 256^2, 8 samples, 96^3, in LDS and in private
// memory: depth 3 2.72 and 2.93 ms, 5 3.85 and 4.06, 6 6.64 and 4.60.
template <int kWalk, bool kLds>
__global__ void __launch_bounds__(kBlockA) k_adj_backward(AArgs A, const float *grad_image, float *grad_albedo,
                                                          float *grad_emission) {
  extern __shared__ Vertex vertices[];
  Vertex own[kLds ? 1 : CT_ADJOINT_MAX_DEPTH + 1];
  __shared__ uint32_t stk[kWalk == kWalkGrid ? 1 : (kStackLds > 0 ? kStackLds : 1) * kBlockA];
  Vertex *path = kLds ? vertices + threadIdx.x : own;
  constexpr uint32_t kStep = kLds ? kBlockA : 1u;
  const uint2 b = A.blocks[blockIdx.x];
  const AView &V = *as_constant(A.views + b.x);
  Path P;
  P.p = b.y + threadIdx.x;
  if (P.p >= V.width * V.height) return;
  P.gpix = V.base + P.p;
  P.pixel_seed = tea(P.gpix, A.seed);
  const float inv = 1.0f / (float)A.spp;
  const F3 G = f3(grad_image[3 * (size_t)P.gpix] * inv, grad_image[3 * (size_t)P.gpix + 1] * inv,
                  grad_image[3 * (size_t)P.gpix + 2] * inv);
  // One sample of every lane at a time (not trace_paths): a voxel of a small
  // scene sums tens of thousands of terms in 32 bits, whose rounding follows
  // the order they come in; this keeps to samples before pixels.
  for (P.s = 0; P.s < A.spp; ++P.s) {
    uint32_t nv = 0;
    start_sample(A, V, P);
    while (P.more) {
      uint32_t g = 0u;
      F3 pos, nrm;
      P.more = segment<kWalk>(A, P, stk + threadIdx.x, g, pos, nrm);
      if (!P.more) break;
      path[P.k * kStep] = Vertex{g, P.beta};
      nv = P.k + 1u;
      P.more = P.k < A.max_depth;
      if (P.more) {
        P.beta = mulv(P.beta, albedo_of(A, g));
        scatter(P, pos, nrm);
      }
    }
    F3 S = f3(0, 0, 0);  // radiance from the vertices after k, relative to vertex k+1
    for (int k = (int)nv - 1; k >= 0; --k) {
      const Vertex v = path[(uint32_t)k * kStep];
      const uint32_t g = v.g;
      const F3 bk = v.beta;
      const float e = A.emission[g];
      atomicAdd(&grad_emission[g], dot(G, bk));
      if ((uint32_t)k < A.max_depth) {
        atomicAdd(&grad_albedo[3 * (size_t)g], G.x * bk.x * S.x);
        atomicAdd(&grad_albedo[3 * (size_t)g + 1], G.y * bk.y * S.y);
        atomicAdd(&grad_albedo[3 * (size_t)g + 2], G.z * bk.z * S.z);
        S = add(f3(e, e, e), mulv(albedo_of(A, g), S));
      } else {
        S = f3(e, e, e);
      }
    }
  }
}

struct AdjPlan {
  DevBuf views, blocks;
  uint32_t nblocks = 0;
};

// ----------------------------------------------------------------------
// Plain (non-ReSTIR) path tracing with the material callables
// (indirect_illumination_path_tracing, indirect_illumination.glsl:454-539;
// scatter by type, rcall_scatter.glsl:11-88 via sample_material,
// light.glsl:231-269).  The path is the adjoint's forward model with a
// material per voxel (PRIMITIVE.material_index): emission is collected at
// every vertex and the scattered direction comes from the material's
// callable; the throughput is multiplied by the callable's attenuation
// (Lambertian and constant medium: diffuse; metal: specular; dielectric: 1).

struct PMat {  // a MATERIAL packed for the kernel
  float4 diffuse_type;    // diffuse rgb, type bits
  float4 specular_rough;  // specular rgb, roughness
  float4 emission_ior;    // emission rgb, ior
};

struct PArgs {
  AArgs A;
  const PMat *mats;
  const ct_primitive *prims;
  uint32_t n_mats;
};

CT_D F3 reflection(F3 v, F3 n) { return sub(v, muls(n, 2.0f * dot(v, n))); }  // prng.glsl:209-211

CT_D float pow5(float x) {  // pow(x, 5.0) of reflectance, as two squarings and a product
  const float x2 = x * x;
  return x2 * x2 * x;
}

CT_D float reflectance(float cosine, float ref_idx) {  // prng.glsl:214-218 (Schlick)
  float r0 = (1.0f - ref_idx) / (1.0f + ref_idx);
  r0 = r0 * r0;
  return r0 + (1.0f - r0) * pow5(1.0f - cosine);
}

CT_D F3 refraction(F3 uv, F3 n, float eta) {  // prng.glsl:220-225
  const float cos_theta = gmin(dot(neg(uv), n), 1.0f);
  const F3 perp = muls(add(uv, muls(n, cos_theta)), eta);
  const float ls = perp.x * perp.x + perp.y * perp.y + perp.z * perp.z;
  const F3 par = muls(n, -sqrtf(fabsf(1.0f - ls)));
  return add(par, perp);
}

// random_unit_vector (prng.glsl:63-74): rejection sampling in the unit
// ball, bounded at 64 draws (then the normal; the chance of reaching the
// bound is below 1e-20).
CT_D F3 random_unit_vector(uint32_t &seed, F3 fallback) {
  for (int k = 0; k < 64; ++k) {
    const float x = -1.0f + rnd(seed) * 2.0f;
    const float y = -1.0f + rnd(seed) * 2.0f;
    const float z = -1.0f + rnd(seed) * 2.0f;
    const float l2 = x * x + y * y + z * z;
    if (l2 >= 1.0f) continue;
    return normalize(f3(x, y, z));
  }
  return fallback;
}

// The callable of the material's type: the new direction, the attenuation,
// and false when the path is absorbed (a metal ray below the surface).
CT_D bool scatter_material(const PMat &m, F3 dir, F3 nrm, uint32_t &seed, F3 &sd, F3 &att) {
  const uint32_t type = __float_as_uint(m.diffuse_type.w) & CT_MATERIAL_TYPE_MASK;
  if (type == 1u) {  // METAL
    const float r = m.specular_rough.w;
    const F3 refl = reflection(dir, nrm);
    sd = add(muls(random_cosine_direction(seed, refl), gmin(r, 1.0f)), muls(refl, 1.0f - r));
    att = f3(m.specular_rough.x, m.specular_rough.y, m.specular_rough.z);
    return dot(sd, nrm) > 0.0f;
  }
  if (type == 2u) {  // DIELECTRIC
    F3 n = nrm;
    float eta = m.emission_ior.w;
    if (dot(dir, n) > 0.0f) {
      n = neg(n);
      eta = 1.0f / eta;
    }
    const float cos_theta = gmin(dot(neg(dir), n), 1.0f);
    const float sin_theta = sqrtf(1.0f - cos_theta * cos_theta);
    const bool cannot_refract = eta * sin_theta > 1.0f;
    if (cannot_refract || reflectance(cos_theta, eta) > rnd(seed)) sd = reflection(dir, n);
    else sd = refraction(dir, n, eta);
    att = f3(1.0f, 1.0f, 1.0f);
    return true;
  }
  if (type == 3u) {  // CONSTANT_MEDIUM
    sd = random_unit_vector(seed, nrm);
    if (normal_near_zero(sd)) sd = nrm;
  } else {  // LAMBERTIAN
    sd = random_cosine_direction(seed, nrm);
    if (normal_near_zero(sd)) sd = nrm;
  }
  att = f3(m.diffuse_type.x, m.diffuse_type.y, m.diffuse_type.z);
  return true;
}

template <int kWalk>
__global__ void __launch_bounds__(kBlockA) k_path_trace(PArgs Q, float *image) {
  const AArgs &A = Q.A;
  trace_paths<kWalk>(
      A,
      [&](Path &P, uint32_t g, F3 pos, F3 nrm) -> bool {
        const uint32_t mi = Q.prims[g].material_index;
        if (mi >= Q.n_mats) return false;  // no material: absorbs
        const PMat m = Q.mats[mi];
        P.L = add(P.L, mulv(P.beta, f3(m.emission_ior.x, m.emission_ior.y, m.emission_ior.z)));
        if (P.k == A.max_depth) return false;
        F3 sd, att;
        if (!scatter_material(m, P.d, nrm, P.seed, sd, att)) return false;
        P.beta = mulv(P.beta, att);
        const uint32_t type = __float_as_uint(m.diffuse_type.w) & CT_MATERIAL_TYPE_MASK;
        const F3 side = (type == 0u || dot(sd, nrm) >= 0.0f) ? nrm : neg(nrm);
        P.d = sd;
        P.o = compute_ray_origin(compute_ray_origin(pos, side), side);
        ++P.k;
        return true;
      },
      [&](Path &P) {
        if (P.s == A.spp) store_pixel(A, P, image);
      });
}

// `stream`: the kernel takes per_lane pixels a lane (trace_paths).
int plan(Accel &a, const ct_adjoint_desc *d, const ct_adjoint_view *views, bool stream, hipStream_t st, AdjPlan &P,
         AArgs &A) {
  if (!d || !views || d->n_views == 0) return fail(CT_E_INVALID, "adjoint: no views");
  if (d->spp == 0 || d->max_depth > CT_ADJOINT_MAX_DEPTH) return fail(CT_E_INVALID, "adjoint: spp 0 or max_depth too large");
  if (a.set.tlas_count == 0) return fail(CT_E_STATE, "adjoint: empty scene");
  std::vector<AView> hv(d->n_views);
  std::vector<uint2> hb;
  uint64_t base = 0, total = 0;
  for (uint32_t v = 0; v < d->n_views; ++v) total += (uint64_t)views[v].width * views[v].height;
  A.S = scene_view(a);
  Reach from;
  from.add(a.set.world_lo, a.set.world_hi);
  for (uint32_t v = 0; v < d->n_views; ++v) keep_served(A.S.grid, from, views[v].inv_view);
  // One lane takes several pixels where that leaves every SIMD 8 waves (256
  // CUs of 4 SIMDs): a wave then refills from 64 * per_lane paths.  Not in
  // the BVH, whose walk a wave runs to its longest ray in any case: there a
  // new pixel's camera ray only joins bounces (path tracing at 1080p with 1
  // sample: 1650 us with 3 pixels a lane, 1100 with 1).
  A.per_lane = stream && A.S.grid.bricks ? (uint32_t)std::min<uint64_t>(std::max<uint64_t>(total / (64u * 8u * 1024u), 1u), 8u) : 1u;
  const uint64_t run = (uint64_t)kBlockA * A.per_lane;
  for (uint32_t v = 0; v < d->n_views; ++v) {
    const ct_adjoint_view &cv = views[v];
    if (cv.width == 0 || cv.height == 0) return fail(CT_E_INVALID, "adjoint: empty view");
    AView &V = hv[v];
    V.width = cv.width;
    V.height = cv.height;
    V.base = (uint32_t)base;
    V.pad = 0;
    std::memcpy(V.inv_view, cv.inv_view, sizeof(V.inv_view));
    std::memcpy(V.inv_proj, cv.inv_proj, sizeof(V.inv_proj));
    const uint64_t np = (uint64_t)cv.width * cv.height;
    for (uint64_t p = 0; p < np; p += run) hb.push_back(make_uint2(v, (uint32_t)p));
    base += np;
    if (base >= (1ull << 31)) return fail(CT_E_INVALID, "adjoint: too many pixels");
  }
  int rc;
  if ((rc = P.views.reserve(sizeof(AView) * hv.size())) || (rc = P.blocks.reserve(sizeof(uint2) * hb.size()))) return rc;
  CT_HIP(hipMemcpyAsync(P.views.p, hv.data(), sizeof(AView) * hv.size(), hipMemcpyHostToDevice, st));
  CT_HIP(hipMemcpyAsync(P.blocks.p, hb.data(), sizeof(uint2) * hb.size(), hipMemcpyHostToDevice, st));
  P.nblocks = (uint32_t)hb.size();
  A.aabbs = a.set.aabbs.as<ct_aabb>();
  A.views = P.views.as<AView>();
  A.blocks = P.blocks.as<uint2>();
  A.spp = d->spp;
  A.max_depth = d->max_depth;
  A.seed = d->seed;
  return CT_OK;
}

}  // namespace
}  // namespace ct

using namespace ct;

extern "C" {

int ct_adjoint_render(ct_accel *a, const ct_adjoint_desc *d, const ct_adjoint_view *views, const float *albedo,
                      const float *emission, float *image, void *stream) {
  if (!a || !albedo || !emission || !image) return fail(CT_E_INVALID, "ct_adjoint_render: null argument");
  CT_HIP(hipSetDevice(a->device));
  hipStream_t st = stream ? static_cast<hipStream_t>(stream) : a->stream;
  AdjPlan P;
  AArgs A;
  int rc;
  if ((rc = plan(*a, d, views, true, st, P, A))) return rc;
  A.albedo = albedo;
  A.emission = emission;
  if (A.S.grid.bricks)
    hipLaunchKernelGGL(k_adj_forward<kWalkGrid>, dim3(P.nblocks), dim3(kBlockA), 0, st, A, image);
  else
    hipLaunchKernelGGL(k_adj_forward<kWalkBvh>, dim3(P.nblocks), dim3(kBlockA), 0, st, A, image);
  CT_HIP(hipGetLastError());
  CT_HIP(hipStreamSynchronize(st));  // the plan's buffers are released on return
  return CT_OK;
}

int ct_path_trace(ct_accel *a, const ct_adjoint_desc *d, const ct_adjoint_view *views, const ct_material *materials,
                  uint32_t material_count, float *image, void *stream) {
  if (!a || !image) return fail(CT_E_INVALID, "ct_path_trace: null argument");
  if (!materials && material_count) return fail(CT_E_INVALID, "ct_path_trace: null materials");
  if (!materials && !a->pt_mats.p) return fail(CT_E_STATE, "ct_path_trace: no materials uploaded yet");
  CT_HIP(hipSetDevice(a->device));
  hipStream_t st = stream ? static_cast<hipStream_t>(stream) : a->stream;
  AdjPlan P;
  PArgs PA;
  int rc;
  if ((rc = plan(*a, d, views, true, st, P, PA.A))) return rc;
  if (materials) {  // pack and keep them for later calls with materials == NULL
    std::vector<PMat> pm(std::max<uint32_t>(material_count, 1));
    for (uint32_t i = 0; i < material_count; ++i) {
      const ct_material &m = materials[i];
      if ((m.type & CT_MATERIAL_TYPE_MASK) > 3u) return fail(CT_E_INVALID, "ct_path_trace: unknown material type");
      float tb;
      std::memcpy(&tb, &m.type, 4);
      pm[i].diffuse_type = make_float4(m.diffuse[0], m.diffuse[1], m.diffuse[2], tb);
      pm[i].specular_rough = make_float4(m.specular[0], m.specular[1], m.specular[2], m.roughness);
      pm[i].emission_ior = make_float4(m.emission[0], m.emission[1], m.emission[2], m.ior);
    }
    if ((rc = a->pt_mats.reserve(sizeof(PMat) * pm.size()))) return rc;
    CT_HIP(hipMemcpyAsync(a->pt_mats.p, pm.data(), sizeof(PMat) * pm.size(), hipMemcpyHostToDevice, st));
    CT_HIP(hipStreamSynchronize(st));  // `pm` is freed on return
    a->pt_mat_count = material_count;
  }
  PA.mats = a->pt_mats.as<PMat>();
  PA.prims = a->set.prims.as<ct_primitive>();
  PA.n_mats = a->pt_mat_count;
  PA.A.albedo = nullptr;
  PA.A.emission = nullptr;
  if (PA.A.S.grid.bricks)
    hipLaunchKernelGGL(k_path_trace<kWalkGrid>, dim3(P.nblocks), dim3(kBlockA), 0, st, PA, image);
  else
    hipLaunchKernelGGL(k_path_trace<kWalkBvh>, dim3(P.nblocks), dim3(kBlockA), 0, st, PA, image);
  CT_HIP(hipGetLastError());
  CT_HIP(hipStreamSynchronize(st));  // the plan's buffers are released on return
  return CT_OK;
}

int ct_adjoint_backward(ct_accel *a, const ct_adjoint_desc *d, const ct_adjoint_view *views, const float *albedo,
                        const float *emission, const float *grad_image, float *grad_albedo, float *grad_emission,
                        void *stream) {
  if (!a || !albedo || !emission || !grad_image || !grad_albedo || !grad_emission)
    return fail(CT_E_INVALID, "ct_adjoint_backward: null argument");
  CT_HIP(hipSetDevice(a->device));
  hipStream_t st = stream ? static_cast<hipStream_t>(stream) : a->stream;
  AdjPlan P;
  AArgs A;
  int rc;
  if ((rc = plan(*a, d, views, false, st, P, A))) return rc;
  A.albedo = albedo;
  A.emission = emission;
  const size_t lds = sizeof(Vertex) * kBlockA * (size_t)(A.max_depth + 1);
  if (A.S.grid.bricks)
    hipLaunchKernelGGL((k_adj_backward<kWalkGrid, true>), dim3(P.nblocks), dim3(kBlockA), lds, st, A, grad_image,
                       grad_albedo, grad_emission);
  else if (A.max_depth <= kBvhLdsDepth)
    hipLaunchKernelGGL((k_adj_backward<kWalkBvh, true>), dim3(P.nblocks), dim3(kBlockA), lds, st, A, grad_image,
                       grad_albedo, grad_emission);
  else
    hipLaunchKernelGGL((k_adj_backward<kWalkBvh, false>), dim3(P.nblocks), dim3(kBlockA), 0, st, A, grad_image,
                       grad_albedo, grad_emission);
  CT_HIP(hipGetLastError());
  CT_HIP(hipStreamSynchronize(st));
  return CT_OK;
}

}  // extern "C"
