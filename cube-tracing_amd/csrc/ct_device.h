// ct_device.h -- device-side math, RNG, ray-box test and BVH traversal.
//
// Every float expression is written as the sequence of single IEEE
// operations the reference GLSL denotes (dot = (x*x' + y*y') + z*z',
// normalize = v / length(v), mix = x*(1-a) + y*a, ...).  The library is
// compiled with -ffp-contract=off and correctly rounded division and
// square root, so nothing is fused or approximated.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ct_internal.h"
#include "grid_reach.h"

namespace ct {
namespace dev {

#define CT_D __device__ __forceinline__

struct F3 {
  float x, y, z;
};
CT_D F3 f3(float x, float y, float z) { return F3{x, y, z}; }
CT_D F3 add(F3 a, F3 b) { return f3(a.x + b.x, a.y + b.y, a.z + b.z); }
CT_D F3 sub(F3 a, F3 b) { return f3(a.x - b.x, a.y - b.y, a.z - b.z); }
CT_D F3 mulv(F3 a, F3 b) { return f3(a.x * b.x, a.y * b.y, a.z * b.z); }
CT_D F3 muls(F3 a, float s) { return f3(a.x * s, a.y * s, a.z * s); }
CT_D F3 divs(F3 a, float s) { return f3(a.x / s, a.y / s, a.z / s); }
CT_D F3 neg(F3 a) { return f3(-a.x, -a.y, -a.z); }
CT_D float dot(F3 a, F3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
CT_D float length(F3 a) { return sqrtf(dot(a, a)); }
CT_D F3 normalize(F3 a) { return divs(a, length(a)); }
// normalize of what is mostly an axis vector already: its length is 1, and
// the square root and the divisions by 1 (45 instructions) are left out.  For
// scattered directions only (a fit's step 14.40 -> 14.19 ms): the branch keeps
// more alive around it, and with it in the material terms k_pt_end (finish,
// hybrid shift) held 232 VGPRs instead of 149.
CT_D F3 normalize_axis(F3 a) {
  const float d = dot(a, a);
  return d == 1.0f ? a : divs(a, sqrtf(d));
}
CT_D F3 cross(F3 a, F3 b) {
  return f3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
CT_D F3 vabs(F3 a) { return f3(fabsf(a.x), fabsf(a.y), fabsf(a.z)); }
CT_D float gmin(float a, float b) { return fminf(a, b); }
CT_D float gmax(float a, float b) { return fmaxf(a, b); }
CT_D float clampf(float x, float lo, float hi) { return gmin(gmax(x, lo), hi); }
CT_D float mixf(float x, float y, float a) { return x * (1.0f - a) + y * a; }
CT_D F3 mix3(F3 x, F3 y, float a) { return f3(mixf(x.x, y.x, a), mixf(x.y, y.y, a), mixf(x.z, y.z, a)); }
CT_D float gsign(float x) { return x > 0.0f ? 1.0f : (x < 0.0f ? -1.0f : 0.0f); }
CT_D F3 xyz(float4 v) { return f3(v.x, v.y, v.z); }

// Saturating conversions (NaN -> 0).
CT_D uint32_t f2u_clamped(float x) {
  if (!(x > 0.0f)) return 0u;
  if (x >= 4294967296.0f) return 0xFFFFFFFFu;
  return (uint32_t)x;
}
CT_D int32_t f2i_clamped(float x) {
  if (!(x == x)) return 0;
  if (x >= 2147483648.0f) return 0x7FFFFFFF;
  if (x <= -2147483648.0f) return (int32_t)0x80000000;
  return (int32_t)x;
}
// The same as the hardware's own instruction (a C++ cast leaves values out of
// range undefined, and guarding it takes 8 instructions; compute_ray_origin
// converts three values, and each pass calls it 2 to 6 times a pixel).  The
// compiler neither leaves out an asm statement whose result nothing uses nor
// moves it into the branch that does: code whose results may go unused takes
// the guarded ones.  (Path reuse, which loads vertices for tests that may not
// need them: k_pt_end held 219 VGPRs in its finish pass and 185 in the request
// pass, instead of 121 and 20.)
#if defined(__HIP_DEVICE_COMPILE__)
CT_D uint32_t f2u_sat(float x) {
  uint32_t r;
  [[clang::noconvergent]] { asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(x)); }
  return r;
}
CT_D int32_t f2i_sat(float x) {
  int32_t r;
  [[clang::noconvergent]] { asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(x)); }
  return r;
}
#else
CT_D uint32_t f2u_sat(float x) { return f2u_clamped(x); }
CT_D int32_t f2i_sat(float x) { return f2i_clamped(x); }
#endif

// Memory that no kernel of the launch writes, as constant memory: uniform
// reads of it are then scalar loads, also after stores and inside loops.
template <class T>
CT_D const T *as_constant(const T *p) {
  return (const T *)(const __attribute__((address_space(4))) T *)p;
}

// Column-major 4x4 (m[c*4 + r]): out_r = ((m0r*v0 + m1r*v1) + m2r*v2) + m3r*v3.
CT_D void mat4_vec(const float *m, float v0, float v1, float v2, float v3, float *o) {
#pragma unroll
  for (int r = 0; r < 4; ++r) o[r] = m[0 * 4 + r] * v0 + m[1 * 4 + r] * v1 + m[2 * 4 + r] * v2 + m[3 * 4 + r] * v3;
}
// 3-row packing (m[c*3 + r]) of the upper three rows.
CT_D F3 xform3(const float *m, F3 p, float w) {
  return f3(m[0] * p.x + m[3] * p.y + m[6] * p.z + m[9] * w,
            m[1] * p.x + m[4] * p.y + m[7] * p.z + m[10] * w,
            m[2] * p.x + m[5] * p.y + m[8] * p.z + m[11] * w);
}

// ---------------------------------------------------------------- RNG
// random.glsl:26-40
CT_D uint32_t tea(uint32_t val0, uint32_t val1) {
  uint32_t v0 = val0, v1 = val1, s0 = 0;
#pragma unroll
  for (uint32_t n = 0; n < 16; n++) {
    s0 += 0x9e3779b9u;
    v0 += ((v1 << 4) + 0xa341316cu) ^ (v1 + s0) ^ ((v1 >> 5) + 0xc8013ea4u);
    v1 += ((v0 << 4) + 0xad90777du) ^ (v0 + s0) ^ ((v0 >> 5) + 0x7e95761eu);
  }
  return v0;
}
// random.glsl:44-56
CT_D uint32_t lcg(uint32_t &prev) {
  prev = 1664525u * prev + 1013904223u;
  return prev & 0x00FFFFFFu;
}
CT_D float rnd(uint32_t &prev) { return (float)lcg(prev) / 16777216.0f; }
CT_D float rnd_interval(uint32_t &prev, float mn, float mx) { return mn + rnd(prev) * (mx - mn); }
// random.glsl:69-77
CT_D uint32_t urnd_interval(uint32_t &prev, uint32_t mn, uint32_t mx) {
  if (mn == mx) return mn;
  if (mn > mx) return f2u_sat(rnd_interval(prev, (float)mx, (float)mn));
  return f2u_sat(rnd_interval(prev, (float)mn, (float)mx));
}

// ------------------------------------------------------------ geometry
CT_D float safe_inverse(float x) { return (x == 0.0f) ? 1e12f : (1.0f / x); }

// primitives.glsl:233-257
// kMaybeUnused: the result may go unused (f2i_sat).
template <bool kMaybeUnused = false>
CT_D F3 compute_ray_origin(F3 pos, F3 n) {
  const float origin = 1.f / 32.f, f_scale = 1.f / 65536.f, i_scale = 256.f;
  auto cvt = [](float x) { return kMaybeUnused ? f2i_clamped(x) : f2i_sat(x); };
  int32_t ix = cvt(n.x * i_scale), iy = cvt(n.y * i_scale), iz = cvt(n.z * i_scale);
  float px = __uint_as_float(__float_as_uint(pos.x) + (uint32_t)(pos.x < 0.0f ? -ix : ix));
  float py = __uint_as_float(__float_as_uint(pos.y) + (uint32_t)(pos.y < 0.0f ? -iy : iy));
  float pz = __uint_as_float(__float_as_uint(pos.z) + (uint32_t)(pos.z < 0.0f ? -iz : iz));
  F3 fo = muls(n, f_scale);
  return f3(fabsf(pos.x) < origin ? pos.x + fo.x : px, fabsf(pos.y) < origin ? pos.y + fo.y : py,
            fabsf(pos.z) < origin ? pos.z + fo.z : pz);
}
// Box.rotation = mat3(1): rotation * v and v * rotation as written.
CT_D F3 rot_mul(F3 v) {
  return f3(1.0f * v.x + 0.0f * v.y + 0.0f * v.z, 0.0f * v.x + 1.0f * v.y + 0.0f * v.z,
            0.0f * v.x + 0.0f * v.y + 1.0f * v.z);
}
CT_D F3 mul_rot(F3 v) {
  return f3(v.x * 1.0f + v.y * 0.0f + v.z * 0.0f, v.x * 0.0f + v.y * 1.0f + v.z * 0.0f,
            v.x * 0.0f + v.y * 0.0f + v.z * 1.0f);
}

// primitives.glsl:273-355 with rotation = identity and radius = h on all
// axes.  `dr` is the (rotated) direction and `sg` = -sign(dr), both
// independent of the box.  oriented: divide by dr; else multiply by inv.
// finite: ro - c is finite, so the rotation leaves it (but for the sign of a
// zero, which no test below sees).
template <bool kCanStart, bool kOriented, bool kFinite = false>
CT_D bool intersect_box(F3 c, F3 ro, F3 dr, F3 sg, F3 inv, float &dist, F3 *normal = nullptr) {
  const float r = kHalfVoxel, ir = 64.0f;  // safeInverse(HALF_VOXEL_EXTENT)
  F3 o = kFinite ? sub(ro, c) : rot_mul(sub(ro, c));
  float winding = 1.0f;
  if (kCanStart) {
    F3 rb = muls(vabs(o), ir);
    winding = (gmax(rb.x, gmax(rb.y, rb.z)) < 1.0f) ? -1.0f : 1.0f;
  }
  float rw = r * winding;
  F3 dtp = sub(f3(rw * sg.x, rw * sg.y, rw * sg.z), o);
  if (kOriented)
    dtp = f3(dtp.x / dr.x, dtp.y / dr.y, dtp.z / dr.z);
  else
    dtp = mulv(dtp, inv);
  // Every term is evaluated (no short circuit): the tests are pure
  // arithmetic, so the result is the same and a wave takes no branches.
  const bool tx = (int)(dtp.x >= 0.0f) & (int)(fabsf(o.y + dr.y * dtp.x) < r) & (int)(fabsf(o.z + dr.z * dtp.x) < r);
  const bool ty = (int)(dtp.y >= 0.0f) & (int)(fabsf(o.z + dr.z * dtp.y) < r) & (int)(fabsf(o.x + dr.x * dtp.y) < r);
  const bool tz = (int)(dtp.z >= 0.0f) & (int)(fabsf(o.x + dr.x * dtp.z) < r) & (int)(fabsf(o.y + dr.y * dtp.z) < r);
  float sx = tx ? sg.x : 0.0f;
  float sy = tx ? 0.0f : (ty ? sg.y : 0.0f);
  float sz = (tx || ty) ? 0.0f : (tz ? sg.z : 0.0f);
  dist = (sx != 0.0f) ? dtp.x : ((sy != 0.0f) ? dtp.y : dtp.z);
  if (normal) *normal = kOriented ? rot_mul(f3(sx, sy, sz)) : f3(sx, sy, sz);
  return (sx != 0.0f) || (sy != 0.0f) || (sz != 0.0f);
}

// primitives.glsl:499-507
CT_D F3 cube_like_normal(F3 n) {
  F3 a = vabs(n);
  float mc = gmax(gmax(a.x, a.y), a.z);
  return (mc == a.x) ? f3(gsign(n.x), 0, 0) : (mc == a.y) ? f3(0, gsign(n.y), 0) : f3(0, 0, gsign(n.z));
}

// mat.glsl:111-202
CT_D F3 sky_grad(F3 dir, F3 a, F3 b) {
  F3 u = normalize(dir);
  float t = 0.5f * (u.y + 1.0f);
  return mix3(a, b, t);
}
CT_D F3 day_color(F3 d) { return sky_grad(d, f3(1.0f, 1.0f, 1.0f), f3(0.5f, 0.7f, 1.0f)); }
CT_D F3 night_color(F3 d) { return sky_grad(d, f3(0.2f, 0.2f, 0.3f), f3(0.2f, 0.2f, 0.5f)); }
CT_D F3 sunset_color(F3 d) { return sky_grad(d, f3(0.8f, 0.4f, 0.0f), f3(1.0f, 0.4f, 0.0f)); }
CT_D F3 sunrise_color(F3 d) { return sky_grad(d, f3(0.7f, 0.35f, 0.0f), f3(0.8f, 0.4f, 0.0f)); }
CT_D F3 sky_color(float t, bool afternoon, F3 dir) {
  const float night_duration = 0.5f, sunrise_duration = 0.10f, full_daylight_transition = 0.10f,
              full_night_transition = 0.10f;
  float sunrise_end = night_duration + sunrise_duration;
  float sunrise_to_daylight = sunrise_end + full_daylight_transition;
  float zenith_transition = 1.0f - sunrise_to_daylight;
  float daylight_end = 1.0f - zenith_transition;
  float sunset_start = 1.0f - zenith_transition - sunrise_duration;
  float sunset_end = 1.0f - zenith_transition - sunrise_duration - full_night_transition;
  if (afternoon) {
    if (t < night_duration) return night_color(dir);
    if (t < sunrise_end) return mix3(night_color(dir), sunrise_color(dir), t);
    if (t < sunrise_to_daylight) return mix3(sunrise_color(dir), sunset_color(dir), t);
    return mix3(sunset_color(dir), day_color(dir), t);
  }
  if (t > daylight_end) return mix3(sunrise_color(dir), day_color(dir), t);
  if (t > sunset_start) return mix3(sunset_color(dir), sunrise_color(dir), t);
  if (t > sunset_end) return mix3(night_color(dir), sunset_color(dir), t);
  return night_color(dir);
}
// light.glsl:78-80
CT_D float luminance(F3 c) { return 0.2126f * c.x + 0.7152f * c.y + 0.0722f * c.z; }

// sin and cos of x in [0, 2*pi).  GLSL leaves their precision to the
// implementation, so the library fixes one: Cody-Waite reduction by pi/2
// (three-part constant) and the single-precision minimax polynomials of
// the Cephes library (S. L. Moshier, sinf.c / cosf.c) on [-pi/4, pi/4].
// Only IEEE add/mul and floor are used, so the CPU restatement computes
// the same bits.
CT_D void sincos_ct(float x, float &s, float &c) {
  const float j = floorf(x * 0.636619772367581343f + 0.5f);
  const int q = (int)j;
  const float r = ((x - j * 1.5703125f) - j * 4.837512969970703125e-4f) - j * 7.54978995489188216e-8f;
  const float z = r * r;
  const float sp = ((-1.9515295891e-4f * z + 8.3321608736e-3f) * z - 1.6666654611e-1f) * z * r + r;
  const float cp = ((2.443315711809948e-5f * z - 1.388731625493765e-3f) * z + 4.166664568298827e-2f) * z * z -
                   0.5f * z + 1.0f;
  switch (q & 3) {
    case 0: s = sp; c = cp; break;
    case 1: s = cp; c = -sp; break;
    case 2: s = -sp; c = -cp; break;
    default: s = -cp; c = sp; break;
  }
}

constexpr float kPi = 3.1415926535897932384626433832795f;  // DAXA_PI, shared.inl:49

CT_D bool normal_near_zero(F3 v) {  // prng.glsl:17-21
  const float s = 1e-8f;
  return fabsf(v.x) < s && fabsf(v.y) < s && fabsf(v.z) < s;
}
// random_cosine_direction, prng.glsl:84-108
CT_D F3 random_cosine_direction(uint32_t &seed, F3 n) {
  const float r1 = rnd(seed);
  const float r2 = rnd(seed);
  const float z = sqrtf(1.0f - r2);
  const float phi = 2.0f * kPi * r1;
  float sp, cp;
  sincos_ct(phi, sp, cp);
  const float x = cp * sqrtf(r2);
  const float y = sp * sqrtf(r2);
  F3 u = fabsf(n.x) > 0.1f ? f3(0.0f, 1.0f, 0.0f) : f3(1.0f, 0.0f, 0.0f);
  u = normalize_axis(cross(n, u));
  F3 v = cross(n, u);
  return add(add(muls(u, x), muls(v, y)), muls(n, z));
}


// A strided loop's next index below `count`, else `count`: base + stride may
// pass 2^32, and a wrapped index would start the loop again.
CT_D uint32_t next_batch(uint32_t base, uint32_t count, uint32_t stride) {
  return count - base > stride ? base + stride : count;
}

// ------------------------------------------------------------ traversal
constexpr uint32_t kMaxTraversalSteps = 1u << 22;

struct TraceCnt {
  uint32_t nodes = 0, leaves = 0, insts = 0;
};

CT_D bool slab(float lx, float ly, float lz, float hx, float hy, float hz, F3 o, F3 inv,
               float limit, float &tn) {
  float t1x = (lx - o.x) * inv.x, t2x = (hx - o.x) * inv.x;
  float t1y = (ly - o.y) * inv.y, t2y = (hy - o.y) * inv.y;
  float t1z = (lz - o.z) * inv.z, t2z = (hz - o.z) * inv.z;
  float n0 = gmax(gmax(gmin(t1x, t2x), gmin(t1y, t2y)), gmin(t1z, t2z));
  float f0 = gmin(gmin(gmax(t1x, t2x), gmax(t1y, t2y)), gmax(t1z, t2z));
  tn = n0;
  return (n0 <= f0) && (f0 >= 0.0f) && (n0 <= limit);
}

// Per-lane traversal stack: the newest kStackReg entries in registers
// (r[0] is the top), older ones in this lane's LDS column.
struct Stack {
  uint32_t r[kStackReg > 0 ? kStackReg : 1];
  uint32_t *lds;
  uint32_t stride;
  int n;
  CT_D void push(uint32_t v, bool &overflow) {
    if (kStackReg == 0) {
      if (n >= kStackLds) { overflow = true; return; }
      lds[(uint32_t)n * stride] = v;
      ++n;
      return;
    }
    if (n >= kStackReg) {
      if (n - kStackReg >= kStackLds) { overflow = true; return; }
      lds[(uint32_t)(n - kStackReg) * stride] = r[kStackReg - 1];
    }
#pragma unroll
    for (int i = kStackReg - 1; i > 0; --i) r[i] = r[i - 1];
    r[0] = v;
    ++n;
  }
  CT_D uint32_t pop() {
    if (kStackReg == 0) {
      --n;
      return lds[(uint32_t)n * stride];
    }
    uint32_t v = r[0];
#pragma unroll
    for (int i = 0; i < kStackReg - 1; ++i) r[i] = r[i + 1];
    --n;
    if (n >= kStackReg) r[kStackReg - 1] = lds[(uint32_t)(n - kStackReg) * stride];
    return v;
  }
};

// A load through a pointer known to address device (global) memory: a
// global load instead of a flat one, which would also count against the
// LDS wait counter that the traversal stack uses.
typedef float gf4 __attribute__((ext_vector_type(4)));
typedef uint32_t gu2 __attribute__((ext_vector_type(2)));
typedef uint32_t gu4 __attribute__((ext_vector_type(4)));
CT_D float gld(const float *p) { return *(const __attribute__((address_space(1))) float *)p; }
CT_D uint32_t gld(const uint32_t *p) { return *(const __attribute__((address_space(1))) uint32_t *)p; }
CT_D float4 gld(const float4 *p) {
  const gf4 v = *(const __attribute__((address_space(1))) gf4 *)p;
  return make_float4(v.x, v.y, v.z, v.w);
}
CT_D uint2 gld(const uint2 *p) {
  const gu2 v = *(const __attribute__((address_space(1))) gu2 *)p;
  return make_uint2(v.x, v.y);
}
CT_D uint4 gld(const uint4 *p) {
  const gu4 v = *(const __attribute__((address_space(1))) gu4 *)p;
  return make_uint4(v.x, v.y, v.z, v.w);
}

// Test both children of a node; returns the next ref (or kInvalid to pop)
// and pushes the other child when both are hit.  Closest-hit walks take the
// near child first (ties to child 0), so the best hit prunes early.  Any-hit
// walks take the far child first (ties to child 1): a shadow ray's
// occluders cluster at its target end, where lights sit among other
// voxels, and the outcome does not depend on the order.
template <bool kFarFirst>
CT_D uint32_t visit_node(const DNode *nodes, uint32_t idx, F3 o, F3 inv, float limit, Stack &stk, bool &overflow) {
  const float4 *p = reinterpret_cast<const float4 *>(nodes + idx);
  float4 a = gld(p), b = gld(p + 1), c = gld(p + 2);
  uint4 d = gld(reinterpret_cast<const uint4 *>(nodes + idx) + 3);
  float tn0, tn1;
  bool h0 = slab(a.x, a.y, a.z, a.w, b.x, b.y, o, inv, limit, tn0);
  bool h1 = slab(b.z, b.w, c.x, c.y, c.z, c.w, o, inv, limit, tn1);
  if (h0 && h1) {
    const bool swap = kFarFirst ? !(tn1 < tn0) : (tn1 < tn0);
    stk.push(swap ? d.x : d.y, overflow);
    return swap ? d.y : d.x;
  }
  if (h0) return d.x;
  if (h1) return d.y;
  return kInvalid;
}

// Leaf semantics of a traversal.
//  kTraceAny:     is_vertex_visible (light.glsl:82-142): is_hit_from_ray
//                 with rayCanStartInBox = false; occluded when a non-target
//                 voxel has 0 <= t <= limit.
//  kTraceClosest: traceRayEXT + rint.glsl:10-43 (rayCanStartInBox = true,
//                 oriented): closest t > 0.
//  kTraceBounce:  intersect() of bounce.glsl:9-130 with its is_hit_from_ray
//                 box test (rayCanStartInBox = true, non-oriented): closest
//                 t >= 0.  The reference commits the first generated hit
//                 (bounce.glsl:118); the closest one is taken here.
// Closest modes break equal t by the smaller (instance, primitive).
constexpr int kTraceAny = 0, kTraceClosest = 1, kTraceBounce = 2;

// Two-level traversal (TLAS in world space, each BLAS in object space) as
// a resumable walker: start() takes a ray, each step() visits one TLAS
// node, BLAS node or voxel leaf (a step that reaches an instance also
// enters it and visits the BLAS root), and `done` is set once the ray is
// finished (for an any-hit query `occluded` tells the outcome).  `stk` is
// the lane's LDS stack column.
// The ray a node test uses (cur_o, cur_inv) is the world ray in the TLAS
// and the object-space ray in a BLAS; it is switched on entering and on
// leaving an instance.  Instance entry comes first in a step and the
// stack update last, so in a wave whose lanes take different branches each
// state register is written after every read of its old value: the
// branches' results merge without register copies.
template <int kMode, bool kCount>
struct Walker {
  static constexpr bool kAny = kMode == kTraceAny;
  F3 o, d, winv, cur_o, cur_inv, dr, sg, sinv;
  float limit, best_t;
  uint32_t ti, tp, best_i, best_p, first, inst, ref, steps;
  int base;
  bool in_blas, done, occluded, overflow;
  const DNode *tlas_nodes, *blas_nodes;  // read once per ray, not per step
  Stack st;

  CT_D void start(const DScene &S, F3 o_, F3 d_, float limit_, uint32_t ti_, uint32_t tp_, uint32_t *stk,
                  uint32_t stride) {
    o = o_;
    d = d_;
    limit = limit_;
    ti = ti_;
    tp = tp_;
    winv = f3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
    cur_o = o; cur_inv = winv; dr = d; sg = d; sinv = d;
    best_t = limit_;
    best_i = kInvalid;
    best_p = kInvalid;
    first = 0;
    inst = 0;
    base = 0;
    steps = 0;
    in_blas = false;
    occluded = false;
    overflow = false;
    st.lds = stk;
    st.stride = stride;
    st.n = 0;
    tlas_nodes = S.tlas_nodes;
    blas_nodes = S.blas_nodes;
    ref = S.tlas_root;
    done = ref == kInvalid;
  }

  CT_D void step(const DScene &S, TraceCnt &cnt) {
    if (++steps > kMaxTraversalSteps) {  // only a malformed tree can get here
      overflow = true;
      done = true;
      return;
    }
    if ((ref & kLeaf) && !in_blas) {
      // Enter the instance: the object-space ray, then its BLAS root below.
      inst = gld(S.tlas_inst + (ref & ~kLeaf));
      if (kCount) cnt.insts++;
      const DInst *I = S.inst + inst;
      float m[12];
#pragma unroll
      for (int k = 0; k < 12; ++k) m[k] = gld(I->w2o + k);
      const F3 oo = xform3(m, o, 1.0f), od = xform3(m, d, 0.0f);
      // An instance without rotation or scale gives back the direction's
      // own bits (its zero terms add signed zeros), and then 1 / od is winv:
      // the three divisions run only for lanes whose direction changed.
      F3 oinv = winv;
      if (__float_as_uint(od.x) != __float_as_uint(d.x) || __float_as_uint(od.y) != __float_as_uint(d.y) ||
          __float_as_uint(od.z) != __float_as_uint(d.z))
        oinv = f3(1.0f / od.x, 1.0f / od.y, 1.0f / od.z);
      if (kMode != kTraceClosest) {
        dr = od;
        // safe_inverse(od) with the quotient above
        sinv = f3(od.x == 0.0f ? 1e12f : oinv.x, od.y == 0.0f ? 1e12f : oinv.y, od.z == 0.0f ? 1e12f : oinv.z);
      } else {
        dr = mul_rot(od);
      }
      sg = f3(-gsign(dr.x), -gsign(dr.y), -gsign(dr.z));
      cur_o = oo;
      cur_inv = oinv;
      first = gld(&I->first);
      in_blas = true;
      base = st.n;
      ref = gld(&I->root);
    }
    uint32_t next = kInvalid;
    bool finished = false;
    if (!(ref & kLeaf)) {
      // TLAS and BLAS nodes take the same code.
      if (kCount) cnt.nodes++;
      const DNode *nodes = in_blas ? blas_nodes + first : tlas_nodes;
      next = visit_node<kAny>(nodes, ref, cur_o, cur_inv, kAny ? limit : best_t, st, overflow);
    } else {
      if (kCount) cnt.leaves++;
      const float4 L = gld(S.blas_leaves + first + (ref & ~kLeaf));
      const uint32_t pid = __float_as_uint(L.w);
      float t;
      if (kAny) {
        const bool hit = intersect_box<false, false>(f3(L.x, L.y, L.z), cur_o, dr, sg, sinv, t);
        if (hit && (t >= 0.0f) && (t <= limit) && !(inst == ti && pid == tp)) {
          occluded = true;
          finished = true;
        }
      } else {
        const bool hit = (kMode == kTraceClosest)
                             ? intersect_box<true, true>(f3(L.x, L.y, L.z), cur_o, dr, sg, sinv, t)
                             : intersect_box<true, false>(f3(L.x, L.y, L.z), cur_o, dr, sg, sinv, t);
        if (hit && ((kMode == kTraceClosest) ? (t > 0.0f) : (t >= 0.0f))) {
          const bool better =
              (t < best_t) || (t == best_t && ((inst < best_i) || (inst == best_i && pid < best_p)));
          if (better) {
            best_t = t;
            best_i = inst;
            best_p = pid;
          }
        }
      }
    }
    if (finished || overflow) {
      done = true;
    } else if (next != kInvalid) {
      ref = next;
    } else {
      if (in_blas && st.n == base) {
        in_blas = false;
        cur_o = o;
        cur_inv = winv;
      }
      if (st.n == 0)
        done = true;
      else
        ref = st.pop();
    }
  }
};

// ------------------------------------------------------------ cell grid
// The walk of one ray through the scene's cell grid (DGrid) instead of its
// BVH: the same voxel tests on the same operands, so the same hits to the
// bit, in far fewer instructions and bytes.  A BVH walk of the noise scenes
// visits about 30 nodes of 64 B per ray; here a ray takes 3 to 4 steps on
// average where a quarter of the cells are voxels and 4 to 7 where an eighth
// are (counted on the host; camera rays that hit 7 and 10, one ray in a
// hundred more than 13 to 28), each over an empty box (a cube of up to
// kGridSkip bricks, 2x2x2 cells of a brick, or a cell), and reads 16 B per
// brick it stops in.
//
// Which voxels can a test accept?  intersect_box() accepts a voxel when the
// ray's computed crossing of the plane of one of its faces lies within the
// face, so up to rounding the ray enters the voxel's cell there (or starts
// in it).  The walk enters every cell the ray enters, except in boxes that
// hold no voxel, and tests it.  Where a crossing lies within p of a cell's
// edge, the cells across that edge are tested too.  p bounds the rounding of
// both sides, in cells, with u = 2^-24, T the ray parameter scaled to 1/2..1
// cells on the fastest axis and iv the crossing times of a cell:
//   walk:  (plane - q) * iv, then q + v T:         3 u T + u |q + v T|
//   test:  ro - c, +-r, * inv, o + dr t:     6 u T + u max(iv) / 2 + 2 u
// hence p = 10 u T + u (1.5 max|position| + max(iv) + 4), cut off at 1/64
// cell.  The term of iv may be cut: an error of u iv in the time a plane is
// crossed at moves the ray by u along that plane's axis, so it is still
// within p of the plane where the test places the crossing.  The other terms
// may not, and where they pass 1/128 cell the BVH's boxes (padded by 2^-12)
// do not bound the test's rounding either, so that what the BVH walk finds
// depends on its boxes.  Rays from far away (about 200 units on) or through
// as much of a grid are therefore walked through the BVH: ray queries look
// at each ray (kChecked, kWalkQuery), frames and path tracing at the camera
// and the scene, whose surfaces every other ray starts from (grid_reach.h).
//
// An empty box may be stepped over when neither its entry nor its exit lies
// within p iv_a of a lattice plane of an axis other than the crossed one, a.
// Take a voxel outside the box whose plane b the ray crosses inside it,
// within p of a face c of the box: positions along the ray only grow, so at
// the exit (or entry) the ray is within p of face c; if c is the crossed
// axis, at most p iv_c of the ray lies between, and there the ray is within
// p iv_c of plane b.  Otherwise the ray takes the cell alone, which has no
// inner planes, with its neighbours.
//
// Coordinates are lattice cells (32 per unit), exact in float, negated on
// the axes the ray runs down (cell i becomes ~i), so every axis runs up.
constexpr float kCellsPerUnit = 32.0f;
constexpr float kU = 5.9604644775390625e-8f;  // 2^-24
constexpr float kNearMax = 0.015625f;
constexpr float kDeadAxis = 9.094947017729282e-13f;  // 2^-40: an axis that is never crossed

// The lanes of the wave where b holds (the same value on every lane).
CT_D uint64_t ballot(bool b) { return __builtin_amdgcn_ballot_w64(b); }
CT_D float med3f(float a, float b, float c) { return __builtin_amdgcn_fmed3f(a, b, c); }
CT_D float fractf(float x) { return __builtin_amdgcn_fractf(x); }  // x - floor(x), below 1
CT_D int32_t imin(int32_t a, int32_t b) { return a < b ? a : b; }
CT_D int32_t imax(int32_t a, int32_t b) { return a > b ? a : b; }
CT_D int32_t clampi(int32_t x, int32_t lo, int32_t hi) { return imax(imin(x, lo), imin(imax(x, lo), hi)); }

// kChecked: rays that this walk does not serve end as kWide.
template <int kMode, bool kChecked = false>
struct GridWalk {
  static constexpr bool kAny = kMode == kTraceAny;
  const DGrid &G;
  F3 oo, dr, sg, sinv;           // object-space ray as the voxel test takes it
  int32_t sx, sy, sz;            // -1 on negated axes
  uint32_t target;               // any hit: the target voxel's cell (DGrid::cells)
  float limit, best_t;
  uint32_t best;                 // index in ids of the closest voxel
  F3 best_n;                     // the normal of the face it is hit at
  bool occluded;

  // The brick record of a (negated) cell and its index (times 64); false
  // outside the grid.
  CT_D bool brick(int32_t ix, int32_t iy, int32_t iz, uint4 &e, uint32_t &base) const {
    const uint32_t x = (uint32_t)((ix ^ sx) - G.org[0]), y = (uint32_t)((iy ^ sy) - G.org[1]),
                   z = (uint32_t)((iz ^ sz) - G.org[2]);
    const uint32_t bx = x >> 4, by = y >> 4, bz = z >> 4;
    if (bx >= G.nblk[0] || by >= G.nblk[1] || bz >= G.nblk[2]) return false;
    const uint32_t b = (bz * G.nblk[1] + by) * G.nblk[0] + bx;
    const uint32_t r = (b << 6) | ((x >> 2) & 3u) | (y & 12u) | ((z & 12u) << 2);
    e = gld(G.bricks + r);
    base = r << 6;
    return true;
  }
  // The bit of a (negated) cell in its brick (the grid starts at a multiple
  // of 16 cells).
  CT_D uint32_t bit_of(int32_t ix, int32_t iy, int32_t iz) const {
    return ((uint32_t)(ix ^ sx) & 3u) | (((uint32_t)(iy ^ sy) & 3u) << 2) | (((uint32_t)(iz ^ sz) & 3u) << 4);
  }

  // The voxel test on an occupied cell.
  CT_D void test(int32_t ix, int32_t iy, int32_t iz, const uint4 &e, uint32_t base, uint32_t bit) {
    const int32_t cx = ix ^ sx, cy = iy ^ sy, cz = iz ^ sz;
    const F3 c = f3(((float)cx + 0.5f) * 0.03125f, ((float)cy + 0.5f) * 0.03125f, ((float)cz + 0.5f) * 0.03125f);
    float t;
    if (kAny) {
      const bool hit = intersect_box<false, false, true>(c, oo, dr, sg, sinv, t);
      if (hit && (t >= 0.0f) && (t <= limit) && (base | bit) != target) occluded = true;
    } else {
      F3 n;
      const bool hit = kMode == kTraceClosest ? intersect_box<true, true, true>(c, oo, dr, sg, sinv, t, &n)
                                              : intersect_box<true, false, true>(c, oo, dr, sg, sinv, t, &n);
      if (hit && (kMode == kTraceClosest ? t > 0.0f : t >= 0.0f) && t <= best_t) {
        const uint64_t mask = ((uint64_t)e.y << 32) | e.x;
        const uint32_t idx = e.z + (uint32_t)__popcll(mask & ((1ull << bit) - 1ull));
        bool better = t < best_t || best == kInvalid;
        if (!better) {  // equal t: the smaller (instance, primitive)
          const uint2 a = gld(G.ids + idx), b = gld(G.ids + best);
          better = a.x < b.x || (a.x == b.x && a.y < b.y);
        }
        if (better) {
          best_t = t;
          best = idx;
          best_n = n;
        }
      }
    }
  }

  // The state of a walk between its steps.
  // kNone: no ray; kWide: walk this ray through the BVH.
  static constexpr uint32_t kStepping = 0, kAtVoxel = 1, kEnded = 2, kNone = 3, kWide = 4;
  uint32_t state;
  uint4 e;                       // the cell's brick, its index and the cell's bit in it
  uint32_t cell_base, cell_bit;
  int32_t box_m, box_ext;        // the empty box: to the cell (i | box_m) + box_ext
  int32_t ix, iy, iz;            // the cell
  float t_in;                    // where the ray entered it
  uint32_t near;                 // 1: within p of a plane there
  float vx, vy, vz, qx, qy, qz, ivx, ivy, ivz, t_unit, t_end, k1;
  uint32_t octant;               // shift of the ray's nibble

  // Whether a position is within `m` of a lattice plane on an axis other
  // than the crossed one (always near its own plane); `any`: on any axis.
  CT_D static bool near_plane(float x, float y, float z, float m, bool any) {
    const float fx = fabsf(fractf(x) - 0.5f), fy = fabsf(fractf(y) - 0.5f), fz = fabsf(fractf(z) - 0.5f);
    return (any ? gmax(gmax(fx, fy), fz) : med3f(fx, fy, fz)) > 0.5f - m;
  }

  // Tests the cells across the edges within p of the position the ray
  // entered the cell at.
  CT_D void test_near() {
    const float p = gmin(__builtin_fmaf(10.0f * kU, t_in, k1), kNearMax), px = __builtin_fmaf(vx, t_in, qx),
                py = __builtin_fmaf(vy, t_in, qy), pz = __builtin_fmaf(vz, t_in, qz);
    const float fx = px - (float)ix, fy = py - (float)iy, fz = pz - (float)iz;
    const int32_t ax = fx < p ? -1 : (fx > 1.0f - p ? 1 : 0), ay = fy < p ? -1 : (fy > 1.0f - p ? 1 : 0),
                  az = fz < p ? -1 : (fz > 1.0f - p ? 1 : 0);
    // bit k: the cell offset on the axes of k's bits
    uint32_t ks = 0xFEu & (ax ? 0xFFu : 0x55u) & (ay ? 0xFFu : 0x33u) & (az ? 0xFFu : 0x0Fu);
    while (ks) {
      const uint32_t k = (uint32_t)__ffs((int)ks) - 1u;
      ks &= ks - 1u;
      const int32_t x = (k & 1u) ? ix + ax : ix, y = (k & 2u) ? iy + ay : iy, z = (k & 4u) ? iz + az : iz;
      uint4 e;
      uint32_t base;
      if (!brick(x, y, z, e, base)) continue;
      const uint32_t bit = bit_of(x, y, z);
      if (((((bit & 32u) ? e.y : e.x) >> (bit & 31u)) & 1u) != 0u) test(x, y, z, e, base, bit);
    }
  }

  // Where the ray leaves the box of cells from its cell to (ex, ey, ez).
  CT_D float leave(int32_t ex, int32_t ey, int32_t ez, float &tx, float &ty, float &tz, float &x, float &y, float &z,
                   float &pn) const {
    tx = ((float)(ex + 1) - qx) * ivx;
    ty = ((float)(ey + 1) - qy) * ivy;
    tz = ((float)(ez + 1) - qz) * ivz;
    const float t = gmin(gmin(tx, ty), tz);
    x = __builtin_fmaf(vx, t, qx);
    y = __builtin_fmaf(vy, t, qy);
    z = __builtin_fmaf(vz, t, qz);
    pn = gmin(__builtin_fmaf(10.0f * kU, t, k1), kNearMax);
    return t;
  }

  // Sets the walk up for a ray and its limit (any hit: of the distance; else
  // of the closest t); ended at once when the ray misses the grid.
  CT_D void start(const DScene &S, F3 o, F3 d, float max_t, uint32_t ti, uint32_t tp) {
    state = kEnded;
    limit = max_t;
    best_t = max_t;
    best = kInvalid;
    best_n = f3(0.0f, 0.0f, 0.0f);
    occluded = false;
    e = make_uint4(0u, 0u, 0u, 0u);
    cell_base = 0u;
    cell_bit = 0u;
    box_m = 0;
    box_ext = 0;
    float m[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) m[k] = G.w2o[k];
    oo = xform3(m, o, 1.0f);
    const F3 od = xform3(m, d, 0.0f);
    target = kInvalid;
    if (kAny && ti < S.n_inst) {
      const DInst *I = S.inst + ti;
      if (tp < gld(&I->count)) target = gld(G.cells + gld(&I->first) + tp);
    }
    const F3 inv = f3(safe_inverse(od.x), safe_inverse(od.y), safe_inverse(od.z));
    sinv = inv;
    dr = kMode == kTraceClosest ? mul_rot(od) : od;
    sg = f3(-gsign(dr.x), -gsign(dr.y), -gsign(dr.z));
    const float qmax = gmax(gmax(fabsf(oo.x), fabsf(oo.y)), fabsf(oo.z)) * kCellsPerUnit;
    const float dmax = gmax(gmax(fabsf(od.x), fabsf(od.y)), fabsf(od.z));
    if (kChecked) {
      state = kWide;
      // the times below are normal floats for these
      if (!(gmax(gmax(fabsf(o.x), fabsf(o.y)), fabsf(o.z)) <= G.max_o) || !(dmax > 1e-20f) ||
          !((fabsf(od.x) + fabsf(od.y)) + fabsf(od.z) < 1e20f))
        return;
    }
    // A direction of zero length or with a term that is not finite hits
    // nothing.
    if (!(dmax > 0.0f) || !((fabsf(od.x) + fabsf(od.y)) + fabsf(od.z) < INFINITY) ||
        !((fabsf(oo.x) + fabsf(oo.y)) + fabsf(oo.z) < 1e9f))
      return;
    int ex;
    (void)frexpf(dmax, &ex);
    sx = od.x < 0.0f ? -1 : 0;
    sy = od.y < 0.0f ? -1 : 0;
    sz = od.z < 0.0f ? -1 : 0;
    octant = ((uint32_t)sx & 4u) | ((uint32_t)sy & 8u) | ((uint32_t)sz & 16u);
    vx = ldexpf(fabsf(od.x), -ex);
    vy = ldexpf(fabsf(od.y), -ex);
    vz = ldexpf(fabsf(od.z), -ex);
    qx = (sx ? -oo.x : oo.x) * kCellsPerUnit;
    qy = (sy ? -oo.y : oo.y) * kCellsPerUnit;
    qz = (sz ? -oo.z : oo.z) * kCellsPerUnit;
    const bool lx = vx > kDeadAxis, ly = vy > kDeadAxis, lz = vz > kDeadAxis;
    ivx = lx ? ldexpf(fabsf(inv.x), ex) : 1e30f;
    ivy = ly ? ldexpf(fabsf(inv.y), ex) : 1e30f;
    ivz = lz ? ldexpf(fabsf(inv.z), ex) : 1e30f;
    // the grid's first and last cells in negated coordinates
    const int32_t dx = (int32_t)(16u * G.nblk[0]), dy = (int32_t)(16u * G.nblk[1]), dz = (int32_t)(16u * G.nblk[2]);
    const int32_t l0x = sx ? -(G.org[0] + dx) : G.org[0], l0y = sy ? -(G.org[1] + dy) : G.org[1],
                  l0z = sz ? -(G.org[2] + dz) : G.org[2];
    const int32_t hx = l0x + dx - 1, hy = l0y + dy - 1, hz = l0z + dz - 1;
    const float tn = gmax(gmax(((float)l0x - qx) * ivx, ((float)l0y - qy) * ivy), ((float)l0z - qz) * ivz);
    const float tf = gmin(gmin(((float)(hx + 1) - qx) * ivx, ((float)(hy + 1) - qy) * ivy), ((float)(hz + 1) - qz) * ivz);
    t_unit = ldexpf(1.0f, ex + 5);  // T of one unit of t
    t_end = (kAny ? limit : best_t) * t_unit;
    const float gm = gmax(gmax(gmax(fabsf((float)l0x), fabsf((float)hx)), gmax(fabsf((float)l0y), fabsf((float)hy))),
                          gmax(fabsf((float)l0z), fabsf((float)hz)));
    if (kChecked) {
      const float last = t_end < tf ? t_end : tf;
      if (!((10.0f * last + 1.5f * gmax(qmax, gm)) + 4.0f <= kWideMax)) return;
      state = kEnded;
    }
    const float t = gmax(tn, 0.0f);
    if (!(t <= tf) || t > t_end + kNearMax) return;
    k1 = kU * (1.5f * gmax(qmax, gm) + gmax(gmax(lx ? ivx : 0.0f, ly ? ivy : 0.0f), lz ? ivz : 0.0f) + 4.0f);
    t_in = t;
    const float px = __builtin_fmaf(vx, t, qx), py = __builtin_fmaf(vy, t, qy), pz = __builtin_fmaf(vz, t, qz);
    ix = clampi((int32_t)floorf(px), l0x, hx);
    iy = clampi((int32_t)floorf(py), l0y, hy);
    iz = clampi((int32_t)floorf(pz), l0z, hz);
    const float p = gmin(__builtin_fmaf(10.0f * kU, t, k1), kNearMax);
    near = near_plane(px, py, pz, p, true) ? 1u : 0u;  // an origin in the grid has crossed no axis
    look(~0);
  }

  // The cell the walk has entered: its brick (when it is another one), the
  // neighbours within p of its edges (rare, tested on the spot), and whether
  // it is a voxel.  Else the empty box to step over: the cell, the 2x2x2
  // cells around it when all are empty, or the empty cube of bricks.
  // Written, as `move`, without early exits: each exit of a divergent loop
  // costs a copy of the walk's state in every step.
  CT_D void look(int32_t moved) {
    bool ended = false;
    if ((moved & ~3) != 0) ended = !brick(ix, iy, iz, e, cell_base);
    if (near != 0u && !ended) {
      test_near();
      if (!kAny) t_end = best_t * t_unit;
      if (kAny) ended = occluded;
    }
    const bool empty = (e.x | e.y) == 0u;
    cell_bit = bit_of(ix, iy, iz);
    const uint32_t w = (uint32_t)((((uint64_t)e.y << 32) | e.x) >> (cell_bit & 0x2Au));
    const bool at_voxel = ((w >> (cell_bit & 0x15u)) & 1u) != 0u;
    box_m = (w & 0x00330033u) == 0u ? 1 : 0;
    box_m = empty ? 3 : box_m;
    box_m = near != 0u ? 0 : box_m;
    box_ext = empty && near == 0u ? (int32_t)((e.w >> octant) & 15u) * 4 - 4 : 0;
    state = ended ? kEnded : (at_voxel ? kAtVoxel : kStepping);
  }

  // One step of a stepping walk: out of the empty box into the next cell.
  CT_D void advance() {
    int32_t fx = (ix | box_m) + box_ext, fy = (iy | box_m) + box_ext, fz = (iz | box_m) + box_ext;
    float tx, ty, tz, x, y, z, pn;
    float t = leave(fx, fy, fz, tx, ty, tz, x, y, z, pn);
    bool nr = near_plane(x, y, z, pn * (tx <= t ? ivx : (ty <= t ? ivy : ivz)), false);
    if (nr && box_m != 0) {
      fx = ix;
      fy = iy;
      fz = iz;
      t = leave(fx, fy, fz, tx, ty, tz, x, y, z, pn);
      nr = near_plane(x, y, z, pn * (tx <= t ? ivx : (ty <= t ? ivy : ivz)), false);
    }
    const int32_t cx = clampi((int32_t)floorf(x), ix, fx), cy = clampi((int32_t)floorf(y), iy, fy),
                  cz = clampi((int32_t)floorf(z), iz, fz);
    const int32_t nx = tx <= t ? fx + 1 : cx, ny = ty <= t ? fy + 1 : cy, nz = tz <= t ? fz + 1 : cz;
    const int32_t moved = (ix ^ nx) | (iy ^ ny) | (iz ^ nz);
    ix = nx;
    iy = ny;
    iz = nz;
    t_in = t;
    near = nr ? 1u : 0u;
    state = kEnded;
    if (!(t > t_end + pn)) look(moved);
  }

  // The test of a walk at a voxel.  A closest walk whose hit lies before the
  // cell's end has ended.
  CT_D void test_voxel() {
    test(ix, iy, iz, e, cell_base, cell_bit);
    near = 0u;  // its neighbours are done too
    box_m = 0;
    box_ext = 0;
    state = kAny && occluded ? kEnded : kStepping;
    if (!kAny) {
      t_end = best_t * t_unit;
      float tx, ty, tz, x, y, z, pn;
      if (leave(ix, iy, iz, tx, ty, tz, x, y, z, pn) > t_end + pn) state = kEnded;
    }
  }

  // Lanes step until each has come to a voxel or ended; the voxel tests then
  // run together, and nearly all accept.  (The ballot also keeps the
  // compiler from testing each lane's voxel inside the stepping loop.)
  CT_D void run() {
    for (;;) {
      while (state == kStepping) advance();
      if (ballot(state == kAtVoxel) == 0ull) return;
      if (state == kAtVoxel) test_voxel();
    }
  }
};

// Walks a stream of rays per lane: `next` starts the lane's next ray (false:
// it has none left) and `done` takes the result of one that has ended.
// The longest ray of a wave takes several times the mean's steps, and a wave
// that waits for it runs at 30% of its lanes.  Here the stepping loop leaves once kWait
// lanes wait, tests those at a voxel and gives those that have ended their
// next ray; kWait balances idle lanes in the loop against the same in the
// (about five times longer) code between the loops.
template <int kMode, int kWait, class Next, class Done>
CT_D void walk_stream(GridWalk<kMode> &w, Next next, Done done) {
  using W = GridWalk<kMode>;
  if (!next()) w.state = W::kNone;
  for (;;) {
    const int keep = __popcll(ballot(w.state != W::kNone)) - kWait;
    if (w.state == W::kStepping) {
      do w.advance();
      while ((int)(w.state == W::kStepping) & (int)(__popcll(ballot(w.state == W::kStepping)) > keep));
    }
    if (w.state == W::kAtVoxel) w.test_voxel();
    const int stepping = __popcll(ballot(w.state == W::kStepping)), ended = __popcll(ballot(w.state == W::kEnded));
    if ((int)(stepping == 0) | (int)(ended >= kWait / 2)) {
      if (w.state == W::kEnded) {
        done();
        if (!next()) w.state = W::kNone;
      }
      if (ballot(w.state != W::kNone) == 0ull) return;
    }
  }
}

// How a kernel is built to walk: the BVH, the BVH with counters, or the cell
// grid (scenes that have one; the counters are the BVH's, so counted
// launches walk it), or the cell grid where it serves the ray and else the
// BVH (queries of any rays).
constexpr int kWalkBvh = 0, kWalkCount = 1, kWalkGrid = 2, kWalkQuery = 3;

// The whole walk of one ray.  Returns true when an any-hit query is
// occluded; a closest query leaves its hit in best_t/best_i/best_p (which
// enter as the current limit and an invalid hit).
template <int kMode, int kWalk>
CT_D bool traverse_mode(const DScene &S, F3 o, F3 d, float limit, uint32_t ti, uint32_t tp,
                        float &best_t, uint32_t &best_i, uint32_t &best_p, uint32_t *stk,
                        uint32_t stride, TraceCnt &cnt, bool &overflow) {
  if constexpr (kWalk == kWalkGrid || kWalk == kWalkQuery) {
    using W = GridWalk<kMode, kWalk == kWalkQuery>;
    W w{S.grid};
    w.start(S, o, d, kMode == kTraceAny ? limit : best_t, ti, tp);
    w.run();
    if (kWalk == kWalkQuery && w.state == W::kWide)
      return traverse_mode<kMode, kWalkBvh>(S, o, d, limit, ti, tp, best_t, best_i, best_p, stk, stride, cnt, overflow);
    if (kMode != kTraceAny && w.best != kInvalid) {
      const uint2 id = gld(S.grid.ids + w.best);
      best_t = w.best_t;
      best_i = id.x;
      best_p = id.y;
    }
    return w.occluded;
  } else {
    Walker<kMode, kWalk == kWalkCount> w;
    w.start(S, o, d, limit, ti, tp, stk, stride);
    w.best_t = best_t;
    w.best_i = best_i;
    w.best_p = best_p;
    while (!w.done) w.step(S, cnt);
    best_t = w.best_t;
    best_i = w.best_i;
    best_p = w.best_p;
    overflow = overflow || w.overflow;
    return w.occluded && !w.overflow;
  }
}

}  // namespace dev
}  // namespace ct
