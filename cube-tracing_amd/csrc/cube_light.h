// cube_light.h -- the random point of a cube light (light.glsl:329-345,
// prng.glsl:198-252) and the ray origin beside it.
#pragma once

#include "ct_device.h"

namespace ct {
namespace dev {

// LCG state after k steps: s * a^k + c * (a^(k-1) + ... + 1) (mod 2^32).
constexpr uint32_t lcg_mul_pow(int k) {
  uint32_t r = 1u;
  for (int i = 0; i < k; ++i) r *= 1664525u;
  return r;
}
constexpr uint32_t lcg_add_sum(int k) {
  uint32_t r = 0u, p = 1u;
  for (int i = 0; i < k; ++i) {
    r += p;
    p *= 1664525u;
  }
  return r * 1013904223u;
}
template <int k>
CT_D uint32_t lcg_skip(uint32_t s) {
  constexpr uint32_t A = lcg_mul_pow(k), C = lcg_add_sum(k);
  return A * s + C;
}
// The axis (0, 1, 2) and sign of a normal that is an axis vector; -1 for
// any other normal.
CT_D int normal_axis(F3 n, float &s) {
  s = 0.0f;
  if (n.y == 0.0f && n.z == 0.0f && fabsf(n.x) == 1.0f) { s = n.x; return 0; }
  if (n.x == 0.0f && n.z == 0.0f && fabsf(n.y) == 1.0f) { s = n.y; return 1; }
  if (n.x == 0.0f && n.y == 0.0f && fabsf(n.z) == 1.0f) { s = n.z; return 2; }
  return -1;
}
CT_D float component(F3 v, int a) { return a == 0 ? v.x : (a == 1 ? v.y : v.z); }
// True when the light voxel lies wholly on the back side of the surface at
// P (normal ns along axis na): then dot(normalize(P - x), n) >= 0 for every
// sample point x of the voxel, light.glsl:343 rejects all draws.  The
// 1e-4 margin covers the rounding of the sample position; near-boundary
// cases take the full loop.
CT_D bool light_behind_surface(F3 P, int na, float ns, F3 c, float half) {
  if (na < 0) return false;
  const float m = half + 1e-4f, p = component(P, na), q = component(c, na);
  return ns > 0.0f ? p >= q + m : p <= q - m;
}

// prng.glsl:198-252: the face random_cube_normal draws (urnd_interval(., 0, 6),
// whose values are below 6) from the state after its LCG step, its normal, and
// the point random_quad draws on it (the normal is an axis vector, so its
// tangents are the exact axis vectors t1, t2: their normalize divides by 1).
CT_D uint32_t random_cube_face(uint32_t s) {
  return min((uint32_t)((float)(s & 0x00FFFFFFu) / 16777216.0f * 6.0f), 5u);
}
CT_D F3 random_on_face(F3 c, uint32_t face, float half, uint32_t &seed) {
  const float u = rnd(seed);
  const float v = rnd(seed);
  const float qx = u * half, qy = v * half;  // light.glsl:335: half the voxel's size
  // c + n * half + t1 * qx + t2 * qy with the zero terms left out but for
  // the sign of a zero: t1, t2 = (0, 0, s), (0, -1, 0) on x, (0, 0, -s),
  // (-1, 0, 0) on y, (0, s, 0), (-1, 0, 0) on z, s the sign of n
  const uint32_t a = face >> 1;
  const bool up = (face & 1u) != 0u;
  const float n = up ? half : -half, q = up ? qx : -qx;
  const F3 c0 = f3(c.x + 0.0f, c.y + 0.0f, c.z + 0.0f);
  return f3(c0.x + (a == 0u ? n : -qy), c0.y + (a == 0u ? -qy : (a == 1u ? n : q)),
            c0.z + (a == 0u ? q : (a == 1u ? -q : n)));
}
// compute_ray_origin(p, n) of the normal n of a face.
CT_D F3 face_ray_origin(F3 p, uint32_t face) {
  const uint32_t a = face >> 1;
  const bool up = (face & 1u) != 0u;
  const float x = a == 0u ? p.x : (a == 1u ? p.y : p.z);
  const float step = up ? 1.f / 65536.f : -1.f / 65536.f;
  const uint32_t ulps = (x < 0.0f) == up ? (uint32_t)-256 : 256u;
  const float m = fabsf(x) < 1.f / 32.f ? x + step : __uint_as_float(__float_as_uint(x) + ulps);
  return f3(a == 0u ? m : p.x + 0.0f, a == 1u ? m : p.y + 0.0f, a == 2u ? m : p.z + 0.0f);
}

// The point on the cube at c that light.glsl:333-345 draws for the surface
// point P: up to 11 draws of a face and a point on it, until one's face looks
// at P and its point lies in front of the surface; returns whether one did.
// `face` and `pos` are the last draw's.
//
// Only that last draw needs its point.  On an axis normal (na, ns) both tests
// are signs: the first depends on the face alone, so a bit per face holds it,
// with the face that looks the way the surface does cleared; the second holds
// for every point when P is behind the whole voxel (P - x has the exact sign,
// and a point's coordinate rounds to no less than its bound's).  So a draw is
// one LCG step of three numbers and a bit test, and only voxels level with P
// compute its point.  A wave draws until its slowest lane is done, about 7
// times, and 11 full draws of 90 instructions each were most of k_ris: at
// 256^2 pixels and 32 candidates 203 us, with this 111 us (one wave a SIMD,
// bound by the chain of dependent instructions and light loads).
CT_D bool draw_cube_point(F3 P, F3 n, int na, float ns, F3 c, float half, uint32_t &seed, uint32_t &face, F3 &pos) {
  uint32_t faces = (P.x < c.x - half ? 1u : 0u) | (P.x > c.x + half ? 2u : 0u) | (P.y < c.y - half ? 4u : 0u) |
                   (P.y > c.y + half ? 8u : 0u) | (P.z < c.z - half ? 16u : 0u) | (P.z > c.z + half ? 32u : 0u);
  bool level = true;
  if (na >= 0) {
    const float p = component(P, na), q = component(c, na), reach = fabsf(half);
    faces &= ~(1u << (2 * na + (ns > 0.0f ? 1 : 0)));
    level = !(ns > 0.0f ? p < q - reach : p > q + reach);
  }
  uint32_t s = lcg_skip<1>(seed), i = 0;  // the state after the draw's first number
  bool vis;
  for (;;) {
    face = random_cube_face(s);
    vis = ((faces >> face) & 1u) != 0u;
    if (vis && level && (int)(face >> 1) != na) {
      uint32_t t = s;
      const F3 w = sub(P, random_on_face(c, face, half, t));
      vis = na >= 0 ? component(w, na) * ns < 0.0f : dot(normalize(w), n) < 0.0f;
    }
    if (vis || i++ >= 10u) break;
    s = lcg_skip<3>(s);
  }
  seed = s;
  pos = random_on_face(c, face, half, seed);
  return vis;
}

}  // namespace dev
}  // namespace ct
