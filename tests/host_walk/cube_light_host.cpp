// Host build of the cube light's draw (csrc/cube_light.h), called through
// ctypes: each draw by draw_cube_point and face_ray_origin and by the text,
// light.glsl:333-350 with prng.glsl:198-252 (random_cube_normal, random_quad),
// which computes every draw's point.
#include "../../cube-tracing_amd/csrc/cube_light.h"

namespace ct {
int fail(int code, const std::string &) { return code; }
}  // namespace ct
using namespace ct;
using namespace ct::dev;

namespace {

F3 cube_normal(uint32_t &seed) {
  switch (std::min(urnd_interval(seed, 0u, 6u), 5u)) {
    case 0: return f3(-1, 0, 0);
    case 1: return f3(1, 0, 0);
    case 2: return f3(0, -1, 0);
    case 3: return f3(0, 1, 0);
    case 4: return f3(0, 0, -1);
    default: return f3(0, 0, 1);
  }
}

F3 quad(F3 n, F3 p, float sx, float sy, uint32_t &seed) {
  const float u = rnd(seed);
  const float v = rnd(seed);
  const F3 t1 = fabsf(n.x) > fabsf(n.y) ? normalize(f3(-n.z, 0.0f, n.x)) : normalize(f3(0.0f, n.z, -n.y));
  const F3 t2 = normalize(cross(n, t1));
  return add(add(p, muls(t1, u * sx)), muls(t2, v * sy));
}

bool text(F3 P, F3 n, F3 c, float size, uint32_t &seed, F3 &pos, F3 &origin) {
  const float half = size * 0.5f;
  F3 nor;
  bool vis;
  uint32_t i = 0;
  do {
    nor = cube_normal(seed);
    pos = quad(nor, add(c, muls(nor, half)), half, half, seed);
    const F3 wi = normalize(sub(P, pos));
    vis = dot(wi, nor) > 0.0f && dot(wi, n) < 0.0f;
  } while (!vis && i++ < 10);
  origin = compute_ray_origin(compute_ray_origin(pos, nor), nor);
  return vis;
}

bool same(F3 a, F3 b) { return std::memcmp(&a, &b, sizeof(F3)) == 0; }

}  // namespace

// P, n, c [count][3], size, seed [count]; returns how many differ (skipping
// lights behind the surface, which draw nothing).  `taken`: by outcome.
extern "C" uint32_t draws_differ(uint32_t count, const float *P, const float *n, const float *c, const float *size,
                                 const uint32_t *seed, uint32_t *taken) {
  uint32_t bad = 0;
  taken[0] = taken[1] = taken[2] = 0;
  for (uint32_t i = 0; i < count; ++i) {
    const F3 p = f3(P[3 * i], P[3 * i + 1], P[3 * i + 2]), nn = f3(n[3 * i], n[3 * i + 1], n[3 * i + 2]),
             q = f3(c[3 * i], c[3 * i + 1], c[3 * i + 2]);
    uint32_t s0 = seed[i], s1 = seed[i], face;
    F3 a, b, o;
    const bool v0 = text(p, nn, q, size[i], s0, a, o);
    float ns;
    const int na = normal_axis(nn, ns);
    if (light_behind_surface(p, na, ns, q, size[i] * 0.5f)) {
      bad += v0 || lcg_skip<33>(s1) != s0;
      ++taken[2];
      continue;
    }
    const bool v1 = draw_cube_point(p, nn, na, ns, q, size[i] * 0.5f, s1, face, b);
    bad += v0 != v1 || s0 != s1 || !same(a, b) || !same(o, face_ray_origin(face_ray_origin(b, face), face));
    ++taken[v0 ? 0 : 1];
  }
  return bad;
}
