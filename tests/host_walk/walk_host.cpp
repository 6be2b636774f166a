// Host build of the cell-grid walk (csrc/ct_device.h), called through ctypes:
// each ray by the walk and by the voxel test on every voxel, with the same
// voxel test on the same operands, or by the walk of ray queries and by the
// BVH walk; and the rays each walk may take (csrc/grid_reach.h).
#include "../../cube-tracing_amd/csrc/ct_device.h"

#include <type_traits>
#include <vector>

namespace ct {
int fail(int code, const std::string &) { return code; }
}  // namespace ct
#include "../../cube-tracing_amd/csrc/grid_plan.h"
using namespace ct;
using namespace ct::dev;

namespace {

struct Scene {
  std::vector<uint4> bricks;
  std::vector<uint2> ids;
  std::vector<float> boxes;
  std::vector<uint32_t> cells;
  std::vector<DInst> inst;
  std::vector<DNode> nodes;
  std::vector<float4> leaves;
  uint32_t tlas_inst = 0;
  DScene S{};
};

// A BVH of the leaves [a, b), split at the median of the longest axis;
// returns the ref of its root (an internal node's index is its split's).
uint32_t build_bvh(Scene &sc, uint32_t a, uint32_t b, float *lo, float *hi) {
  auto axis = [](const float4 &v, int k) { return k == 0 ? v.x : (k == 1 ? v.y : v.z); };
  for (int k = 0; k < 3; ++k) {
    lo[k] = hi[k] = axis(sc.leaves[a], k);
    for (uint32_t i = a; i < b; ++i) {
      lo[k] = std::min(lo[k], axis(sc.leaves[i], k));
      hi[k] = std::max(hi[k], axis(sc.leaves[i], k));
    }
  }
  int k = 0;
  for (int c = 1; c < 3; ++c)
    if (hi[c] - lo[c] > hi[k] - lo[k]) k = c;
  for (int c = 0; c < 3; ++c) {
    lo[c] -= kHalfVoxel + kLeafPad;
    hi[c] += kHalfVoxel + kLeafPad;
  }
  if (b - a == 1) return kLeaf | a;
  const uint32_t m = (a + b) / 2;
  std::nth_element(sc.leaves.begin() + a, sc.leaves.begin() + m, sc.leaves.begin() + b,
                   [&](const float4 &p, const float4 &q) { return axis(p, k) < axis(q, k); });
  float l[6], h[6];
  const uint32_t c0 = build_bvh(sc, a, m, l, h), c1 = build_bvh(sc, m, b, l + 3, h + 3);
  DNode &n = sc.nodes[m];
  n.a = float4{l[0], l[1], l[2], h[0]};
  n.b = float4{h[1], h[2], l[3], l[4]};
  n.c = float4{l[5], h[3], h[4], h[5]};
  n.d = uint4{c0, c1, 0u, 0u};
  return m;
}

// cells [n][3] of one instance's voxels (object space lattice), each once
void build(Scene &sc, const int32_t *cells, uint32_t n, const float *w2o) {
  int32_t lo[3], hi[3];
  for (int a = 0; a < 3; ++a) {
    lo[a] = hi[a] = cells[a];
    for (uint32_t i = 0; i < n; ++i) {
      lo[a] = std::min(lo[a], cells[3 * i + a]);
      hi[a] = std::max(hi[a], cells[3 * i + a]);
    }
  }
  DGrid &G = sc.S.grid;
  uint32_t nb = 1;
  for (int a = 0; a < 3; ++a) {
    G.org[a] = (lo[a] - 4) & ~15;
    G.nblk[a] = (uint32_t)(((hi[a] + 4) | 15) + 1 - G.org[a]) / 16;
    nb *= G.nblk[a];
  }
  std::memcpy(G.w2o, w2o, sizeof(G.w2o));
  sc.bricks.assign((size_t)nb * 64, uint4{0, 0, 0, 0});
  auto at = [&](int32_t x, int32_t y, int32_t z) -> uint4 * {
    const uint32_t ux = (uint32_t)(x - G.org[0]), uy = (uint32_t)(y - G.org[1]), uz = (uint32_t)(z - G.org[2]);
    if (ux >= 16 * G.nblk[0] || uy >= 16 * G.nblk[1] || uz >= 16 * G.nblk[2]) return nullptr;
    const uint32_t b = ((uz >> 4) * G.nblk[1] + (uy >> 4)) * G.nblk[0] + (ux >> 4);
    return &sc.bricks[((size_t)b << 6) | ((ux >> 2) & 3u) | (uy & 12u) | ((uz & 12u) << 2)];
  };
  auto bit = [](int32_t x, int32_t y, int32_t z) { return (uint32_t)((x & 3) | ((y & 3) << 2) | ((z & 3) << 4)); };
  for (uint32_t i = 0; i < n; ++i) {
    uint4 *e = at(cells[3 * i], cells[3 * i + 1], cells[3 * i + 2]);
    const uint32_t b = bit(cells[3 * i], cells[3 * i + 1], cells[3 * i + 2]);
    (b < 32 ? e->x : e->y) |= 1u << (b & 31u);
  }
  uint32_t total = 0;
  for (uint4 &e : sc.bricks) {
    e.z = total;
    total += (uint32_t)(__builtin_popcount(e.x) + __builtin_popcount(e.y));
  }
  // the largest empty cube of bricks into each octant, by its definition
  auto occupied = [&](int32_t x, int32_t y, int32_t z) {
    const uint4 *e = at(x, y, z);
    return e && (e->x | e->y) != 0u;
  };
  for (uint32_t b = 0; b < nb; ++b)
    for (uint32_t l = 0; l < 64; ++l) {
      uint4 &e = sc.bricks[(size_t)b * 64 + l];
      if (e.x | e.y) continue;
      const int32_t x = G.org[0] + 16 * (int32_t)(b % G.nblk[0]) + 4 * (int32_t)(l & 3),
                    y = G.org[1] + 16 * (int32_t)((b / G.nblk[0]) % G.nblk[1]) + 4 * (int32_t)((l >> 2) & 3),
                    z = G.org[2] + 16 * (int32_t)(b / (G.nblk[0] * G.nblk[1])) + 4 * (int32_t)(l >> 4);
      for (uint32_t o = 0; o < 8; ++o) {
        uint32_t side = 1;
        for (int32_t s = 2; s <= (int32_t)kGridSkip; ++s) {
          bool empty = true;
          for (int32_t k = 0; k < s * s * s && empty; ++k)
            empty = !occupied(x + ((o & 1u) ? -4 : 4) * (k % s), y + ((o & 2u) ? -4 : 4) * (k / s % s),
                              z + ((o & 4u) ? -4 : 4) * (k / (s * s)));
          if (!empty) break;
          side = (uint32_t)s;
        }
        e.w |= side << (4 * o);
      }
    }
  sc.ids.resize(n);
  sc.boxes.resize(6 * (size_t)n);
  sc.cells.resize(n);
  for (uint32_t i = 0; i < n; ++i) {
    const int32_t *c = cells + 3 * i;
    const uint4 *e = at(c[0], c[1], c[2]);
    const uint64_t mask = ((uint64_t)e->y << 32) | e->x;
    sc.ids[e->z + (uint32_t)__builtin_popcountll(mask & ((1ull << bit(c[0], c[1], c[2])) - 1ull))] = uint2{0u, i};
    sc.cells[i] = (uint32_t)((e - sc.bricks.data()) << 6) | bit(c[0], c[1], c[2]);
    for (int a = 0; a < 3; ++a) {
      sc.boxes[6 * (size_t)i + a] = (float)c[a] * 0.03125f;
      sc.boxes[6 * (size_t)i + 3 + a] = (float)(c[a] + 1) * 0.03125f;
    }
  }
  sc.inst.resize(1);
  std::memset(sc.inst.data(), 0, sizeof(DInst));
  std::memcpy(sc.inst[0].w2o, w2o, sizeof(sc.inst[0].w2o));
  sc.inst[0].count = n;
  sc.S.inst = sc.inst.data();
  sc.S.n_inst = 1;
  for (uint32_t i = 0; i < n; ++i) {
    const float *b = &sc.boxes[6 * (size_t)i];
    sc.leaves.push_back(float4{(b[0] + b[3]) * 0.5f, (b[1] + b[4]) * 0.5f, (b[2] + b[5]) * 0.5f, __uint_as_float(i)});
  }
  sc.nodes.resize(n);
  float lo3[3], hi3[3];
  sc.inst[0].root = build_bvh(sc, 0, n, lo3, hi3);
  sc.S.blas_nodes = sc.nodes.data();
  sc.S.blas_leaves = sc.leaves.data();
  sc.S.tlas_inst = &sc.tlas_inst;
  sc.S.tlas_root = kLeaf;
  G.max_o = INFINITY;
  G.bricks = sc.bricks.data();
  G.ids = sc.ids.data();
  G.cells = sc.cells.data();
}

template <int kMode>
void both(const Scene &sc, const int32_t *cells, uint32_t n, F3 o, F3 d, float limit, uint32_t target, float *t_out,
          uint32_t *id_out, float *t_ref, uint32_t *id_ref) {
  float bt = limit;
  uint32_t bi = kInvalid, bp = kInvalid;
  TraceCnt cnt;
  bool ovf = false;
  const bool occ = traverse_mode<kMode, kWalkGrid>(sc.S, o, d, limit, target == kInvalid ? kInvalid : 0u, target, bt, bi,
                                                   bp, nullptr, 0u, cnt, ovf);
  // the same ray three times in one stream
  GridWalk<kMode> w{sc.S.grid};
  int left = 3, off = 0;
  walk_stream<kMode, 1>(
      w,
      [&]() -> bool {
        if (left-- == 0) return false;
        w.start(sc.S, o, d, limit, target == kInvalid ? kInvalid : 0u, target);
        return true;
      },
      [&]() {
        if (kMode == kTraceAny) off += w.occluded != occ;
        else off += (w.best == kInvalid) != (bp == kInvalid) || (bp != kInvalid && (sc.ids[w.best].y != bp || w.best_t != bt));
      });
  if (off != 0 || left != -1) bp = kInvalid - 1u;  // reported as a difference
  *t_out = kMode == kTraceAny || bp == kInvalid ? 0.0f : bt;
  *id_out = kMode == kTraceAny && bp == kInvalid ? (uint32_t)occ : bp;
  const float *m = sc.S.grid.w2o;
  const F3 oo = xform3(m, o, 1.0f), od = xform3(m, d, 0.0f);
  const F3 dr = kMode == kTraceClosest ? mul_rot(od) : od;
  const F3 sg = f3(-gsign(dr.x), -gsign(dr.y), -gsign(dr.z));
  const F3 inv = f3(safe_inverse(od.x), safe_inverse(od.y), safe_inverse(od.z));
  float rt = limit;
  uint32_t rp = kInvalid, hit_any = 0;
  for (uint32_t i = 0; i < n; ++i) {
    const float *b = &sc.boxes[6 * (size_t)i];
    const F3 c = f3((b[0] + b[3]) * 0.5f, (b[1] + b[4]) * 0.5f, (b[2] + b[5]) * 0.5f);
    float t;
    if (kMode == kTraceAny) {
      if (intersect_box<false, false>(c, oo, dr, sg, inv, t) && t >= 0.0f && t <= limit && i != target) hit_any = 1;
    } else {
      const bool hit = kMode == kTraceClosest ? intersect_box<true, true>(c, oo, dr, sg, inv, t)
                                              : intersect_box<true, false>(c, oo, dr, sg, inv, t);
      if (hit && (kMode == kTraceClosest ? t > 0.0f : t >= 0.0f) && (t < rt || (t == rt && i < rp))) {
        rt = t;
        rp = i;
      }
    }
  }
  *t_ref = kMode == kTraceAny || rp == kInvalid ? 0.0f : rt;
  *id_ref = kMode == kTraceAny ? hit_any : rp;
}

// A ray query's walk against the BVH walk; whether the query took the BVH.
template <int kMode>
bool query(const Scene &sc, F3 o, F3 d, float limit, uint32_t target, float *t_out, uint32_t *id_out, float *t_ref,
           uint32_t *id_ref) {
  const uint32_t ti = target == kInvalid ? kInvalid : 0u;
  auto one = [&](auto walk, float *t, uint32_t *id) {
    uint32_t stk[kStackLds], bi = kInvalid, bp = kInvalid;
    float bt = limit;
    TraceCnt cnt;
    bool ovf = false;
    const bool occ = traverse_mode<kMode, decltype(walk)::value>(sc.S, o, d, limit, ti, target, bt, bi, bp, stk, 1u, cnt, ovf);
    *t = kMode == kTraceAny || bp == kInvalid ? 0.0f : bt;
    *id = kMode == kTraceAny ? (uint32_t)occ : bp;
    if (ovf) *id = kInvalid - 1u;
  };
  one(std::integral_constant<int, kWalkQuery>{}, t_out, id_out);
  one(std::integral_constant<int, kWalkBvh>{}, t_ref, id_ref);
  GridWalk<kMode, true> w{sc.S.grid};
  w.start(sc.S, o, d, limit, ti, target);
  return w.state == GridWalk<kMode, true>::kWide;
}

}  // namespace

extern "C" void query_and_bvh(const int32_t *cells, uint32_t n, const float *w2o, int mode, uint32_t rays, const float *o,
                              const float *d, const float *limit, const uint32_t *target, float *t_out, uint32_t *id_out,
                              float *t_ref, uint32_t *id_ref, uint8_t *wide) {
  Scene sc;
  build(sc, cells, n, w2o);
#pragma omp parallel for schedule(dynamic, 64)
  for (uint32_t i = 0; i < rays; ++i) {
    const F3 ro = f3(o[3 * i], o[3 * i + 1], o[3 * i + 2]), rd = f3(d[3 * i], d[3 * i + 1], d[3 * i + 2]);
    auto fn = mode == kTraceAny ? query<kTraceAny> : mode == kTraceClosest ? query<kTraceClosest> : query<kTraceBounce>;
    wide[i] = fn(sc, ro, rd, limit[i], target[i], t_out + i, id_out + i, t_ref + i, id_ref + i);
  }
}

// Memory a scene can do without, refused: no buffer and no error left (0).
extern "C" int refused_memory() {
  DevBuf b;
  const bool got = reserve_optional(b, (size_t)1 << 30);
  return (got ? 1 : 0) | (b.p ? 2 : 0) | (b.bytes ? 4 : 0) | (hipGetLastError() != hipSuccess ? 8 : 0);
}

// Batches a wave takes, from `base` on (at most `most`, so that a loop without
// an end shows).
extern "C" uint32_t batches(uint32_t base, uint32_t count, uint32_t stride, uint32_t most) {
  uint32_t n = 0;
  for (; base < count && n < most; base = next_batch(base, count, stride)) ++n;
  return n;
}

// Updates of a scene's grid, planned (csrc/grid_plan.h): `count` instances of
// 8^3 cells side by side along x, all marked.  Then, by instance: first slots,
// counts, boxes' shifts in cells along x, bits (1 used, 2 changed, 4 bad, 8 turned).
// Returns the kind; lists and region as the plan has them.
extern "C" int plan_update(uint32_t count, const uint32_t *first, const uint32_t *prims, const float *shift,
                           const uint8_t *bits, int everything, int given_up, uint32_t *lists, uint32_t *region) {
  GridState g;
  std::vector<ct_instance> inst(count);
  std::vector<uint8_t> used(count);
  std::vector<float> w2o(16 * count, 0.0f), boxes(6 * count);
  const uint4 some{};
  g.lay.bricks = &some;
  g.given_up = given_up != 0;
  for (int a = 0; a < 3; ++a) {
    g.lay.org[a] = -16;
    g.lay.nblk[a] = a == 0 ? (8 * count + 15) / 16 + 2 : 3;
  }
  GridScene s{&inst, &used, w2o.data(), boxes.data(), {}, everything != 0};
  g.inst.resize(count);
  for (uint32_t i = 0; i < count; ++i) {
    inst[i] = ct_instance{};
    for (int k = 0; k < 16; k += 5) inst[i].transform[k] = w2o[16 * i + k] = 1.0f;
    inst[i].first_primitive_index = first[i];
    inst[i].primitive_count = prims[i];
    used[i] = bits[i] & 1u;
    if (bits[i] & 2u) s.changed.push_back(i);
    if (bits[i] & 8u) inst[i].transform[12] = w2o[16 * i + 12] = 0.5f;
    for (int a = 0; a < 3; ++a) {
      const float lo = a == 0 ? 8.0f * (float)i : 0.0f;
      g.inst[i].box[a] = lo / 32.0f;
      g.inst[i].box[3 + a] = (lo + 8.0f) / 32.0f;
      boxes[6 * i + a] = (lo + (a == 0 ? shift[i] : 0.0f)) / 32.0f;
      boxes[6 * i + 3 + a] = (lo + 8.0f + (a == 0 ? shift[i] : 0.0f)) / 32.0f;
    }
    g.inst[i].first = 64 * i;
    g.inst[i].count = 64;
    g.inst[i].bad = (bits[i] & 4u) != 0u;
  }
  const GridPlan p = plan_grid(s, g);
  for (uint32_t i = 0; i < count; ++i) lists[i] = 0;
  for (uint32_t i : p.unmark) lists[i] |= 1u;
  for (uint32_t i : p.mark) lists[i] |= 2u;
  for (uint32_t i : p.retry) lists[i] |= 4u;
  region[0] = p.lo[0];
  region[1] = p.hi[0];
  return (int)p.kind | (p.one_transform ? 16 : 0) | (p.give_up ? 32 : 0);
}

extern "C" float reach_of(const float *m, const float *w, const float *lo, const float *hi) { return world_reach(m, w, lo, hi); }

// Whether a scene's grid stays for rays from its surfaces and a camera.
extern "C" int served(const int32_t *cells, uint32_t n, const float *w2o, float max_o, const float *lo, const float *hi,
                      const float *inv_view) {
  Scene sc;
  build(sc, cells, n, w2o);
  sc.S.grid.max_o = max_o;
  Reach from;
  from.add(lo, hi);
  keep_served(sc.S.grid, from, inv_view);
  return sc.S.grid.bricks != nullptr;
}

extern "C" void walk_and_brute(const int32_t *cells, uint32_t n, const float *w2o, int mode, uint32_t rays,
                               const float *o, const float *d, const float *limit, const uint32_t *target, float *t_out,
                               uint32_t *id_out, float *t_ref, uint32_t *id_ref) {
  Scene sc;
  build(sc, cells, n, w2o);
#pragma omp parallel for schedule(dynamic, 64)
  for (uint32_t i = 0; i < rays; ++i) {
    const F3 ro = f3(o[3 * i], o[3 * i + 1], o[3 * i + 2]), rd = f3(d[3 * i], d[3 * i + 1], d[3 * i + 2]);
    auto fn = mode == kTraceAny ? both<kTraceAny> : mode == kTraceClosest ? both<kTraceClosest> : both<kTraceBounce>;
    fn(sc, cells, n, ro, rd, limit[i], target[i], t_out + i, id_out + i, t_ref + i, id_ref + i);
  }
}
