// grid_plan.h -- (host) what an update has to do to the scene's cell grid.
#pragma once

#include <cmath>
#include <cstring>
#include <vector>

#include "ct_internal.h"

namespace ct {

constexpr float kGridMaxCell = 4194304.0f;  // 2^22: cell centres and planes are exact floats

// What the update works from, by instance id.
struct GridScene {
  const std::vector<ct_instance> *instances;
  const std::vector<uint8_t> *used;
  const float *w2o;         // [id][16]
  const float *boxes;       // [id][6], object space
  std::vector<uint32_t> changed;  // instances whose voxels may have changed
  bool everything = false;  // the slots themselves are new
};

// kNone: the scene can have no grid.  kKeep: the grid's arrays are right as
// they are.  kPart: unmark the voxels of `unmark` (as last marked), mark
// those of `mark`, mark what `retry` has left unmarked, and link the blocks
// [lo, hi) again.  kFull: build it.
struct GridPlan {
  enum { kNone, kKeep, kPart, kFull } kind = kNone;
  bool one_transform = false;  // the walk may use the grid
  bool give_up = false;        // kNone, and until everything is new
  std::vector<uint32_t> unmark, mark, retry;
  int32_t org[3] = {0, 0, 0};  // the grid, whole blocks of 16 cells
  uint32_t nblk[3] = {0, 0, 0};
  uint32_t lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
  uint32_t n = 0;              // voxels of the scene
};

// Cells of a box with an empty brick at least around it; false out of range.
inline bool grid_cells(const float *box, int32_t *l, int32_t *h) {
  for (int c = 0; c < 3; ++c) {
    if (!(std::fabs(box[c]) < kGridMaxCell / 64.0f) || !(std::fabs(box[3 + c]) < kGridMaxCell / 64.0f)) return false;
    l[c] = (int32_t)std::floor(box[c] * 32.0f) - 5;
    h[c] = (int32_t)std::floor(box[3 + c] * 32.0f) + 5;
  }
  return true;
}

// A grid needs one transform for every instance, voxels on the 2^-5 lattice,
// one to a cell (both found while marking), and bricks that are few against
// the voxels.  The cost of an update is that of the instances it changed:
// building the whole grid anew took 0.35 ms of an update of 256^3 voxels
// whatever it changed (0.48 -> 0.83 ms for one that moves no voxel).  A
// change of half of the voxels is built anew, which also closes the gaps
// that parts leave in `ids`.  Where bad instances that the update leaves alone
// hold an eighth of the voxels, looking at them again each time would cost
// more than it promises.
inline GridPlan plan_grid(const GridScene &s, const GridState &g) {
  GridPlan p;
  const std::vector<ct_instance> &inst = *s.instances;
  std::vector<uint32_t> ids;
  for (uint32_t i = 0; i < inst.size(); ++i)
    if ((*s.used)[i]) ids.push_back(i);
  if (ids.empty()) return p;
  p.one_transform = true;
  std::vector<uint8_t> changed(inst.size(), 0);
  for (uint32_t id : s.changed)
    if (id < changed.size()) changed[id] = 1;
  bool same = g.lay.bricks && !s.everything, inside = same;
  uint64_t n = 0, moved = 0, retried = 0;
  float box[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  int32_t rl[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, rh[3] = {INT32_MIN, INT32_MIN, INT32_MIN};
  auto link = [&](const float *b) {
    int32_t l[3], h[3];
    if (!grid_cells(b, l, h)) return false;
    for (int c = 0; c < 3; ++c) {
      rl[c] = std::min(rl[c], l[c]);
      rh[c] = std::max(rh[c], h[c]);
    }
    return true;
  };
  for (uint32_t id : ids) {
    const ct_instance &in = inst[id];
    const float *b = s.boxes + 6 * (size_t)id;
    p.one_transform = p.one_transform && std::memcmp(s.w2o + 16 * (size_t)ids[0], s.w2o + 16 * (size_t)id, 64) == 0 &&
                      std::memcmp(inst[ids[0]].transform, in.transform, 64) == 0;
    for (int c = 0; c < 3; ++c) {
      box[c] = std::fmin(box[c], b[c]);
      box[3 + c] = std::fmax(box[3 + c], b[3 + c]);
    }
    n += in.primitive_count;
    if (!same) continue;
    const GridInst was = id < g.inst.size() ? g.inst[id] : GridInst{};
    if (changed[id] || was.first != in.first_primitive_index || was.count != in.primitive_count) {
      p.mark.push_back(id);
      inside = inside && link(b);
      moved += in.primitive_count;
      if (was.count) {
        p.unmark.push_back(id);
        inside = inside && link(was.box);
      }
    } else if (was.bad) {
      p.retry.push_back(id);
      retried += in.primitive_count;
      inside = inside && link(b);
    }
  }
  if (same)
    for (uint32_t id = 0; id < g.inst.size(); ++id)
      if (g.inst[id].count && !(id < inst.size() && (*s.used)[id])) {
        p.unmark.push_back(id);
        inside = inside && link(g.inst[id].box);
      }
  p.n = (uint32_t)n;
  if (same && p.mark.empty() && p.unmark.empty()) {
    p.retry.clear();  // nothing has made room
    p.kind = GridPlan::kKeep;
    return p;
  }
  if (!p.one_transform) return p;  // nothing would use it
  if (!s.everything && (g.given_up || 8 * retried > n)) {
    p.give_up = true;
    return p;
  }
  if (same && inside && 2 * moved <= n) {
    bool in_grid = true;
    for (int c = 0; c < 3; ++c) {
      p.org[c] = g.lay.org[c];
      p.nblk[c] = g.lay.nblk[c];
      in_grid = in_grid && rl[c] >= p.org[c] && rh[c] < p.org[c] + (int32_t)(16 * p.nblk[c]);
      if (!in_grid) break;
      // and what may step over the changed bricks: bricks within kGridSkip - 1
      const int32_t halo = 4 * ((int32_t)kGridSkip - 1);
      p.lo[c] = (uint32_t)std::max(rl[c] - halo - p.org[c], 0) / 16u;
      p.hi[c] = std::min((uint32_t)(rh[c] + halo - p.org[c]) / 16u + 1u, p.nblk[c]);
    }
    if (in_grid) {
      p.kind = GridPlan::kPart;
      return p;
    }
  }
  p.unmark.clear();
  p.retry.clear();
  p.mark = ids;
  int32_t l[3], h[3];
  if (!grid_cells(box, l, h)) return p;
  uint64_t nblk = 1;
  for (int c = 0; c < 3; ++c) {
    p.org[c] = l[c] & ~15;
    p.nblk[c] = (uint32_t)((h[c] | 15) + 1 - p.org[c]) / 16u;
    p.hi[c] = p.nblk[c];
    p.lo[c] = 0;
    nblk *= p.nblk[c];
    if (p.nblk[c] > 1024u || nblk > (1u << 19)) return p;
  }
  if (64 * nblk > 4 * n + (1u << 20)) return p;
  p.kind = GridPlan::kFull;
  return p;
}

}  // namespace ct
