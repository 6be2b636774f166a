// grid_reach.h -- (host) which ray origins the cell-grid walk serves with the
// BVH walk's hits to the bit.  The walk's own bound is GridWalk's in
// ct_device.h: in cells, 10 T + 1.5 max|position| + 4 <= kWideMax.
#pragma once

#include <algorithm>
#include <cmath>

#include "ct_internal.h"

namespace ct {

constexpr float kWideMax = 131072.0f;  // 2^-7 (half the padding of the BVH's boxes, in cells) / 2^-24

// The largest |world coordinate| of a ray origin for which the TLAS, whose
// boxes are padded by 2^-12 in world space, keeps every instance that the
// object-space ray hits.  `m` takes the instances to the world, `w` back
// (4x4, column-major), [lo, hi] bounds the instances there.  The object-space
// ray is off the world ray by the rounding of w, of its product with the ray
// and of the test of the boxes: 19 u (K |o| + |m| |w_t|) + 5 u K B + 4 u B for
// K the largest row sum of |m| |w| and B the largest coordinate of the boxes.
// An identity rounds nothing.  0: no ray (the transforms are not each
// other's inverses, or not affine, or of a size whose products leave the
// normal floats).
inline float world_reach(const float *m, const float *w, const float *lo, const float *hi) {
  const double u = 5.9604644775390625e-8;
  bool identity = true;
  for (int c = 0; c < 4; ++c)
    for (int r = 0; r < 4; ++r) {
      const float e = c == r ? 1.0f : 0.0f;
      identity = identity && m[c * 4 + r] == e && w[c * 4 + r] == e;
      if (r == 3 && !(m[c * 4 + r] == e)) return 0.0f;
    }
  if (identity) return INFINITY;
  double K = 0.0, wt = 0.0, B = 0.0, mmax = 0.0, wmax = 0.0;
  for (int r = 0; r < 3; ++r) {
    double row = 0.0, t = 0.0, tr = m[12 + r];
    for (int j = 0; j < 3; ++j) {
      double s = 0.0, a = 0.0;
      for (int c = 0; c < 3; ++c) {
        const double p = (double)m[c * 4 + r] * w[j * 4 + c];
        s += p;
        a += std::fabs(p);
      }
      if (!(std::fabs(s - (j == r ? 1.0 : 0.0)) <= 8.0 * u * a)) return 0.0f;
      row += a;
      const double q = (double)m[j * 4 + r] * w[12 + j];
      tr += q;
      t += std::fabs(q);
      mmax = std::max<double>(mmax, std::fabs(m[j * 4 + r]));
      wmax = std::max<double>(wmax, std::fabs(w[j * 4 + r]));
    }
    if (!(std::fabs(tr) <= 8.0 * u * (t + std::fabs(m[12 + r])))) return 0.0f;
    K = std::max(K, row);
    wt = std::max(wt, t);
    for (const double x : {(double)lo[r], (double)hi[r], (double)m[12 + r]}) {
      if (!(std::fabs(x) < INFINITY)) return 0.0f;
      B = std::max(B, std::fabs(x));
    }
  }
  if (!(mmax > 1e-9) || !(mmax < 1e9) || !(wmax > 1e-9) || !(wmax < 1e9)) return 0.0f;
  const double reach = (0.000244140625 / (19.0 * u) - wt - (1.0 + K) * B) / K;
  return reach > 0.0 ? (float)reach : 0.0f;
}

// Whether the grid walk serves every ray whose origin lies in the world box
// [lo, hi], whatever its direction.
inline bool grid_serves(const DGrid &g, const float *lo, const float *hi) {
  if (!g.bricks) return false;
  double extent = 0.0, pos = 0.0;
  for (int r = 0; r < 3; ++r) {
    double c = g.w2o[9 + r], e = 0.0;
    for (int j = 0; j < 3; ++j) {
      const float reach = std::max(std::fabs(lo[j]), std::fabs(hi[j]));
      if (!(reach <= g.max_o) || !(reach < 1e9f) || !(lo[j] <= hi[j])) return false;
      c += (double)g.w2o[j * 3 + r] * 0.5 * ((double)lo[j] + hi[j]);
      e += std::fabs((double)g.w2o[j * 3 + r]) * 0.5 * ((double)hi[j] - lo[j]);
    }
    const double a = std::min(32.0 * (c - e), (double)g.org[r]),
                 b = std::max(32.0 * (c + e), (double)g.org[r] + 16.0 * g.nblk[r]);
    extent = std::max(extent, b - a);
    pos = std::max(pos, std::max(std::fabs(a), std::fabs(b)));
  }
  // T runs over 1/2 to 1 cell of the fastest axis
  return 1.01 * (20.0 * extent + 1.5 * pos + 4.0) <= kWideMax;
}

// Whether a camera's matrix makes rays of ordinary lengths: its axes are
// about at right angles and neither tiny nor huge.
inline bool camera_regular(const float *inv_view) {
  double len[3];
  for (int c = 0; c < 3; ++c) {
    const float *a = inv_view + 4 * c;
    len[c] = std::sqrt((double)a[0] * a[0] + (double)a[1] * a[1] + (double)a[2] * a[2]);
    if (!(len[c] > 1e-9) || !(len[c] < 1e9)) return false;
  }
  for (int c = 0; c < 3; ++c) {
    const float *a = inv_view + 4 * c, *b = inv_view + 4 * ((c + 1) % 3);
    if (!(std::fabs((double)a[0] * b[0] + (double)a[1] * b[1] + (double)a[2] * b[2]) <= 0.01 * len[c] * len[(c + 1) % 3]))
      return false;
  }
  return true;
}

// The grid of a scene for rays from its surfaces (within `from`) and from a
// camera; null bricks: walk its BVH.
inline void keep_served(DGrid &g, const Reach &from, const float *inv_view) {
  Reach r = from;
  r.add(inv_view + 12, inv_view + 12);
  if (!camera_regular(inv_view) || !grid_serves(g, r.lo, r.hi)) g.bricks = nullptr;
}

}  // namespace ct
