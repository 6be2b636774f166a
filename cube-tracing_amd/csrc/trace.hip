// trace.hip -- ct_trace_closest / ct_trace_any on caller-owned arrays: the
// traversal kernels of the frame path, exposed for tests and tools.

#include <hip/hip_runtime.h>

#include <cstring>
#include <functional>
#include <vector>

#include "ct_internal.h"

using namespace ct;

namespace ct {

// The block is kept between calls up to this size; a larger one is the call's
// own.  The copies are pageable: pinned memory halves their time, but its
// allocation and release (3 ms) would be paid by every accel, and one that is
// built, asked once and closed is a usual one.
// 100 k rays through closest, bounce and any hit took 490, 880 and 640 us with
// an allocation and a repacking loop on the host per array.
constexpr size_t kIoKeep = (size_t)64 << 20;

int through_device(Accel &a, const std::vector<HostIn> &in, const std::vector<HostOut> &out,
                   const std::function<int(const std::vector<void *> &)> &launch) {
  std::vector<size_t> at;
  size_t total = 0;
  auto place = [&](size_t bytes) {
    at.push_back(total);
    total += (bytes + 15) & ~(size_t)15;
  };
  for (const HostIn &i : in) place(i.bytes);
  for (const HostOut &o : out) place(o.bytes);
  const std::lock_guard<std::mutex> lock(a.io_mu);
  DevBuf own;
  DevBuf &dev = total <= kIoKeep ? a.io_dev : own;
  int rc;
  if ((rc = dev.reserve(total))) return rc;
  std::vector<void *> ptr;
  for (size_t o : at) ptr.push_back(dev.as<unsigned char>() + o);
  for (size_t k = 0; k < in.size(); ++k) CT_HIP(hipMemcpy(ptr[k], in[k].p, in[k].bytes, hipMemcpyHostToDevice));
  rc = launch(ptr);
  const hipError_t e = hipStreamSynchronize(a.stream);  // the block is the next call's
  if (!rc && e != hipSuccess) rc = fail(CT_E_HIP, std::string("hipStreamSynchronize: ") + hipGetErrorString(e));
  if (rc) return rc;
  for (size_t k = 0; k < out.size(); ++k)
    CT_HIP(hipMemcpy(out[k].p, ptr[in.size() + k], out[k].bytes, hipMemcpyDeviceToHost));
  return CT_OK;
}

}  // namespace ct

namespace {

constexpr uint32_t kNoAllocMaxRays = 1u << 20;

// Counters of an instrumented launch, which start at zero.
struct Counters {
  unsigned long long v[3] = {0, 0, 0};
  void store(uint32_t n, ct_trace_stats *stats) const {
    stats->rays = n;
    stats->nodes = v[0];
    stats->leaves = v[1];
    stats->instances = v[2];
  }
};

}  // namespace

extern "C" {

int ct_trace_any_noalloc(ct_accel *a, uint32_t n, const float *origins, const float *directions,
                         const float *distances, const uint32_t *targets, uint8_t *occluded_out, void *stream) {
  if (!a || (n && (!origins || !directions || !distances || !occluded_out)))
    return fail(CT_E_INVALID, "ct_trace_any_noalloc: null argument");
  if (n > kNoAllocMaxRays) return fail(CT_E_CAPACITY, "ct_trace_any_noalloc: more than 2^20 rays in one call");
  if (a->set.tlas_count == 0) return fail(CT_E_STATE, "ct_trace_any_noalloc: empty scene");
  if (n == 0) return CT_OK;
  CT_HIP(hipSetDevice(a->device));
  hipStream_t st = stream ? static_cast<hipStream_t>(stream) : a->stream;
  const TraceAnyArgs t{origins, directions, distances, targets, occluded_out, nullptr, n};
  DScene s = scene_view(*a);
  if (recording(st)) s.grid.bricks = nullptr;
  return launch_trace_any(s, t, st);
}

int ct_trace_closest(ct_accel *a, uint32_t n, const float *origins, const float *directions, float tmax,
                     float *t_out, uint32_t *ids_out, ct_trace_stats *stats) {
  if (!a || (n && (!origins || !directions || !t_out || !ids_out)))
    return fail(CT_E_INVALID, "ct_trace_closest: null argument");
  if (a->set.tlas_count == 0) return fail(CT_E_STATE, "ct_trace_closest: empty scene");
  if (n == 0) return CT_OK;
  CT_HIP(hipSetDevice(a->device));
  const size_t m = n;
  Counters c;
  std::vector<HostIn> in{{origins, 12 * m}, {directions, 12 * m}};
  std::vector<HostOut> out{{t_out, 4 * m}, {ids_out, 8 * m}};
  if (stats) {
    in.push_back({c.v, sizeof(c.v)});
    out.push_back({c.v, sizeof(c.v)});
  }
  const int rc = through_device(*a, in, out, [&](const std::vector<void *> &p) -> int {
    TraceClosestArgs t;
    t.o = static_cast<float *>(p[0]);
    t.d = static_cast<float *>(p[1]);
    t.tmax = tmax;
    t.n = n;
    t.t = static_cast<float *>(p[in.size()]);
    t.ids = static_cast<uint32_t *>(p[in.size() + 1]);
    t.stats = nullptr;
    if (stats) {
      t.stats = static_cast<unsigned long long *>(p.back());
      CT_HIP(hipMemcpyAsync(t.stats, p[2], sizeof(c.v), hipMemcpyDeviceToDevice, a->stream));
    }
    return launch_trace_closest(scene_view(*a), t, a->stream);
  });
  if (!rc && stats) c.store(n, stats);
  return rc;
}

int ct_trace_any(ct_accel *a, uint32_t n, const float *origins, const float *directions, const float *distances,
                 const uint32_t *targets, uint8_t *occluded_out, ct_trace_stats *stats) {
  if (!a || (n && (!origins || !directions || !distances || !occluded_out)))
    return fail(CT_E_INVALID, "ct_trace_any: null argument");
  if (a->set.tlas_count == 0) return fail(CT_E_STATE, "ct_trace_any: empty scene");
  if (n == 0) return CT_OK;
  CT_HIP(hipSetDevice(a->device));
  const size_t m = n;
  Counters c;
  std::vector<HostIn> in{{origins, 12 * m}, {directions, 12 * m}, {distances, 4 * m}};
  std::vector<HostOut> out{{occluded_out, m}};
  if (targets) in.push_back({targets, 8 * m});
  if (stats) {
    in.push_back({c.v, sizeof(c.v)});
    out.push_back({c.v, sizeof(c.v)});
  }
  const int rc = through_device(*a, in, out, [&](const std::vector<void *> &p) -> int {
    TraceAnyArgs t;
    t.o = static_cast<float *>(p[0]);
    t.d = static_cast<float *>(p[1]);
    t.dist = static_cast<float *>(p[2]);
    t.targets = targets ? static_cast<uint32_t *>(p[3]) : nullptr;
    t.occ = static_cast<uint8_t *>(p[in.size()]);
    t.stats = nullptr;
    t.n = n;
    if (stats) {
      t.stats = static_cast<unsigned long long *>(p.back());
      CT_HIP(hipMemcpyAsync(t.stats, p[in.size() - 1], sizeof(c.v), hipMemcpyDeviceToDevice, a->stream));
    }
    return launch_trace_any(scene_view(*a), t, a->stream);
  });
  if (!rc && stats) c.store(n, stats);
  return rc;
}

}  // extern "C"
