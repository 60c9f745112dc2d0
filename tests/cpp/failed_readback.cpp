// Read-backs that fail: the library over a stand-in for the HIP runtime that
// needs no GPU.  Memory is host memory, launches do nothing (every header stays
// zero), and the n-th copy to the host fails on request.  A call that fails so
// has to give back what it allocated.
//
// The executable's own definitions of the HIP calls replace the runtime's (it is
// linked with its symbols exported).

#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "gdict.h"

namespace {
int copies_until_failure = -1;  // -1: none fails

hipError_t copy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind) {
  if (kind == hipMemcpyDeviceToHost && copies_until_failure >= 0 &&
      copies_until_failure-- == 0)
    return hipErrorUnknown;
  std::memcpy(dst, src, bytes);
  return hipSuccess;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t bytes) {
  *p = std::aligned_alloc(256, (bytes + 255) / 256 * 256);
  std::memset(*p, 0, bytes);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes,
                          hipMemcpyKind kind, hipStream_t) {
  return copy(dst, src, bytes, kind);
}
hipError_t hipMemcpy(void *dst, const void *src, size_t bytes,
                     hipMemcpyKind kind) {
  return copy(dst, src, bytes, kind);
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t,
                           hipStream_t) {
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) {
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(1);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
}

namespace {
int failures = 0;

void check(bool ok, const char *what) {
  std::printf("%s %s\n", ok ? "PASS" : "FAIL", what);
  failures += ok ? 0 : 1;
}

uint64_t live(gd_lsm *h) {
  gd_memory_stats m;
  if (gd_lsm_memory(h, &m) != GD_OK) std::abort();
  return m.live_bytes;
}

// A call whose n-th read-back fails for n = 0, 1, ... until none is left.
template <class Call>
void fail_each(gd_lsm *h, const char *what, Call call) {
  char line[128];
  for (int n = 0; n < 16; ++n) {
    const uint64_t before = live(h);
    copies_until_failure = n;
    const gd_status st = call();
    const bool failed = copies_until_failure == -1;
    copies_until_failure = -1;
    std::snprintf(line, sizeof(line), "%s: read-back %d %s, memory given back",
                  what, n, failed ? "fails" : "is not made");
    check((st != GD_OK) == failed && live(h) == before, line);
    if (!failed) return;
  }
  check(false, what);
}
}  // namespace

int main() {
  for (int runs = 1; runs <= 3; ++runs) {
    gd_config cfg{};
    cfg.max_elements = 1 << 16;
    cfg.batch_capacity = 1 << 12;
    gd_lsm *h = nullptr;
    if (gd_lsm_create(&cfg, &h) != GD_OK) return 1;
    static uint32_t keys[1024], values[1024];
    // batches of falling size stay runs of their own
    for (int r = 0; r < runs; ++r)
      if (gd_lsm_insert(h, keys, values, 1000 >> r, nullptr) != GD_OK) return 1;
    uint32_t got_runs = 0;
    uint64_t rows = 0, out = 0;
    if (gd_lsm_shape(h, &got_runs, &rows) != GD_OK) return 1;
    check(got_runs == static_cast<uint32_t>(runs), "runs as inserted");
    fail_each(h, "dump", [&] {
      return gd_lsm_dump_sorted(h, keys, values, 1024, &out, nullptr);
    });
    fail_each(h, "snapshot", [&] {
      return gd_lsm_snapshot_save(h, "/dev/null", &out, nullptr);
    });
    gd_lsm_destroy(h);
  }
  std::printf("FAILURES %d\n", failures);
  return failures != 0;
}
