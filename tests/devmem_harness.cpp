// The device block pool (vrad_amd/csrc/devmem.cpp) over a stand-in for the HIP
// calls it makes: memory is numbers, and every call is recorded.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <map>

#include "../vrad_amd/csrc/vr_internal.h"

namespace {
int64_t g_total = 0, g_used = 0, g_next = 0;
int g_dev = 0, g_sync_error = 0;
int64_t g_syncs[4];  // synchronisations of each device
struct Block {
  int64_t bytes;
  int dev;
};
std::map<void *, Block> g_blocks;
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  if (g_used + (int64_t)n > g_total) return hipErrorOutOfMemory;
  *p = reinterpret_cast<void *>((uintptr_t)(0x1000 * ++g_next));
  g_blocks[*p] = Block{(int64_t)n, g_dev};
  g_used += (int64_t)n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  g_used -= g_blocks.at(p).bytes;
  g_blocks.erase(p);
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  if (g_sync_error) return hipErrorStreamCaptureUnsupported;
  ++g_syncs[g_dev];
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
  *f = (size_t)(g_total - g_used);
  *t = (size_t)g_total;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
  *d = g_dev;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  g_dev = d;
  return hipSuccess;
}

void t_setup(int64_t total) { g_total = total; }
void t_sync_error(int on) { g_sync_error = on; }
void t_device(int d) { g_dev = d; }
int t_current() { return g_dev; }
int64_t t_syncs(int dev) { return g_syncs[dev]; }
int64_t t_used() { return g_used; }
int64_t t_bytes(void *p) { return g_blocks.count(p) ? g_blocks[p].bytes : -1; }
int t_block_device(void *p) { return g_blocks.count(p) ? g_blocks[p].dev : -1; }
void *t_alloc(int64_t n) {
  void *p = nullptr;
  return vr::dev_alloc(&p, (size_t)n) == 0 ? p : nullptr;
}
void t_free(void *p) { vr::dev_free(p); }
void t_free_idle(void *p) { vr::dev_free(p, true); }
int64_t t_release() { return (int64_t)vr::dev_release(); }
void t_holder(int delta) { vr::dev_holder(delta); }
}
