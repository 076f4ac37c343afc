// Device memory of the library's calls: blocks given back by one call are kept
// for the next.  hipMalloc and hipFree cost 15-100 us each, and memory that
// the driver takes back is cleared before it is handed out again, at some 60
// GB/s: a level's bake frees 36 GB, and repeated bakes waited up to a second
// each for that once the whole of HBM had been handed out.
//
// What is kept: up to 256 MiB at any time, and up to an eighth of the device's
// memory while a scene, a transfer set or a server is alive; the rest, and
// everything above 256 MiB when the last of them is destroyed, goes back to
// the driver.  When the driver has no memory left, what is kept goes back
// first.
//
// A block that was given back may still be read by work in flight (a caller's
// stream, the other MakeTransfers stream), so it waits in a list of its own
// and is handed out only after a device synchronisation, which the first
// request that could use such a block pays for all of them.  hipFree, which
// this stands in for, waits in the same way.
#include <hip/hip_runtime_api.h>

#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "vr_internal.h"

namespace vr {
namespace {

constexpr size_t kKeepAlways = (size_t)256 << 20;

struct Pool {
  std::mutex mu;
  std::multimap<size_t, void *> ready;               // blocks no work can touch
  std::vector<std::pair<size_t, void *>> waiting;    // given back since the last synchronisation
  std::unordered_map<void *, size_t> size;           // every block handed out or kept
  size_t kept = 0, cap = 0;
  int holders = 0;

  size_t limit() {
    if (cap == 0) {
      size_t free_b = 0, total = 0;
      if (hipMemGetInfo(&free_b, &total) != hipSuccess) {
        (void)hipGetLastError();
        total = 0;
      }
      cap = total / 8 > kKeepAlways ? total / 8 : kKeepAlways;
    }
    return holders > 0 ? cap : kKeepAlways;
  }
  void drop(std::multimap<size_t, void *>::iterator it) {
    kept -= it->first;
    size.erase(it->second);
    (void)hipFree(it->second);
    ready.erase(it);
  }
  // The waiting blocks become ready, unless the synchronisation fails (a stream
  // of the caller is capturing, say): then their work may still run, and they
  // wait on.
  void settle() {
    if (waiting.empty()) return;
    if (hipDeviceSynchronize() != hipSuccess) {
      (void)hipGetLastError();
      return;
    }
    for (auto &w : waiting) ready.emplace(w.first, w.second);
    waiting.clear();
  }
  // gives back the largest blocks until at most `most` bytes are kept (or only
  // waiting ones are left that do not settle)
  void trim(size_t most) {
    if (kept <= most) return;
    settle();
    while (kept > most && !ready.empty()) drop(std::prev(ready.end()));
  }
  // a kept block for a request of n bytes: at most an eighth (and a page) larger
  std::multimap<size_t, void *>::iterator fit(size_t n) {
    auto it = ready.lower_bound(n);
    return it != ready.end() && it->first <= n + n / 8 + 65536 ? it : ready.end();
  }
};
Pool &pool() {
  static Pool *p = new Pool;  // outlives every handle
  return *p;
}

}  // namespace

int dev_alloc(void **out, size_t n) {
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  // sizes step by a sixteenth, so that calls of similar sizes share blocks
  size_t step = 4096;
  while (step * 32 <= n) step *= 2;
  n = (n + step - 1) / step * step;
  auto it = P.fit(n);
  if (it == P.ready.end()) {
    for (auto &w : P.waiting)
      if (w.first >= n && w.first <= n + n / 8 + 65536) {
        P.settle();
        it = P.fit(n);
        break;
      }
  }
  if (it != P.ready.end()) {
    *out = it->second;
    P.kept -= it->first;
    P.ready.erase(it);
    return 0;
  }
  hipError_t e = hipMalloc(out, n);
  if (e == hipErrorOutOfMemory && P.kept > 0) {
    (void)hipGetLastError();
    P.trim(0);
    e = hipMalloc(out, n);
  }
  if (e != hipSuccess) {
    *out = nullptr;
    (void)hipGetLastError();
    return (int)e;
  }
  P.size[*out] = n;
  return 0;
}

void dev_free(void *p) {
  if (!p) return;
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  auto it = P.size.find(p);
  if (it == P.size.end()) return;
  const size_t n = it->second, lim = P.limit();
  if (n > lim) {
    P.size.erase(it);
    (void)hipFree(p);
    return;
  }
  P.trim(lim - n);
  P.waiting.emplace_back(n, p);
  P.kept += n;
}

void dev_holder(int delta) {
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  P.holders += delta;
  if (P.holders <= 0) P.trim(kKeepAlways);
}

}  // namespace vr
