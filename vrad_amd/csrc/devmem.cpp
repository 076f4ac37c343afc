// Device memory of the library's calls: blocks given back by one call are kept
// for the next.  hipMalloc and hipFree cost 15-100 us each, and memory that
// the driver takes back is cleared before it is handed out again, at some 60
// GB/s: a level's bake frees 36 GB, and repeated bakes waited up to a second
// each for that once the whole of HBM had been handed out.
//
// What is kept on a device: up to 256 MiB at any time, and up to an eighth of its
// memory while a scene, a transfer set or a server is alive; the rest, and
// everything above 256 MiB when the last of them is destroyed, goes back to
// the driver.  When the driver has no memory left, what is kept goes back
// first, and dev_release gives it back at any time.
//
// A block that was given back may still be read by work in flight (a caller's
// or a server's stream), so it waits in a list of its own and is handed out
// only after a synchronisation of its device, which the first request that
// could use such a block pays for all of them.  hipFree, which this stands in
// for, waits in the same way.  A block that the caller says is idle (it has
// waited for the stream of the block's only work) is available at once: the
// device synchronisation costs a call 7-11 us after pageable copies.  Each device has its own blocks: a thread's
// current device need not be the one a block lies on.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "vr_internal.h"

namespace vr {
namespace {

constexpr size_t kKeepAlways = (size_t)256 << 20;

// The blocks of one device.
struct Device {
  int id = 0;
  std::multimap<size_t, void *> ready;             // blocks no work can touch
  std::vector<std::pair<size_t, void *>> waiting;  // given back since the last synchronisation
  size_t kept = 0, cap = 0;
  size_t spare = 0;  // bytes of handed-out blocks beyond what was asked for
};
struct Block {
  size_t bytes, spare;
  Device *dev;
};

struct Pool {
  std::mutex mu;
  std::map<int, Device> devices;
  std::unordered_map<void *, Block> blocks;  // every block handed out or kept
  int holders = 0;

  // the device that hipMalloc allocates on in this thread
  Device &current() {
    int id = 0;
    if (hipGetDevice(&id) != hipSuccess) {
      (void)hipGetLastError();
      id = 0;
    }
    Device &D = devices[id];
    D.id = id;
    if (D.cap == 0) {
      size_t free_b = 0, total = 0;
      if (hipMemGetInfo(&free_b, &total) != hipSuccess) {
        (void)hipGetLastError();
        total = 0;
      }
      D.cap = std::max(total / 8, kKeepAlways);
    }
    return D;
  }
  size_t limit(const Device &D) const { return holders > 0 ? D.cap : kKeepAlways; }
  void drop(Device &D, std::multimap<size_t, void *>::iterator it) {
    D.kept -= it->first;
    blocks.erase(it->second);
    (void)hipFree(it->second);
    D.ready.erase(it);
  }
  // The waiting blocks become ready, unless the synchronisation fails (a stream
  // of the caller is capturing, say): then their work may still run, and they
  // wait on.
  void settle(Device &D) {
    if (D.waiting.empty()) return;
    int was = D.id;
    (void)hipGetDevice(&was);
    if (was != D.id) (void)hipSetDevice(D.id);
    const hipError_t e = hipDeviceSynchronize();
    if (was != D.id) (void)hipSetDevice(was);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return;
    }
    for (auto &w : D.waiting) D.ready.emplace(w.first, w.second);
    D.waiting.clear();
  }
  // gives back the largest blocks until at most `most` bytes are kept (or only
  // waiting ones are left that do not settle)
  void trim(Device &D, size_t most) {
    if (D.kept <= most) return;
    settle(D);
    while (D.kept > most && !D.ready.empty()) drop(D, std::prev(D.ready.end()));
  }
  // Whether n more bytes than asked for may be handed out: 1/128 of the device
  // in all, so that a set of blocks near its capacity still fits; 64 KiB always.
  static bool can_spare(const Device &D, size_t n) {
    return n <= 65536 || D.spare + n <= D.cap / 16;
  }
  // a kept block for a request of n bytes rounded to r: at most an eighth (and
  // a page) larger
  static std::multimap<size_t, void *>::iterator fit(Device &D, size_t n, size_t r) {
    auto it = D.ready.lower_bound(n);
    return it != D.ready.end() && fits(D, it->first, n, r) ? it : D.ready.end();
  }
  static bool fits(const Device &D, size_t have, size_t n, size_t r) {
    return have >= n && have <= r + r / 8 + 65536 && can_spare(D, have - n);
  }
  void hand_out(Device &D, void *p, size_t bytes, size_t n) {
    blocks[p] = Block{bytes, bytes - n, &D};
    D.spare += bytes - n;
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
  Device &D = P.current();
  // sizes step by a sixteenth, so that calls of similar sizes share blocks
  size_t step = 4096;
  while (step * 32 <= n) step *= 2;
  const size_t r = (n + step - 1) / step * step;
  auto it = P.fit(D, n, r);
  if (it == D.ready.end()) {
    for (auto &w : D.waiting)
      if (P.fits(D, w.first, n, r)) {
        P.settle(D);
        it = P.fit(D, n, r);
        break;
      }
  }
  if (it != D.ready.end()) {
    *out = it->second;
    P.hand_out(D, it->second, it->first, n);
    D.kept -= it->first;
    D.ready.erase(it);
    return 0;
  }
  size_t bytes = P.can_spare(D, r - n) ? r : n;
  hipError_t e = hipMalloc(out, bytes);
  if (e == hipErrorOutOfMemory && D.kept > 0) {
    (void)hipGetLastError();
    P.trim(D, 0);
    e = hipMalloc(out, bytes);
  }
  if (e == hipErrorOutOfMemory && bytes > n) {
    (void)hipGetLastError();
    e = hipMalloc(out, bytes = n);
  }
  if (e != hipSuccess) {
    *out = nullptr;
    (void)hipGetLastError();
    return (int)e;
  }
  P.hand_out(D, *out, bytes, n);
  return 0;
}

void dev_free(void *p, bool idle) {
  if (!p) return;
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  auto it = P.blocks.find(p);
  if (it == P.blocks.end()) return;
  Device &D = *it->second.dev;
  const size_t n = it->second.bytes, lim = P.limit(D);
  D.spare -= it->second.spare;
  it->second.spare = 0;
  if (n > lim) {
    P.blocks.erase(it);
    (void)hipFree(p);
    return;
  }
  P.trim(D, lim - n);
  if (idle) D.ready.emplace(n, p);
  else D.waiting.emplace_back(n, p);
  D.kept += n;
}

int dev_holder(int delta) {
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  P.holders += delta;
  if (P.holders <= 0)
    for (auto &d : P.devices) P.trim(d.second, kKeepAlways);
  return P.holders;
}

size_t dev_release() {
  Pool &P = pool();
  std::lock_guard<std::mutex> lock(P.mu);
  size_t left = 0;
  for (auto &d : P.devices) {
    P.trim(d.second, 0);
    left += d.second.kept;
  }
  return left;
}

}  // namespace vr
