// g5_pool.hip -- device memory with freed blocks kept for reuse.
//
// A freed block joins its device's list (after the wait for the device that
// hipFree makes, or the owner's own wait for all work on it, so whoever takes it next, on whatever stream or thread,
// finds no work of the previous owner on it) and serves a later request of
// at least 4/5 of its size.  The list holds at most 1/8 of the device's
// memory; older blocks go back to the driver first, larger ones at once.  A
// request the driver cannot fill empties the list and tries again.  With the
// last context of a device gone everything goes back.
#include "g5_internal.hpp"

#include <list>
#include <mutex>
#include <unordered_map>

namespace g5 {
namespace {

struct Block {
  void* p;
  size_t bytes;
};

constexpr int kMaxDevices = 64;

struct Pool {
  std::list<Block> kept;  // oldest first
  size_t total = 0, limit = 0;
  int contexts = 0;
};

struct Live {
  size_t bytes;
  int device;
};

std::mutex g_mu;
Pool g_pool[kMaxDevices];
std::unordered_map<void*, Live> g_live;  // blocks handed out, with their real sizes

void trim(Pool& pl, size_t to) {
  while (pl.total > to) {
    (void)hipFree(pl.kept.front().p);
    pl.total -= pl.kept.front().bytes;
    pl.kept.pop_front();
  }
}

// The current device, -1 if unknown or beyond the table.
int current() {
  int dev = 0;
  return hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices ? dev : -1;
}

}  // namespace

hipError_t pool_alloc(void** p, size_t bytes) {
  std::lock_guard<std::mutex> lk(g_mu);
  const int dev = current();
  Pool* pl = dev >= 0 ? &g_pool[dev] : nullptr;
  if (pl) {
    auto best = pl->kept.end();
    for (auto it = pl->kept.begin(); it != pl->kept.end(); ++it)
      if (it->bytes >= bytes && it->bytes - bytes <= it->bytes / 5 &&
          (best == pl->kept.end() || it->bytes < best->bytes))
        best = it;
    if (best != pl->kept.end()) {
      g_live[best->p] = {best->bytes, dev};
      *p = best->p;
      pl->total -= best->bytes;
      pl->kept.erase(best);
      return hipSuccess;
    }
  }
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();  // or a launch's check finds it, though the next try succeeds
    if (pl && !pl->kept.empty()) {
      trim(*pl, 0);
      e = hipMalloc(p, bytes);
      if (e != hipSuccess) (void)hipGetLastError();
    }
  }
  if (e == hipSuccess) g_live[*p] = {bytes, dev};
  return e;
}

void pool_free(void* p, bool idle) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    const auto it = g_live.find(p);
    const Live b = it != g_live.end() ? it->second : Live{0, -1};
    if (it != g_live.end()) g_live.erase(it);
    if (b.device >= 0 && b.device == current()) {
      Pool& pl = g_pool[b.device];
      if (pl.contexts > 0 && b.bytes <= pl.limit && (idle || hipDeviceSynchronize() == hipSuccess)) {
        trim(pl, pl.limit - b.bytes);
        pl.kept.push_back({p, b.bytes});
        pl.total += b.bytes;
        return;
      }
    }
  }
  (void)hipFree(p);
}

void pool_context(int device, int delta) {
  if (device < 0 || device >= kMaxDevices) return;
  std::lock_guard<std::mutex> lk(g_mu);
  Pool& pl = g_pool[device];
  pl.contexts += delta;
  if (!pl.limit) {
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) == hipSuccess) pl.limit = total_b / 8;
  }
  if (pl.contexts == 0) trim(pl, 0);
}

}  // namespace g5
