// g5_pool.hip -- device memory with freed blocks kept for reuse.
//
// A freed block joins its device's list (after the wait for the device that
// hipFree makes, or the owner's own wait for all work on it, so whoever takes
// it next, on whatever stream or thread, finds no work of the previous owner
// on it) and serves a later request of at least 4/5 of its size.  The list
// holds at most 1/8 of the device's memory; older blocks go back to the driver
// first, larger ones at once.  A request the driver cannot fill empties the
// list and tries again.  With the last context of a device gone everything
// goes back.
//
// Calls that wait for the device or for the driver (hipMalloc of memory that
// is still being cleared, hipFree) run without g_mu, so that no thread's
// request waits for another thread's work.  Kept blocks go back under
// g_driver, which a refused request takes before it tries again: it finds
// what was on its way back when it was refused.
#include "g5_internal.hpp"

#include <list>
#include <mutex>
#include <new>
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

std::mutex g_mu;      // the tables below
std::mutex g_driver;  // kept blocks on their way back to the driver; taken before g_mu
Pool g_pool[kMaxDevices];
std::unordered_map<void*, Live> g_live;  // blocks handed out, with their real sizes

// The oldest kept blocks, until the rest is at most `to`.
std::list<Block> take(Pool& pl, size_t to) {
  std::list<Block> out;
  while (pl.total > to) {
    pl.total -= pl.kept.front().bytes;
    out.splice(out.end(), pl.kept, pl.kept.begin());
  }
  return out;
}

void give_back(const std::list<Block>& blocks) {
  for (const Block& b : blocks) (void)hipFree(b.p);
}

// The current device, -1 if unknown or beyond the table.
int current() {
  int dev = 0;
  return hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDevices ? dev : -1;
}

}  // namespace

hipError_t pool_alloc(void** p, size_t bytes) {
  const int dev = current();
  if (dev >= 0) {
    std::lock_guard<std::mutex> lk(g_mu);
    Pool& pl = g_pool[dev];
    auto best = pl.kept.end();
    for (auto it = pl.kept.begin(); it != pl.kept.end(); ++it)
      if (it->bytes >= bytes && it->bytes - bytes <= it->bytes / 5 &&
          (best == pl.kept.end() || it->bytes < best->bytes))
        best = it;
    if (best != pl.kept.end()) {
      g_live[best->p] = {best->bytes, dev};
      *p = best->p;
      pl.total -= best->bytes;
      pl.kept.erase(best);
      return hipSuccess;
    }
  }
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();  // or a launch's check finds it, though the next try succeeds
    if (dev >= 0) {
      std::lock_guard<std::mutex> driver(g_driver);
      std::list<Block> back;
      {
        std::lock_guard<std::mutex> lk(g_mu);
        back = take(g_pool[dev], 0);
      }
      give_back(back);
      e = hipMalloc(p, bytes);
      if (e != hipSuccess) (void)hipGetLastError();
    }
  }
  if (e == hipSuccess) {
    try {
      std::lock_guard<std::mutex> lk(g_mu);
      g_live[*p] = {bytes, dev};
    } catch (const std::bad_alloc&) {
      (void)hipFree(*p);
      e = hipErrorOutOfMemory;
    }
  }
  return e;
}

void pool_free(void* p, bool idle) {
  Live b{0, -1};
  bool keep = false;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    const auto it = g_live.find(p);
    if (it != g_live.end()) {
      b = it->second;
      g_live.erase(it);
    }
    if (b.device >= 0 && b.device == current()) {
      const Pool& pl = g_pool[b.device];
      keep = pl.contexts > 0 && b.bytes <= pl.limit;
    }
  }
  // the list's entry: without host memory the block goes back at once (this
  // runs in destructors)
  std::list<Block> entry;
  if (keep) {
    try {
      entry.push_back({p, b.bytes});
    } catch (const std::bad_alloc&) {
      keep = false;
    }
  }
  if (keep && (idle || hipDeviceSynchronize() == hipSuccess)) {
    Pool& pl = g_pool[b.device];
    const auto add = [&] {
      pl.kept.splice(pl.kept.end(), entry);
      pl.total += b.bytes;
    };
    {
      std::lock_guard<std::mutex> lk(g_mu);
      if (pl.contexts > 0 && pl.total <= pl.limit - b.bytes) {
        add();
        return;
      }
    }
    std::lock_guard<std::mutex> driver(g_driver);
    std::list<Block> back;
    {
      std::lock_guard<std::mutex> lk(g_mu);
      keep = pl.contexts > 0;
      if (keep) {
        back = take(pl, pl.limit - b.bytes);
        add();
      }
    }
    give_back(back);
    if (keep) return;
  }
  (void)hipFree(p);
}

void pool_context(int device, int delta) {
  if (device < 0 || device >= kMaxDevices) return;
  std::unique_lock<std::mutex> driver(g_driver, std::defer_lock);
  if (delta < 0) driver.lock();  // blocks may go back
  std::list<Block> back;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    Pool& pl = g_pool[device];
    pl.contexts += delta;
    if (!pl.limit) {
      size_t free_b = 0, total_b = 0;
      if (hipMemGetInfo(&free_b, &total_b) == hipSuccess) pl.limit = total_b / 8;
    }
    if (pl.contexts == 0) back = take(pl, 0);
  }
  give_back(back);
}

}  // namespace g5
