// Checks of the block pool (g5_pool.hip) on the CPU; argv[1] names one.
#include "g5_internal.hpp"

#include <stdlib.h>
#include <string.h>

#include <functional>
#include <future>
#include <map>
#include <mutex>
#include <new>

// Host allocations fail while this is set.
static bool no_memory;
void* operator new(size_t n) {
  void* p = no_memory ? nullptr : malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

namespace {

constexpr size_t kTotal = 8000;  // the pool keeps up to an eighth
std::mutex mu;
std::map<void*, size_t> blocks;
size_t used;
int mallocs, frees, waits;
thread_local int device;
thread_local hipError_t last;
uintptr_t next_p = 0x1000;
bool fail_after_malloc;  // host memory ends with the next device allocation
std::function<void()> on_wait;  // runs while a call waits for the device (a free waits for it too)

void wait_for_device() {
  std::function<void()> f;
  std::swap(f, on_wait);
  if (f) f();
}

}  // namespace

const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "out of memory"; }
hipError_t hipMalloc(void** p, size_t bytes) {
  std::lock_guard<std::mutex> lk(mu);
  ++mallocs;
  if (used + bytes > kTotal) return last = hipErrorOutOfMemory;
  *p = (void*)next_p;
  next_p += 0x1000;
  blocks[*p] = bytes;
  used += bytes;
  no_memory = fail_after_malloc;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  wait_for_device();
  std::lock_guard<std::mutex> lk(mu);
  ++frees;
  const auto it = blocks.find(p);
  if (it == blocks.end()) {
    fprintf(stderr, "freed twice\n");
    abort();
  }
  used -= it->second;
  blocks.erase(it);
  return hipSuccess;
}
hipError_t hipGetDevice(int* dev) {
  *dev = device;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  ++waits;
  wait_for_device();
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t hipMemGetInfo(size_t* free_b, size_t* total_b) {
  *free_b = kTotal - used;
  *total_b = kTotal;
  return hipSuccess;
}

using namespace g5;

#define CHECK(x)                                              \
  do {                                                        \
    if (!(x)) {                                               \
      fprintf(stderr, "line %d: %s\n", __LINE__, #x);         \
      exit(1);                                                \
    }                                                         \
  } while (0)

static void* get(size_t bytes) {
  void* p = nullptr;
  CHECK(pool_alloc(&p, bytes) == hipSuccess && p);
  return p;
}

// A request takes the smallest kept block it fills to 4/5.
static void sizes() {
  pool_context(0, 1);
  void *a = get(500), *b = get(450);
  pool_free(a);
  pool_free(b);
  CHECK(frees == 0 && waits == 2 && used == 950);
  CHECK(get(400) == b);
  CHECK(get(400) == a);
  void* c = get(399);
  CHECK(c != a && c != b && mallocs == 3);
  pool_free(a);
  CHECK(get(501) != a);
  CHECK(get(399) != a);
  CHECK(get(500) == a);
}

// At most an eighth is kept: older blocks go back first, a larger one at once.
static void bound() {
  pool_context(0, 1);
  void *a = get(400), *b = get(410), *c = get(420), *d = get(1001);
  pool_free(a);
  pool_free(b, true);
  CHECK(waits == 1);
  pool_free(c);
  CHECK(frees == 1 && blocks.count(a) == 0 && blocks.count(b) == 1);
  pool_free(d);
  CHECK(blocks.count(d) == 0 && used == 830);
}

// A request the device cannot fill takes back what is kept, and leaves no
// error for the next call's check to find; one beyond that fails, likewise.
static void refill() {
  pool_context(0, 1);
  void *a = get(900), *b = get(6900);
  pool_free(a);
  CHECK(used == 7800);
  void* c = get(1000);
  CHECK(hipGetLastError() == hipSuccess);
  CHECK(blocks.count(a) == 0 && used == 7900);
  void* d = nullptr;
  CHECK(pool_alloc(&d, 200) == hipErrorOutOfMemory);
  CHECK(hipGetLastError() == hipSuccess);
  pool_free(b);
  pool_free(c);
}

// Nothing is kept without a context, beside other devices, or past the last one.
static void contexts() {
  void* a = get(100);
  pool_free(a);
  CHECK(blocks.empty());
  pool_context(0, 1);
  pool_context(0, 1);
  pool_context(1, 1);
  a = get(100);
  device = 1;
  pool_free(a);
  CHECK(blocks.empty());
  a = get(100);
  pool_free(a);
  device = 0;
  void* b = get(100);
  CHECK(b != a);
  pool_free(b);
  pool_context(0, -1);
  CHECK(used == 200);
  pool_context(0, -1);
  CHECK(used == 100);
  pool_context(1, -1);
  CHECK(blocks.empty());
}

// While one thread waits for the device (a free, a block that goes back to the
// driver, the last context), others get and return blocks; none of it is lost.
static void threads() {
  bool ran = false;
  const auto other_goes_on = [&ran] {
    ran = true;
    auto f = std::async(std::launch::async, [] { pool_free(get(50), true); });
    if (f.wait_for(std::chrono::seconds(5)) == std::future_status::timeout) {
      fprintf(stderr, "a request waited for another thread's wait for the device\n");
      _Exit(1);
    }
  };
  const auto check = [&](const std::function<void()>& call) {
    ran = false;
    on_wait = other_goes_on;
    call();
    CHECK(ran && !on_wait);
  };
  pool_context(0, 1);
  pool_free(get(50));
  void *a = get(500), *b = get(600), *c = get(5000);
  check([&] { pool_free(a); });        // kept
  check([&] { pool_free(b, true); });  // kept, a goes back
  CHECK(blocks.count(a) == 0 && blocks.count(b) == 1);
  check([&] { pool_free(c); });        // too large to be kept
  CHECK(blocks.count(c) == 0);
  c = get(7250);
  check([&] { pool_free(get(640)); });  // the kept blocks go back and the request succeeds
  CHECK(blocks.count(b) == 0 && hipGetLastError() == hipSuccess);
  pool_free(c);
  check([&] { pool_context(0, -1); });
  CHECK(used <= 50);  // what the other thread may have kept before the context was gone
}

// Without host memory a returned block goes to the driver (it comes from
// destructors: an exception there ends the process), and so does a new one that
// cannot be entered: the request fails as one for device memory.
static void host_memory() {
  pool_context(0, 1);
  void *a = get(500), *b = get(600);
  no_memory = true;
  pool_free(a);
  no_memory = false;
  CHECK(blocks.count(a) == 0 && used == 600);
  void *c = get(500), *d = get(500);
  pool_free(c);
  no_memory = true;
  pool_free(d, true);  // where an older block would have to go back for it
  no_memory = false;
  CHECK(blocks.count(d) == 0 && blocks.count(c) == 1);
  fail_after_malloc = true;
  void* e = nullptr;
  const hipError_t rc = pool_alloc(&e, 450 + 300);
  no_memory = fail_after_malloc = false;
  CHECK(rc == hipErrorOutOfMemory && used == 1100);
  CHECK(get(500) == c);
  pool_free(b);
  pool_free(c);
}

// The wrapper: a buffer that cannot be had is an error of the library, and
// what it held before has gone back.
static void buffer() {
  pool_context(0, 1);
  DevBuf<uint64_t> x;
  x.alloc(100);
  const void* p = x.p;
  x.alloc(90);
  CHECK(x.p == p && x.bytes() == 800);
  try {
    x.alloc(2000);
    CHECK(false);
  } catch (const Error& e) {
    CHECK(e.code == G5_ERR_MEM);
  }
  CHECK(!x.p && x.n == 0 && hipGetLastError() == hipSuccess && blocks.empty());
}

int main(int argc, char** argv) {
  const struct {
    const char* name;
    void (*f)();
  } checks[] = {{"sizes", sizes}, {"bound", bound}, {"refill", refill}, {"contexts", contexts}, {"buffer", buffer},
                {"threads", threads}, {"host_memory", host_memory}};
  for (const auto& c : checks)
    if (argc > 1 && !strcmp(argv[1], c.name)) {
      c.f();
      return 0;
    }
  return 2;
}
