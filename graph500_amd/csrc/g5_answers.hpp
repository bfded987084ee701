// g5_answers.hpp -- answers on their way to the host.
//
// A kernel that makes an answer stores it straight into host memory where the
// GPU can: the caller's buffer if it is pinned, else, for small answers, a
// pinned buffer of the context that the host copies from.  Making the values
// and moving them then overlap, and a small answer costs one launch and one
// wait instead of a launch, a copy command and the wait.  Other buffers are
// filled by a copy from device memory.
#pragma once

#include "g5_ctx.hpp"
#include "g5_prims.hpp"

#include <cstring>

namespace g5 {

// Where a kernel writes an answer of `bytes` for host memory `host`.
struct HostOut {
  // Up to here the host's copy out of the pinned buffer (about 10 GB/s) costs
  // less than the copy command it replaces (15-20 us with its kernel).
  static constexpr size_t kStageBytes = size_t(256) << 10;
  void* p = nullptr;  // the kernel's output, 16-byte aligned
  // dev is used only for answers the GPU does not store to the host itself:
  // those for memory it cannot address, and those of more than `direct` bytes
  template <class T>
  HostOut(T* host, size_t count, HostStage& stage, DevBuf<T>& dev, hipStream_t s, size_t direct = SIZE_MAX)
      : host_(host), bytes_(count * sizeof(T)), s_(s) {
    if (bytes_ <= direct && pinned(host, bytes_)) {
      p = host;
    } else if (bytes_ <= kStageBytes) {
      p = stage.get(kStageBytes);
      staged_ = true;
    } else {
      dev.alloc(count);
      p = dev.p;
      copied_ = true;
    }
  }
  // after the kernel's launch: the answer is in the caller's buffer on return
  void finish() {
    if (copied_) G5_HIP(hipMemcpyAsync(host_, p, bytes_, hipMemcpyDeviceToHost, s_));
    G5_HIP(hipStreamSynchronize(s_));
    if (staged_) std::memcpy(host_, p, bytes_);
  }

 private:
  // one allocation of host memory that the GPU addresses by the same pointer
  static bool pinned(const void* q, size_t bytes) {
    hipPointerAttribute_t at{};
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if ((uintptr_t)q % 16 || !bytes) return false;
    if (hipPointerGetAttributes(&at, q) != hipSuccess || at.type != hipMemoryTypeHost || at.devicePointer != q ||
        hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)q) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    return (const char*)base <= (const char*)q && (const char*)q + bytes <= (const char*)base + size;
  }
  void* host_;
  size_t bytes_;
  hipStream_t s_;
  bool staged_ = false, copied_ = false;
};

// Levels by original id from levels by row: 16 consecutive ids per thread,
// so that 16 lookups are in flight and a wave stores 1 KiB at a time.  Large
// answers are bound by the link to the host (S28: 5.2 ms for 268 MB).
void launch_make_levels(const uint32_t* old2new, const uint8_t* row_level, int64_t n, int64_t rows, int64_t root,
                        uint8_t* out, hipStream_t s);

}  // namespace g5
