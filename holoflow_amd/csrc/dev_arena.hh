// Device allocations of one owner, released together.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <utility>
#include <vector>

#include "../../include/hfx.h"

namespace hfx {

void set_last_error(const std::string &msg);

// Small tables share blocks of kBlock bytes: a plan has a dozen of them.
struct DevArena {
  static constexpr size_t kBlock = 128 << 10, kSmall = 32 << 10;
  std::vector<std::pair<void *, size_t>> ptrs;  // with their sizes
  size_t bytes = 0;  // device memory held: whole blocks, whatever is used of them
  char *block = nullptr;
  size_t used = 0;

  DevArena() = default;
  DevArena(const DevArena &) = delete;
  DevArena &operator=(const DevArena &) = delete;
  ~DevArena() {
    release_to(0);
  }

  template <typename T> hfx_status alloc(T **p, size_t count) {
    const size_t want = count * sizeof(T), b = want ? want : 16;
    const bool small = b <= kSmall;
    const size_t padded = (b + 255) & ~(size_t)255;
    if (small && block && used + padded <= kBlock) {
      *p = reinterpret_cast<T *>(block + used);
      used += padded;
      return HFX_OK;
    }
    const size_t held = small ? kBlock : b;
    void *v = nullptr;
    if (hipMalloc(&v, held) != hipSuccess) {
      (void)hipGetLastError();  // reported here; not to be found again by the next launch's check
      set_last_error("hipMalloc of " + std::to_string(held) + " bytes failed");
      return HFX_E_NOMEM;
    }
    ptrs.emplace_back(v, held);
    bytes += held;
    if (small) {
      block = static_cast<char *>(v);
      used = padded;
    }
    *p = static_cast<T *>(v);
    return HFX_OK;
  }

  // Gives back all but the first n allocations.
  void release_to(size_t n) {
    for (; ptrs.size() > n; ptrs.pop_back()) {
      if (ptrs.back().first == block) block = nullptr;
      bytes -= ptrs.back().second;
      (void)hipFree(ptrs.back().first);
    }
  }
};

// Runs alloc(n) (allocations from `a`); where the device has no room for them, gives back what it got
// and runs alloc(1), with n = 1 from then on.
template <typename F> hfx_status alloc_or_one(DevArena &a, int &n, F alloc) {
  const size_t mark = a.ptrs.size();
  hfx_status rc = alloc(n);
  if (rc == HFX_E_NOMEM && n > 1) {
    a.release_to(mark);
    n = 1;
    rc = alloc(n);
  }
  return rc;
}

}  // namespace hfx
