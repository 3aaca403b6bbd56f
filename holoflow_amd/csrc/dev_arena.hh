// Device allocations of one owner, released together.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/hfx.h"

namespace hfx {

void set_last_error(const std::string &msg);

// Small tables share blocks of kBlock bytes: a plan has a dozen of them.
struct DevArena {
  static constexpr size_t kBlock = 128 << 10, kSmall = 32 << 10;
  std::vector<void *> ptrs;
  size_t bytes = 0;  // device memory held: whole blocks, whatever is used of them
  char *block = nullptr;
  size_t used = 0;

  DevArena() = default;
  DevArena(const DevArena &) = delete;
  DevArena &operator=(const DevArena &) = delete;
  ~DevArena() {
    for (void *p : ptrs) (void)hipFree(p);
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
    ptrs.push_back(v);
    bytes += held;
    if (small) {
      block = static_cast<char *>(v);
      used = padded;
    }
    *p = static_cast<T *>(v);
    return HFX_OK;
  }
};

// Makes a plan by create(d); where the device has no room for the windows per launch that the library
// would choose (batch_windows 0), for one.
template <typename F> hfx_status create_or_one_window(const hfx_plan_desc &d, F create) {
  const hfx_status rc = create(d);
  if (rc != HFX_E_NOMEM || d.batch_windows != 0) return rc;
  hfx_plan_desc one = d;
  one.batch_windows = 1;
  return create(one);
}

}  // namespace hfx
