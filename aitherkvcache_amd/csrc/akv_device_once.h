// What is said once on every device of a process, such as the dynamic LDS a kernel may use: a flag per process leaves the second
// device without it.  (Devices past 64 are told at every call, and a call that fails is made again.)
#pragma once
#include <stdint.h>

#include <atomic>

struct akv_device_once {
  std::atomic<uint64_t> told{0};
  template <class Tell>
  int operator()(int device, Tell&& tell) {
    const uint64_t bit = device >= 0 && device < 64 ? (uint64_t)1 << device : 0;
    if ((told.load(std::memory_order_acquire) & bit) != 0) return 0;
    const int rc = tell();
    if (rc == 0) told.fetch_or(bit, std::memory_order_release);
    return rc;
  }
};
