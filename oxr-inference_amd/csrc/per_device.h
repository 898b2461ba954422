// Settings that are made once per device (host code; plain C++).
#pragma once

#include <atomic>
#include <cstdint>

namespace oxr {

// Calls set() unless it has succeeded for `device` with this `done` before; returns its status (0: made).  A failed
// call is tried again by the next one, devices from 64 on are set every time.  Safe from several threads: set() may run
// more than once, which does no harm to a setting.
template <class Set>
int once_per_device(std::atomic<uint64_t>& done, int device, Set set) {
  const uint64_t bit = device >= 0 && device < 64 ? (uint64_t)1 << device : 0;
  if (done.load(std::memory_order_relaxed) & bit) return 0;
  const int status = set();
  if (status == 0) done.fetch_or(bit, std::memory_order_relaxed);
  return status;
}

}  // namespace oxr
