// host_memory.h -- what kind of memory a caller's buffer is, from what the
// runtime says of it.  No HIP call here: the look-up is a parameter, so that the
// rule can be run without a GPU.
#pragma once
#include <cstddef>
#include <cstdint>

namespace afid {

enum class HostKind {
  ordinary,   // memory that the runtime does not know
  pinned,     // wholly inside one pinned host allocation
  other       // anything else (managed or device memory, part of it unknown): the runtime's own copy
};

// One allocation as the runtime reports it.
struct Allocation {
  bool host = false;                     // pinned host memory
  uintptr_t base = 0;                    // its first byte, as the host sees it
  size_t size = 0;
  uintptr_t device = 0;                  // the device address of `base`
};

// lookup(address, Allocation *) -> whether the runtime knows the address.  A
// buffer is pinned only if it ends inside the allocation that it begins in: two
// pinned allocations may have unmapped memory between them.  `device` receives
// the device address of p then.
template <typename Lookup>
HostKind host_kind(const void *p, size_t bytes, Lookup &&lookup, uintptr_t *device) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  Allocation lo, hi;
  const bool klo = lookup(a, &lo), khi = lookup(a + bytes - 1, &hi);
  if (!klo && !khi) return HostKind::ordinary;
  if (!klo || !lo.host || !lo.device || a < lo.base || a - lo.base >= lo.size || bytes > lo.size - (a - lo.base))
    return HostKind::other;
  *device = lo.device + (a - lo.base);
  return HostKind::pinned;
}

}  // namespace afid
