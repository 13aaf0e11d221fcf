// nsm_copy_plan.h -- how a staged device-to-host copy is cut (internal).
#pragma once

#include <stddef.h>

namespace nsm {

constexpr size_t kStaged = (size_t)2 << 20;   // below, one hipMemcpy is as fast
constexpr size_t kShared = (size_t)16 << 20;  // from here on helper threads take chunks too
constexpr size_t kLarge  = (size_t)32 << 20;  // the allocator's mmap threshold: fresh memory every time
constexpr int    kHelperSlots = 2, kMaxOwnSlots = 4, kMaxHelpers = 7;
constexpr int    kMaxSlots = kMaxOwnSlots + kMaxHelpers * kHelperSlots;

// The caller's pinned slots and two for each helper, of a chunk each.  New
// pinned memory costs its first touch by the host 370 us per MB, so small
// copies use few and small slots (1 MB; with 4 MB the first read of a process
// took 0.8 to 1.8 ms longer than hipMemcpy's), copies in between 9 MB, and
// only from kLarge on, where every page of the destination faults, 18 MB.
// First read of a process, hipMemcpy / these: 2.2 MB 0.56 / 0.65 ms, 6.6 MB
// 1.02 / 1.29, 15 MB 1.79 / 1.86, 18 MB 2.05 / 2.21, 32 MB 3.13 / 2.64, 51.5 MB
// 5.1 / 2.9; the first one after another model's end, 18 MB 1.13 / 0.68, 32 MB
// 2.10 / 1.23 (18 MB of slots: 2.84 and 3.37).  Three slots of 256 KB make the
// first read 0.1 ms shorter and eight results of 2.8 MB that the caller keeps
// 1.57 ms instead of 1.41 (hipMemcpy 1.68); 21.9 MB take 0.97 ms through 11
// slots of 512 KB, 0.90 through 18 of 1 MB and 0.86 through these 9.
struct CopyPlan {
  size_t chunk;
  int    own, helpers;

  constexpr int    slots() const { return own + helpers * kHelperSlots; }
  constexpr size_t pinned() const { return (size_t)slots() * chunk; }
};

constexpr CopyPlan copy_plan(size_t bytes)
{
  if (bytes < kShared) return {(size_t)512 << 10, 2, 0};
  if (bytes < kLarge) return {(size_t)1 << 20, 3, 3};
  return {(size_t)1 << 20, kMaxOwnSlots, kMaxHelpers};
}

}  // namespace nsm
