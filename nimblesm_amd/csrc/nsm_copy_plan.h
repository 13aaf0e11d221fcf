// nsm_copy_plan.h -- how a staged device-to-host copy is cut (internal).
#pragma once

#include <stddef.h>

namespace nsm {

constexpr size_t kStaged = (size_t)2 << 20;   // below, one hipMemcpy is as fast
constexpr size_t kShared = (size_t)16 << 20;  // from here on helper threads take chunks too
constexpr size_t kLarge  = (size_t)40 << 20;
constexpr int    kHelperSlots = 2, kMaxOwnSlots = 4, kMaxHelpers = 7;
constexpr int    kMaxSlots = kMaxOwnSlots + kMaxHelpers * kHelperSlots;

// The caller's pinned slots and two for each helper, of a chunk each.  New
// pinned memory costs its first touch by the host 370 us per MB, so small
// copies use few and small slots (1 MB; with 4 MB the first read of a process
// took 0.8 to 1.8 ms longer than hipMemcpy's), copies in between 5.5 MB, and
// only from kLarge on, where hipMemcpy takes 4 ms and more, 18 MB.  First read
// of a process, hipMemcpy / these: 2.2 MB 0.56 / 0.65 ms, 6.6 MB 1.02 / 1.29,
// 15 MB 1.79 / 1.86, 18 MB 2.03 / 1.66, 32 MB 3.49 / 2.03, 51.5 MB 5.1 / 2.9;
// the first one after another model's end, 18 MB 1.17 / 0.77, 32 MB 2.13 /
// 1.56.  Three slots of 256 KB make the first read 0.1 ms shorter and eight
// results of 2.8 MB that the caller keeps 1.57 ms instead of 1.41 (hipMemcpy
// 1.68).
struct CopyPlan {
  size_t chunk;
  int    own, helpers;

  constexpr int    slots() const { return own + helpers * kHelperSlots; }
  constexpr size_t pinned() const { return (size_t)slots() * chunk; }
};

constexpr CopyPlan copy_plan(size_t bytes)
{
  if (bytes < kShared) return {(size_t)512 << 10, 2, 0};
  if (bytes < kLarge) return {(size_t)512 << 10, 3, 4};
  return {(size_t)1 << 20, kMaxOwnSlots, kMaxHelpers};
}

}  // namespace nsm
