// gx_slots.hpp -- values that are their own flags, exchanged by the workgroups
// of a launch whose workgroups are all resident.
//
// A value is written and read by relaxed device-scope atomics of 64 bits, at
// the level that all XCDs share; a slot holds kSlotEmpty (a NaN that
// arithmetic does not produce) until its owner has published, and a reader
// repeats its load while it sees that.
#pragma once

#include <hip/hip_runtime.h>

namespace gx {
namespace {

typedef unsigned long long Slot;
constexpr Slot kSlotEmpty = 0xfff8dead5a5a0001ull;
constexpr Slot kSlotNan = 0x7ff8000000000000ull;

__device__ __forceinline__ void put_slot(Slot* p, Slot v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void put_slot(Slot* p, double v) {
  put_slot(p, v == v ? (Slot)__double_as_longlong(v) : kSlotNan);
}
__device__ __forceinline__ Slot get_slot(const Slot* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// `seen` was read from p.  All workgroups are resident and take the same
// decisions, so every one publishes for every meeting and every wait ends.
__device__ __forceinline__ Slot await_bits(const Slot* p, Slot seen) {
  while (seen == kSlotEmpty) {
    __builtin_amdgcn_s_sleep(1);
    seen = get_slot(p);
  }
  return seen;
}
__device__ __forceinline__ double await_slot(const Slot* p, Slot seen) {
  return __longlong_as_double((long long)await_bits(p, seen));
}

}  // namespace
}  // namespace gx
