// Reads of pinned host memory, which the host writes anew between launches.
#pragma once
#include "common.h"

namespace {

// At system scope, past the scalar cache and what other caches may hold of an earlier
// use: pinned memory is fine-grained unless it was asked for otherwise (bindings.cpp
// looks, and copies what is not), so that such a load has what the host wrote before
// the launch.  (A fence that drops the caches'
// lines as well was 2 us a workgroup, one after another: 23 rows 45 us, now 4.)
template <class T>
DEV_INLINE T host_read(const T* from) {
  return __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace
