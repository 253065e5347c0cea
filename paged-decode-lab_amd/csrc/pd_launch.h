// Host helpers of the launchers in the HIP sources.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "pd_internal.h"

namespace pd {

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
template <typename... Ts>
inline bool all_aligned16(Ts... p) { return (aligned16(p) && ...); }

// The status of the launch just made.
inline int launch_status(const char* what) {
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess)
    return fail(PD_ELAUNCH, "%s launch failed: %s", what, hipGetErrorString(err));
  return PD_OK;
}

inline hipStream_t as_stream(pd_stream_t s) { return reinterpret_cast<hipStream_t>(s); }
inline const uint16_t* u16(const void* p) { return static_cast<const uint16_t*>(p); }
inline uint16_t* u16(void* p) { return static_cast<uint16_t*>(p); }

}  // namespace pd
