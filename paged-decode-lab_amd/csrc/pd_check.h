// The check of a packed prefill's metadata, which only the device holds, made by
// the first workgroups of a kernel that is launched anyway: the K/V write ahead
// of the attention, where there is one, so that its verdict is there when the
// host has prepared the attention's launch; else the attention.
//
// Each wavefront of theirs writes kChecked and the bits it found to its word of
// pinned memory, which the host polls while that kernel and the next ones run.
// Measured on MI355X, a call of 5 rows: 15 us unchecked, 20 checked by the
// attention, 27 with a kernel and an event of the check's own, which also cost
// the stream 3 to 5 us a call, 22 with a kernel and the poll.  A layer's call of 3
// rows, with its write: 23.5 us unchecked, 27.5 to 28.6 checked by the write (1 us
// of it the wait), 30.8 by the attention.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "paged_decode.h"

namespace pdk {

struct PackedCheck {
  const int32_t *cu_q, *cu_k, *table;
  int64_t total_q, total_k, num_pages, tsb;
  int num_seqs, table_width, page_size;
  int32_t* verdicts;  // or null: no check
};

constexpr int kChecked = 4, kCheckGroups = PD_CHECK_WORDS / 4;  // of 256 threads

// Args: PackedCheck, or a kernel's own arguments of these names.
template <bool kPaged, typename Args>
__device__ __forceinline__ void check_packed(const Args& a, int tid) {
  const int width = kPaged ? a.table_width : 1;
  const int64_t total = int64_t(a.num_seqs) * width;
  const int step = min(int(gridDim.x), kCheckGroups) * 256;
  bool odd = false, outside = false;
  for (int64_t at = blockIdx.x * 256 + tid; at < total; at += step) {
    const int64_t i = at / width;
    const int entry = int(at - i * width);
    const int64_t k0 = a.cu_k[i], k1 = a.cu_k[i + 1], nk = k1 - k0;
    if (entry == 0) {
      const int64_t q0 = a.cu_q[i], q1 = a.cu_q[i + 1];
      odd |= q0 < 0 || q1 < q0 || q1 > a.total_q || nk < 0 || (nk == 0 && q1 > q0);
      if (kPaged)
        outside |= nk > int64_t(width) * a.page_size;
      else
        odd |= k0 < 0 || k1 > a.total_k;
    }
    if (kPaged && int64_t(entry) * a.page_size < nk) {
      const int64_t page = a.table[i * a.tsb + entry];
      odd |= page < 0;
      outside |= page >= a.num_pages || page < -a.num_pages;
    }
  }
  const int found =
      kChecked | (__any(odd) ? PD_CHECK_ODD : 0) | (__any(outside) ? PD_CHECK_OUTSIDE : 0);
  if ((tid & 63) == 0)
    __hip_atomic_store(a.verdicts + 4 * blockIdx.x + (tid >> 6), found, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

// Whether this workgroup has a share of the check.
__device__ __forceinline__ bool has_share(const int32_t* verdicts) {
  return verdicts && blockIdx.x < kCheckGroups && blockIdx.y == 0;
}

// Before the launch: the words of workgroups that the grid does not have.
inline void mark_absent(int32_t* verdicts, int64_t grid_x) {
  if (verdicts)
    for (int64_t word = 4 * grid_x; word < PD_CHECK_WORDS; ++word) verdicts[word] = kChecked;
}

}  // namespace pdk
