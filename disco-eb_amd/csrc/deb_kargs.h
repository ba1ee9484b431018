// The parameter block read where the launch put it.
#pragma once

#include "deb_device.h"

namespace deb {

// The kernel-argument segment's first argument, a Params<NS>.  Reading it
// through this pointer rather than through the by-value argument matters
// because its arrays are indexed per lane and pointed into: the compiler then
// copied the whole block into every lane's private memory, and each value
// loaded back from there counted as different from lane to lane (branches on
// launch constants by execution mask, loads by vector registers).
template <int NS>
__device__ __forceinline__ const Params<NS> &kernel_params() {
  return *(const Params<NS> *)__builtin_amdgcn_kernarg_segment_ptr();
}

}  // namespace deb
