// Zero fill of device memory (kernels_misc.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace pcfd {

// n 4-byte words of zeros from p, by a kernel on `stream`: ordered with the
// work that follows there.  (hipMemset runs on the null stream, which the
// library's non-blocking streams do not wait for.)
void launch_zero(hipStream_t stream, void* p, size_t n);

}  // namespace pcfd
