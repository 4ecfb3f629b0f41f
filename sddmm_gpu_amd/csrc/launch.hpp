// Kernel launches that return their own error: hipLaunchKernelGGL leaves it to be fetched by hipGetLastError, a call
// that costs 0.4 us next to 2.6 us for the launch itself -- on a small matrix the calls take as long as the kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>

namespace sddmm {

template <class... P>
inline hipError_t launch(void (*fn)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, std::type_identity_t<P>... args)
{
    void *p[] = {(void *)&args...};
    return hipLaunchKernel((const void *)fn, grid, block, p, lds, stream);
}

}  // namespace sddmm
