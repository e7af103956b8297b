// Counts where the kernels' short forms of a reciprocal root and of a division
// by a constant differ from the compiler's own, over every argument they take.
#include <hip/hip_runtime.h>

#include "hip/dev_shading.h"

using namespace mrt;

// All 2^32 floats: 4096 blocks of 256 lanes take 4096 each.
__global__ __launch_bounds__(256) void kCountRsq(unsigned long long* differ) {
    const uint32_t lane = blockIdx.x * 256u + threadIdx.x;
    uint32_t n = 0;
    for (uint32_t k = 0; k < 4096u; k++) {
        const float x = __uint_as_float((k << 20) | lane);
        n += __float_as_uint(rsq(x)) != __float_as_uint(1.0f / sqrtf(x));
    }
    if (n) atomicAdd(differ, (unsigned long long)n);
}

// Whole numbers of 16 bits: 256 blocks of 256 lanes take one each.
template <int N>
__global__ __launch_bounds__(256) void kCountDiv(unsigned long long* differ) {
    const float v = (float)((int)(blockIdx.x * 256u + threadIdx.x) - 32768), n = (float)N;
    if (__float_as_uint(divConst<N>(v)) != __float_as_uint(v / n)) atomicAdd(differ, 1ull);
}

// which: 0 = rsq, else divConst<which>. Returns the number of differing arguments, or -1.
extern "C" long long device_math_differences(int which) {
    unsigned long long *dev = nullptr, count = 0;
    if (hipMalloc(&dev, sizeof(count)) != hipSuccess) return -1;
    bool ok = hipMemcpy(dev, &count, sizeof(count), hipMemcpyHostToDevice) == hipSuccess;
    if (which == 0)
        hipLaunchKernelGGL(kCountRsq, dim3(4096), dim3(256), 0, 0, dev);
    else if (which == 32767)
        hipLaunchKernelGGL(kCountDiv<32767>, dim3(256), dim3(256), 0, 0, dev);
    else if (which == 16383)
        hipLaunchKernelGGL(kCountDiv<16383>, dim3(256), dim3(256), 0, 0, dev);
    else
        ok = false;
    ok = hipGetLastError() == hipSuccess && ok;
    ok = hipMemcpy(&count, dev, sizeof(count), hipMemcpyDeviceToHost) == hipSuccess && ok;
    (void)hipFree(dev);
    return ok ? (long long)count : -1;
}
