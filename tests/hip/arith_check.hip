// arith_check.hip -- the FP64 quotients and roots of afd_device.hpp, element by element (tests only).
#include <hip/hip_runtime.h>

#include "afd_device.hpp"

using namespace afd;

// op 0: a / b, 1: sqrt(a), 2: 1 / sqrt(a)
__global__ __launch_bounds__(256) void k_arith(int op, unsigned n, const double *a, const double *b, double *out) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    out[i] = op == 0 ? fdiv(a[i], b[i]) : (op == 1 ? fsqrt(a[i]) : finvsqrt(a[i]));
}

// Host arrays of n values each (1 <= n <= 2^24; b is read for op 0 only).  Returns 0, or a HIP error code.
extern "C" int arith_check(int op, int n, const double *a, const double *b, double *out) {
    if (op < 0 || op > 2 || n < 1 || n > (1 << 24) || !a || !out || (op == 0 && !b)) return -1;
    const size_t bytes = (size_t)n * 8;
    double *d = nullptr;
    hipError_t e = hipMalloc(&d, 3 * bytes);
    if (e != hipSuccess) return (int)e;
    e = hipMemcpy(d, a, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d + n, op == 0 ? b : a, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_arith, dim3(((unsigned)n + 255) / 256), dim3(256), 0, 0, op, (unsigned)n, d, d + n,
                           d + 2 * (size_t)n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, d + 2 * (size_t)n, bytes, hipMemcpyDeviceToHost);
    (void)hipFree(d);
    return (int)e;
}
