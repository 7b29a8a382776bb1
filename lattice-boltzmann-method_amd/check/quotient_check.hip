// Runs chem_device.h's device quotients on arrays, for tests/test_gpu_quotient.py.
#include "chem_device.h"

using namespace lbm::chem;

// q = a / b and y = 1 / b as the kernels form them
__global__ void k_quotients(const double* a, const double* b, double* q, double* y, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const Divisor d = divisor(b[i]);
    q[i] = quot(a[i], d);
    y[i] = d.y;
}

extern "C" int quotient_check(const double* a, const double* b, double* q, double* y, int64_t n)
{
    if (n <= 0 || n > (1 << 24)) return -1;
    double* dev = nullptr;
    const size_t bytes = sizeof(double) * (size_t)n;
    hipError_t e = hipMalloc((void**)&dev, 4 * bytes);
    if (e == hipSuccess) e = hipMemcpy(dev, a, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dev + n, b, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_quotients, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, dev, dev + n, dev + 2 * n,
                           dev + 3 * n, n);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(q, dev + 2 * n, bytes, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(y, dev + 3 * n, bytes, hipMemcpyDeviceToHost);
    if (dev) (void)hipFree(dev);
    return (int)e;
}
