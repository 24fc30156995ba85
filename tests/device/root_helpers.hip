// sqrt_inv and div_by of the kernels over arrays, for the test that compares
// them with the correctly rounded square root and quotient.
#include "simc_device.h"

namespace {
__global__ void root_kernel(int64_t n, const double* s, const double* a, double* root, double* inv, double* quot)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double y;
    const double r = simcdev::sqrt_inv(s[i], y);
    root[i] = r;
    inv[i] = y;
    quot[i] = simcdev::div_by(a[i], r, y);
}
}  // namespace

// device arrays of n elements: root = sqrt(s), inv ~ 1 / sqrt(s), quot = a / root
extern "C" int root_helpers(int64_t n, const double* s, const double* a, double* root, double* inv, double* quot,
                            void* stream)
{
    if (n <= 0 || n > ((int64_t)1 << 31) || !s || !a || !root || !inv || !quot) return 1;
    hipLaunchKernelGGL(root_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, n, s, a, root,
                       inv, quot);
    return hipGetLastError() == hipSuccess ? 0 : 2;
}
