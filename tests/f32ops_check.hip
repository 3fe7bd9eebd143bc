// f32ops_check.hip -- TEST INFRASTRUCTURE ONLY: the all-f32 event loop's
// division and square root (3photons-rust_amd/csrc/tp_math.h) beside '/' and
// sqrtf() on the device, for tests/test_gpu_f32_range.py.
#include "tp_math.h"

__global__ void f32ops(const float *a, const float *b, int64_t n, float *out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    out[i] = tpm::div_f(a[i], b[i]);
    out[n + i] = a[i] / b[i];
    out[2 * n + i] = tpm::sqrt_f(a[i]);
    out[3 * n + i] = sqrtf(a[i]);
}

// out: 4 n values, device pointers all.
extern "C" int f32ops_run(const float *a, const float *b, int64_t n, float *out)
{
    hipLaunchKernelGGL(f32ops, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, nullptr, a, b, n, out);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? (int)hipDeviceSynchronize() : (int)e;
}
