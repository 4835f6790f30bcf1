// device_math.hip -- gam_math.h and gam_erfc.h evaluated on the device for
// tests/test_gpu_device_math.py: y (and e) of n values x, host arrays.
#include <hip/hip_runtime.h>
#include "gam_erfc.h"

__global__ void k_eval(int fn, int n, const double *x, double *y, double *e)
{
    const int q = (int)(blockIdx.x * 256 + threadIdx.x);
    if (q >= n) return;
    double a = 0.0, b = 0.0;
    if (fn == 0) a = gam_rcp(x[q]);
    else if (fn == 1) gam_sqrt_rsqrt(x[q], a, b);
    else if (fn == 2) a = gam_sqrt(x[q]);
    else if (fn == 3) a = gam_exp_neg(x[q]);
    else a = gam_erfc_exp(x[q], b);
    y[q] = a;
    e[q] = b;
}

extern "C" int dev_math(int fn, int n, const double *x, double *y, double *e)
{
    double *d = nullptr;
    const size_t b = (size_t)n * sizeof(double);
    if (n < 1 || hipMalloc((void **)&d, 3 * b) != hipSuccess) return 1;
    hipError_t err = hipMemcpy(d, x, b, hipMemcpyHostToDevice);
    if (err == hipSuccess) {
        k_eval<<<dim3((unsigned)((n + 255) / 256)), dim3(256)>>>(fn, n, d, d + n, d + 2 * (size_t)n);
        err = hipGetLastError();
    }
    if (err == hipSuccess) err = hipMemcpy(y, d + n, b, hipMemcpyDeviceToHost);
    if (err == hipSuccess) err = hipMemcpy(e, d + 2 * (size_t)n, b, hipMemcpyDeviceToHost);
    hipFree(d);
    return err != hipSuccess;
}
