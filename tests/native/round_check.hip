// The functions of nse_round.hpp on arrays, for tests/test_gpu_nse_round.py.
#include <hip/hip_runtime.h>

#include "nse_round.hpp"

namespace {

// kind 0: sqrt_rn(a); 1: quot_rn(a, b, 1 / b); 2: quot_rn(a, b)
__global__ void k_float(int kind, long n, const float *a, const float *b, float *out) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    if (kind == 0) out[t] = saras::nse::sqrt_rn(a[t]);
    else if (kind == 1) out[t] = saras::nse::quot_rn(a[t], b[t], 1.0f / b[t]);
    else out[t] = saras::nse::quot_rn(a[t], b[t]);
}
__global__ void k_by6(long n, const double *a, double *out) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) out[t] = saras::nse::by6(a[t]);
}

// `bytes` of `src` on the device
void *put(const void *src, size_t bytes) {
    void *p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) return nullptr;
    if (src && hipMemcpy(p, src, bytes, hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(p);
        return nullptr;
    }
    return p;
}

}  // namespace

// host arrays of n values (b may be null for kind 0); 0 on success
extern "C" int round_check_float(int kind, long n, const float *a, const float *b, float *out) {
    if (n <= 0 || kind < 0 || kind > 2 || !a || !out || (kind > 0 && !b)) return 1;
    const size_t bytes = (size_t)n * sizeof(float);
    float *da = (float *)put(a, bytes), *db = (float *)put(b ? b : a, bytes), *d = (float *)put(nullptr, bytes);
    int rc = 1;
    if (da && db && d) {
        hipLaunchKernelGGL(k_float, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, kind, n, da, db, d);
        rc = hipGetLastError() != hipSuccess || hipMemcpy(out, d, bytes, hipMemcpyDeviceToHost) != hipSuccess;
    }
    (void)hipFree(da);
    (void)hipFree(db);
    (void)hipFree(d);
    return rc;
}

extern "C" int round_check_by6(long n, const double *a, double *out) {
    if (n <= 0 || !a || !out) return 1;
    const size_t bytes = (size_t)n * sizeof(double);
    double *da = (double *)put(a, bytes), *d = (double *)put(nullptr, bytes);
    int rc = 1;
    if (da && d) {
        hipLaunchKernelGGL(k_by6, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, 0, n, da, d);
        rc = hipGetLastError() != hipSuccess || hipMemcpy(out, d, bytes, hipMemcpyDeviceToHost) != hipSuccess;
    }
    (void)hipFree(da);
    (void)hipFree(d);
    return rc;
}
