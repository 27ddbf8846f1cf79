// The short reciprocal and square root of csrc/vsdmo_numerics.h against the
// correctly rounded division and square root: every mantissa of a range of
// exponents.  out[0]: values whose bits differ, out[1]: values compared.
#include <hip/hip_runtime.h>

#include "vsdmo_numerics.h"

using namespace vsdmo;

// biased exponents [e0, e1), 2^23 mantissas each
template <bool SQRT>
__global__ __launch_bounds__(256) void k_compare(unsigned e0, unsigned e1, unsigned long long* out)
{
    const unsigned long long n = (unsigned long long)(e1 - e0) << 23, step = (unsigned long long)gridDim.x * 256;
    unsigned long long bad = 0, all = 0;
    for (unsigned long long i = (unsigned long long)blockIdx.x * 256 + threadIdx.x; i < n; i += step) {
        const float x = bitsf((unsigned)(i + ((unsigned long long)e0 << 23)));
        const float got = SQRT ? sqrt_rn(x) : recip_rn(x), want = SQRT ? sqrtf(x) : 1.0f / x;
        bad += fbits(got) != fbits(want);
        ++all;
    }
    if (bad) atomicAdd(out, bad);
    atomicAdd(out + 1, all);
}

extern "C" int rounding_compare(int root, unsigned e0, unsigned e1, unsigned long long* out)
{
    if (!out || e0 < 1 || e1 > 255 || e0 >= e1) return -1;
    unsigned long long* d = nullptr;
    const unsigned long long zero[2] = { 0, 0 };
    hipError_t e = hipMalloc(&d, sizeof(zero));
    if (e != hipSuccess) return (int)e;
    e = hipMemcpy(d, zero, sizeof(zero), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        if (root) k_compare<true><<<2048, 256>>>(e0, e1, d);
        else k_compare<false><<<2048, 256>>>(e0, e1, d);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, d, sizeof(zero), hipMemcpyDeviceToHost);
    (void)hipFree(d);
    return (int)e;
}
