// qpso_rcp_check.hip -- the fast reciprocals of qpso_math.h against the division
// over all 2^32 inputs, on this device.  They rest on what its v_rcp_f32
// returns (one Newton step from an estimate alone need not round correctly), so
// the comparison belongs to the device and the compiler, not to the arithmetic.
// Prints one count a line; a wrong one is 0 where all is well.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "qpso_internal.h"
#include "qpso_math.h"

namespace {

enum { kNewton, kAny, kNormal, kDivision, kRejected, kAccepted, kCounts };
const char* const kNames[kCounts] = {
    "newton_wrong",      // accepted by its residual, not 1.0f / x
    "any_wrong",         // rcp_any is not 1.0f / x
    "normal_wrong",      // rcp_normal is not 1.0f / x for 1 <= x <= 2^31
    "division_wrong",    // 1.0f / x is not the rounded quotient (x and 1 / x normal)
    "normal_rejected",   // x and 1 / x normal, but the residual fails
    "other_accepted",    // not so, and the residual passes
};

__device__ bool same(float a, float b) { return __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b); }
__device__ bool normal(float x) { return __builtin_fabsf(x) >= 0x1p-126f && __builtin_fabsf(x) <= 0x1.fffffep127f; }

__global__ __launch_bounds__(256) void k_check(unsigned long long* counts) {
    unsigned long long c[kCounts] = {};
    for (unsigned long long i = blockIdx.x * 256ull + threadIdx.x; i < (1ull << 32); i += gridDim.x * 256ull) {
        const float x = __uint_as_float((unsigned)i);
        const float want = 1.0f / x;
        float e;
        const float r = qpso::rcp_newton(x, e);
        const bool ok = __builtin_fabsf(e) < qpso::kRcpOk, nn = normal(x) && normal(want);
        c[kNewton] += ok && !same(r, want);
        c[kAny] += !same(qpso::rcp_any(x), want);
        c[kNormal] += x >= 1.0f && x <= 0x1p31f && !same(qpso::rcp_normal(x), want);
        // the binary64 quotient rounded again is the rounded quotient (53 >= 2 24 + 2)
        c[kDivision] += nn && !same(want, (float)(1.0 / (double)x));
        c[kRejected] += nn && !ok;
        c[kAccepted] += !nn && ok;
    }
    for (int k = 0; k < kCounts; ++k)
        if (c[k]) atomicAdd(&counts[k], c[k]);
}

}  // namespace

int main() {
    unsigned long long *d = nullptr, h[kCounts] = {};
    if (hipMalloc(&d, sizeof(h)) != hipSuccess || hipMemcpy(d, h, sizeof(h), hipMemcpyHostToDevice) != hipSuccess) return 1;
    hipLaunchKernelGGL(k_check, dim3(8192), dim3(256), 0, 0, d);
    if (hipGetLastError() != hipSuccess || hipMemcpy(h, d, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return 1;
    for (int k = 0; k < kCounts; ++k) std::printf("%s %llu\n", kNames[k], h[k]);
    if (hipFree(d) != hipSuccess) return 1;
    return 0;
}
