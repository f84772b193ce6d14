// recip_test.hip -- the device reciprocal of recon_common.hpp (v_rcp_f32 and
// one Newton step) against the division, over every float32 significand at
// binary exponents across the range the kernels accept, and over whole
// numbers.  Prints the number of values that differ where the residual is
// within kRecipBad (0 expected), and how many of the out-of-range values
// (denormal or with a denormal reciprocal) were not reported by it.
#include "recon_common.hpp"

#include <cstdio>

#pragma clang fp contract(off)

namespace {

__global__ __launch_bounds__(256) void check_kernel(unsigned* wrong) {
    const unsigned i = blockIdx.x * 256u + threadIdx.x;  // significand
    for (unsigned e = 1; e < 254; e += 7) {
        const float x = __uint_as_float((e << 23) | i);
        for (int s = 0; s < 2; ++s) {
            const float v = s ? -x : x;
            float bad = 0.0f, sum = 0.0f;
            const float y = recon::recip(v, bad), z = recon::recip_sum(v, sum);
            const float t = 1.0f / v;
            if (bad <= recon::kRecipBad && __float_as_uint(y) != __float_as_uint(t)) atomicAdd(wrong, 1u);
            if (sum <= recon::kRecipBad && __float_as_uint(z) != __float_as_uint(t)) atomicAdd(wrong, 1u);
        }
    }
    if (i < (1u << 20)) {
        const float v = (float)(i + 1);
        float bad = 0.0f;
        if (__float_as_uint(recon::recip(v, bad)) != __float_as_uint(1.0f / v) || bad > recon::kRecipBad)
            atomicAdd(wrong + 1, 1u);
    }
    // denormal x: the estimate is infinite, the residual must say so
    if (i) {
        float bad = 0.0f;
        const float x = __uint_as_float(i);
        const float y = recon::recip(x, bad);
        if (bad <= recon::kRecipBad && __float_as_uint(y) != __float_as_uint(1.0f / x)) atomicAdd(wrong + 2, 1u);
    }
}

}  // namespace

int main() {
    unsigned* d = nullptr;
    unsigned h[3] = {0, 0, 0};
    if (hipMalloc((void**)&d, sizeof(h)) != hipSuccess) return 1;
    if (hipMemcpy(d, h, sizeof(h), hipMemcpyHostToDevice) != hipSuccess) return 1;
    hipLaunchKernelGGL(check_kernel, dim3((1u << 23) / 256), dim3(256), 0, nullptr, d);
    if (hipGetLastError() != hipSuccess) return 1;
    if (hipMemcpy(h, d, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return 1;
    std::printf("significands %u whole %u denormal %u\n", h[0], h[1], h[2]);
    return (h[0] || h[1] || h[2]) ? 1 : 0;
}
