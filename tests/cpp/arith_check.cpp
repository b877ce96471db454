// Device check of the renderer's short exact forms (swegl_amd/csrc/core.h)
// against the compiler's IEEE '/' and sqrtf: rcp_rn and sqrt_rn for every
// float from 2^-96 to 2^96, div_rn for every 4,099th significand of a against
// every 4,093rd of b and the ends of both, at exponents across its range.
// Prints the counts; exits 1 on any mismatch, 2 without a device.
#include <cstdio>

#include "../../swegl_amd/csrc/core.h"

__global__ void unary(uint32_t lo, uint32_t n, unsigned long long *bad)
{
    unsigned long long r = 0, s = 0;
    for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += gridDim.x * 256ull) {
        const float x = __uint_as_float(lo + (uint32_t)i);
        r += sw::rcp_rn(x) != 1.0f / x;
        r += sw::rcp_rn(-x) != -1.0f / x;
        s += sw::sqrt_rn(x) != sqrtf(x);
    }
    if (r)
        atomicAdd(&bad[0], r);
    if (s)
        atomicAdd(&bad[1], s);
}

__device__ uint32_t significand(uint32_t k, uint32_t step, uint32_t count)
{
    return k < 8 ? k : k < 16 ? 0x7FFFFFu - (k - 8) : k + 16 <= count ? (k - 15) * step % 0x800000u : 0u;
}
__global__ void quotients(uint32_t count, unsigned long long *bad)
{
    const uint32_t j = blockIdx.x * 256u + threadIdx.x;
    if (j >= count)
        return;
    unsigned long long d = 0;
    const int eb[] = {-47, -20, 0, 21, 46}, ea[] = {-90, -26, 0, 40, 70};
    for (int p = 0; p < 5; p++) {
        const float b = __uint_as_float((uint32_t)(127 + eb[p]) << 23 | significand(j, 4093, count));
        const float r = sw::rcp_rn(b);
        for (uint32_t i = 0; i < count; i++) {
            const float a = __uint_as_float((uint32_t)(127 + ea[(i + p) % 5]) << 23 | significand(i, 4099, count));
            const float q = a / b;
            if (q >= 0x1p-120f && q <= 0x1p120f)
                d += (sw::div_rn(a, b, r) != q) + (sw::div_rn(-a, b, r) != -q);
        }
        d += __float_as_uint(sw::div_rn(0.0f, b, r)) != 0u;
    }
    if (d)
        atomicAdd(&bad[2], d);
}

__global__ void means(unsigned long long *bad)
{
    const uint32_t c = blockIdx.x + 1;
    const float rc = __builtin_amdgcn_rcpf((float)c);
    unsigned long long d = 0;
    for (uint32_t x = threadIdx.x; x <= 255u * c; x += 256u)
        d += sw::tap_mean(x, rc) != x / c;
    if (d)
        atomicAdd(&bad[3], d);
}

int main()
{
    unsigned long long *bad = nullptr, h[4] = {1, 1, 1, 1};
    if (hipMalloc((void **)&bad, sizeof h) != hipSuccess || hipMemset(bad, 0, sizeof h) != hipSuccess) {
        std::printf("no device\n");
        return 2;
    }
    const uint32_t lo = (127u - 96u) << 23, n = 192u << 23, count = 2048;
    for (uint32_t part = 0; part < 4; part++)
        unary<<<4096, 256>>>(lo + part * (n / 4), n / 4 + (part == 3), bad);
    quotients<<<count / 256, 256>>>(count, bad);
    means<<<1024, 256>>>(bad);
    if (hipMemcpy(h, bad, sizeof h, hipMemcpyDeviceToHost) != hipSuccess) {
        std::printf("device error\n");
        return 2;
    }
    std::printf("mismatches: reciprocal %llu, square root %llu, quotient %llu, mean %llu\n", h[0], h[1], h[2],
                h[3]);
    return h[0] || h[1] || h[2] || h[3] ? 1 : 0;
}
