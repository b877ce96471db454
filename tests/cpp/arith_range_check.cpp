// Device check of the short exact division (swegl_amd/csrc/core.h) down to
// the smallest numerators it is used with, against the compiler's IEEE '/':
// div_rn for numerators from 2^-102 and quotients from 2^-62 (the lights'
// second quotient, scaled by 2^64), then that quotient scaled back under the
// lights' own guard for highlights s from the smallest denormal to 2^10.
// Also runs arith_check's comparisons again, each launch checked.
// Prints the counts; exits 1 on any mismatch or comparison not made, 2
// without a device.
#define main arith_check_main
#include "arith_check.cpp"
#undef main

// every `step`-th significand, from the smallest, and the largest
__device__ float number(uint32_t i, uint32_t count, int exponent)
{
    const uint32_t m = i + 1 < count ? i * (0x800000u / (count - 1)) : 0x7FFFFFu;
    return __uint_as_float((uint32_t)(127 + exponent) << 23 | m);
}

// n: comparisons made, mismatches
__global__ void small_quotients(uint32_t count, unsigned long long *n)
{
    const uint32_t j = blockIdx.x * 256u + threadIdx.x;
    if (j >= count)
        return;
    unsigned long long made = 0, bad = 0;
    const int eb[] = {-40, -39, -20, 0, 21, 39};
    for (int k = 0; k < 6; k++) {
        const float b = number(j, count, eb[k]), r = sw::rcp_rn(b);
        for (int ea = -102; ea <= -102 + 64; ea += 4)
            for (uint32_t i = 0; i < count; i += 7) {
                const float a = number(i, count, ea), q = a / b;
                made++;
                bad += q >= 0x1p-62f && q <= 0x1p120f && sw::div_rn(a, b, r) != q;
            }
    }
    atomicAdd(&n[0], made);
    if (bad)
        atomicAdd(&n[1], bad);
}

__global__ void highlights(uint32_t count, unsigned long long *n)
{
    const uint32_t j = blockIdx.x * 256u + threadIdx.x;
    if (j >= count)
        return;
    unsigned long long made = 0, bad = 0;
    for (int e = -40; e < 40; e += 5) {
        const float d2 = number(j, count, e), r2 = sw::rcp_rn(d2);
        // 0 and every 2^17 or so of the floats up to 2^10
        for (uint32_t w = 0; w <= (127u + 10) << 23; w += 131071u + j) {
            const float s = __uint_as_float(w), q = sw::div_rn(s * 0x1p64f, d2, r2);
            made++;
            if (q >= 0x1p-62f || s == 0.0f)
                bad += __float_as_uint(q * 0x1p-64f) != __float_as_uint(s / d2);
        }
    }
    atomicAdd(&n[0], made);
    if (bad)
        atomicAdd(&n[1], bad);
}

static bool ran(const char *what)
{
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = hipDeviceSynchronize();
    if (e != hipSuccess)
        std::printf("%s: %s\n", what, hipGetErrorString(e));
    return e == hipSuccess;
}

int main()
{
    int devices = 0;
    if (hipGetDeviceCount(&devices) != hipSuccess || devices == 0) {
        std::printf("no device\n");
        return 2;
    }
    unsigned long long *n = nullptr, h[8] = {};
    if (hipMalloc((void **)&n, sizeof h) != hipSuccess ||
        hipMemcpy(n, h, sizeof h, hipMemcpyHostToDevice) != hipSuccess)
        return 2;
    const uint32_t lo = (127u - 96u) << 23, all = 192u << 23, count = 2048;
    bool ok = true;
    for (uint32_t part = 0; ok && part < 4; part++) {
        unary<<<4096, 256>>>(lo + part * (all / 4), all / 4 + (part == 3), n + 4);
        ok = ran("unary");
    }
    if (ok) {
        quotients<<<count / 256, 256>>>(count, n + 4);
        ok = ran("quotients");
    }
    if (ok) {
        means<<<1024, 256>>>(n + 4);
        ok = ran("means");
    }
    if (ok) {
        small_quotients<<<count / 256, 256>>>(count, n);
        ok = ran("small quotients");
    }
    if (ok) {
        highlights<<<count / 256, 256>>>(count, n + 2);
        ok = ran("highlights");
    }
    if (!ok || hipMemcpy(h, n, sizeof h, hipMemcpyDeviceToHost) != hipSuccess)
        return 1;
    unsigned long long want[2] = {count * 6ull * 17 * ((count + 6) / 7), 0};
    for (uint32_t j = 0; j < count; j++)
        want[1] += 16ull * (((127u + 10) << 23) / (131071u + j) + 1);
    std::printf("small quotients: %llu of %llu compared, %llu differ\nhighlights: %llu of %llu compared, %llu differ\n"
                "mismatches: reciprocal %llu, square root %llu, quotient %llu, mean %llu\n",
                h[0], want[0], h[1], h[2], want[1], h[3], h[4], h[5], h[6], h[7]);
    return h[0] != want[0] || h[2] != want[1] || h[1] || h[3] || h[4] || h[5] || h[6] || h[7];
}
