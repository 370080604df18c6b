// sigmoid_check.hip -- TEST INFRASTRUCTURE (built into libsigmoidcheck.so by
// __graft_entry__.build(); loaded only by tests/test_gpu_sigmoid.py).
//
// Exhaustive check that the product's sigmoid (et::sigmoid in
// peer-review-agents_amd/csrc/et_common.hpp: reciprocal, Newton step and residual
// correction) equals the specified one for every one of the 2^32 binary32
// inputs.  The specification is written here on its own, with the language's
// division (correctly rounded, HIP's default) and the special cases branched on:
//     NaN: the input; l >= 0: 1 / (1 + exp(-l)); l < 0: exp(l) / (1 + exp(l));
//     exp(x) for x <= 0: 0 below -87, else the degree-7 polynomial of the reduced
//     argument times 2^n through the exponent field.
#include "../../peer-review-agents_amd/csrc/et_common.hpp"

namespace {

__device__ float rule_exp(float x)
{
    if (x < -87.0f) return 0.0f;
    const float n = __builtin_rintf(x * __uint_as_float(0x3FB8AA3Bu));
    const float hi = __builtin_fmaf(-n, __uint_as_float(0x3F317200u), x);
    const float r = __builtin_fmaf(-n, __uint_as_float(0x35BFBE8Eu), hi);
    const float c[8] = {1.0f / 5040.0f, 1.0f / 720.0f, 1.0f / 120.0f, 1.0f / 24.0f, 1.0f / 6.0f, 0.5f, 1.0f, 1.0f};
    float p = c[0];
    for (int i = 1; i < 8; ++i) p = __builtin_fmaf(p, r, c[i]);
    return p * __uint_as_float((uint32_t)((int)n + 127) << 23);
}

__device__ float rule_sigmoid(float l)
{
    if (l != l) return l;
    if (l >= 0.0f) return 1.0f / (1.0f + rule_exp(-l));
    const float z = rule_exp(l);
    return z / (1.0f + z);
}

__global__ __launch_bounds__(256) void sigmoid_check_kernel(uint64_t base, unsigned long long* mismatches,
                                                            unsigned int* first_bad)
{
    const uint32_t u = (uint32_t)(base + (uint64_t)blockIdx.x * 256 + threadIdx.x);
    const float l = __uint_as_float(u);
    if (__float_as_uint(et::sigmoid(l)) != __float_as_uint(rule_sigmoid(l))) {
        atomicAdd(mismatches, 1ull);
        atomicMin(first_bad, u);
    }
}

}  // namespace

// Runs the check over all 2^32 inputs on the current device and stream 0.
// Returns 0 and fills *mismatches and *first_bad (the lowest differing input,
// 0xffffffff if none); a negative value on a HIP error.
extern "C" int sigmoid_check(unsigned long long* mismatches, unsigned int* first_bad)
{
    struct Result {
        unsigned long long mismatches;
        unsigned int first_bad;
    } h = {0, 0xffffffffu}, *d = nullptr;
    if (hipMalloc(&d, sizeof(h)) != hipSuccess) return -1;
    int rc = hipMemcpy(d, &h, sizeof(h), hipMemcpyHostToDevice) == hipSuccess ? 0 : -2;
    const uint64_t per_launch = uint64_t(1) << 30;
    for (uint64_t base = 0; rc == 0 && base < (uint64_t(1) << 32); base += per_launch) {
        sigmoid_check_kernel<<<dim3((unsigned)(per_launch / 256)), dim3(256)>>>(base, &d->mismatches, &d->first_bad);
        if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) rc = -3;
    }
    if (rc == 0 && hipMemcpy(&h, d, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) rc = -4;
    (void)hipFree(d);
    *mismatches = h.mismatches;
    *first_bad = h.first_bad;
    return rc;
}
