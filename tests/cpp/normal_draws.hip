// The device forms of the Box-Muller functions against the general division and square root and the quadrant
// taken from the product, over every 24-bit argument a draw can have.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "../../dynamic-occupancy-grid-map_amd/csrc/dogm_numerics.h"

using namespace dogm_num;

constexpr unsigned COUNT = 1u << 24;

__global__ void k_compare(unsigned* differ)
{
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= COUNT)
        return;
    // The logarithm's quotient, at the significand of every uniform and, beyond them, of every float.
    const float m = f32_from_bits(0x3f800000u | (i & 0x7fffffu)) * (i >> 23 ? 0.5f : 1.0f);
    if (m > 0.70710677f && m <= 1.41421354f && f32_bits(log_quotient(m - 1.0f, m + 1.0f)) != f32_bits((m - 1.0f) / (m + 1.0f)))
        atomicAdd(&differ[0], 1u);
    // The radius of every first word.
    const float x = -2.0f * log_f32(uniform01_oc(i << 8));
    if (f32_bits(box_muller_sqrt(x)) != f32_bits(sqrtf(x)))
        atomicAdd(&differ[1], 1u);
    // The angle of every second word.
    const uint32_t a = 0x12345678u, b = (i << 8) | 0xffu;
    const float r = sqrtf(-2.0f * log_f32(uniform01_oc(a)));
    float s, c, z0, z1;
    sincos_2pi_f32(uniform01(b), &s, &c);
    box_muller(a, b, &z0, &z1);
    if (f32_bits(z0) != f32_bits(r * c) || f32_bits(z1) != f32_bits(r * s))
        atomicAdd(&differ[2], 1u);
}

int main()
{
    unsigned host[3] = {0u, 0u, 0u};
    unsigned* differ = nullptr;
    if (hipMalloc(reinterpret_cast<void**>(&differ), sizeof(host)) != hipSuccess)
        return 2;
    if (hipMemcpy(differ, host, sizeof(host), hipMemcpyHostToDevice) != hipSuccess)
        return 2;
    hipLaunchKernelGGL(k_compare, dim3(COUNT / 256), dim3(256), 0, nullptr, differ);
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess)
        return 2;
    if (hipMemcpy(host, differ, sizeof(host), hipMemcpyDeviceToHost) != hipSuccess)
        return 2;
    std::printf("differ: quotient %u root %u normals %u\n", host[0], host[1], host[2]);
    return host[0] || host[1] || host[2] ? 1 : 0;
}
