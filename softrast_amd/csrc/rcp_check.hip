// rcp_check.hip -- stand-alone check of sr_device.h's RCPPS and RSQRTPS on the
// device: every cell of leading mantissa bits at every exponent and sign, with
// the lowest, a middle and the highest value of the cell, and the special
// values, against the recorded tables. Prints the number of differing results
// and exits with 0 when there is none.
#include <cstdio>

#include "sr_device.h"

using namespace srg;

__device__ const uint32_t c_rcp[2048] = {
#include "rcpps_table.inc"
};
__device__ const uint32_t c_rsqrt[4096] = {
#include "rsqrtps_table.inc"
};

__device__ uint32_t want_rcp(uint32_t u)
{
    const uint32_t sign = u & 0x80000000u, e = (u >> 23) & 255u;
    if (e == 255u) return (u & 0x7FFFFFu) ? (u | 0x00400000u) : sign;
    if (e == 0u) return sign | 0x7F800000u;
    const uint32_t t = c_rcp[(u >> 12) & 2047u];
    const int ne = (int)((t >> 23) & 255u) - ((int)e - 127);
    return ne <= 0 ? sign : (sign | ((uint32_t)ne << 23) | (t & 0x7FFFFFu));
}

__device__ uint32_t want_rsqrt(uint32_t u)
{
    const uint32_t e = (u >> 23) & 255u;
    if (e == 255u && (u & 0x7FFFFFu)) return u | 0x00400000u;
    if (e == 0u) return (u & 0x80000000u) | 0x7F800000u;
    if (u & 0x80000000u) return 0xFFC00000u;
    if (e == 255u) return 0u;
    const int ub = (int)e - 127, p = ub & 1;
    const uint32_t t = c_rsqrt[(uint32_t)p * 2048u + ((u >> 12) & 2047u)];
    return ((uint32_t)((int)((t >> 23) & 255u) - (ub - p) / 2) << 23) | (t & 0x7FFFFFu);
}

// grid (8, 512): 2,048 cells x sign and exponent
__global__ void k_check(uint32_t* bad)
{
    const uint32_t cell = ((blockIdx.y & 511u) << 23) | ((blockIdx.x * 256u + threadIdx.x) << 12);
    const uint32_t low[3] = { 0u, 0x5A3u, 0xFFFu };
    for (int k = 0; k < 3; ++k) {
        const uint32_t u = cell | low[k], e = (u >> 23) & 255u;
        const float x = ffrom(u);
        uint32_t n = (fbits(rcpps(x)) != want_rcp(u)) + (fbits(rsqrtps(x)) != want_rsqrt(u));
        if (!(u >> 31) && e >= 1u && e <= 251u) n += fbits(rcpps_pos(x)) != want_rcp(u);
        if (!(u >> 31) && e >= 1u && e <= 254u) n += fbits(rsqrtps_pos(x)) != want_rsqrt(u);
        if (n) atomicAdd(bad, n);
    }
}

int main()
{
    uint32_t *bad = nullptr, n = 0;
    if (hipMalloc((void**)&bad, 4) != hipSuccess || hipMemcpy(bad, &n, 4, hipMemcpyHostToDevice) != hipSuccess) return 2;
    hipLaunchKernelGGL(k_check, dim3(8, 512), dim3(256), 0, 0, bad);
    if (hipGetLastError() != hipSuccess || hipMemcpy(&n, bad, 4, hipMemcpyDeviceToHost) != hipSuccess) return 2;
    std::printf("differing results: %u\n", n);
    return n ? 1 : 0;
}
