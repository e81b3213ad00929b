// Makes the calls it reads (m n k weight_bits, one per line) by bfaintb_gemm_prepacked without scratch, as a device's first calls, under capture, on a
// stand-in for the HIP runtime, and prints what each returned, how many kernels it launched and the workgroups of the first.
#include "stand_in_runtime.hpp"

#include <cstdio>

#include "../../include/bfaintb_gemm.h"

static int g_launches = 0;
static unsigned g_workgroups = 0;

extern "C" hipError_t hipLaunchKernel(const void*, dim3 grid, dim3, void**, size_t, hipStream_t)
{
    if (g_launches++ == 0) g_workgroups = grid.x * grid.y * grid.z;
    return hipSuccess;
}

int main()
{
    void* const p = reinterpret_cast<void*>(0x10000);  // never dereferenced
    unsigned m, n, k;
    int bits;
    while (scanf("%u %u %u %d", &m, &n, &k, &bits) == 4) {
        g_launches = 0;
        g_workgroups = 0;
        g_capturing = true;
        const int rc = bfaintb_gemm_prepacked(p, p, p, p, nullptr, m, n, k, k, n, bits, 0, nullptr, 0, nullptr);
        printf("%d %d %u\n", rc, g_launches, g_workgroups);
    }
    return 0;
}
