// Makes the calls it reads (m n k weight_bits kind workspace_bytes, one per line; kind 0: bfaintb_gemm, 1: bfaintb_gemm_prepacked,
// 2: bfaintb_gemm_static under capture, 3: bfaintb_gemm_reference, 4: as 0 and 5: as 1, under capture; 0 bytes: no workspace) on a stand-in for the HIP runtime and prints what each returned,
// how many kernels it launched and the workgroups of the first.
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
    int bits, kind;
    size_t bytes;
    while (scanf("%u %u %u %d %d %zu", &m, &n, &k, &bits, &kind, &bytes) == 6) {
        void* const ws = bytes ? p : nullptr;
        g_launches = 0;
        g_workgroups = 0;
        g_capturing = kind == 2 || kind > 3;
        if (kind > 3) kind -= 4;
        const int rc = kind == 3   ? bfaintb_gemm_reference(p, p, p, static_cast<float*>(p), m, n, k, k, n, n, ws, bytes, nullptr)
                       : kind == 2   ? bfaintb_gemm_static(p, p, p, p, m, n, k, k, n, n, bits, 0, nullptr)
                       : kind == 1 ? bfaintb_gemm_prepacked(p, p, p, p, nullptr, m, n, k, k, n, bits, 0, ws, bytes, nullptr)
                                   : bfaintb_gemm(p, p, p, p, m, n, k, k, n, n, bits, 0, ws, bytes, nullptr);
        printf("%d %d %u\n", rc, g_launches, g_workgroups);
    }
    return 0;
}
