// Makes the calls it reads (m n k weight_bits packed workspace_bytes, one per line; 0 bytes: no workspace) on a stand-in for the
// HIP runtime and prints what each returned and how many kernels it launched.
#include "stand_in_runtime.hpp"

#include <cstdio>

#include "../../include/bfaintb_gemm.h"

static int g_launches = 0;

extern "C" hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t)
{
    ++g_launches;
    return hipSuccess;
}

int main()
{
    void* const p = reinterpret_cast<void*>(0x10000);  // never dereferenced
    unsigned m, n, k;
    int bits, packed;
    size_t bytes;
    while (scanf("%u %u %u %d %d %zu", &m, &n, &k, &bits, &packed, &bytes) == 6) {
        void* const ws = bytes ? p : nullptr;
        g_launches = 0;
        const int rc = packed ? bfaintb_gemm_prepacked(p, p, p, p, nullptr, m, n, k, k, n, bits, 0, ws, bytes, nullptr)
                              : bfaintb_gemm(p, p, p, p, m, n, k, k, n, n, bits, 0, ws, bytes, nullptr);
        printf("%d %d\n", rc, g_launches);
    }
    return 0;
}
