// Reads questions (m n k weight_bits group_size packed variant ldb, one per line; ldb 0: n) and prints, of each, what bfaintb_gemm_plan says (variant,
// kernel, tile rows and columns, waves, splits, workgroups, workgroups of further launches, launches) and what the call then launches on a
// stand-in for the HIP runtime (return code, launches, waves and workgroups of the first, workgroups of the others).
#include "stand_in_runtime.hpp"

#include <cstdio>
#include <cstdlib>

#include "../../include/bfaintb_gemm.h"

static unsigned g_launches = 0, g_waves = 0, g_workgroups = 0, g_others = 0;

extern "C" hipError_t hipLaunchKernel(const void*, dim3 grid, dim3 block, void**, size_t, hipStream_t)
{
    const unsigned workgroups = grid.x * grid.y * grid.z;
    if (g_launches++ == 0) g_waves = block.x / 64u, g_workgroups = workgroups;
    else g_others += workgroups;
    return hipSuccess;
}

int main()
{
    void* const p = reinterpret_cast<void*>(0x10000);  // never dereferenced
    unsigned m, n, k, group, ldb;
    int bits, packed, variant;
    while (scanf("%u %u %u %d %u %d %d %u", &m, &n, &k, &bits, &group, &packed, &variant, &ldb) == 8) {
        bfaintb_plan t;
        if (bfaintb_gemm_plan(m, n, k, bits, group, packed, variant, 0, &t) != 0) return 1;
        g_launches = g_waves = g_workgroups = g_others = 0;
        const int rc = packed ? bfaintb_gemm_prepacked_ex(p, p, p, p, nullptr, m, n, k, k, n, bits, group, p, t.workspace_bytes, nullptr, variant)
                              : bfaintb_gemm_ex(p, p, p, p, m, n, k, k, ldb ? ldb : n, n, bits, group, p, t.workspace_bytes, nullptr, variant, 0);
        printf("%d %u %u %u %u %u %u %u %u %d %u %u %u %u\n", t.variant, t.kernel, t.tile_rows, t.tile_cols, t.waves, t.splits, t.workgroups, t.tail_workgroups,
               t.launches, rc, g_launches, g_waves, g_workgroups, g_others);
    }
    return 0;
}
