// Prints the host's time for a known call (m n k weight_bits packed, one per line), in ns, on a stand-in for the HIP runtime: the least of several runs.
#include "stand_in_runtime.hpp"

#include <chrono>
#include <cstdio>

#include "../../include/bfaintb_gemm.h"

extern "C" hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }

int main()
{
    void* const p = reinterpret_cast<void*>(0x10000);  // never dereferenced
    unsigned m, n, k;
    int bits, packed;
    while (scanf("%u %u %u %d %d", &m, &n, &k, &bits, &packed) == 5) {
        double least = 1e30;
        for (int run = 0; run < 15; ++run) {
            const auto from = std::chrono::steady_clock::now();
            for (int i = 0; i < 2000; ++i) {
                const int rc = packed ? bfaintb_gemm_prepacked(p, p, p, p, nullptr, m, n, k, k, n, bits, 0, nullptr, 0, nullptr)
                                      : bfaintb_gemm(p, p, p, p, m, n, k, k, n, n, bits, 0, nullptr, 0, nullptr);
                if (rc != 0) return 1;
            }
            const double ns = std::chrono::duration<double, std::nano>(std::chrono::steady_clock::now() - from).count() / 2000;
            if (ns < least) least = ns;
        }
        printf("%.0f\n", least);
    }
    return 0;
}
