// Calls from two host threads that share a stream and a workspace, on a stand-in for the HIP runtime that only writes down
// who launches what: the launches of one call that meet in the workspace follow one another, with no other launch that uses
// it in between.  (The executable's own definitions of the runtime's functions come before the runtime's.)
#include "stand_in_runtime.hpp"

#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

#include "../../include/bfaintb_gemm.h"

static std::mutex g_mutex;
static std::condition_variable g_cond;
static std::vector<int> g_order;        // the thread of every launch
static thread_local int t_thread = 0;   // 0: launches of the main thread pass unseen

extern "C" {
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t)
{
    if (t_thread == 0) return hipSuccess;
    std::unique_lock<std::mutex> lock(g_mutex);
    g_order.push_back(t_thread);
    const size_t seen = g_order.size();
    g_cond.notify_all();
    // every launch leaves the other thread the time to put one of its own behind it
    g_cond.wait_for(lock, std::chrono::milliseconds(100), [&] { return g_order.size() > seen && g_order.back() != t_thread; });
    return hipSuccess;
}
}

static void* const kDev = reinterpret_cast<void*>(0x10000);        // never dereferenced
static void* const kWorkspace = reinterpret_cast<void*>(0x200000);
static const size_t kBytes = 64u << 20;

static int tiles(uint32_t m, uint32_t n, uint32_t k)
{
    return bfaintb_gemm_ex(kDev, kDev, kDev, kDev, m, n, k, k, n, n, 8, 0, kWorkspace, kBytes, nullptr, BFAINTB_VARIANT_PREFILL_128, 0);
}
static int packed_tiles() { return bfaintb_gemm_prepacked_ex(kDev, kDev, kDev, kDev, nullptr, 96, 4096, 11008, 11008, 4096, 8, 0, kWorkspace, kBytes, nullptr, BFAINTB_VARIANT_PREFILL_128); }
static int decode() { return bfaintb_gemm_ex(kDev, kDev, kDev, kDev, 1, 4096, 4096, 4096, 4096, 4096, 8, 0, kWorkspace, kBytes, nullptr, BFAINTB_VARIANT_DECODE, 0); }
static int init() { return bfaintb_workspace_init(kWorkspace, kBytes, nullptr); }
static int on_scratch() { return bfaintb_gemm_static(kDev, kDev, kDev, kDev, 96, 4096, 11008, 11008, 4096, 4096, 8, 0, nullptr); }
static int reset_scratch() { return bfaintb_static_scratch_reset(nullptr); }

struct Call {
    const char* name;
    size_t launches;
    std::function<int()> run;
};

// `calls` calls on each of two threads: every call's launches are adjacent.
static int check(const Call& first, const Call& second)
{
    g_order.clear();
    int rc[2] = {0, 0};
    const Call* what[2] = {&first, &second};
    std::vector<std::thread> threads;
    for (int i = 0; i < 2; ++i)
        threads.emplace_back([&, i] {
            t_thread = i + 1;
            for (int rep = 0; rep < 2; ++rep) rc[i] |= what[i]->run();
        });
    for (auto& t : threads) t.join();
    bool ok = rc[0] == 0 && rc[1] == 0 && g_order.size() == 2 * (first.launches + second.launches);
    for (size_t at = 0; ok && at < g_order.size();) {
        const size_t launches = what[g_order[at] - 1]->launches;
        for (size_t i = 0; i < launches; ++i) ok = ok && at + i < g_order.size() && g_order[at + i] == g_order[at];
        at += launches;
    }
    printf("%s | %s: return codes %d %d, launches by thread:", first.name, second.name, rc[0], rc[1]);
    for (int t : g_order) printf(" %d", t);
    printf("%s\n", ok ? "" : "   <-- a launch between those of one call");
    return ok ? 0 : 1;
}

int main()
{
    bfaintb_plan plan{};
    if (bfaintb_gemm_plan(96, 4096, 11008, 8, 0, 0, BFAINTB_VARIANT_PREFILL_128, 0, &plan) != 0 || plan.launches != 2 || bfaintb_init(nullptr) != 0) {
        printf("the shape this test is about is one launch\n");
        return 1;
    }
    const Call wide{"tiles 96 x 4096 x 11008", 2, [] { return tiles(96, 4096, 11008); }}, small{"tiles 64 x 1024 x 14336", 2, [] { return tiles(64, 1024, 14336); }};
    const Call packed{"packed tiles 96 x 4096 x 11008", 2, packed_tiles}, one{"decode 1 x 4096 x 4096", 1, decode}, fill{"workspace_init", 2, init};
    const Call fixed{"static 96 x 4096 x 11008", 2, on_scratch}, reset{"static_scratch_reset", 2, reset_scratch};
    int bad = check(wide, small) + check(wide, one) + check(packed, wide) + check(packed, one) + check(wide, fill) + check(fixed, fixed) + check(fixed, reset);
    printf("%s\n", bad ? "FAILED" : "all checks passed");
    return bad ? 1 : 0;
}
