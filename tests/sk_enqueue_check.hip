// Host-only check that the two launches of a prefill GEMM call with partial
// tiles (xinfer_amd/csrc/gemm_sk_int4.hip) are neighbours on their stream when
// several host threads call on it: the second launch adds up what the first
// left in the stream's area.  Launches are recorded instead of made.  Built and
// run by tests/test_plan_invariants.py.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdio>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

struct Launch {
    std::thread::id by;
    bool sum;
    const void* part;
};
static std::mutex g_log_mu;
static std::map<hipStream_t, std::vector<Launch>> g_log;
template <typename P>
static void record(dim3 block, hipStream_t st, const P& p) {
    {
        std::lock_guard<std::mutex> lock(g_log_mu);
        g_log[st].push_back({std::this_thread::get_id(), block.x == 256, p.part});
    }
    std::this_thread::sleep_for(std::chrono::microseconds(200));  // another thread's chance to come between
}
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(k, grid, block, lds, st, p) record(block, st, p)
#define hipFuncSetAttribute(k, a, v) hipSuccess
#define hipGetDevice(p) (*(p) = 0, hipSuccess)
#define hipGetSymbolAddress(p, s) (*(p) = (void*)0x1000, hipSuccess)
#include "../xinfer_amd/csrc/scratch.hip"
#include "../xinfer_amd/csrc/gemm_sk_int4.hip"
namespace xhip_host {
int num_cus() { return 256; }
int launch_status() { return 0; }
int gemm_ws_linear(hipStream_t, void*, const void*, const uint8_t*, const uint16_t*, const float*, int64_t, int64_t,
                   int64_t, bool, int*) { return 1; }
template <> float* sk_group_base<0>() { return (float*)0x10000000; }
template <> float* sk_group_base<1>() { return (float*)0x20000000; }
template <> float* sk_group_base<2>() { return (float*)0x30000000; }
template <> float* sk_group_base<3>() { return (float*)0x50000000; }
template <> float* sk_group_base<4>() { return (float*)0x90000000; }
template <> float* sk_group_base<5>() { return (float*)0x190000000; }
}

int main() {
    const hipStream_t streams[2] = {nullptr, reinterpret_cast<hipStream_t>((uintptr_t)0x10000)};
    std::vector<std::thread> threads;
    for (int t = 0; t < 6; ++t)
        threads.emplace_back([&, t] {
            const xinfer_fused_desc d = {(void*)0x100, (const uint8_t*)0x100, (const void*)0x100, nullptr, 5120};
            for (int i = 0; i < 20; ++i)
                xhip_host::prefill_gemm(streams[t % 2], &d, 1, nullptr, nullptr, (const void*)0x100, false, 17 + 100 * t,
                                        17408, false);
        });
    for (auto& t : threads) t.join();
    int bad = 0, pairs = 0;
    for (auto& [st, log] : g_log)
        for (size_t i = 0; i < log.size(); i += 2, ++pairs)
            if (i + 1 == log.size() || log[i].sum || !log[i + 1].sum || log[i].by != log[i + 1].by ||
                log[i].part != log[i + 1].part || !log[i].part)
                ++bad;
    printf("pairs %d, parted %d\n", pairs, bad);
    return bad || pairs != 120 ? 1 : 0;
}
