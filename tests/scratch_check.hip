// Host-only check of who owns the scratch of xinfer_amd/csrc/scratch.hip: the
// split-K slots and the prefill GEMM's areas are owned apart, areas of
// different streams do not overlap, a group of areas is looked up (and thereby
// placed) only when one of its areas is first asked for, streams past the last
// area get none, a released area is handed out again, and the per-thread
// stream's handle means another stream on every host thread.  Built and run by
// tests/test_plan_invariants.py; the runtime's lookups are replaced below.
#include <hip/hip_runtime.h>
#define hipGetDevice(p) (*(p) = 0, hipSuccess)
#define hipGetSymbolAddress(p, s) (*(p) = (void*)0x1000, hipSuccess)
#include "../xinfer_amd/csrc/scratch.hip"
static int asked[xhip::kSkGroups];
static float* base(int g) {
    ++asked[g];
    return reinterpret_cast<float*>((uintptr_t)(g + 1) << 40);
}
namespace xhip_host {
template <> float* sk_group_base<0>() { return base(0); }
template <> float* sk_group_base<1>() { return base(1); }
template <> float* sk_group_base<2>() { return base(2); }
template <> float* sk_group_base<3>() { return base(3); }
template <> float* sk_group_base<4>() { return base(4); }
template <> float* sk_group_base<5>() { return base(5); }
}
#include <cstdio>
#include <set>
#include <thread>
using namespace xhip_host;
static int bad = 0;
#define CHECK(c) ((c) ? 0 : (printf("FAILED line %d: %s\n", __LINE__, #c), ++bad))
static hipStream_t stream(int i) { return reinterpret_cast<hipStream_t>((uintptr_t)(0x10000 + 64 * i)); }

int main() {
    float* part;
    size_t floats;
    uint32_t* cnt;
    int ncnt;
    for (int i = 100; i < 140; ++i)  // streams that only decode
        CHECK(splitk_slot(stream(i), &part, &floats, &cnt, &ncnt) == (i < 100 + xhip::kSplitSlots));
    for (int g = 0; g < xhip::kSkGroups; ++g) CHECK(asked[g] == 0);
    int areas = 0;
    for (int g = 0; g < xhip::kSkGroups; ++g) areas += xhip::sk_group_areas(g);
    CHECK(areas == xhip::kSkAreas);
    std::set<void*> seen;
    float* of[xhip::kSkAreas];
    for (int i = 0; i < xhip::kSkAreas; ++i) {
        const SkArea a = sk_area(stream(i));
        of[i] = a.part;
        CHECK(a.part && a.enqueue && seen.insert(a.part).second && seen.insert(a.enqueue).second);
        int placed = 0;
        for (int g = 0; g < xhip::kSkGroups; ++g) {
            CHECK(asked[g] <= 1);
            placed += asked[g] * xhip::sk_group_areas(g);
        }
        CHECK(placed > i && placed <= 2 * (i + 1));
        const int g = (int)((uintptr_t)of[i] >> 40) - 1;
        const size_t at = ((uintptr_t)of[i] & (((uintptr_t)1 << 40) - 1)) / 4;
        CHECK(at % xhip::kSkAreaFloats == 0 && (int)(at / xhip::kSkAreaFloats) < xhip::sk_group_areas(g));
    }
    for (int i = 0; i < xhip::kSkAreas; ++i) CHECK(sk_area(stream(i)).part == of[i]);
    CHECK(sk_area(stream(50)).part == nullptr);
    splitk_release(stream(7));
    CHECK(sk_area(stream(50)).part == of[7]);
    CHECK(sk_area(stream(7)).part == nullptr);
    for (int i = 0; i < xhip::kSkAreas; ++i) splitk_release(stream(i));
    for (int i = 100; i < 110; ++i) splitk_release(stream(i));
    const SkArea here = sk_area(hipStreamPerThread);
    float* part_here = nullptr;
    CHECK(splitk_slot(hipStreamPerThread, &part_here, &floats, &cnt, &ncnt));
    for (int t = 0; t < 2; ++t)
        std::thread([&] {
            float* part_there = nullptr;
            CHECK(splitk_slot(hipStreamPerThread, &part_there, &floats, &cnt, &ncnt) && part_there != part_here);
            const SkArea there = sk_area(hipStreamPerThread);
            CHECK(there.part && there.part != here.part && there.enqueue != here.enqueue);
            CHECK(sk_area(hipStreamPerThread).part == there.part);
            splitk_release(hipStreamPerThread);  // this thread's, not the other's
        }).join();
    CHECK(sk_area(hipStreamPerThread).part == here.part);
    CHECK(splitk_slot(hipStreamPerThread, &part, &floats, &cnt, &ncnt) && part == part_here);
    printf("bad %d\n", bad);
    return bad != 0;
}
