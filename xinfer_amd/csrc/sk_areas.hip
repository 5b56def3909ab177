// The prefill GEMM's partial tiles: one group of 64 MiB areas (room for two
// partial tiles of 128 x 256 per CU), a code object of its own.
//
// Compiled once per group (XHIP_SK_GROUP, build.py): groups of 1, 1, 2, 4, 8
// and 16 areas, an area for each of 32 streams.  The code object loader places
// a group when its address is first asked for, so a program holds the areas of
// at most twice the streams that have needed one, and one that only decodes
// holds none; nothing is allocated through the HIP allocator, so the call that
// asks may be under capture.

#include "sk_areas.h"

#define XHIP_SK_CAT2(a, b) a##b
#define XHIP_SK_CAT(a, b) XHIP_SK_CAT2(a, b)
#define XHIP_SK_ARRAY XHIP_SK_CAT(g_sk_areas_, XHIP_SK_GROUP)

namespace xhip {
__device__ __align__(256) float XHIP_SK_ARRAY[sk_group_areas(XHIP_SK_GROUP)][kSkAreaFloats];
}

namespace xhip_host {

// The device address of the group on the current device, or null.
template <>
float* sk_group_base<XHIP_SK_GROUP>() {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(xhip::XHIP_SK_ARRAY)) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return reinterpret_cast<float*>(p);
}

}  // namespace xhip_host
