// Partial-tile areas of the prefill GEMM (sk_areas.hip, owned in scratch.hip).
#pragma once

#include <mutex>

#include "common.h"

namespace xhip {
constexpr size_t kSkAreaFloats = (size_t)1 << 24;  // 64 MiB
constexpr int kSkGroups = 6;
constexpr int sk_group_areas(int group) { return group < 2 ? 1 : 1 << (group - 1); }
constexpr int kSkAreas = 1 << (kSkGroups - 1);  // of all groups
}  // namespace xhip

namespace xhip_host {

// A stream's area.  A call that leaves partial tiles is two launches, and the
// second reads what the first wrote: `enqueue` is held from before the first
// until after the second is enqueued (the host does not wait for either), so
// that a call of another host thread on the same stream cannot put its own
// between them.
struct SkArea {
    float* part;  // kSkAreaFloats floats; null: the stream has no area
    std::mutex* enqueue;
};
SkArea sk_area(hipStream_t st);  // scratch.hip

template <int GROUP>
float* sk_group_base();
// clang-format off
template <> float* sk_group_base<0>();
template <> float* sk_group_base<1>();
template <> float* sk_group_base<2>();
template <> float* sk_group_base<3>();
template <> float* sk_group_base<4>();
template <> float* sk_group_base<5>();
// clang-format on
}
