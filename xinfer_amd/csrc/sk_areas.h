// Partial-tile areas of the prefill GEMM (sk_areas.hip, owned in scratch.hip).
#pragma once

#include "common.h"

namespace xhip {
constexpr size_t kSkAreaFloats = (size_t)1 << 24;  // 64 MiB
constexpr int kSkGroups = 6;
constexpr int sk_group_areas(int group) { return group < 2 ? 1 : 1 << (group - 1); }
constexpr int kSkAreas = 1 << (kSkGroups - 1);  // of all groups
}  // namespace xhip

namespace xhip_host {
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
