// Split-K workspace of the small-batch kernel without run-time allocation.
//
// The reference's projections allocate nothing per call: its split-K
// partials live in SLM (src/ops/linear.cpp:25-27) and every buffer a call
// touches is the caller's.  The small-batch MFMA kernel splits long K over
// several blocks, so its partial sums cross blocks and need device memory.
// That memory is a file-scope __device__ array here: the code object loader
// places it when the library's kernels are first loaded on a device, so no
// projection call runs hipMalloc, hipMemset or a device synchronisation, and
// the first call of a shape can be captured into a hipGraph.
//
// The array holds kSplitSlots independent slots (partials + arrival
// counters), 32 x (4 MiB + 16 KiB) = 128.5 MiB on every device the library
// runs on.  A slot belongs to one stream of a device until
// xinfer_stream_release gives it back: calls on one stream run in order, so
// they never share a slot concurrently, and calls on different streams use
// different slots.  (A call that uses a slot is one launch, so host threads
// that share a stream need no more than the stream's own order.)  Every counter
// is zero at load time and is returned to zero by the block that finishes its
// tile range, so a slot needs no clearing between calls.  When every slot of a device is taken (more live
// streams than slots) the caller plans without a cross-block split instead.
//
// The prefill GEMM's partial tiles have areas of their own (sk_areas.hip), 64
// MiB for each stream whose calls leave such tiles, for up to kSkAreas streams
// of a device, owned and given back as the slots are; with every area owned
// its calls run as whole tiles.  Such a call is two launches, which the area's
// lock keeps together where several host threads enqueue to one stream.

#include <atomic>

#include "sk_areas.h"

namespace xhip {
constexpr int kSplitSlots = 32;  // torch's stream pool alone hands out 32 streams per device
constexpr size_t kSplitPartialFloats = (size_t)1 << 20;  // 4 MiB of FP32 partials per slot
constexpr int kSplitCounters = 4096;                       // tile ranges per slot

__device__ __align__(256) float g_splitk_partials[kSplitSlots][kSplitPartialFloats];
__device__ __align__(256) uint32_t g_splitk_counters[kSplitSlots][kSplitCounters];
}  // namespace xhip

namespace xhip_host {

namespace {
constexpr int kMaxDev = 64;

// A stream by its handle, and hipStreamPerThread, one handle for a stream of
// every host thread, by its thread too (numbers are not used again, so a thread
// that ended without xinfer_stream_release keeps what it owned).
struct StreamKey {
    hipStream_t st = nullptr;
    uint64_t thread = 0;
    bool operator==(const StreamKey& o) const { return st == o.st && thread == o.thread; }
};

StreamKey stream_key(hipStream_t st) {
    if (st != hipStreamPerThread) return {st, 0};
    static std::atomic<uint64_t> threads{0};
    thread_local const uint64_t mine = ++threads;
    return {st, mine};
}

// Which streams own the N slots of one kind on a device.
template <int N>
struct Owners {
    int nused = 0;
    StreamKey owner[N] = {};
    bool released[N] = {};

    // The slot of `st`, now its own if it had none; -1 when other streams own
    // all of them.
    int take(const StreamKey& st) {
        int freed = -1;
        for (int i = 0; i < nused; ++i) {
            if (!released[i] && owner[i] == st) return i;
            if (released[i] && freed < 0) freed = i;
        }
        if (freed < 0 && nused == N) return -1;
        const int slot = freed >= 0 ? freed : nused++;
        owner[slot] = st;
        released[slot] = false;
        return slot;
    }
    void release(const StreamKey& st) {
        for (int i = 0; i < nused; ++i)
            if (owner[i] == st && !released[i]) {
                released[i] = true;
                owner[i] = {};
            }
    }
};

struct DevSlots {
    bool resolved = false;
    float* partials = nullptr;    // device address of g_splitk_partials on this device
    uint32_t* counters = nullptr; // device address of g_splitk_counters on this device
    Owners<xhip::kSplitSlots> slots;
    float* group[xhip::kSkGroups] = {};  // device addresses of the area groups placed so far
    Owners<xhip::kSkAreas> areas;
    std::mutex enqueue[xhip::kSkAreas];
};
std::mutex g_mu;
DevSlots g_devs[kMaxDev];

int current_device() {
    int dev = 0;
    return hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kMaxDev ? dev : -1;
}

typedef float* (*GroupBase)();
const GroupBase kGroupBase[xhip::kSkGroups] = {sk_group_base<0>, sk_group_base<1>, sk_group_base<2>,
                                               sk_group_base<3>, sk_group_base<4>, sk_group_base<5>};
}  // namespace

// The split-K slot of `st` on the current device: its partials (capacity in
// floats) and counters (count).  Returns false when the device's slots are
// all owned by other streams or the symbol lookup failed.
bool splitk_slot(hipStream_t st, float** partials, size_t* partial_floats, uint32_t** counters,
                 int* ncounters) {
    const int dev = current_device();
    if (dev < 0) return false;
    std::lock_guard<std::mutex> lock(g_mu);
    DevSlots& d = g_devs[dev];
    if (!d.resolved) {
        void* pa = nullptr;
        void* ca = nullptr;
        if (hipGetSymbolAddress(&pa, HIP_SYMBOL(xhip::g_splitk_partials)) != hipSuccess ||
            hipGetSymbolAddress(&ca, HIP_SYMBOL(xhip::g_splitk_counters)) != hipSuccess || !pa || !ca) {
            (void)hipGetLastError();
            return false;
        }
        d.partials = reinterpret_cast<float*>(pa);
        d.counters = reinterpret_cast<uint32_t*>(ca);
        d.resolved = true;
    }
    const int slot = d.slots.take(stream_key(st));
    if (slot < 0) return false;
    *partials = d.partials + (size_t)slot * xhip::kSplitPartialFloats;
    *partial_floats = xhip::kSplitPartialFloats;
    *counters = d.counters + (size_t)slot * xhip::kSplitCounters;
    *ncounters = xhip::kSplitCounters;
    return true;
}

// The area of `st` on the current device for the prefill GEMM's partial tiles.
SkArea sk_area(hipStream_t st) {
    const int dev = current_device();
    if (dev < 0) return {nullptr, nullptr};
    std::lock_guard<std::mutex> lock(g_mu);
    DevSlots& d = g_devs[dev];
    const int area = d.areas.take(stream_key(st));
    if (area < 0) return {nullptr, nullptr};
    int group = 0, first = 0;
    while (area >= first + xhip::sk_group_areas(group)) first += xhip::sk_group_areas(group++);
    if (!d.group[group] && !(d.group[group] = kGroupBase[group]())) {
        d.areas.release(stream_key(st));
        return {nullptr, nullptr};
    }
    return {d.group[group] + (size_t)(area - first) * xhip::kSkAreaFloats, &d.enqueue[area]};
}

// Gives the split-K slot and the area of `st` on the current device back (the
// slot's counters are zero once the stream's work has finished).
void splitk_release(hipStream_t st) {
    const int dev = current_device();
    if (dev < 0) return;
    std::lock_guard<std::mutex> lock(g_mu);
    g_devs[dev].slots.release(stream_key(st));
    g_devs[dev].areas.release(stream_key(st));
}

}  // namespace xhip_host
