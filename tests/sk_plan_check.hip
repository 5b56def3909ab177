// Host-only check of the prefill GEMM's work split (sk_plan and the cut into
// runs, xinfer_amd/csrc/gemm_sk_int4.hip) over random calls: the runs cover
// every step once, a plan with partial sums fits the scratch slot, the pieces
// the main kernel leaves are exactly the ones the second launch adds (each
// split tile once, its pieces in order), and the kernels' float division
// agrees with integer division; and the calls given as arguments are cut.  Built and run by
// tests/test_plan_invariants.py; no GPU is touched.
#include "../xinfer_amd/csrc/gemm_sk_int4.hip"
namespace xhip_host {
int num_cus() { return 256; }
int launch_status() { return 0; }
SkArea sk_area(hipStream_t) { return {nullptr, nullptr}; }
int gemm_ws_linear(hipStream_t, void*, const void*, const uint8_t*, const uint16_t*, const float*, int64_t, int64_t,
                   int64_t, bool, int*) { return 1; }
}
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <random>
#include <set>
#include <vector>

static int quotient(int n, int d) {  // sk_div of the kernels
    const float inv = 1.0f / (float)d;
    int q = (int)((float)n * inv);
    const int rest = n - q * d;
    q += rest >= d ? 1 : 0;
    q -= rest < 0 ? 1 : 0;
    return q;
}

// A call whose plan a GPU test relies on, "MT,M,K,swiglu,N[,N..]": cut, with MT
// row tiles, at least one tile in pieces and one run that starts inside a tile.
static bool cut_as_said(const char* arg) {
    int v[8] = {}, n = 0;
    for (const char* c = arg; c && n < 8; c = strchr(c, ',') ? strchr(c, ',') + 1 : nullptr) v[n++] = atoi(c);
    xinfer_fused_desc d[4] = {};
    for (int i = 4; i < n; ++i) d[i - 4].N = v[i];
    const SkPlan pl = sk_plan(d, n - 4, v[3] != 0, v[1], v[2], xhip::kSkAreaFloats, 256);
    const int64_t ns = (v[2] / 128 + sk::kwaves(pl.mt) - 1) / sk::kwaves(pl.mt), steps = pl.tiles * pl.mb * ns;
    const bool ok = n > 4 && !pl.whole && pl.mt == v[0] && (steps % pl.nb || steps / pl.nb % ns);
    if (!ok) printf("BAD %s: mt %d, runs %d of %lld steps, whole %d\n", arg, pl.mt, pl.nb, (long long)steps, pl.whole);
    return ok;
}

int main(int argc, char** argv) {
    std::mt19937_64 rng(2024);
    int bad = 0, whole = 0, cut = 0;
    for (int i = 1; i < argc; ++i) bad += !cut_as_said(argv[i]);
    for (int it = 0; it < 2000000; ++it) {
        const int d = 1 + (int)(rng() % (rng() % 2 ? 64 : 200000));
        const int n = (int)(rng() % (1 << 24));
        if (quotient(n, d) != n / d && ++bad < 5) printf("BAD division %d / %d\n", n, d);
    }
    for (int it = 0; it < 20000; ++it) {
        const bool swiglu = rng() % 4 == 0;
        const int nd = swiglu ? 1 : 1 + (int)(rng() % 4);
        xinfer_fused_desc d[4] = {};
        for (int i = 0; i < nd; ++i) d[i].N = 1 + (int64_t)(rng() % (rng() % 2 ? 40000 : 300));
        const int64_t M = 1 + (int64_t)(rng() % (rng() % 2 ? 600 : 70)), K = 128 * (1 + (int64_t)(rng() % 140));
        const size_t caps[3] = {(size_t)1 << 24, (size_t)1 << 20, 0};
        const size_t cap = caps[rng() % 3];
        const SkPlan pl = sk_plan(d, nd, swiglu, M, K, cap, 256);
        const int ng = (int)(K / 128), ns = (ng + sk::kwaves(pl.mt) - 1) / sk::kwaves(pl.mt);
        const int64_t tiles = sk_tiles(d, nd, swiglu, pl.mt) * pl.mb, steps = tiles * ns;
        const int grain = pl.whole ? ns : 1;
        const int q = (int)(steps / grain / pl.nb), r = (int)(steps / grain % pl.nb);
        bool ok = pl.mt >= 1 && pl.mt <= 4 && (int64_t)pl.mt * pl.mb * 32 >= M && pl.nb >= 1 && pl.nb <= 256 && q >= 1 &&
                  (pl.whole || (size_t)2 * pl.nb * sk::piece(pl.mt) <= cap) && pl.tiles * pl.mb == tiles;
        (pl.whole ? whole : cut)++;
        // the main kernel's walk
        auto start = [&](int b) { return b * q + (b < r ? b : r); };
        std::map<int, std::vector<int>> pieces;  // tile -> slots (2 * run + slot)
        int64_t done = 0, full = 0;
        for (int b = 0; b < pl.nb && ok; ++b) {
            int u = start(b) * grain, rem = (q + (b < r ? 1 : 0)) * grain;
            const int u0 = u;
            ok = ok && u == done;
            while (rem > 0) {
                const int t = quotient(u, ns), g = u - t * ns, n = rem < ns - g ? rem : ns - g;
                if (n == ns) ++full;
                else pieces[t].push_back(2 * b + (u == u0 ? 0 : 1));
                u += n, rem -= n, done += n;
            }
        }
        ok = ok && done == steps && full + (int64_t)pieces.size() == tiles;
        // the second launch's walk
        std::set<int> summed;
        if (!pl.whole) {
            for (int x = 0; x < pl.nb - 1 && ok; ++x) {
                const int b1 = x + 1, t = quotient(start(b1), ns), t0 = t * ns, t1 = t0 + ns;
                if (start(b1) == t0 || start(b1 - 1) > t0) continue;
                std::vector<int> got;
                for (int b = b1 - 1; start(b) < t1; ++b)
                    got.push_back(2 * b + (b == b1 - 1 && start(b) != t0 ? 1 : 0));
                ok = ok && summed.insert(t).second && pieces.count(t) && pieces[t] == got;
            }
        }
        ok = ok && summed.size() == pieces.size();
        if (!ok && ++bad < 10)
            printf("BAD M=%lld K=%lld nd=%d N0=%lld swiglu=%d: mt %d mb %d nb %d whole %d\n", (long long)M, (long long)K,
                   nd, (long long)d[0].N, swiglu, pl.mt, pl.mb, pl.nb, pl.whole);
    }
    printf("plans of whole tiles %d, cut %d, bad %d\n", whole, cut, bad);
    return bad || !whole || !cut ? 1 : 0;
}
