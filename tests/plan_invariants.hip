// Host-only check of the small-batch planner (plan_mb in
// xinfer_amd/csrc/gemv_mb_int4.hip) over random shapes: every descriptor gets
// between one range and one range per tile, the ranges sum to the plan's
// count, no range holds more tiles than the LDS result area was sized for,
// the grid is ranges x k-slices, the LDS request fits a CU, and a plan that
// splits K fits the stream's split-K slot (partials and counters); and
// small_batch keeps the calls of 9-16 rows on the kernel that measured faster.  Built and
// run by tests/test_plan_invariants.py; no GPU is touched (the planner's
// device queries are replaced below by a 256-CU stand-in).
#include "../xinfer_amd/csrc/gemv_mb_int4.hip"
namespace xhip_host {
int num_cus() { return 256; }
int launch_status() { return 0; }
bool gemv_stages_x(int64_t M, int64_t K) { return K <= 6144; }  // decides only M = 2
bool splitk_slot(hipStream_t, float**, size_t*, uint32_t**, int*) { return false; }
}
constexpr size_t kCap = (size_t)1 << 20;  // the slot sizes of scratch.hip
constexpr int kCnt = 4096;
#include <cstdio>
#include <random>
template <int EPI>
int check(std::mt19937_64& rng, int iters) {
    int bad = 0, planned = 0;
    for (int it = 0; it < iters; ++it) {
        MbParams p = {};
        const int nd = EPI == MB_PLAIN ? 1 + (int)(rng() % 4) : 1;
        for (int i = 0; i < nd; ++i) p.d[i].N = 1 + (int)(rng() % (rng() % 2 ? 200000 : 300));
        p.ndesc = nd;
        p.M = 2 + (int)(rng() % (EPI == MB_ARGMAX ? 7 : 15));
        p.K = 128 * (1 + (int)(rng() % (rng() % 2 ? 300 : 60)));
        xhip_host::MbPlan pl;
        const bool raise = rng() % 2;
        if (!xhip_host::plan_mb<EPI, f16>(p, pl, kCap, kCnt, raise)) continue;
        ++planned;
        int64_t sum = 0;
        bool ok = pl.blocks == pl.nranges * pl.ks && pl.lds <= 160 * 1024 && pl.kw >= 1 && (pl.nw % pl.kw) == 0 &&
                  (pl.ks == 1 || (pl.ws_floats <= kCap && pl.nranges <= kCnt));
        for (int i = 0; i < nd; ++i) {
            const int t = (p.d[i].N + 15) / 16;
            const int nr = p.d[i].nr;
            ok = ok && nr >= 1 && nr <= t && (t + nr - 1) / nr <= pl.tiles_blk;
            sum += nr;
        }
        ok = ok && sum == pl.nranges && p.nranges == pl.nranges;
        if (!ok) {
            if (bad < 5) printf("BAD epi=%d M=%d K=%d nd=%d N0=%d blocks=%d ranges=%d ks=%d tiles_blk=%d kw=%d lds=%zu\n", EPI, p.M, p.K, nd, p.d[0].N, pl.blocks, pl.nranges, pl.ks, pl.tiles_blk, pl.kw, pl.lds);
            ++bad;
        }
    }
    printf("epi=%d planned %d of %d, bad %d\n", EPI, planned, iters, bad);
    return bad;
}
// Calls of M = 9..16 (weight rows * K in millions) whose two kernels were timed and differ.
int check_routes() {
    struct Route {
        int M, K, millions;
        bool swiglu, small;
    };
    static const Route routes[] = {
        {9, 8192, 85, true, true},    {9, 10240, 100, true, true},   {10, 14336, 100, true, true},
        {9, 16384, 140, true, true},  {10, 6144, 140, true, true},   {12, 10240, 85, true, true},
        {12, 16384, 85, true, true},  {9, 6144, 180, true, false},   {16, 8192, 85, true, false},
        {13, 12288, 140, true, false}, {13, 8192, 82, true, false}, {9, 17408, 100, true, false}, {12, 5248, 140, true, false},
        {12, 17408, 45, true, true},  {12, 17408, 85, false, false}, {9, 9216, 85, false, false},
        {16, 12288, 100, false, false}, {12, 8192, 30, false, true}, {16, 2560, 89, false, true},
    };
    int bad = 0;
    for (const Route& r : routes)
        if (xhip_host::small_batch(r.M, (int64_t)r.millions * 1000000 / r.K, r.K, r.swiglu) != r.small) {
            printf("BAD route M=%d K=%d %d M swiglu=%d\n", r.M, r.K, r.millions, r.swiglu);
            ++bad;
        }
    for (int M = 1; M <= 20; ++M)  // other rows: never, and always for 2-8
        if ((M < 9 || M > 16) && xhip_host::small_batch(M, 100000, 8192, M & 1) != (M >= 2 && M <= 8)) ++bad;
    return bad;
}
int main() {
    std::mt19937_64 rng(12345);
    int bad = check<MB_PLAIN>(rng, 20000) + check<MB_SWIGLU>(rng, 20000) + check<MB_ARGMAX>(rng, 20000) + check_routes();
    return bad ? 1 : 0;
}
