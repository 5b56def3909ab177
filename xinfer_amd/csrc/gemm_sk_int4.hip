// INT4-G128-SYM projection GEMM for prefill rows on gfx950 (M > 16, and M =
// 9-16 where small_batch() of gemv_mb_int4.hip sends many weights here):
// weights decoded in registers, work split evenly over the CUs.
//
// Same contract as the reference's linear_int4 / linear_int4_fused /
// mlp_gate_up_swiglu_int4 at M > 8 (src/ops/linear.h:30-139; chunked prefill
// calls them with M = chunk, src/targets/qwen3_8/forward.cpp:112-125, 229,
// 276-287): q is exact in fp16, a group's products are summed in FP32 by the
// matrix cores and the group's fp16 scale is applied to that sum in FP32.
//
// Work: a tile is 32 * MT activation rows x 128 or 256 weight rows (half of
// them gate and half up rows for the SwiGLU) of one projection, a step one or
// two 128-k groups of a tile.  The steps of all tiles of all projections of
// the call, in tile order, are cut into equal runs, one per block, so every CU
// has the same work whatever the number of tiles is.  A run that starts or ends
// inside a tile leaves FP32 partial sums; a second launch adds those of each
// split tile in order.  (Adding them in the block that arrives last, by a
// counter per tile, measured slower everywhere: one CU then reads all pieces
// of a tile, e.g. 13 x 128 KB for N = 5120, K = 17408, M = 128: 74.0 against
// 41.2 us.)
//
// What bounds it (N = 69632, K = 5120, test builds without a part; M = 32 / 64 /
// 96 / 128, full 58.7 / 75.5 / 89.8 / 109.5 us): up to M = 64 the copies to LDS
// and the barriers between them (55.3 / 67.6 us without MFMA and decode), at
// larger M these (73.9 / 88.8) and the rest (without copies 72.6 / 90.6) take
// about four fifths of the time each and overlap only in part; the decode is
// hidden (111.8 at M = 128 without it), the matrix cores are busy 55 % of the
// M = 128 launch.
// N = 17408, K = 5120, M = 17 / 64 / 128: 21.7 / 26.4 / 39.9 us = 2.1 / 1.7 /
// 1.1 TB/s of weights, 140 / 432 / 572 TFLOP/s (the 128-row GEMM with a block
// per tile and rounded weights that it replaced: 49.3 / 55.0 / 68.2);
// N = 5120, K = 17408, M = 23 / 512: 23.2 / 107 us (157 / 201); K = 3456,
// N = 5003, M = 200, fp32 outputs: 27.1 us (214 as GEMV slabs of 8 rows).
// Before the run cut, those long-K, small-N shapes left two thirds of the CUs
// without a block.

#include <stdlib.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "sk_areas.h"

namespace xhip {

struct SkDesc {
    const uint8_t* W;    // [N][K/2] (gate)
    const uint16_t* S;   // [N][K/128]
    const uint8_t* W2;   // up (SwiGLU)
    const uint16_t* S2;
    const float* bias;   // optional [N]
    void* Y;             // [M][N]
    int32_t N;
    int32_t tile_begin;  // first column tile
    int32_t y16;         // fp16 Y: 16-byte aligned and N % 8 == 0
    int32_t pad;
};

struct SkParams {
    SkDesc d[4];
    const f16* X;     // [M][K]
    float* part;      // partial tiles, two slots per block
    int32_t M, K, ng, ns;  // ns: steps of a tile
    int32_t mb;       // row blocks
    int32_t ndesc;
    int32_t q, r;     // granules per run (the first r runs have one more)
    int32_t grain;    // steps per granule: 1, or ns (runs of whole tiles)
    int32_t residual; // fp16 Y = fp16(Y + fp16(result))
    float inv_ns, inv_mb;
};

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void* sk_lds_ptr_t;

namespace sk {
constexpr int kWaves = 8;      // of a block; the first half copies X, the other half weights
constexpr int kXRing = 3;      // steps of X (and of scales) in LDS: one in use, two on their way
constexpr int kOutWave = 32 * 64;  // bytes of a staged 32 x 32 fp16 tile
// where 16-byte piece ch of row r of it is
__device__ __forceinline__ int out_at(int r, int ch) { return r * 64 + ((ch ^ ((r >> 1) & 3)) * 16); }
// Shape of a block by row tiles: KW waves share 32 weight rows and take one
// group each of a step's KW groups.
constexpr int kwaves(int mt) { return mt <= 2 ? 2 : 1; }
constexpr int colgroups(int mt) { return kWaves / kwaves(mt); }
constexpr int bn(int mt) { return 32 * colgroups(mt); }         // weight rows of a tile
constexpr int xbytes(int mt) { return mt * 8192 * kwaves(mt); }  // X of a step
constexpr int wbytes(int mt) { return bn(mt) * 64 * kwaves(mt); }
constexpr int wring(int mt) { return mt == 1 ? 6 : mt == 3 ? 5 : 3; }  // steps of weights
constexpr int piece(int mt) { return 32 * mt * bn(mt); }         // floats of a partial tile
constexpr int kScales = kWaves / 2 * 64;                         // scales of a step: bn * KW
constexpr int off_w(int mt) { return kXRing * xbytes(mt); }
constexpr int off_s(int mt) { return off_w(mt) + wring(mt) * wbytes(mt); }
constexpr int lds_bytes(int mt) { return off_s(mt) + kXRing * kScales * 2; }
static_assert(kScales == bn(1) * kwaves(1) && kScales == bn(4) * kwaves(4), "a scale per lane of the X waves");
static_assert(lds_bytes(1) <= 160 * 1024 && lds_bytes(2) <= 160 * 1024 && lds_bytes(3) <= 160 * 1024 &&
                  lds_bytes(4) <= 160 * 1024,
              "LDS of one CU");
// the X just used makes room for the wave sums, then for staged output rows
static_assert(colgroups(1) * 4096 <= xbytes(1) && colgroups(2) * 8192 <= xbytes(2), "sums that cross waves");
static_assert(colgroups(1) * kOutWave <= xbytes(1) && colgroups(4) * kOutWave <= xbytes(3), "staged rows");
}  // namespace sk

// Natural-order decode of one dword (8 nibbles, k0 in bits 0-3) into the 8
// exact integers of an MFMA operand (k0 .. k7).
__device__ __forceinline__ f16x8 sk_decode8(uint32_t w) {
    const f16x2 kMul = {(f16)1.0f, (f16)0.0625f};
    const f16x2 kAdd = {(f16)-1032.0f, (f16)-72.0f};
    f16x8 o;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const uint32_t sel = 0x0C000C00u | ((uint32_t)b << 16) | (uint32_t)b;
        const uint32_t bb = __builtin_amdgcn_perm(w, w, sel);  // [byte b, 0, byte b, 0]
        const f16x2 q = as_h2((bb & 0x00F0000Fu) ^ 0x64806408u) * kMul + kAdd;
        o[2 * b] = q.x;
        o[2 * b + 1] = q.y;
    }
    return o;
}

#define XHIP_SK_VMCNT(n) \
    __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

// Stores a 32 x 32 tile of sums from the MFMA layout (lane (li, lh), register
// e: column li, row 8 (e / 4) + 4 lh + e % 4) at row m0 and output column n0.
// SwiGLU: columns 0-15 are gate, 16-31 up rows of 16 output columns.  `st`:
// kOutWave bytes of LDS of this wave.
template <bool SWIGLU, typename OutT, bool HALVES>
__device__ __forceinline__ void sk_store(const SkDesc& d, const f32x16& sum, int m0, int n0, int M, bool residual,
                                         unsigned char* st, int lane) {
    using namespace sk;
    constexpr int COLS = SWIGLU ? 16 : 32;
    const int li = lane & 31, lh = lane >> 5;
    const int N = d.N;
    if (n0 >= N || m0 >= M) return;
    const int col = SWIGLU ? (lane & 15) : li;
    const float bn = (!SWIGLU && d.bias && n0 + col < N) ? d.bias[n0 + col] : 0.0f;
    OutT* const Y = reinterpret_cast<OutT*>(d.Y);
    // SwiGLU: lanes 16 apart hold gate and up of the same outputs.  HALVES:
    // each of the two takes half of them (in the second launch, whose waves
    // do little else: N = 3000, K = 2176, M = 40 18.9 -> 17.9 us, N = 1100,
    // K = 5120, M = 77 22.8 -> 20.2); in the main kernel, where it costs the
    // loop its registers (N = 17408, K = 5120, M = 60 45.7 -> 52.8), the lane
    // with the gate row computes all 16.
    constexpr bool BOTH = SWIGLU && HALVES;
    constexpr int NV = BOTH ? 8 : 16;
    const int up16 = BOTH ? (lane & 16) : 0;  // the upper half's rows
    const bool live = !SWIGLU || BOTH || !(lane & 16);
    auto row_of = [&](int e) { return 8 * (e >> 2) + 4 * lh + (e & 3) + up16; };
    float v[NV];
#pragma unroll
    for (int e = 0; e < NV; ++e) {
        if constexpr (BOTH) {
            const float mine = up16 ? sum[e + 8] : sum[e];
            const float other = __shfl_xor(up16 ? sum[e] : sum[e + 8], 16);
            const float g = up16 ? other : mine, u = up16 ? mine : other;
            v[e] = g / (1.0f + expf(-g)) * u;
        } else if constexpr (SWIGLU) {
            const float u = __shfl_xor(sum[e], 16);
            v[e] = sum[e] / (1.0f + expf(-sum[e])) * u;
        } else {
            v[e] = sum[e] + bn;
        }
    }
    if constexpr (sizeof(OutT) == 2) {
        if (d.y16) {  // whole 16-byte pieces of rows, through LDS
            if (live) {
#pragma unroll
                for (int e = 0; e < NV; ++e)
                    *reinterpret_cast<f16*>(st + out_at(row_of(e), col >> 3) + 2 * (col & 7)) = (f16)v[e];
            }
            constexpr int CH = COLS / 8;  // pieces of a row
            constexpr int RPS = 64 / CH;  // rows per store
#pragma unroll
            for (int r0 = 0; r0 < 32; r0 += RPS) {
                const int rr = r0 + lane / CH, ch = lane % CH;
                const int m = m0 + rr, n = n0 + 8 * ch;
                if (m < M && n < N) {
                    u32x4 o = *reinterpret_cast<const u32x4*>(st + out_at(rr, ch));
                    u32x4* y = reinterpret_cast<u32x4*>(Y + (size_t)m * N + n);
                    if (residual) {
                        const u32x4 b = *y;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const f16x2 a2 = as_h2(b[i]), c2 = as_h2(o[i]);
                            f16x2 s2;
                            s2.x = (f16)((float)a2.x + (float)c2.x);
                            s2.y = (f16)((float)a2.y + (float)c2.y);
                            o[i] = as_u32(s2);
                        }
                    }
                    *y = o;
                }
            }
            return;
        }
    }
#pragma unroll
    for (int e = 0; e < NV; ++e) {
        const int m = m0 + row_of(e);
        if (live && m < M && n0 + col < N) {
            OutT* y = Y + (size_t)m * N + n0 + col;
            if (sizeof(OutT) == 2 && residual)
                *y = (OutT)((float)*y + (float)(OutT)v[e]);
            else
                *y = (OutT)v[e];
        }
    }
}

// The projection of a column tile.
__device__ __forceinline__ const SkDesc& sk_desc(const SkParams& p, int ct) {
    int di = 0;
#pragma unroll
    for (int i = 1; i < 4; ++i)
        if (i < p.ndesc && ct >= p.d[i].tile_begin) di = i;
    return p.d[di];
}

// n / d of wave-uniform n < 2^24 (the host keeps the step count below that):
// the float quotient is off by one at most.
__device__ __forceinline__ int sk_div(int n, int d, float inv) {
    int q = __builtin_amdgcn_readfirstlane((int)((float)n * inv));
    const int rest = n - q * d;
    q += rest >= d ? 1 : 0;
    q -= rest < 0 ? 1 : 0;
    return q;
}

// A run's partial tile is its first tile (slot 0 of the block) or its last
// (slot 1; a run inside one tile has slot 0 only): byte offset of a column
// group's sums.
template <int MT>
__device__ __forceinline__ size_t sk_piece_at(int run, int slot, int cgr) {
    return (size_t)(2 * run + slot) * (sk::piece(MT) * 4) + (size_t)cgr * (MT * 4096);
}

template <int MT, bool SWIGLU, typename OutT>
__global__ __launch_bounds__(64 * sk::kWaves) void gemm_sk_int4_kernel(const SkParams p) {
    using namespace sk;
    constexpr int BM = 32 * MT;
    constexpr int KW = kwaves(MT), CG = colgroups(MT), RW = wring(MT), HALF = kWaves / 2;
    constexpr int XB = xbytes(MT), WB = wbytes(MT);
    constexpr int COLS = SWIGLU ? 16 : 32;         // output columns of a wave
    constexpr int XPW = XB / 1024 / HALF;          // copies of a wave per step, 1 KB each
    constexpr int WPW = WB / 1024 / HALF;
    constexpr int CPW = XPW > WPW ? XPW : WPW;
    constexpr int WRI = 16 / KW;                   // weight rows of a copy
    static_assert(XPW * HALF * 1024 == XB && WPW * HALF * 1024 == WB && CPW <= 8, "copies split evenly");
    extern __shared__ __align__(16) unsigned char smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const int cgr = wave % CG, kw = wave / CG;  // column group, group of a step

    // runs of consecutive steps on one XCD (blocks go to the XCDs in turn)
    const int nb = gridDim.x;
    const int l = (nb & 7) ? (int)blockIdx.x : ((int)blockIdx.x & 7) * (nb >> 3) + ((int)blockIdx.x >> 3);
    const int M = p.M, ng = p.ng, ns = p.ns, mbs = p.mb;
    const uint32_t row_bytes = (uint32_t)(p.K >> 1);
    const int u0 = (l * p.q + min(l, p.r)) * p.grain;
    int rem = (p.q + (l < p.r ? 1 : 0)) * p.grain;  // steps still to compute
    int left = rem;                                  // steps still to copy

    // ---- copies of a step to LDS ----------------------------------------------
    // A copy is 1 KB.  Weights: 16 / KW rows, of each the step's KW * 64
    // bytes; X: 8 rows of 64 k.  Lanes go along a row, so a copy takes the
    // address unit about half as long as one with a row per lane (13 against
    // 27 ns measured); a row's 16-byte chunks are stored in an order that
    // depends on the row, so that the operand reads, a row per lane, spread
    // over all banks.  Loads of a wave land in order, so X (from L2, two
    // steps ahead) and weights (from HBM, up to five steps ahead) are copied
    // by different waves: neither waits for the other's.
    const int role = wave & (HALF - 1);
    // The whole run, for the waves that copy X or for those that copy weights:
    // each has its own count of loads in flight.
    auto block = [&](auto xw) {
        constexpr bool xwave = decltype(xw)::value;
        int pt = sk_div(u0, ns, p.inv_ns), pg = u0 - pt * ns;  // the step this wave copies next
        __amdgpu_buffer_rsrc_t r0, r1;
        const uint16_t* sp = nullptr;
        uint32_t off[CPW];
        int to = 0;  // its place in the ring
        // Where a row's chunk is stored: LDS serves 16 lanes of 16 bytes a cycle from
        // 64 banks, so a chunk of 16 consecutive rows takes every place of 256 bytes
        // once (with the order of 8 rows repeated, half of the LDS cycles were bank
        // conflicts).
        auto xchunk = [](int row, int ch) { return ch ^ (row & 7) ^ ((row >> 3) & 1); };
        auto wchunk = [&](int row, int ch) {
            return KW == 2 ? xchunk(row, ch) : ch ^ ((row >> 2) & 3);
        };
        // Lane-dependent addresses of rare work are computed where they are used
        // and not kept in registers through the loop.
        auto here = [&]() {
            int v = lane;
            asm volatile("" : "+v"(v));
            return v;
        };
        auto set_tile = [&]() {
            const int lane = here();
            const int ct = mbs == 1 ? pt : sk_div(pt, mbs, p.inv_mb);
            const SkDesc& d = sk_desc(p, ct);
            const int N = d.N;
            const int c0 = (ct - d.tile_begin) * (CG * COLS);
            // weight row v of the tile (32 per column group; the SwiGLU's are 16
            // gate and 16 up rows)
            auto row_of = [&](int v) { return min(c0 + (SWIGLU ? (v >> 5) * 16 + (v & 15) : v), N - 1); };
            if constexpr (xwave) {
                r0 = r1 = __builtin_amdgcn_make_buffer_rsrc((void*)p.X, (short)0, (int)((uint32_t)M * (uint32_t)p.K * 2u),
                                                            0x00020000);
                const int m0 = (pt - ct * mbs) * BM;
#pragma unroll
                for (int j = 0; j < XPW; ++j) {
                    const int q = role * XPW + j;                          // copy of the step
                    const int gq = q / (8 * MT), qq = q - gq * (8 * MT);   // group of the step, copy of the group
                    const int rg = qq / (4 * MT), rb = qq - rg * (4 * MT);
                    const int xr = min(m0 + rb * 8 + (lane >> 3), M - 1);
                    off[j] = ((uint32_t)xr * (uint32_t)p.K + 128u * gq + 64u * rg + 8u * xchunk(rb * 8 + (lane >> 3), lane & 7)) * 2u;
                }
                const int v = (role * 64 + lane) % bn(MT);
                sp = ((SWIGLU && (v & 16)) ? d.S2 : d.S) + (size_t)row_of(v) * ng;
            } else {
                r0 = __builtin_amdgcn_make_buffer_rsrc((void*)d.W, (short)0, (int)((uint32_t)N * row_bytes), 0x00020000);
                r1 = SWIGLU ? __builtin_amdgcn_make_buffer_rsrc((void*)d.W2, (short)0, (int)((uint32_t)N * row_bytes), 0x00020000)
                            : r0;
#pragma unroll
                for (int j = 0; j < WPW; ++j) {
                    const int v = (role * WPW + j) * WRI + lane / (4 * KW);
                    off[j] = (uint32_t)row_of(v) * row_bytes + 16u * wchunk(v, lane % (4 * KW));
                }
            }
        };
        auto copy = [&](const int j) {
            if (j < (xwave ? XPW : WPW)) {
                const int at = xwave ? to * XB + (role * XPW + j) * 1024 : off_w(MT) + to * WB + (role * WPW + j) * 1024;
                const int go = pg * (xwave ? 256 * KW : 64 * KW);
                __builtin_amdgcn_raw_ptr_buffer_load_lds((j * WRI) & 16 ? r1 : r0, (sk_lds_ptr_t)(smem + at), 16,
                                                         (int)off[j], go, 0, 0);
            }
        };
        auto advance = [&]() {  // to the next step; past the run's end: the last one again
            to = to + 1 == (xwave ? kXRing : RW) ? 0 : to + 1;
            if (left > 1) {
                --left;
                if (++pg == ns) {
                    pg = 0;
                    ++pt;
                    set_tile();
                }
            }
        };
        // scales: a lane of the X waves has one of the step's, group role * 64 / bn
        auto scale_load = [&]() { return sp[min(pg * KW + (role * 64) / bn(MT), ng - 1)]; };
        uint16_t* const sbuf = reinterpret_cast<uint16_t*>(smem + off_s(MT));

        // operand addresses in a stage: X chunk c of row r, weight chunk of row li
        int xa[4], wa[2];
#pragma unroll
        for (int d = 0; d < 4; ++d)
            xa[d] = kw * (MT * 8192) + (li >> 3) * 1024 + (li & 7) * 128 + xchunk(li, 4 * lh + d) * 16;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            wa[j] = off_w(MT) + (cgr * 32 + li) * (64 * KW) + 16 * wchunk(li, 4 * kw + 2 * j + lh);

        f32x16 acc[MT];
        // One step: k = 64 j + 32 lh + 8 d of dword d of weight chunk j.  16-k
        // steps of two row tiles at a time, the operands of the next one read and
        // decoded between the MFMAs; the second pair of row tiles reuses the
        // decoded weights.  The first operands of the next step are read at this
        // one's end, so no wave starts a step with a wait for LDS.
        // The copies of a later step go out one or two at a time between the
        // first MFMAs: a wave waits at a copy until the address unit takes it,
        // so all of them at the start of the step would hold every wave for as
        // long as the unit needs for the block's copies (measured: a step then
        // took the sum of its copies' and its arithmetic's time).
        constexpr int P0 = MT < 2 ? MT : 2, P1 = MT - P0;
        u32x4 w[2];
        f16x8 b[P1 > 0 ? 8 : 2];
        f16x8 a[2][2];
        auto opread = [&](const unsigned char* xs, int k, int mt0, int n, int into) {
#pragma unroll
            for (int t = 0; t < n; ++t)
                a[into][t] = *reinterpret_cast<const f16x8*>(xs + xa[k & 3] + ((k >> 2) * MT + mt0 + t) * 4096);
        };
        auto first = [&](int xat, int wat) {
            w[0] = *reinterpret_cast<const u32x4*>(smem + wat + wa[0]);
            opread(smem + xat, 0, 0, P0, 0);
            w[1] = *reinterpret_cast<const u32x4*>(smem + wat + wa[1]);
        };
        auto mfma = [&](f16x8 x, f16x8 y, f32x16 c, bool zero) {
            if (zero) {
#pragma unroll
                for (int e = 0; e < 16; ++e) c[e] = 0.0f;
            }
            return __builtin_amdgcn_mfma_f32_32x32x16_f16(x, y, c, 0, 0, 0);
        };
        // `mid` runs once all copies of the step are out
        auto compute = [&](int xat, float s, auto mid, auto next) {
            const unsigned char* xs = smem + xat;
            f32x16 pa[P0], pb[P1 > 0 ? P1 : 1];
            constexpr int CPK = P1 > 0 ? 1 : 2;  // copies per 16-k step
            static_assert(CPW <= (P1 > 0 ? 8 : 4) * CPK, "copies before the middle");
            b[0] = sk_decode8(w[0][0]);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int cur = k & 1;
                if (k < 7) opread(xs, k + 1, 0, P0, cur ^ 1);
                else if (P1) opread(xs, 0, P0, P1, cur ^ 1);
                else next();
#pragma unroll
                for (int t = 0; t < P0; ++t) pa[t] = mfma(a[cur][t], b[P1 > 0 ? k : cur], pa[t], k == 0);
#pragma unroll
                for (int c = 0; c < CPK; ++c)
                    if (k * CPK + c < CPW) copy(k * CPK + c);
                if (k < 7) b[P1 > 0 ? k + 1 : cur ^ 1] = sk_decode8(w[(k + 1) >> 2][(k + 1) & 3]);
                __builtin_amdgcn_sched_barrier(0);
                if (k == (P1 > 0 ? 7 : 3)) mid();
            }
            if constexpr (P1 > 0) {
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const int cur = k & 1;
                    if (k < 7) opread(xs, k + 1, P0, P1, cur ^ 1);
                    else next();
#pragma unroll
                    for (int t = 0; t < P1; ++t) pb[t] = mfma(a[cur][t], b[k], pb[t], k == 0);
#pragma unroll
                    for (int t = 0; t < P0; ++t)
#pragma unroll
                        for (int e = 2 * k; e < 2 * k + 2; ++e) acc[t][e] = __builtin_fmaf(s, pa[t][e], acc[t][e]);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int t = 0; t < P1; ++t)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[P0 + t][e] = __builtin_fmaf(s, pb[t][e], acc[P0 + t][e]);
            } else {
#pragma unroll
                for (int t = 0; t < P0; ++t)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[t][e] = __builtin_fmaf(s, pa[t][e], acc[t][e]);
            }
        };

        // the second wave's sums of a column group onto the first's, through LDS
        auto sum_waves = [&](unsigned char* at) {
            const int lane = here();
            if (kw == 1) {
#pragma unroll
                for (int v = 0; v < MT * 4; ++v)
                    *reinterpret_cast<f32x4*>(at + (cgr * MT * 4 + v) * 1024 + lane * 16) =
                        f32x4{acc[v / 4][(v % 4) * 4], acc[v / 4][(v % 4) * 4 + 1], acc[v / 4][(v % 4) * 4 + 2],
                              acc[v / 4][(v % 4) * 4 + 3]};
            }
            __builtin_amdgcn_s_waitcnt(0xC07F);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (kw == 0) {
#pragma unroll
                for (int v = 0; v < MT * 4; ++v) {
                    const f32x4 f = *reinterpret_cast<const f32x4*>(at + (cgr * MT * 4 + v) * 1024 + lane * 16);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[v / 4][(v % 4) * 4 + e] += f[e];
                }
            }
        };
        auto store_piece = [&](int slot) {
            f32x4* const at = reinterpret_cast<f32x4*>(reinterpret_cast<unsigned char*>(p.part) + sk_piece_at<MT>(l, slot, cgr)) + here();
#pragma unroll
            for (int v = 0; v < MT * 4; ++v)
                at[v * 64] = f32x4{acc[v / 4][(v % 4) * 4], acc[v / 4][(v % 4) * 4 + 1], acc[v / 4][(v % 4) * 4 + 2],
                                   acc[v / 4][(v % 4) * 4 + 3]};
        };
        auto store_tile = [&](int t, unsigned char* st) {
            const int lane = here();
            const int ct = mbs == 1 ? t : sk_div(t, mbs, p.inv_mb), mb = t - ct * mbs;
            const SkDesc& d = sk_desc(p, ct);
            const int n0 = (ct - d.tile_begin) * (CG * COLS) + cgr * COLS;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                sk_store<SWIGLU, OutT, false>(d, acc[mt], mb * BM + mt * 32, n0, M, p.residual != 0, st + cgr * kOutWave, lane);
        };

        int ct = pt, cg = pg;
        int end = min(rem, ns - cg);  // steps of this tile in the run
        int i = end;
        int g = cg * KW + kw;         // this wave's group of the step
        int xat = 0, wat = 0;         // the step's places in the rings
        int sat = 0;
        set_tile();
        auto clear = [&]() {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[mt][e] = 0.0f;
        };
        clear();
        // the steps on their way before the first one: X 2 (with their scales),
        // weights RW - 1
        auto ahead = [&]() {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < CPW; ++j) copy(j);
            advance();
            __builtin_amdgcn_sched_barrier(0);
        };
        uint16_t s_next;  // X waves: the scale of the step after the one in use
        if constexpr (xwave) {
            const uint16_t sa = scale_load();
            ahead();
            s_next = scale_load();
            ahead();
            sbuf[role * 64 + lane] = sa;
        } else {
            for (int k = 0; k < RW - 1; ++k) ahead();
        }
        auto landed = [&]() {  // this wave's copies of the next step
            if constexpr (xwave) {
                XHIP_SK_VMCNT(XPW);
            } else {
                XHIP_SK_VMCNT((RW - 2) * WPW);
            }
        };
        auto barrier = [&]() {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        landed();
        __builtin_amdgcn_s_waitcnt(0xC07F);  // the scale is stored
        barrier();
        first(0, 0);
        for (;;) {
            // here every wave is past the step before this one, whose places the
            // copies may take
            const int xnx = xat == 2 * XB ? 0 : xat + XB;
            const int wnx = wat == (RW - 1) * WB ? 0 : wat + WB;
            const int snx = sat == 2 * kScales ? 0 : sat + kScales;
            __builtin_amdgcn_sched_barrier(0);
            // The middle of a step: the next one's copies and scales are in LDS.
            auto mid = [&]() {
                landed();
                if constexpr (xwave) sbuf[snx + role * 64 + lane] = s_next;
                __builtin_amdgcn_s_waitcnt(0xC07F);
                barrier();
                if constexpr (xwave) s_next = scale_load();
                advance();
                __builtin_amdgcn_sched_barrier(0);
            };
            auto next = [&]() { first(xnx, wnx); };
            if (KW == 1 || g < ng) {
                compute(xat, h2f(sbuf[sat + kw * bn(MT) + cgr * 32 + li]), mid, next);
            } else {  // a dead group is not read
#pragma unroll
                for (int j = 0; j < CPW; ++j) copy(j);
                mid();
                next();
            }
            __builtin_amdgcn_sched_barrier(0);
            g += KW;
            if (--i == 0) {
                unsigned char* const used = smem + xat;  // free once every wave is past its reads
                barrier();
                if (KW > 1) {
                    sum_waves(used);
                    __builtin_amdgcn_s_waitcnt(0xC07F);  // the sums are read before staged rows take their place
                    barrier();
                }
                if (kw == 0) {
                    if (end == ns) store_tile(ct, used);
                    else store_piece(ct * ns + cg == u0 ? 0 : 1);
                }
                rem -= end;
                if (rem <= 0) break;
                ++ct;
                cg = 0;
                g = kw;
                i = end = min(rem, ns);
                clear();
                __builtin_amdgcn_s_waitcnt(0xC07F);  // reads of the staged rows
            }
            barrier();
            xat = xnx;
            wat = wnx;
            sat = snx;
        }
        XHIP_SK_VMCNT(0);  // no copy is left in flight
    };
    if (wave < HALF)
        block(std::true_type{});
    else
        block(std::false_type{});
}

// Adds the pieces of split tiles and stores them: a wave takes one 32 x 32
// tile of sums.  Block x stands for the start of run x + 1: where that start
// is the first one inside a tile, the block has that tile.
template <int MT, bool SWIGLU, typename OutT>
__global__ __launch_bounds__(256) void gemm_sk_sum_kernel(const SkParams p) {
    using namespace sk;
    constexpr int CG = colgroups(MT), COLS = SWIGLU ? 16 : 32;
    __shared__ __align__(16) unsigned char smem[4 * kOutWave];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    auto start = [&](int b) { return b * p.q + min(b, p.r); };
    const int b1 = blockIdx.x + 1;
    const int t = sk_div(start(b1), p.ns, p.inv_ns);
    const int t0 = t * p.ns, t1 = t0 + p.ns;
    if (start(b1) == t0 || start(b1 - 1) > t0) return;
    const int first = b1 - 1;
    const int slot0 = start(first) == t0 ? 0 : 1;
    const int sub = blockIdx.y * 4 + wave;
    const int cgr = sub / MT, mt = sub - cgr * MT;
    const unsigned char* const part = reinterpret_cast<const unsigned char*>(p.part);
    auto at = [&](int b) {
        return reinterpret_cast<const f32x4*>(part + sk_piece_at<MT>(b, b == first ? slot0 : 0, cgr)) + mt * 256 + lane;
    };
    f32x16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
    constexpr int PB = 4;  // pieces in flight
    for (int b = first; start(b) < t1; b += PB) {
        f32x4 x[PB][4];
#pragma unroll
        for (int c = 0; c < PB; ++c) {
            const f32x4* q = at(start(b + c) < t1 ? b + c : b);
#pragma unroll
            for (int v = 0; v < 4; ++v) x[c][v] = q[v * 64];
        }
#pragma unroll
        for (int c = 0; c < PB; ++c) {
            if (start(b + c) >= t1) break;
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[e] += x[c][e >> 2][e & 3];
        }
    }
    const int ct = p.mb == 1 ? t : sk_div(t, p.mb, p.inv_mb);
    const SkDesc& d = sk_desc(p, ct);
    sk_store<SWIGLU, OutT, true>(d, acc, (t - ct * p.mb) * (32 * MT) + mt * 32, (ct - d.tile_begin) * (CG * COLS) + cgr * COLS,
                           p.M, p.residual != 0, smem + wave * kOutWave, lane);
}

}  // namespace xhip

// ------------------------------------------------------------------ host ----

using namespace xhip;

namespace xhip_host {
int gemm_ws_linear(hipStream_t st, void* Y, const void* X, const uint8_t* W, const uint16_t* S, const float* bias,
                   int64_t M, int64_t N, int64_t K, bool residual, int* rc);  // gemm_ws_int4.hip
}

namespace {

typedef void (*SkKernel)(SkParams);
struct SkKernels {
    SkKernel main, sum;
};

template <bool SWIGLU, typename OutT>
SkKernels sk_kernels(int mt) {
    switch (mt) {
        case 1: return {gemm_sk_int4_kernel<1, SWIGLU, OutT>, gemm_sk_sum_kernel<1, SWIGLU, OutT>};
        case 2: return {gemm_sk_int4_kernel<2, SWIGLU, OutT>, gemm_sk_sum_kernel<2, SWIGLU, OutT>};
        case 3: return {gemm_sk_int4_kernel<3, SWIGLU, OutT>, gemm_sk_sum_kernel<3, SWIGLU, OutT>};
        default: return {gemm_sk_int4_kernel<4, SWIGLU, OutT>, gemm_sk_sum_kernel<4, SWIGLU, OutT>};
    }
}

bool sk_allow_lds(SkKernel k, int lds) {
    static std::mutex mu;
    static SkKernel done[16];
    static int ndone = 0;
    std::lock_guard<std::mutex> lock(mu);
    for (int i = 0; i < ndone; ++i)
        if (done[i] == k) return true;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
        return false;
    if (ndone < 16) done[ndone++] = k;
    return true;
}

// How the work is cut: row tiles per block, row blocks, runs, and whether a
// run is whole tiles (no partial sums).
struct SkPlan {
    int mt, mb, nb;
    bool whole;
    int64_t tiles;  // column tiles of all projections
};

int64_t sk_tiles(const xinfer_fused_desc* descs, int nd, bool swiglu, int mt) {
    const int bn = swiglu ? sk::bn(mt) / 2 : sk::bn(mt);
    int64_t tiles = 0;
    for (int i = 0; i < nd; ++i) tiles += (descs[i].N + bn - 1) / bn;
    return tiles;
}

// Smallest estimated time, in us: a step of MT row tiles takes kStep[MT][0]
// with few blocks running and kStep[MT][1] with one on every CU (they share
// HBM, L2 and power); start, first loads and stores 5.5; the second launch 3
// and 0.35 per piece of a tile.  kStep is from before a step's first operands
// were read ahead and the LDS order changed; with a block on every CU a step
// now takes 1.10 / 1.46 / 1.70 / 2.06 at MT = 1 .. 4.  A piece is counted alike
// at 16 KB (MT = 1) and 128 KB (MT = 4): sums of N = 5003, K = 3456, M = 200
// take 9.2 us where 5.2 are estimated, of {10240, 6144, 48, 48} x 5120, M = 77
// 7.2 where 4.6.  Measured, chosen plan first: N = 1024, K = 5120, M = 128 14.8,
// 32 runs 18.3, 16 runs 25.5; N = 3000, K = 1024, M = 64 whole tiles 8.0, 96
// runs 10.7; N = 17408, K = 5120, M = 17 / 64 256 runs 21.6 / 26.4, whole tiles
// 23.3 / 29.8.
SkPlan sk_plan(const xinfer_fused_desc* descs, int nd, bool swiglu, int64_t M, int64_t K, size_t part_floats, int cus) {
    static const double kStep[5][2] = {{0, 0}, {0.8, 1.1}, {1.0, 1.5}, {1.2, 1.85}, {1.45, 2.2}};
    const int64_t ng = K / kGroup, rows = (M + 31) / 32;
    SkPlan best = {0, 0, 0, false, 0};
    double best_t = 1e300;
    for (int64_t mb = (rows + 3) / 4; mb <= (rows + 3) / 4 + 1 && mb <= rows; ++mb) {
        const int mt = (int)((rows + mb - 1) / mb);
        const int64_t ns = (ng + sk::kwaves(mt) - 1) / sk::kwaves(mt);
        const int64_t tiles = sk_tiles(descs, nd, swiglu, mt), all = tiles * mb, steps = all * ns;
        auto step_us = [&](int64_t nb) { return kStep[mt][0] + (kStep[mt][1] - kStep[mt][0]) * (double)nb / cus; };
        auto take = [&](int64_t nb, bool whole, double t) {
            if (t < best_t) {
                best_t = t;
                best = {mt, (int)mb, (int)nb, whole, tiles};
            }
        };
        const int64_t wb = std::min<int64_t>(cus, all);
        take(wb, true, 5.5 + (double)((all + wb - 1) / wb * ns) * step_us(wb));
        // a run of the cut plans: every CU its share, or at least 1 .. 24 steps
        const int64_t cap = std::min<int64_t>(cus, (int64_t)(part_floats / (2 * (size_t)sk::piece(mt))));
        for (int per = 1; per <= 24 && cap >= 1; ++per) {
            const int64_t nb = std::min<int64_t>(cap, (steps + per - 1) / per);
            if (nb <= 1) break;
            const double pieces = (double)nb / (double)all + 1.0;
            take(nb, false, 8.5 + (double)((steps + nb - 1) / nb) * step_us(nb) + 0.35 * pieces);
        }
    }
    return best;
}

int sk_launch(hipStream_t st, const xinfer_fused_desc* descs, int nd, const uint8_t* W2, const uint16_t* S2,
              const void* X, bool y_f32, int64_t M, int64_t K, bool residual) {
    using namespace xhip_host;
    const bool swiglu = W2 != nullptr;
    SkPlan pl = sk_plan(descs, nd, swiglu, M, K, kSkAreaFloats, num_cus());
    SkArea area = {};
    if (!pl.whole && !(area = sk_area(st)).part) pl = sk_plan(descs, nd, swiglu, M, K, 0, num_cus());
    SkParams p = {};
    p.X = reinterpret_cast<const f16*>(X);
    p.part = area.part;
    p.M = (int32_t)M;
    p.K = (int32_t)K;
    p.ng = (int32_t)(K / kGroup);
    const int kw = sk::kwaves(pl.mt);
    p.ns = (p.ng + kw - 1) / kw;
    p.mb = pl.mb;
    p.inv_ns = 1.0f / (float)p.ns;
    p.inv_mb = 1.0f / (float)p.mb;
    p.ndesc = nd;
    p.residual = residual ? 1 : 0;
    for (int i = 0; i < nd; ++i) {
        SkDesc& d = p.d[i];
        d.W = descs[i].W_int4;
        d.S = reinterpret_cast<const uint16_t*>(descs[i].scales);
        d.W2 = W2;
        d.S2 = S2;
        d.bias = descs[i].bias;
        d.Y = descs[i].Y;
        d.N = (int32_t)descs[i].N;
        d.tile_begin = (int32_t)sk_tiles(descs, i, swiglu, pl.mt);
        d.y16 = ((d.N & 7) == 0 && aligned(d.Y, 16)) ? 1 : 0;
    }
    for (int i = nd; i < 4; ++i) p.d[i] = p.d[0];
    p.grain = pl.whole ? p.ns : 1;
    const int64_t grains = pl.tiles * pl.mb * (pl.whole ? 1 : p.ns);
    p.q = (int32_t)(grains / pl.nb);
    p.r = (int32_t)(grains % pl.nb);
    const SkKernels k = swiglu  ? sk_kernels<true, f16>(pl.mt)
                        : y_f32 ? sk_kernels<false, float>(pl.mt)
                                : sk_kernels<false, f16>(pl.mt);
    const int lds = sk::lds_bytes(pl.mt);
    if (!sk_allow_lds(k.main, lds)) return XINFER_ERR_HIP;
    // the two launches of a cut call stay together on the stream
    std::unique_lock<std::mutex> together;
    if (!pl.whole) together = std::unique_lock<std::mutex>(*area.enqueue);
    hipLaunchKernelGGL(k.main, dim3((unsigned)pl.nb), dim3(64 * sk::kWaves), lds, st, p);
    if (int rc = launch_status()) return rc;
    if (pl.whole || (p.r == 0 && p.q % p.ns == 0)) return XINFER_OK;  // every run starts with a tile
    hipLaunchKernelGGL(k.sum, dim3((unsigned)(pl.nb - 1), (unsigned)(sk::colgroups(pl.mt) * pl.mt / 4)), dim3(256), 0,
                       st, p);
    return launch_status();
}

}  // namespace

namespace xhip_host {

// Prefill rows: up to four projections of one X, or one gate/up pair (W2,
// S2).  Every M; shapes were checked by the caller.
int prefill_gemm(hipStream_t st, const xinfer_fused_desc* descs, int nd, const uint8_t* W2, const uint16_t* S2,
                 const void* X, bool y_f32, int64_t M, int64_t K, bool residual) {
    // XINFER_GEMM_EXACT=1: never the kernel that rounds q * s to fp16
    static const bool exact = [] {
        const char* v = getenv("XINFER_GEMM_EXACT");
        return v && *v && atoi(v) != 0;
    }();
    if (!exact && nd == 1 && !y_f32 && !W2) {
        const xinfer_fused_desc& d = descs[0];
        int rc = XINFER_OK;
        if (!gemm_ws_linear(st, d.Y, X, d.W_int4, reinterpret_cast<const uint16_t*>(d.scales), d.bias, M, d.N, K,
                            residual, &rc))
            return rc;
    }
    // Slabs of rows: 32-bit offsets into X and fewer than 2^24 steps
    // (weights are below 4 GiB, so a row block has at most 2^21).
    const int64_t steps = sk_tiles(descs, nd, W2 != nullptr, 1) * (K / kGroup);
    int64_t slab = std::min<int64_t>(((1LL << 32) - 4096) / (2 * K), 32 * (((1LL << 24) - 1) / steps));
    slab = std::min<int64_t>(slab, 1 << 16) / 128 * 128;
    if (slab < 128) slab = 32;
    for (int64_t m0 = 0; m0 < M; m0 += slab) {
        const int64_t mm = std::min<int64_t>(slab, M - m0);
        xinfer_fused_desc part[4];
        for (int i = 0; i < nd; ++i) {
            part[i] = descs[i];
            part[i].Y = reinterpret_cast<char*>(descs[i].Y) + (size_t)m0 * descs[i].N * (y_f32 ? 4 : 2);
        }
        const int rc = sk_launch(st, part, nd, W2, S2, reinterpret_cast<const char*>(X) + (size_t)m0 * K * 2, y_f32, mm, K,
                                 residual);
        if (rc) return rc;
    }
    return XINFER_OK;
}

}  // namespace xhip_host
