// Dispatch of the one-tile-per-workgroup GEMM (gemm_tile.hpp): which tile, how
// wide its column blocks are and into how many K ranges it is cut.
#include <algorithm>

#include "gemm_tile.hpp"
#include "internal.hpp"

namespace fp8lin {
namespace {

using gemm_tile::Cfg;
using gemm_tile::Grid;

typedef hipError_t (*LaunchFn)(const uint16_t*, const void*, const float*, int, const uint16_t*, uint16_t*, int64_t,
                               int, int, int, const Grid&, float*, hipStream_t);

// One tile configuration and what a round of workgroups costs: `fixed` us for
// its first loads and last stores, tau for 128 K with the whole chip running
// it, `low` of that with one workgroup alone (`slots` 2: two workgroups per CU,
// tau for both, tau1 where one per CU is enough).
struct Tile {
    int bm, bn, slots;
    float fixed, tau, tau1, low;
    LaunchFn plain, swiglu;
};

template <class C, bool FP8>
constexpr Tile tile(int slots, float fixed, float tau, float tau1, float low) {
    static_assert(C::BM * C::BN != 128 * 128 || C::WK > 1 || 2 * C::LDS_BYTES <= gemm_tile::kLds, "two per CU");
    return {C::BM, C::BN, slots, fixed, tau, tau1, low, gemm_tile::launch<C, false>, FP8 ? gemm_tile::launch<C, FP8> : nullptr};
}

// BF16 weights, M x N x K in us (torch's mm, hipBLASLt, beside it): 1036 x 3456
// x 1152 13.9 (24.5), 1036 x 4304 x 1152 18.1 (21.1), 1036 x 1152 x 4304 28
// (31), 40 x 7168 x 5120 16.5 (22.3), 300 x 5120 x 5120 30.2 (35.8), 4096 x
// 8192 x 8192 447 (355: the library's large tile is the better one).  The
// 256x256-only kernel this replaced took 45, 45, 570 (K % 64 != 0), 156, 168
// and 597.  192x128 and 256x160 stand where 128x128 would need another round
// of workgroups or 256x256 leave CUs idle: 1036 x 4304 x 1152 18.0 (19.7
// without them), 1036 x 5120 x 5120 60 (76), 2048 x 4304 x 1152 28.5 (34.2),
// 2048 x 5120 x 5120 101 (124), 4096 x 5120 x 5120 203 (236).
// E4M3FN codes, M x N x K in us (the persistent GEMM without these tiles or,
// at K % 256, the general template): 93 x 17408 x 5120 36.8 (38.8), 93 x 5120 x
// 8704 21.6 (28.5), 200 x 7168 x 5120 29.2 (37.1), 512 x 2048 x 2048 10.8
// (26.1), 320 x 5120 x 3072 20.6 (33.7), 128 x 6000 x 1152 8.1 (18.8), 128 x
// 5000 x 4304 18.4 (581, byte loads), row scales 27 x 8192 x 5120 14.1 (56.5).
// What bounds them: at 128 rows or fewer the activations, which every
// workgroup reads in full, share its 64 B/clk of DMA with the codes that come
// from HBM (about 40 KB/us per CU against 29 for codes alone); above, LDS
// reads and MFMA issue that one barrier per step does not let overlap fully.
// Small tiles split a step's K over the waves of the workgroup, so that a
// wave's tile stays deep enough for its LDS reads; FP8 tiles keep WM = 1 up
// to 128 rows, where every code is dequantized once.
// The FP8 constants are fitted to 40000 timed calls of every tile at M 9..4096,
// N 257..34816, K 256..13696, weights from HBM, with 3 us for a split's second
// launch (4 in the estimate: calls this short are bound by the host, which it
// costs as much again) and 0.8e-6 us per partial.  Four fifths of the estimates
// are within 12%; the tile that they pick is 0.7% slower than the fastest one
// timed, in one call of a hundred by more than 11% (2.9% and 50% with constants
// taken from one shape per tile).
const Tile kBf16[] = {
    tile<Cfg<false, 32, 32, 1, 1, 4, 128, 6, false>, false>(1, 2.1f, 0.25f, 0.25f, 0.65f),
    tile<Cfg<false, 64, 32, 1, 1, 4, 128, 3, false>, false>(1, 2.2f, 0.39f, 0.39f, 0.65f),
    tile<Cfg<false, 64, 64, 1, 2, 4, 128, 3, false>, false>(1, 2.4f, 0.49f, 0.49f, 0.65f),
    tile<Cfg<false, 128, 64, 2, 1, 4, 128, 3, false>, false>(1, 2.75f, 0.68f, 0.68f, 0.65f),
    tile<Cfg<false, 128, 128, 2, 2, 2, 64, 4, true>, false>(1, 3.5f, 0.98f, 0.98f, 0.65f),
    tile<Cfg<false, 128, 128, 2, 2, 1, 64, 2, false>, false>(2, 3.5f, 1.80f, 1.15f, 0.65f),
    tile<Cfg<false, 192, 128, 2, 2, 2, 64, 4, true>, false>(1, 4.25f, 1.33f, 1.33f, 0.65f),
    tile<Cfg<false, 256, 160, 4, 1, 1, 64, 3, true>, false>(1, 5.75f, 2.35f, 2.35f, 0.65f),
    tile<Cfg<false, 256, 256, 2, 4, 1, 64, 2, false>, false>(1, 8.0f, 3.10f, 3.10f, 0.65f),
};
const Tile kFp8[] = {
    tile<Cfg<true, 32, 32, 1, 1, 4, 128, 8, false>, true>(1, 1.95f, 0.28f, 0.28f, 0.77f),
    tile<Cfg<true, 64, 32, 1, 1, 4, 128, 4, false>, true>(1, 2.85f, 0.35f, 0.35f, 0.77f),
    tile<Cfg<true, 64, 64, 1, 2, 4, 128, 4, false>, true>(1, 2.75f, 0.44f, 0.44f, 0.68f),
    tile<Cfg<true, 96, 64, 1, 2, 4, 128, 4, false>, true>(1, 3.55f, 0.54f, 0.54f, 0.66f),
    tile<Cfg<true, 128, 64, 1, 2, 4, 128, 3, false>, true>(1, 4.0f, 0.68f, 0.68f, 0.66f),
    tile<Cfg<true, 64, 128, 1, 2, 4, 128, 4, false>, true>(1, 4.15f, 0.70f, 0.70f, 0.64f),
    tile<Cfg<true, 96, 192, 1, 6, 2, 64, 5, true>, true>(1, 4.05f, 1.34f, 1.34f, 0.53f),
    tile<Cfg<true, 128, 128, 1, 4, 2, 64, 5, true>, true>(1, 3.95f, 1.19f, 1.19f, 0.57f),
    tile<Cfg<true, 128, 128, 1, 4, 1, 64, 2, false>, true>(2, 2.15f, 2.02f, 1.66f, 0.66f),
    tile<Cfg<true, 256, 256, 2, 4, 1, 64, 2, false>, true>(1, 5.05f, 4.11f, 4.11f, 0.55f),
};
constexpr int kMaxTileSplits = 8;

int ceil_div(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }

// Microseconds of tile t over M x N x K in `splits` K ranges: per round of
// workgroups its fixed part and its steps, whose time grows with the share of
// the chip that runs them, and for a split the partials written and read back
// and the second launch.
float estimate(const Tile& t, int M, int N, int K, int splits, int cus) {
    const int64_t units = (int64_t)ceil_div(M, t.bm) * ceil_div(N, t.bn) * splits;
    const float steps = (float)ceil_div(ceil_div(K, 128), splits);
    const int64_t whole = units / ((int64_t)cus * t.slots), rest = units - whole * cus * t.slots;
    float us = 2.0f + (float)whole * (t.fixed + steps * t.tau);
    if (rest > cus)
        us += t.fixed + steps * t.tau;
    else if (rest > 0)
        us += t.fixed + steps * t.tau1 * (t.low + (1.0f - t.low) * (float)rest / (float)cus);
    return splits == 1 ? us : us + 4.0f + 0.8e-6f * (float)splits * (float)M * (float)N;
}

const Tile& tile_of(bool fp8, int i) { return fp8 ? kFp8[i] : kBf16[i]; }

Grid grid_of(const Tile& t, int M, int N, int64_t ldy, const uint16_t* y, const uint16_t* bias, int splits, bool swiglu,
             int cus) {
    Grid g;
    g.mtiles = ceil_div(M, t.bm);
    g.nblocks = ceil_div(N, t.bn);
    g.splits = splits;
    g.group_m = 8;
    g.ldp = ceil_div(N, 8) * 8 + 8;
    g.wide = (ldy % 8 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0 ? 1 : 0) |
             (ldy % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 8 == 0 ? 4 : 0) |
             (ldy % 2 == 0 && reinterpret_cast<uintptr_t>(y) % 4 == 0 ? 8 : 0) |
             (reinterpret_cast<uintptr_t>(bias) % 16 == 0 ? 2 : 0);
    // One round: spread the columns evenly over the CUs.
    g.per = t.bn;
    const int fit = cus / (g.mtiles * splits);
    if (fit >= g.nblocks) {
        g.per = std::min(t.bn, ceil_div(ceil_div(N, fit), 16) * 16);
        g.nblocks = ceil_div(N, g.per);
    }
    if (swiglu && splits == 1) g.per /= 2;
    return g;
}

}  // namespace

bool tile_supported(const uint16_t* x, const void* w, bool fp8, int S, int64_t M, int64_t N, int64_t K) {
    const int64_t lim = (int64_t)1 << 31;
    return M > 0 && K % (fp8 ? 16 : 8) == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(w) % 16 == 0 && N * K * (fp8 ? 1 : 2) < lim && 256 * K * 2 < lim &&
           N + 16 < lim / 8 && M < lim / 8 && (!fp8 || S == 1 || S == (K + 127) / 128);
}

// The plan with the smallest estimate.  It depends on M, N, K and whether a
// split may be taken, not on the epilogue, so that the SwiGLU form sums as the
// plain one.
TilePlan tile_plan(bool fp8, int M, int N, int K, bool may_split) {
    const int cus = compute_units(), count = fp8 ? (int)(sizeof(kFp8) / sizeof(Tile)) : (int)(sizeof(kBf16) / sizeof(Tile));
    TilePlan best{-1, 1, 0.0f};
    for (int i = 0; i < count; ++i) {
        const Tile& t = tile_of(fp8, i);
        const int64_t tiles = (int64_t)ceil_div(M, t.bm) * ceil_div(N, t.bn);
        const int most = may_split ? std::min(kMaxTileSplits, ceil_div(K, 128)) : 1;
        for (int s = 1; s <= most && (s == 1 || tiles * s <= cus); ++s) {
            const float us = estimate(t, M, N, K, s, cus);
            if (best.cfg < 0 || us < best.us) best = {i, s, us};
        }
    }
    return best;
}

bool tile_is_block(const TilePlan& p) { return p.splits == 1 && kFp8[p.cfg].bm == 256 && kFp8[p.cfg].bn == 256; }

void tile_shape(const TilePlan& p, bool fp8, int& bm, int& bn, int& slots) {
    slots = tile_of(fp8, p.cfg).slots;
    bm = tile_of(fp8, p.cfg).bm;
    bn = tile_of(fp8, p.cfg).bn;
}

size_t tile_plan_bytes(const TilePlan& p, int M, int N) {
    return p.splits <= 1 ? 0 : (size_t)p.splits * M * (ceil_div(N, 8) * 8 + 8) * sizeof(float);
}

hipError_t launch_tile(const TilePlan& p, bool fp8, const uint16_t* x, const void* w, const float* scales, int S,
                       const uint16_t* bias, uint16_t* y, int64_t ldy, int M, int N, int K, bool swiglu, void* ws,
                       hipStream_t stream) {
    const Tile& t = tile_of(fp8, p.cfg);
    const Grid g = grid_of(t, M, N, ldy, y, bias, p.splits, swiglu, compute_units());
    float* part = static_cast<float*>(ws);
    if (p.splits == 1) return (swiglu ? t.swiglu : t.plain)(x, w, scales, S, bias, y, ldy, M, N, K, g, nullptr, stream);
    const hipError_t e = t.plain(x, w, scales, S, nullptr, y, ldy, M, N, K, g, part, stream);
    if (e != hipSuccess) return e;
    const int64_t threads = (int64_t)M * ceil_div(swiglu ? N >> 1 : N, 8);
    const dim3 grid((unsigned)((threads + 255) / 256));
    auto reduce = [&]<int SPLITS>() {
        if (swiglu)
            hipLaunchKernelGGL((gemm_tile::split_reduce_kernel<true, SPLITS>), grid, dim3(256), 0, stream, part, g.ldp, bias, y,
                               ldy, M, N, g.wide);
        else
            hipLaunchKernelGGL((gemm_tile::split_reduce_kernel<false, SPLITS>), grid, dim3(256), 0, stream, part, g.ldp, bias, y,
                               ldy, M, N, g.wide);
    };
    static_assert(kMaxTileSplits == 8, "a reduce for every number of ranges");
    switch (p.splits) {
        case 2: reduce.operator()<2>(); break;
        case 3: reduce.operator()<3>(); break;
        case 4: reduce.operator()<4>(); break;
        case 5: reduce.operator()<5>(); break;
        case 6: reduce.operator()<6>(); break;
        case 7: reduce.operator()<7>(); break;
        default: reduce.operator()<8>(); break;
    }
    return hipGetLastError();
}

}  // namespace fp8lin
