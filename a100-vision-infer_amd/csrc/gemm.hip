// Prefill GEMM dispatch.  FP8 weights with K % 256 == 0 run gemm_fp8_kernel
// (gemm_fp8.hpp) or, where its estimate is lower, one tile per workgroup
// (gemm_tile.hip); other K whose rows start on 16 bytes and BF16 weights run
// the tiles, the largest FP8 ones by the template of gemm_kernel.hpp where K %
// 64 == 0, and what is left (unaligned operands, K off the 16-byte grid, 2 GiB
// operands) that template with element-wise loads.
#include <algorithm>
#include <atomic>

#include "../../include/fp8lin.h"
#include "gemm_fp8.hpp"
#include "gemm_kernel.hpp"
#include "internal.hpp"

namespace fp8lin {
namespace {

constexpr int kGroupM = 8;  // XCD-local tile patch height

using Block = gemm::Cfg<256, 256, 64, 2, 4>;

// The template with element-wise loads.
template <bool FP8, bool SWIGLU>
hipError_t run(const uint16_t* x, const void* w, const float* scales, int S, const uint16_t* bias, uint16_t* y,
               int64_t ldy, int M, int N, int K, hipStream_t stream) {
    return gemm::launch<Block, FP8, true, SWIGLU, kGroupM, 1>(x, w, scales, S, bias, y, ldy, M, N, K, stream);
}

// The template with 16-byte loads two K steps ahead, the next stage's
// dequantization and LDS store after the second MFMA group.
template <bool SWIGLU>
hipError_t run_block(const uint16_t* x, const void* w, const float* scales, int S, const uint16_t* bias, uint16_t* y,
                     int64_t ldy, int M, int N, int K, hipStream_t stream) {
    return gemm::launch<Block, true, false, SWIGLU, kGroupM, 1, 2, 1>(x, w, scales, S, bias, y, ldy, M, N, K, stream);
}

// Work plan of the persistent FP8 GEMM (see gemm_fp8.hpp).  Without a
// workspace every tile is computed whole.  With one, K is split where the
// tile count leaves CUs idle:
//  - fewer tiles than half the CUs (e.g. the prefill QKV-gate and down
//    projections at M = 512): every tile, into min(G / T, K / 256, 8)
//    ranges;
//  - otherwise a last round of at most half the CUs (M = 1024: 16 of 272
//    tiles; M = 4096: 64 of 1088; the M = 512 output head: 82 of 594): those
//    tiles, into min(G / R, K / 256, 8) ranges.  A last round over more than
//    half the CUs stays whole: splitting it would not shorten the CUs that
//    run an unsplit tile.
gemm_fp8::Plan plan_for(int bm, int M, int N, int K, bool swiglu, int G, bool split) {
    using namespace gemm_fp8;
    Plan p;
    p.bm = bm;
    p.mtiles = (M + bm - 1) / bm;
    p.ntiles = swiglu ? ((N >> 1) + BN / 2 - 1) / (BN / 2) : (N + BN - 1) / BN;
    const int T = p.mtiles * p.ntiles;
    p.full = T;
    p.rtiles = 0;
    p.splits = 1;
    if (split) {
        const int chunks = K / 256;
        if (2 * T <= G) {
            const int s = std::min(std::min(G / T, chunks), kMaxSplits);
            if (s > 1) {
                p.full = 0;
                p.rtiles = T;
                p.splits = s;
            }
        } else if (T > G && T % G != 0 && 2 * (T % G) <= G) {
            const int R = T % G;
            const int s = std::min(std::min(G / R, chunks), kMaxSplits);
            if (s > 1) {
                p.full = T - R;
                p.rtiles = R;
                p.splits = s;
            }
        }
    }
    p.fpad = (p.full + kXcds - 1) / kXcds * kXcds;
    p.units = p.fpad + p.rtiles * p.splits;
    return p;
}

size_t plan_bytes(const gemm_fp8::Plan& p) {
    return (size_t)p.rtiles * p.splits * p.bm * gemm_fp8::BN * sizeof(float);
}

// The plan of a launch.  M <= 128 (one tile row) takes 128-row tiles: the
// same outputs at half the MFMA work of a 256-row tile that is at least half
// padding.  Above that the 256-row tile stays: measured on MI355X, a 128-row
// tile costs 0.62 (whole chip) to 0.77 (one partial round) of a 256-row tile
// (its K loop issues 4 dequant VALU per MFMA instead of 2, with the same
// per-step waits), so two of them cost more than the one they replace; 192-row
// tiles stand where they pay (route).  Every height gives each output the same
// FP32 sum over a K range.
gemm_fp8::Plan make_plan(int M, int N, int K, bool swiglu, int G, bool split) {
    return plan_for(M <= 128 ? 128 : 256, M, N, K, swiglu, G, split);
}

template <int MT, bool SWIGLU>
hipError_t run_fp8_mt(const uint16_t* x, const uint8_t* w, const float* scales, int S, uint16_t* y, int64_t ldy,
                      int M, int N, int K, const gemm_fp8::Plan& plan, int G, float* part, hipStream_t stream) {
    using namespace gemm_fp8;
    using Gm = Geo<MT>;
    if (!Gm::SPLIT && plan.rtiles != 0) return hipErrorInvalidValue;
    auto kern = gemm_fp8_kernel<MT, SWIGLU>;
    static const hipError_t attr = gemm::allow_lds(reinterpret_cast<const void*>(kern), Gm::LDS_BYTES);
    if (attr != hipSuccess) return attr;
    const int grid = std::min(plan.units, G);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(THREADS), Gm::LDS_BYTES, stream, x, w, scales, S, y, (int)ldy, M, N,
                       K, plan, part);
    hipError_t e = hipGetLastError();
    if constexpr (Gm::SPLIT) {
        if (e != hipSuccess || plan.rtiles == 0) return e;
        const int64_t threads = (int64_t)plan.rtiles * Gm::BM * (SWIGLU ? 32 : 64);
        hipLaunchKernelGGL((tail_reduce_kernel<MT, SWIGLU>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
                           stream, part, plan, M, N, y, ldy);
        e = hipGetLastError();
    }
    return e;
}

template <bool SWIGLU>
hipError_t run_fp8(const uint16_t* x, const uint8_t* w, const float* scales, int S, uint16_t* y, int64_t ldy,
                   int M, int N, int K, const gemm_fp8::Plan& plan, int G, float* part, hipStream_t stream) {
    if (plan.bm == 128) return run_fp8_mt<4, SWIGLU>(x, w, scales, S, y, ldy, M, N, K, plan, G, part, stream);
    if (plan.bm == 192) return run_fp8_mt<6, SWIGLU>(x, w, scales, S, y, ldy, M, N, K, plan, G, part, stream);
    return run_fp8_mt<8, SWIGLU>(x, w, scales, S, y, ldy, M, N, K, plan, G, part, stream);
}

// Shapes and alignments the FP8 kernel takes.
bool fp8_kernel_ok(const uint16_t* x, const void* w, int S, int64_t ldy, int M, int N, int K) {
    return gemm_fp8::supported(x, w, S, ldy, M, N, K);
}

// A few weight rows (N <= kSkinnyRows, as the GDN in_proj_all group's 48 BF16
// rows): 256x256 tiles would run M/256 workgroups, so the skinny MFMA kernel
// takes them (16 x 16 output tiles, K split over 4 waves; skinny.hip), or,
// for K % 32 != 0 or unaligned operands, the GEMV's prefill form (8
// activation rows per workgroup row).  N counts weight rows in both forms, so
// the fused SwiGLU GEMM and the plain GEMM of one weight take the same kernel
// (and give the same sums).
bool skinny(int M, int N, bool /*swiglu*/) { return M > 8 && N <= kSkinnyRows; }

hipError_t launch_skinny(const uint16_t* x, const void* w, const float* scales, int S, uint16_t* y, int64_t ldy,
                         int M, int N, int K, bool swiglu, hipStream_t stream) {
    if (skinny_mfma_supported(x, w, scales != nullptr, S, M, N, K))
        return launch_skinny_mfma(x, w, scales != nullptr, scales, S, y, ldy, M, N, K, swiglu, stream);
    const bool wide = K % 16 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                      reinterpret_cast<uintptr_t>(w) % 16 == 0;
    return launch_gemv_rows(x, w, scales != nullptr, scales, S, y, ldy, M, N, K, wide, swiglu, stream);
}

// 9..16 activation rows of a block-FP8 weight of more than 1024 rows: the
// small-M matrix-core kernels (small_m.hip), whose 16x16 MFMA tile holds all
// of them, stream the codes once with each dequantized once (the wide
// row-staged form up to 64 rows per CU, else the row-range form or the
// K-split 16-row tiles); a GEMM tile would be at least seven eighths
// padding.  17..32 rows in the wide row-staged form with 32 staged
// activation rows (up to 32 weight rows per CU), else in the row-range form
// with two activation tiles (K <= 5120) or the K-split 16-row tiles with two
// activation tiles.  33..64 rows where the row-staged form holds them (64
// staged rows in 256-byte stages, up to 32 weight rows per CU), else the
// GEMM.  Its geometry limits are those of the decode routing (block scales
// [N, K/128], 16-byte aligned x and codes).
bool mid_rows(const uint16_t* x, const void* w, int S, int64_t M, int64_t N, int64_t K) {
    const int64_t lim = (int64_t)1 << 31;
    if (M > 32 && !(M <= 64 && N < lim && K < lim && small_m_wide_rows((int)M, (int)N, (int)K))) return false;
    return M > 8 && N > 1024 && K % 128 == 0 && S == K / 128 &&
           reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 && 16 * K < lim &&
           N * S * 4 < lim && M * K * 2 < lim;
}

}  // namespace

bool gemm_mid_rows(const uint16_t* x, const void* w, int S, int64_t M, int64_t N, int64_t K) {
    return mid_rows(x, w, S, M, N, K);
}

namespace {

// 65..128 rows where both halves are mid rows (narrow weights) and the GEMM
// would run its tiles whole (no split-K workspace): two passes of the small-M
// kernels, each half as a call of its own rows.  Whole tiles run one
// workgroup per 128x256 tile (20 on the 5120-row down projection: 144 us
// against about 50 for the halves); where a workspace lets the GEMM split K
// it stays, being faster (29-38 us there).
bool halves(const uint16_t* x, const void* w, int S, int M, int N, int K) {
    return M > 64 && M <= 128 && mid_rows(x, w, S, M / 2, N, K) && mid_rows(x, w, S, M - M / 2, N, K);
}

hipError_t launch_halves(const uint16_t* x, const uint8_t* codes, const float* scales, uint16_t* y, int64_t ldy,
                         int M, int N, int K, bool swiglu, hipStream_t stream) {
    const int h = M - M / 2;
    const hipError_t e = launch_small_m(x, codes, scales, y, ldy, h, N, K, 1, swiglu, stream);
    if (e != hipSuccess) return e;
    return launch_small_m(x + (int64_t)h * K, codes, scales, y + (int64_t)h * ldy, ldy, M - h, N, K, 1, swiglu,
                          stream);
}

}  // namespace

// Compute units of the current device (cached per device), rounded down to a
// multiple of the 8 XCDs: the persistent kernels' grid size.
int compute_units() {
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int v = cached[dev].load(std::memory_order_relaxed);
    if (v == 0) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 8) cus = 256;
        v = cus / gemm_fp8::kXcds * gemm_fp8::kXcds;
        cached[dev].store(v, std::memory_order_relaxed);
    }
    return v;
}

namespace {

// Estimated us of the persistent FP8 GEMM under plan p, fitted to 1900 calls of
// it with weights from HBM (half of them within 4%, nine tenths within 13%): us
// per 256 K of a round of tiles, which grows with the share of the CUs that run
// one; for each round after the first its fill and drain; and for a split the
// partials' round trip and the second launch.
float estimate(const gemm_fp8::Plan& p, int K, int G) {
    const int chunks = K / 256, rounds = p.full / G;
    const float share = (float)(p.full - rounds * G) / (float)G;
    const float round = p.bm == 128 ? 3.2f : p.bm == 192 ? 5.0f : 6.05f;
    const float last = p.bm == 128   ? 3.3f + 2.0f * std::max(0.0f, share - 0.5f)
                       : p.bm == 192 ? 3.5f + 5.5f * std::max(0.0f, share - 0.66f)
                                     : 4.6f + 4.2f * std::max(0.0f, share - 0.53f);
    float us = 7.2f + (float)chunks * ((float)rounds * round + (share > 0.0f ? last : 0.0f));
    us += 8.0f * (float)std::max(0, rounds + (share > 0.0f) + (p.rtiles > 0) - 1);
    const float c = p.bm == 128 ? 3.4f : p.full >= G ? 5.75f : 5.35f;
    if (p.rtiles > 0)
        us += c * (float)((chunks + p.splits - 1) / p.splits) + 1.15f +
              0.95e-6f * (float)p.rtiles * (float)p.splits * (float)(p.bm * gemm_fp8::BN);
    return us;
}

// How an FP8 call of more than 8 rows that is neither skinny nor mid rows
// runs: the persistent GEMM under `plan`, the tiles under `tile`, or (neither)
// the general template.  have: the bytes of workspace that K-split partials
// may take; a plan that needs more is made without a split.  block: the
// template's 256x256 tiles in the place of gemm_tile.hip's, where K allows and
// they are one round on more than 0.6 of the CUs: 512 x 25088 x 5056 (SwiGLU)
// 135 us against 147, 466 x 25656 x 4224 120 against 130; median of 80 such
// shapes 0.97, and 1.05 on fewer CUs, 1.03 over more rounds.  The persistent
// GEMM's unsplit sums do not depend on the row count or the tile height, and
// the entry points that take no workspace (any false) keep them: there the
// tiles only run the K that it does not.
struct Route {
    bool gemm, tiles, block;
    gemm_fp8::Plan plan;
    TilePlan tile;
};

Route route(const uint16_t* x, const void* w, int S, int64_t ldy, int M, int N, int K, bool swiglu, bool any, size_t have) {
    Route r{fp8_kernel_ok(x, w, S, ldy, M, N, K), false, false, {}, {}};
    const int G = compute_units();
    // 192-row tiles, unsplit, where their round is the cheaper one: 256-row
    // tiles that fill half the CUs to two thirds, or are half padding.  M x N x
    // K without a workspace, 256-row tiles and 192: 512 x 17408 x 5120 91.6 and
    // 87.6 us, 576 x 17408 x 5120 105.3 and 90.0, 300 x 17408 x 5120 87.9 and
    // 72.4, 960 x 10240 x 5120 94.6 and 86.7, 1152 x 8704 x 5120 97.5 and 88.8.
    // The required workspace stays the 256-row plan's.
    auto fitting = [&](bool sw) {
        gemm_fp8::Plan p = make_plan(M, N, K, sw, G, any);
        if (plan_bytes(p) > have) p = make_plan(M, N, K, sw, G, false);
        const gemm_fp8::Plan low = plan_for(192, M, N, K, sw, G, false);
        return p.bm == 256 && estimate(low, K, G) < 0.99f * estimate(p, K, G) ? low : p;
    };
    if (r.gemm) r.plan = fitting(swiglu);
    if (tile_supported(x, w, true, S, M, N, K) && (!r.gemm || any)) {
        r.tile = tile_plan(true, M, N, K, any);
        if (tile_plan_bytes(r.tile, M, N) > have) r.tile = tile_plan(true, M, N, K, false);
        // against the plain form's plan for both epilogues: one route for both
        r.tiles = (!r.gemm || r.tile.us < estimate(fitting(false), K, G));
    }
    if (r.tiles) r.gemm = false;
    const int64_t blocks = (int64_t)((M + 255) / 256) * ((N + 255) / 256);
    r.block = r.tiles && tile_is_block(r.tile) && gemm::aligned(x, w, true, M, N, K) && blocks <= G && 10 * blocks > 6 * G;
    return r;
}

}  // namespace

size_t gemm_split_bytes(int S, int64_t ldy, int M, int N, int K, bool swiglu) {
    if (skinny(M, N, swiglu) || mid_rows(nullptr, nullptr, S, M, N, K) || !fp8_kernel_ok(nullptr, nullptr, S, ldy, M, N, K))
        return 0;
    return plan_bytes(make_plan(M, N, K, swiglu, compute_units(), true));
}

size_t gemm_workspace_bytes(int S, int64_t ldy, int M, int N, int K, bool swiglu) {
    if (skinny(M, N, swiglu) || mid_rows(nullptr, nullptr, S, M, N, K)) return 0;
    const Route r = route(nullptr, nullptr, S, ldy, M, N, K, swiglu, true, SIZE_MAX);
    const size_t gemm = gemm_split_bytes(S, ldy, M, N, K, swiglu);
    return r.tiles ? std::max(gemm, tile_plan_bytes(r.tile, M, N)) : gemm;
}

void gemm_plan(int S, int M, int N, int K, bool split, int& kind, int& bm, int& bn, int& splits, int& slots) {
    bm = bn = splits = slots = 0;
    kind = skinny(M, N, false) ? FP8LIN_GEMM_FEW_ROWS : FP8LIN_GEMM_ELEMENTS;
    if (kind == FP8LIN_GEMM_FEW_ROWS) return;
    if (S == 0) {
        if (!tile_supported(nullptr, nullptr, false, 1, M, N, K)) return;
        kind = FP8LIN_GEMM_TILES;
        splits = 1;
        return tile_shape(tile_plan(false, M, N, K, false), false, bm, bn, slots);
    }
    const Route r = route(nullptr, nullptr, S, N, M, N, K, false, split, split ? SIZE_MAX : 0);
    if (mid_rows(nullptr, nullptr, S, M, N, K) || (r.gemm && r.plan.rtiles == 0 && halves(nullptr, nullptr, S, M, N, K))) {
        kind = FP8LIN_GEMM_SMALL_M;
    } else if (r.tiles) {
        kind = r.block ? FP8LIN_GEMM_BLOCK : FP8LIN_GEMM_TILES;
        splits = r.tile.splits;
        tile_shape(r.tile, true, bm, bn, slots);
    } else if (r.gemm) {
        kind = FP8LIN_GEMM_PERSISTENT;
        bm = r.plan.bm;
        bn = gemm_fp8::BN;
        slots = 1;
        splits = r.plan.rtiles > 0 ? r.plan.splits : 1;
    }
}

hipError_t launch_gemm_ws(const uint16_t* x, const void* w, const float* scales, int S, uint16_t* y, int64_t ldy,
                          int M, int N, int K, bool swiglu, bool may_split, void* ws, size_t ws_bytes,
                          const uint16_t* bias, bool* bias_added, hipStream_t stream) {
    if (skinny(M, N, swiglu)) return launch_skinny(x, w, scales, S, y, ldy, M, N, K, swiglu, stream);
    const uint8_t* codes = static_cast<const uint8_t*>(w);
    if (mid_rows(x, w, S, M, N, K)) return launch_small_m(x, codes, scales, y, ldy, M, N, K, 1, swiglu, stream);
    const size_t have = ws != nullptr && reinterpret_cast<uintptr_t>(ws) % 16 == 0 ? ws_bytes : 0;
    const Route r = route(x, w, S, ldy, M, N, K, swiglu, may_split, have);
    if (r.gemm && r.plan.rtiles == 0 && halves(x, w, S, M, N, K))
        return launch_halves(x, codes, scales, y, ldy, M, N, K, swiglu, stream);
    if (r.block) {
        if (bias) *bias_added = true;
        return swiglu ? run_block<true>(x, w, scales, S, nullptr, y, ldy, M, N, K, stream)
                      : run_block<false>(x, w, scales, S, bias, y, ldy, M, N, K, stream);
    }
    if (r.tiles) {
        if (bias) *bias_added = true;
        return launch_tile(r.tile, true, x, w, scales, S, bias, y, ldy, M, N, K, swiglu, ws, stream);
    }
    if (r.gemm) {
        const int G = compute_units();
        float* part = static_cast<float*>(ws);
        return swiglu ? run_fp8<true>(x, codes, scales, S, y, ldy, M, N, K, r.plan, G, part, stream)
                      : run_fp8<false>(x, codes, scales, S, y, ldy, M, N, K, r.plan, G, part, stream);
    }
    if (bias) *bias_added = true;
    return swiglu ? run<true, true>(x, w, scales, S, nullptr, y, ldy, M, N, K, stream)
                  : run<true, false>(x, w, scales, S, bias, y, ldy, M, N, K, stream);
}

hipError_t launch_gemm_bf16(const uint16_t* x, const uint16_t* w, const uint16_t* bias, uint16_t* y, int64_t ldy, int M,
                            int N, int K, hipStream_t stream) {
    if (!skinny(M, N, false) && tile_supported(x, w, false, 1, M, N, K))
        return launch_tile(tile_plan(false, M, N, K, false), false, x, w, nullptr, 1, bias, y, ldy, M, N, K, false,
                           nullptr, stream);
    if (!skinny(M, N, false)) return run<false, false>(x, w, nullptr, 1, bias, y, ldy, M, N, K, stream);
    const hipError_t e = launch_skinny(x, w, nullptr, 1, y, ldy, M, N, K, false, stream);
    return e != hipSuccess || !bias ? e : launch_bias(y, ldy, bias, M, N, stream);
}

}  // namespace fp8lin
