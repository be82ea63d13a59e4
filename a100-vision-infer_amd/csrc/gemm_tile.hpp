// GEMM over one output tile per workgroup: y[M,N] = x[M,K] * W^T (+ bias) on
// the BF16 matrix cores, W as BF16 or as E4M3FN codes with FP32 scales (per
// row or per 128-K block), any K whose rows start on 16 bytes.
//
// Orientation: the weights are the MFMA's A operand and the activations its B
// operand, so a lane's 16 accumulator values are outputs of one activation
// row.  Weight row n of a 32-row fragment sits at fragment row i(n) with
// n = 16 h + 4 q + t for i = 8 q + 4 h + t, which makes the 16 values
// consecutive columns: two 16-byte stores per fragment.
//
// A workgroup of WM x WN x WK waves computes a BM x BN tile; a wave owns
// (BM / WM) x (BN / WN) of it as 32x32 accumulators, over every WK-th 32-K
// slice of a step (WK > 1: the WK partial tiles are added in LDS in wave
// order at the end).  Splitting K over waves instead of splitting the tile
// keeps the wave's tile, and with it the LDS reads per MFMA, while a second
// wave per SIMD hides the first one's LDS and barrier waits; with WM == 1 it
// also dequantizes every FP8 code once per workgroup.
//
// Data movement: BK of K per step through a ring of ST stages, filled by
// direct-to-LDS DMA ST - 1 steps ahead, one wait and one barrier per step.
// The 16-byte chunks of a row are XOR-swizzled so that the 16 rows of a
// fragment read fall in distinct LDS banks.  K is cut in 16-byte chunks:
// chunks at or past K, rows past M and weight rows past N read zeros, and
// every step issues the same number of DMAs, so the waits are fixed numbers.
#pragma once
#include "device.hpp"
#include "gemm_fp8.hpp"

namespace fp8lin {
namespace gemm_tile {

using gemm_fp8::dma16;
using gemm_fp8::i32x4;
using gemm_fp8::make_desc;

constexpr int kLds = 160 * 1024;

// PIPE: the next slice's fragments are read (and dequantized) into a second
// register set while the current ones are multiplied; stage t + 1 must then
// have landed before step t, one stage less in flight.  It gains 5-8% where a
// step has enough MFMAs to cover the reads (128 x 128 tiles at ST >= 4) and
// loses a few percent on small tiles, and on tiles that only fit two stages.
template <bool FP8_, int BM_, int BN_, int WM_, int WN_, int WK_, int BK_, int ST_, bool PIPE_>
struct Cfg {
    static constexpr bool PIPE = PIPE_;
    static constexpr bool FP8 = FP8_;
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, WK = WK_, BK = BK_, ST = ST_;
    static constexpr int WAVES = WM * WN * WK, THREADS = 64 * WAVES;
    static constexpr int MT = BM / WM / 32, NT = BN / WN / 32;  // 32x32 accumulators per wave
    static constexpr int XROW = 2 * BK, WROW = FP8 ? BK : 2 * BK;  // LDS row bytes of a stage
    static constexpr int X_STAGE = BM * XROW, W_STAGE = BN * WROW, STAGE = X_STAGE + W_STAGE;
    static constexpr int XD = X_STAGE / 1024 / WAVES, WD = W_STAGE / 1024 / WAVES;  // DMAs per wave and step
    static constexpr int ND = XD + WD;
    static constexpr int RING = ST * STAGE;
    static constexpr int SLICES = BK / 32;  // 32-K slices (two MFMAs deep) of a step
    static_assert(BK == 64 || BK == 128, "steps of half a 128-K block or a whole one");
    static_assert(ST >= (PIPE ? 3 : 2), "a stage in flight beside the ones read");
    static_assert(BM % (32 * WM) == 0 && BN % (32 * WN) == 0 && SLICES % WK == 0, "wave tile");
    static_assert(X_STAGE % (1024 * WAVES) == 0 && W_STAGE % (1024 * WAVES) == 0, "equal DMA shares");
    static_assert(WK == 1 || BM * BN * 4 <= RING, "a partial tile fits the ring");
    static_assert(RING <= kLds, "LDS");
    // Waves per SIMD to leave registers for: a workgroup's own, or as many as the
    // 128x128 FP8 tile of four waves has in LDS (two of them: 10% slower).
    static constexpr int EU = FP8 && WAVES == 4 && RING <= kLds / 3 ? kLds / RING : (WAVES + 3) / 4;
    // FP8: the rows' scales, in two windows of SWB 128-K blocks beside the ring:
    // while the SPW steps of one run, SQ DMAs a wave fill the other.  Scales of
    // the whole K in LDS left no room for the large tiles at K above 8064
    // (256x256): 1016 x 29884 x 11392 took 1074 us in smaller ones, 634 in 256x256.
    // A DMA's 256 bytes hold 64 / SWB rows; the next ones start on another bank,
    // so that 32 rows at one block fall in distinct banks.
    static constexpr int SWB = BK == 128 ? 8 : 4, SPW = SWB * 128 / BK, SQ = FP8 ? BN * SWB / 64 / WAVES : 0;
    static constexpr int SCHUNK = 260, SWIN = BN * SWB / 64 * SCHUNK;
    static constexpr int LDS_BYTES = RING + (FP8 ? 2 * SWIN : 0);
    static_assert(!FP8 || BN * SWB % (64 * WAVES) == 0, "equal scale DMA shares");
    static_assert(ST <= SPW && SPW % 2 == 0, "a window's scales, issued in the one before, land before its first step");
    static_assert(LDS_BYTES <= kLds, "LDS");
    // Output rows off the 16-byte grid go through LDS (store_staged), in the part
    // of the ring that each wave then has to itself; 4 is rows on 8 bytes, which
    // the smaller tiles store as they are.  Lane's own rows and staged, us: 512 x
    // 15137 x 1152 45.8 and 24.5, 2048 x 562 x 1152 14.8 and 12.2, 1036 x 625 x
    // 1152 (FP8) 11.5 and 9.2; on 8 bytes 2048 x 9740 x 1152 66.5 and 58.9 (large
    // tiles), 40 x 11004 x 1152 7.5 and 8.0 (64x64).
    static constexpr bool STAGED = BM * BN >= 64 * 64;
    static constexpr int DIRECT = BM * BN >= 128 * 128 ? 1 : 1 | 4;
    static constexpr int STORE_BYTES = WK > 1 ? MT * NT * 4096 : 32 * (NT * 64 + 16);
    static_assert(!STAGED || (STORE_BYTES >= 32 * (NT * 64 + 16) && WM * WN * STORE_BYTES <= RING), "32 rows of a wave's tile");
};

// o = bf16(y + bias) of eight rounded outputs from column c on, as the separate
// bias kernel adds it; wide: eight bias values in one load where all are below lim.
__device__ __forceinline__ void add_bias8(uint32_t* o, const uint16_t* __restrict__ bias, int c, int lim, bool wide) {
    uint32_t v[4];
    if (wide && c + 8 <= lim) {
        const u32x4 q = load_u32x4(bias + c);
        v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            v[r] = (c + 2 * r < lim ? (uint32_t)bias[c + 2 * r] : 0u) |
                   (c + 2 * r + 1 < lim ? (uint32_t)bias[c + 2 * r + 1] << 16 : 0u);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        o[r] = pack_bf16x2(f32x2{bf16_bits_to_f32(o[r] & 0xffffu) + bf16_bits_to_f32(v[r] & 0xffffu),
                                 bf16_bits_to_f32(o[r] >> 16) + bf16_bits_to_f32(v[r] >> 16)});
}

// The first `left` (at most eight) of the outputs o to dst, in the widest
// stores that dst's alignment allows (Grid::wide).
__device__ __forceinline__ void store8(uint16_t* dst, const uint32_t* o, int left, int wide) {
    if ((wide & 1) && left >= 8) {
        *reinterpret_cast<u32x4*>(dst) = u32x4{o[0], o[1], o[2], o[3]};
        return;
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        if ((wide & 4) && left >= 4 * q + 4) {
            *reinterpret_cast<u32x2*>(dst + 4 * q) = u32x2{o[2 * q], o[2 * q + 1]};
        } else {
#pragma unroll
            for (int r = 4 * q; r < 4 * q + 4; ++r)
                if (r < left) dst[r] = (uint16_t)(o[r >> 1] >> (16 * (r & 1)));
        }
    }
}

// The first `left` of COLS columns and `rows` of 32 rows that the wave has just
// put in LDS (rows of 2 COLS + 16 bytes) to dst, E outputs a lane, neighbouring
// lanes on neighbouring outputs.  Where y's rows start off the 16-byte grid a
// lane's own row in narrow stores touches a cache line per lane and store.  The
// reads of a batch are all under way before its first store.
template <int E, int COLS>
__device__ __forceinline__ void store_staged(uint16_t* dst, int64_t ldy, const uint8_t* stage, int rows, int left) {
    typedef uint16_t Out __attribute__((ext_vector_type(E)));
    constexpr int LPR = COLS / E, ITER = LPR / 2;  // lanes a row, instructions
    constexpr int B = ITER % 8 == 0 ? 8 : ITER % 4 == 0 ? 4 : 2;  // of a batch
    static_assert(ITER % B == 0, "whole batches");
    const int lane = threadIdx.x & 63;
    asm volatile("" ::: "memory");  // the other lanes' rows, in the wave's own order
#pragma unroll 1
    for (int p0 = 0; p0 < ITER; p0 += B) {
        Out v[B];
#pragma unroll
        for (int p = 0; p < B; ++p) {
            const int id = (p0 + p) * 64 + lane;
            v[p] = *reinterpret_cast<const Out*>(stage + id / LPR * (2 * COLS + 16) + 2 * E * (id % LPR));
        }
#pragma unroll
        for (int p = 0; p < B; ++p) {
            const int id = (p0 + p) * 64 + lane, r = id / LPR, c = id % LPR * E;
            uint16_t* out = dst + (int64_t)r * ldy + c;
            if (r < rows && c + E <= left) {
                *reinterpret_cast<Out*>(out) = v[p];
            } else if (r < rows) {
#pragma unroll
                for (int e = 0; e + 1 < E; ++e)
                    if (c + e < left) out[e] = v[p][e];
            }
        }
    }
    asm volatile("" ::: "memory");
}

// Position of chunk ch of row r in a row of CH chunks.
template <int CH>
__device__ __forceinline__ int swz(int r, int ch) {
    if constexpr (CH == 16) return ch ^ (r & 15);
    if constexpr (CH == 8) return ch ^ gemm_fp8::ga(r);
    return ch ^ gemm_fp8::gb(r);
}

// Column of fragment row i (0..31) in its 32-column block (see the header).
__device__ __forceinline__ int frag_col(int i) { return 16 * ((i >> 2) & 1) + 4 * (i >> 3) + (i & 3); }

// Waits until at most N of the wave's DMAs are in flight and its LDS reads are
// done, then for the workgroup.
template <int N>
__device__ __forceinline__ void wait_vm_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(N) : "memory");
}

// 64 lanes x 4 B from global (voff + soff, bounds-checked) into LDS
// [m0v, m0v + 256), lane l at m0v + 4 l.
__device__ __forceinline__ void dma4(uint32_t m0v, uint32_t voff, i32x4 desc, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 ::"s"(m0v), "v"(voff), "s"(desc), "s"(soff) : "memory", "m0");
}

// 16-byte chunk at LDS byte address a.
__device__ __forceinline__ u32x4 lds16(uint32_t a) {
    return *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>((uintptr_t)a);
}

__device__ __forceinline__ float lds4(uint32_t a) {
    return *reinterpret_cast<const __attribute__((address_space(3))) float*>((uintptr_t)a);
}

// Weight row of tile row b (fragment order) of the column block that starts at
// row (SWIGLU: output) n0 and holds `per` of them, or -1.  SWIGLU: the 32 rows
// of a fragment are 16 outputs; lane half h's 16 values are the gates of
// outputs 8 h + [0, 8), then their ups.
template <bool SWIGLU>
__device__ __forceinline__ int64_t weight_row(int n0, int per, int b, int N) {
    const int c = frag_col(b & 31);
    if constexpr (SWIGLU) {
        const int D = N >> 1, r = (b >> 5) * 16 + 8 * (c >> 4) + (c & 7), o = n0 + r;
        return r < per && o < D ? ((c & 8) ? (int64_t)D + o : (int64_t)o) : -1;
    } else {
        const int r = (b & ~31) + c;
        return r < per && n0 + r < N ? (int64_t)n0 + r : -1;
    }
}

// Work of one launch: column blocks of `per` outputs (SWIGLU: output pairs),
// at most a tile's width, and `splits` K ranges of whole steps each, whose
// FP32 sums go to part[split][M][ldp] for split_reduce_kernel.  per below the
// tile's width lets the blocks match the CU count; the rows past it cost no
// memory traffic.
struct Grid {
    int mtiles, nblocks, per, splits;
    int group_m;  // tile rows walked together (x and W rows shared in an XCD's L2)
    int ldp;      // row stride of the partials
    int wide;     // y's rows start on 16 bytes (1), 8 (4) or 4 (8); bias on 16 (2)
};

// Requirements (checked by the launcher): x, w 16-byte aligned; K % 8 == 0
// (BF16) or K % 16 == 0 (FP8); BM * K * 2 and N * K * (FP8 ? 1 : 2) below
// 2^31; S == 1 or ceil(K / 128); per % 8 == 0 and per <= BN (SWIGLU: BN / 2).
// With SWIGLU, N counts weight rows and y is [M, N/2].
template <class C, bool SWIGLU>
__global__ __launch_bounds__(C::THREADS, C::EU) void gemm_tile_kernel(const uint16_t* __restrict__ x, const void* __restrict__ w,
                                                               const float* __restrict__ scales, int S,
                                                               const uint16_t* __restrict__ bias,
                                                               uint16_t* __restrict__ y, int64_t ldy, int M, int N, int K,
                                                               Grid gr, float* __restrict__ part) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr int CHX = C::BK / 8, CHW = C::FP8 ? C::BK / 16 : C::BK / 8;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = lane >> 5, l32 = lane & 31;
    const int wk = wave / (C::WM * C::WN), wm = wave / C::WN % C::WM, wn = wave % C::WN;
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

    // Unit of this workgroup: each XCD (workgroup % 8) takes a contiguous run
    // of the units (split, tile), a split's tiles walked group_m tile rows at
    // a time, so that the tiles an XCD runs together share x and W rows in
    // its L2.
    const int tiles = gr.mtiles * gr.nblocks, units = tiles * gr.splits;
    const int per_xcd = (units + 7) / 8;
    const int u = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= per_xcd || u >= units) return;
    const int split = u / tiles, L = u - split * tiles;
    const int per_group = gr.group_m * gr.nblocks, g = L / per_group;
    const int gsize = min(gr.group_m, gr.mtiles - g * gr.group_m), rem = L - g * per_group;
    const int m0 = (g * gr.group_m + rem % gsize) * C::BM, n0 = rem / gsize * gr.per;
    const int ksteps = (K + C::BK - 1) / C::BK;
    const int t0 = (int)((int64_t)ksteps * split / gr.splits), KT = (int)((int64_t)ksteps * (split + 1) / gr.splits) - t0;

    const int rows = min(C::BM, M - m0);
    const i32x4 dx = make_desc(x + (int64_t)m0 * K, (uint32_t)((int64_t)rows * K * 2));
    const i32x4 dw = make_desc(w, (uint32_t)((int64_t)N * K * (C::FP8 ? 1 : 2)));

    // DMA d of this wave fills 1 KiB of a stage: lane -> byte 16 * lane of it.
    uint32_t xoff[C::XD], woff[C::WD];
    int xk[C::XD], wk0[C::WD];  // first K of the lane's chunk within a step
#pragma unroll
    for (int d = 0; d < C::XD; ++d) {
        const int q = (wave * C::XD + d) * 64 + lane, r = q / CHX, ch = swz<CHX>(r, q % CHX);
        xk[d] = 8 * ch;
        xoff[d] = r < rows ? (uint32_t)(r * K * 2 + ch * 16) : kBufferOob;
    }
#pragma unroll
    for (int d = 0; d < C::WD; ++d) {
        const int q = (wave * C::WD + d) * 64 + lane, r = q / CHW, ch = swz<CHW>(r, q % CHW);
        const int64_t n = weight_row<SWIGLU>(n0, gr.per, r, N);
        wk0[d] = (C::FP8 ? 16 : 8) * ch;
        woff[d] = n >= 0 ? (uint32_t)(n * K * (C::FP8 ? 1 : 2) + ch * 16) : kBufferOob;
    }
    const uint32_t m0x = __builtin_amdgcn_readfirstlane(lds0 + wave * C::XD * 1024);
    const uint32_t m0w = __builtin_amdgcn_readfirstlane(lds0 + C::X_STAGE + wave * C::WD * 1024);
    // FP8: scale DMA q of this wave fills 64 / SWB rows of a window: lane l ->
    // row l / SWB, block l % SWB.  The range's step 0 is step tt0 of window 0.
    // Row scales are block 0 of window 0, which nothing overwrites.
    const int kb0 = S == 1 ? 0 : (t0 * C::BK) >> 7, tt0 = t0 % (128 / C::BK);
    const i32x4 ds = make_desc(scales, C::FP8 ? (uint32_t)((int64_t)N * S * 4) : 0u);
    uint32_t soff[C::FP8 ? C::SQ : 1];
    const int sblk = kb0 + lane % C::SWB;
    const uint32_t m0s = __builtin_amdgcn_readfirstlane(lds0 + C::RING + wave * C::SQ * C::SCHUNK);
    auto scale_window = [&](int wd) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < C::SQ; ++q)
            dma4(m0s + (wd & 1) * C::SWIN + q * C::SCHUNK, sblk + wd * C::SWB < S ? soff[q] + (uint32_t)(wd * C::SWB * 4) : kBufferOob, ds, 0);
    };
    auto issue = [&](int t, uint32_t slot) __attribute__((always_inline)) {
        // past the range's last step: nothing (the same number of DMAs)
        const int k = (t0 + t) * C::BK, kend = t < KT ? K : 0;
#pragma unroll
        for (int d = 0; d < C::XD; ++d)
            dma16(m0x + slot + d * 1024, k + xk[d] < kend ? xoff[d] : kBufferOob, dx, k * 2);
#pragma unroll
        for (int d = 0; d < C::WD; ++d)
            dma16(m0w + slot + d * 1024, k + wk0[d] < kend ? woff[d] : kBufferOob, dw, C::FP8 ? k : k * 2);
    };
    if constexpr (C::FP8) {
#pragma unroll
        for (int q = 0; q < C::SQ; ++q) {
            const int64_t n = weight_row<SWIGLU>(n0, gr.per, (wave * C::SQ + q) * (64 / C::SWB) + lane / C::SWB, N);
            soff[q] = n >= 0 ? (uint32_t)((n * S + sblk) * 4) : kBufferOob;
        }
        scale_window(0);
    }
#pragma unroll
    for (int p = 0; p < C::ST - 1; ++p) issue(p, p * C::STAGE);

    f32x16 acc[C::MT][C::NT];
#pragma unroll
    for (int i = 0; i < C::MT; ++i)
#pragma unroll
        for (int j = 0; j < C::NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    // Fragment row bases; the swizzle of a row depends on the row mod 16 only.
    const uint32_t xrow = lds0 + (wm * (C::BM / C::WM) + l32) * C::XROW;
    const uint32_t wrow = lds0 + C::X_STAGE + (wn * (C::BN / C::WN) + l32) * C::WROW;
    const uint32_t srow = lds0 + C::RING + l32 / (64 / C::SWB) * C::SCHUNK + l32 % (64 / C::SWB) * C::SWB * 4 +
                          wn * (C::BN / C::WN / 32) * (C::SWB / 2) * C::SCHUNK;
    // A slice of 32 K: lane half h holds K [16 h, 16 h + 16) of it, its first
    // 8 in the first MFMA and the rest in the second, for x and W alike.
    constexpr int SETS = C::PIPE ? 2 : 1;
    u32x4 a[SETS][C::NT][2], b[SETS][C::MT][2], raw[C::NT];
    float scl[C::NT];
    const int klim = K - 16 * h;
    // Byte offset of step t's scale block in the windows.
    auto scale_at = [&](int t) __attribute__((always_inline)) {
        const uint32_t kb = S == 1 ? 0u : (uint32_t)(t + tt0) * C::BK / 128;  // block within the range
        return (kb / C::SWB & 1) * C::SWIN + kb % C::SWB * 4;
    };
    // MASK: K may end in this step.  sa: scale_at(t), worked out a step ahead, and
    // the scales are read first: the conversions wait for them.
    auto fetch = [&]<bool MASK>(int set, uint32_t stage, int s, int t, uint32_t sa) __attribute__((always_inline)) {
        if constexpr (C::FP8) {
#pragma unroll
            for (int j = 0; j < C::NT; ++j) {
                scl[j] = lds4(srow + sa + j * (C::SWB / 2) * C::SCHUNK);
                raw[j] = lds16(wrow + stage + j * 32 * C::WROW + 16 * swz<CHW>(l32, 2 * s + h));
                // a chunk past K holds zero codes; its scale must be zero too (0 * inf)
                if constexpr (MASK) scl[j] = (t0 + t) * C::BK + 32 * s < klim ? scl[j] : 0.0f;
            }
        } else {
#pragma unroll
            for (int j = 0; j < C::NT; ++j)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    a[set][j][e] = lds16(wrow + stage + j * 32 * C::WROW + 16 * swz<CHW>(l32, 4 * s + 2 * h + e));
        }
#pragma unroll
        for (int i = 0; i < C::MT; ++i)
#pragma unroll
            for (int e = 0; e < 2; ++e)
                b[set][i][e] = lds16(xrow + stage + i * 32 * C::XROW + 16 * swz<CHX>(l32, 4 * s + 2 * h + e));
    };
    auto convert = [&](int set) __attribute__((always_inline)) {
        if constexpr (C::FP8) {
#pragma unroll
            for (int j = 0; j < C::NT; ++j) {
                uint32_t o[8];
                dequant4(raw[j].x, scl[j], o[0], o[1]);
                dequant4(raw[j].y, scl[j], o[2], o[3]);
                dequant4(raw[j].z, scl[j], o[4], o[5]);
                dequant4(raw[j].w, scl[j], o[6], o[7]);
                a[set][j][0] = u32x4{o[0], o[1], o[2], o[3]};
                a[set][j][1] = u32x4{o[4], o[5], o[6], o[7]};
            }
        }
    };
    auto multiply = [&](int set) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int i = 0; i < C::MT; ++i)
#pragma unroll
                for (int j = 0; j < C::NT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[set][j][e]),
                                                                        __builtin_bit_cast(bf16x8, b[set][i][e]),
                                                                        acc[i][j], 0, 0, 0);
    };
    constexpr int SL = C::SLICES / C::WK;  // slices of a wave per step
    uint32_t sa = C::FP8 ? scale_at(0) : 0u, sn = C::FP8 ? scale_at(1) : 0u;  // of this step and the next
    uint32_t rd = 0, nx = C::STAGE, wr = (C::ST - 1) * C::STAGE;
    auto next = [&](uint32_t v) __attribute__((always_inline)) { return v == (C::ST - 1) * C::STAGE ? 0u : v + C::STAGE; };
    // Steps that need no mask (PIPE: step t also fetches from step t + 1).
    const int plain = C::FP8 && (t0 + KT) * C::BK > K ? max(KT - (C::PIPE ? 2 : 1), 0) : KT;
    // Runs body(first, last) over the steps [0, plain), with window w + 1's
    // scale DMAs between two of them: behind the barrier of window w's first
    // step, where every wave is done with window w - 1.  (Asked for in every
    // step, the same DMAs cost the loop 7 to 10% of its time.)  They come on
    // top of the ND a step that the waits count, which only makes those wait
    // for no less than they should.  An even step for PIPE's pairs.
    auto windows = [&](auto body) __attribute__((always_inline)) {
        if constexpr (!C::FP8) {
            body(0, plain);
        } else {
            const int at = C::PIPE ? 2 - 2 * tt0 : 1 - tt0;
            int t = 0;
            for (int w = 0;; ++w) {
                const int stop = S == 1 ? plain : min(plain, at + w * C::SPW);
                body(t, stop);
                if (stop == plain) break;
                t = stop;
                scale_window(w + 1);
            }
        }
    };
    if constexpr (C::PIPE) {
        static_assert(SL == 1 || SL % 2 == 0, "register sets alternate");
        // Step t: stages t and t + 1 have landed for every wave, and every
        // wave is done reading stage t - 1, whose slot takes stage t + ST - 1.
        auto step = [&]<bool MASK>(int t, int p) __attribute__((always_inline)) {
            wait_vm_barrier<(C::ST - 3) * C::ND>();
            issue(t + C::ST - 1, wr);
#pragma unroll
            for (int s0 = 0; s0 < SL; ++s0) {
                const int cur = (p + s0) & 1;
                if (s0 + 1 < SL)
                    fetch.template operator()<MASK>(cur ^ 1, rd, (s0 + 1) * C::WK + wk, t, sa);
                else
                    fetch.template operator()<MASK>(cur ^ 1, nx, wk, t + 1, sn);
                multiply(cur);
                convert(cur ^ 1);
            }
            rd = nx;
            nx = next(nx);
            wr = next(wr);
            sa = sn;
            if constexpr (C::FP8) sn = scale_at(t + 2);
        };
        wait_vm_barrier<(C::ST - 2) * C::ND>();
        fetch.template operator()<true>(0, rd, wk, 0, sa);
        convert(0);
        int t = 0;
        if constexpr (SL == 1) {
            windows([&](int first, int last) __attribute__((always_inline)) {
                for (t = first; t + 1 < last; t += 2) {
                    step.template operator()<false>(t, 0);
                    step.template operator()<false>(t + 1, 1);
                }
            });
            for (; t < KT; t += 2) {
                step.template operator()<C::FP8>(t, 0);
                if (t + 1 < KT) step.template operator()<C::FP8>(t + 1, 1);
            }
        } else {
            windows([&](int first, int last) __attribute__((always_inline)) {
                for (t = first; t < last; ++t) step.template operator()<false>(t, 0);
            });
            if constexpr (C::FP8)
                for (; t < KT; ++t) step.template operator()<true>(t, 0);
        }
    } else {
        auto step = [&]<bool MASK>(int t) __attribute__((always_inline)) {
            wait_vm_barrier<(C::ST - 2) * C::ND>();
            issue(t + C::ST - 1, wr);
#pragma unroll
            for (int s0 = 0; s0 < SL; ++s0) {
                fetch.template operator()<MASK>(0, rd, s0 * C::WK + wk, t, sa);
                convert(0);
                multiply(0);
            }
            rd = next(rd);
            wr = next(wr);
            if constexpr (C::FP8) sa = scale_at(t + 1);
        };
        int t = 0;
        windows([&](int first, int last) __attribute__((always_inline)) {
            for (t = first; t < last; ++t) step.template operator()<false>(t);
        });
        if constexpr (C::FP8)
            if (t < KT) step.template operator()<true>(t);
    }
    // The last steps prefetched zeros past K; they must land before the ring
    // is reused or the workgroup's LDS is freed.
    wait_vm_barrier<0>();

    if constexpr (C::WK > 1) {
        // Wave (wk, q) leaves its tile at [q][fragment quad][lane]; wave (0, q)
        // adds the partials in wk order, one wk at a time.
        constexpr int Q = C::WM * C::WN, QUADS = C::MT * C::NT * 4;
        f32x4* part = reinterpret_cast<f32x4*>(smem) + (wave % Q) * QUADS * 64 + lane;
        for (int k = 1; k < C::WK; ++k) {
            if (wk == k) {
#pragma unroll
                for (int i = 0; i < C::MT; ++i)
#pragma unroll
                    for (int j = 0; j < C::NT; ++j)
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            part[((i * C::NT + j) * 4 + q) * 64] = f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1],
                                                                         acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
            }
            __syncthreads();
            if (wk == 0) {
#pragma unroll
                for (int i = 0; i < C::MT; ++i)
#pragma unroll
                    for (int j = 0; j < C::NT; ++j)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const f32x4 p = part[((i * C::NT + j) * 4 + q) * 64];
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[i][j][4 * q + e] += p[e];
                        }
            }
            if (k + 1 < C::WK) __syncthreads();
        }
        if (wk != 0) return;
    }

    // ---- epilogue: lane (h, l32) of fragment (i, j) holds row
    // m0 + 32 (wm MT + i) + l32 and tile columns 32-block + 16 h + [0, 16)
    // (SWIGLU: outputs 16-block + 8 h + [0, 8)).
    constexpr int OW = SWIGLU ? 8 : 16, COLS = C::NT * 2 * OW;  // outputs of a lane and fragment, columns of a wave
    const int lim = min(n0 + gr.per, SWIGLU ? N >> 1 : N);
    auto outputs = [&](uint32_t (&o)[OW / 2], int i, int j, int col) __attribute__((always_inline)) {
        if constexpr (SWIGLU) {
            uint32_t gu[8];
            uint16_t v[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) gu[r] = pack_bf16x2(f32x2{acc[i][j][r], acc[i][j][r + 8]});
            swiglu_bf16_batch<8>(gu, v);
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = (uint32_t)v[2 * r] | ((uint32_t)v[2 * r + 1] << 16);
        } else {
#pragma unroll
            for (int r = 0; r < 8; ++r) o[r] = pack_bf16x2(f32x2{acc[i][j][2 * r], acc[i][j][2 * r + 1]});
            if (bias) {
                add_bias8(o, bias, col, lim, gr.wide & 2);
                add_bias8(o + 4, bias, col + 8, lim, gr.wide & 2);
            }
        }
    };
    if constexpr (C::STAGED) {
        if (!(gr.wide & C::DIRECT) && gr.splits == 1) {
            uint8_t* own = smem + wave % (C::WM * C::WN) * C::STORE_BYTES;
            const int cb = n0 + wn * COLS;
#pragma unroll
            for (int i = 0; i < C::MT; ++i) {
                const int mb = m0 + wm * (C::BM / C::WM) + 32 * i;
                if (mb >= M || cb >= lim) break;
#pragma unroll
                for (int j = 0; j < C::NT; ++j) {
                    const int col = cb + j * 2 * OW + OW * h;
                    if (col >= lim) continue;
                    uint32_t o[OW / 2];
                    outputs(o, i, j, col);
                    u32x4* dst = reinterpret_cast<u32x4*>(own + l32 * (2 * COLS + 16) + 2 * (col - cb));
#pragma unroll
                    for (int q = 0; q < OW / 8; ++q) dst[q] = u32x4{o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]};
                }
                uint16_t* dst = y + (int64_t)mb * ldy + cb;
                if (gr.wide & 4)
                    store_staged<4, COLS>(dst, ldy, own, min(32, M - mb), lim - cb);
                else if (gr.wide & 8)
                    store_staged<2, COLS>(dst, ldy, own, min(32, M - mb), lim - cb);
                else
                    store_staged<1, COLS>(dst, ldy, own, min(32, M - mb), lim - cb);
            }
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < C::MT; ++i) {
        const int m = m0 + wm * (C::BM / C::WM) + 32 * i + l32;
#pragma unroll
        for (int j = 0; j < C::NT; ++j) {
            const int col = n0 + wn * COLS + j * 2 * OW + OW * h;
            if (m >= M || col >= lim) continue;
            if constexpr (!SWIGLU) {
                if (gr.splits > 1) {
                    float* dst = part + ((int64_t)split * M + m) * gr.ldp + col;
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        if (col + 4 * q < lim)
                            reinterpret_cast<f32x4*>(dst)[q] = f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1],
                                                                     acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                    continue;
                }
            }
            uint32_t o[OW / 2];
            outputs(o, i, j, col);
            uint16_t* dst = y + (int64_t)m * ldy + col;
#pragma unroll
            for (int q = 0; q < OW / 8; ++q) store8(dst + 8 * q, o + 4 * q, lim - col - 8 * q, gr.wide);
        }
    }
}

// y = bf16(sum over splits, in order) (+ bias), or SWIGLU y = swiglu of the
// gate and up sums: eight outputs per thread.
template <bool SWIGLU, int SPLITS>
__global__ __launch_bounds__(256) void split_reduce_kernel(const float* __restrict__ part, int ldp,
                                                           const uint16_t* __restrict__ bias, uint16_t* __restrict__ y,
                                                           int64_t ldy, int M, int N, int wide) {
    const int D = SWIGLU ? N >> 1 : N, groups = (D + 7) / 8;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)M * groups) return;
    const int m = (int)(idx / groups), col = 8 * (int)(idx % groups);
    const int64_t stride = (int64_t)M * ldp;
    // D % 4 != 0: up's groups start off the 16-byte grid
    typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
    auto sum8 = [&](int c, float (&v)[8]) __attribute__((always_inline)) {
        const float* p = part + (int64_t)m * ldp + c;
        f32x4 a[SPLITS], b[SPLITS];  // all under way before the first sum
#pragma unroll
        for (int s = 0; s < SPLITS; ++s) {
            a[s] = *reinterpret_cast<const f32x4_any*>(p + s * stride);
            b[s] = *reinterpret_cast<const f32x4_any*>(p + s * stride + 4);
        }
#pragma unroll
        for (int s = 1; s < SPLITS; ++s) a[0] += a[s], b[0] += b[s];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = a[0][r], v[4 + r] = b[0][r];
    };
    float a[8];
    uint32_t o[4];
    sum8(col, a);
    if constexpr (SWIGLU) {
        float b[8];
        uint32_t gu[8];
        uint16_t v[8];
        sum8(D + col, b);
#pragma unroll
        for (int r = 0; r < 8; ++r) gu[r] = pack_bf16x2(f32x2{a[r], b[r]});
        swiglu_bf16_batch<8>(gu, v);
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (uint32_t)v[2 * r] | ((uint32_t)v[2 * r + 1] << 16);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = pack_bf16x2(f32x2{a[2 * r], a[2 * r + 1]});
        if (bias) add_bias8(o, bias, col, N, wide & 2);
    }
    uint16_t* dst = y + (int64_t)m * ldy + col;
    store8(dst, o, D - col, wide);
}

inline hipError_t allow_lds(const void* kern, int bytes) {
    return hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

// The launch of config C over grid gr (part: splits > 1, gr.splits x M x
// gr.ldp floats).
template <class C, bool SWIGLU>
hipError_t launch(const uint16_t* x, const void* w, const float* scales, int S, const uint16_t* bias, uint16_t* y,
                  int64_t ldy, int M, int N, int K, const Grid& gr, float* part, hipStream_t stream) {
    auto kern = gemm_tile_kernel<C, SWIGLU>;
    static const hipError_t attr = allow_lds(reinterpret_cast<const void*>(kern), kLds);
    if (attr != hipSuccess) return attr;
    const int units = gr.mtiles * gr.nblocks * gr.splits;
    hipLaunchKernelGGL(kern, dim3((unsigned)((units + 7) / 8 * 8)), dim3(C::THREADS), C::LDS_BYTES, stream,
                       x, w, scales, S, bias, y, ldy, M, N, K, gr, part);
    return hipGetLastError();
}

}  // namespace gemm_tile
}  // namespace fp8lin
