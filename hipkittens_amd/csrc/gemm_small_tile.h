// Small-tile GEMM kernel body shared by the FP8 and BF16 GEMMs (a K-step is 128 bytes per operand
// row in both; only the MFMA differs).
#pragma once
#include "gemm_tile.h"
#include "hk_host.h"
#include "../../include/hk355.h"

namespace hk {

// 128x128-tile kernel body for problems with too few 256x256 tiles to occupy the chip (a 1024^3
// GEMM has 16 of them for 256 CUs): 4 waves, each a 64x64 patch (16 MFMA tiles), four LDS
// stages of 2 x 16 KiB (MXFP4: three). Same tile format, B-row permutation and epilogue as the
// large-tile kernels.
constexpr int kSmallTile = 128;
constexpr int kSmallTileBytes = kSmallTile * BK;          // 16 KiB per operand
constexpr int kSmallStageBytes = 2 * kSmallTileBytes;
constexpr int kSmallStages = 4, kSmallStagesScaled = 3;
// the same kernel with 64x64 tiles and four 16 KiB stages (two workgroups per CU): for problems
// with so few 128x128 tiles that a quarter of the tile is needed to give every CU work
constexpr int kTinyTile = 64;
constexpr int kTinyStages = 4;
constexpr int kTinyLdsBytes = kTinyStages * 2 * kTinyTile * BK;  // 64 KiB

// SPLIT: blockIdx.y selects a range of `kps` K-steps; the tile's fp32 partial sums go to
// partial[blockIdx.y][M][N] (plain stores; splitk_reduce_kernel adds the ranges in order, so the
// result does not depend on timing). For problems with few tiles and a long K (decode-like
// shapes), where a single workgroup per tile walks K one K-step latency at a time.
// MMA: the operand type's MFMA on one 16-row x 128-byte fragment pair, `MMA::mma(acc, b, a)`. K is
// the operands' row length in BYTES (a multiple of 16); smem: the workgroup's dynamic LDS.
// MMA::kScaled (MXFP4): every operand row also has e8m0 block scales, 8 bytes per K-step, in rows of
// sa_pitch / sb_pitch bytes (multiples of 8); `MMA::mma(acc, b, a, sb, sa)` then takes, per fragment,
// the lane's scale bytes of the K-step's two halves in bits [7:0] of .x / .y.
// tail_pair / tail_shift: the pair of K-steps whose scale fetch starts tail_shift bytes early (rows that do not
// hold whole groups of 16 scale bytes; see mxfp4_gemm.hip), -1 / 0: none.
// row_bytes: scale bytes of a row that may be fetched (0: the whole pitch); the last row of an operand is in
// the descriptor's range up to there.
struct SmallTileScales {
    const uint8_t* SA; const uint8_t* SB; int sa_pitch, sb_pitch; int tail_pair = -1, tail_shift = 0, row_bytes = 0;
};
// bytes of the scale rows [row0, row0 + rows) that a descriptor covers
__device__ __forceinline__ uint32_t scale_rows_bytes(int rows, int pitch, int row_bytes) {
    return (uint32_t)(rows - 1) * (uint32_t)pitch + (uint32_t)(row_bytes ? row_bytes : pitch);
}
template <int TILE, int STAGES>
constexpr int small_tile_lds_bytes(bool scaled) { return STAGES * 2 * TILE * BK + (scaled ? 4 * 2 * TILE * 16 : 0); }

template <typename MMA, int TILE, int STAGES, bool EDGE, bool SPLIT>
__device__ __forceinline__ void gemm_small_tile_body(
    uint8_t* smem, const uint8_t* __restrict__ A, const uint8_t* __restrict__ B, uint16_t* __restrict__ C,
    int M, int N, int K, float alpha, int tiles_m, int tiles_n, int kps, float* __restrict__ partial,
    SmallTileScales sc = SmallTileScales{nullptr, nullptr, 0, 0}) {
    constexpr int NW = 4, TM = TILE / 2, TN = TILE / 2, MT = TM / 16, NT = TN / 16;
    constexpr int kTB = TILE * BK, kSB = 2 * kTB;    // bytes of one operand tile / of one stage
    constexpr int NDMA = kTB / (NW * 1024);          // loads per wave per operand per K-step
    constexpr bool kScaled = MMA::kScaled;
    constexpr int LPT = 2 * NDMA;                    // operand loads per wave per K-step
    // scales: four slots, each the 16 bytes (two K-steps) of the TILE rows of A, then of B
    constexpr int kScaleSlot = 2 * TILE * 16, kScaleBase = STAGES * kSB;
    static_assert(STAGES >= 3 && STAGES <= 8 && (STAGES - 1) * LPT < 64, "vmcnt range");
    static_assert(!kScaled || STAGES <= 5, "four scale slots cover the K-step pairs of at most five stages");
    const int lane = lane_id(), w = wave_id();
    const int wm = w >> 1, wn = w & 1;

    int pm, pn;
    {
        // An XCD's run of fewer than 32 tiles is the squarer patch with groups of four rows; with 32 it is 8 x 4 or 4 x 8. us,
        // tiles round robin over the XCDs / runs in groups of eight rows / of four: FP8 1000 x 3000 x 4096 20.4 / 20.3 / 19.5,
        // 3438 x 640 x 1024 6.9 / 7.0 / 6.95; BF16 775 x 2176 x 2752 20.8 / 17.9 / 17.9.
        const int id = xcd_chunk_order(blockIdx.x, tiles_m * tiles_n, kCuPerXcd);
        grouped_raster(id, tiles_m, tiles_n, tiles_m * tiles_n < kNumXcd * kCuPerXcd ? 4 : 8, pm, pn);
    }
    const int row0 = pm * TILE, col0 = pn * TILE;
    const int a_rows = min(M - row0, TILE), b_rows = min(N - col0, TILE);
    const v4i srd_a = make_srd(A + (size_t)row0 * K, (uint32_t)a_rows * (uint32_t)K);
    const v4i srd_b = make_srd(B + (size_t)col0 * K, (uint32_t)b_rows * (uint32_t)K);

    uint32_t voff_a[NDMA], voff_b[NDMA];
#pragma unroll
    for (int i = 0; i < NDMA; ++i) {
        const int R = 8 * (i * NW + w) + (lane >> 3);
        const uint32_t c = swz_chunk(R, lane & 7);
        int ra = R, rb = b_row_to_col(R);
        if (EDGE) {
            ra = min(ra, a_rows - 1);
            rb = min(rb, b_rows - 1);
        }
        voff_a[i] = (uint32_t)ra * (uint32_t)K + c * 16u;
        voff_b[i] = (uint32_t)rb * (uint32_t)K + c * 16u;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    const uint32_t lds_wave = to_sgpr(lds0 + (uint32_t)w * 1024u);
    const int nk = (K + BK - 1) / BK;
    // last K-step of a K that is not a multiple of 128: lanes whose 16-byte chunk lies past the
    // end of the row are moved out of the buffer's range (bit 31) and write zeros to LDS
    const uint32_t tail_or =
        (int)(swz_chunk(8 * w + (lane >> 3), lane & 7) * 16u) >= K - (nk - 1) * BK ? 0x80000000u : 0u;
    // this workgroup's K-steps: [kt0, kt0 + nkt)
    const int kt0 = SPLIT ? (int)blockIdx.y * kps : 0;
    const int nkt = SPLIT ? min(kps, nk - kt0) : nk;
    // Scale loads (kScaled): wave w fetches operand w & 1 (0 = A), lane l the 16 bytes of row 64 (w >> 1) + l (TILE = 64:
    // waves 0 and 1 only), i.e. the scales of the pair of K-steps kt / 2, in front of the even K-step's operands. A scale
    // load touches a cache line per lane, where the 1 KiB loads of operands touch eight: with every K-step and from every
    // wave, which keeps the waits' counts the same, the scales cost more of a CU's vector-memory path than the operands.
    // The waits leave the scale loads out: one among the loads behind a K-step makes its wait stricter, never weaker.
    // (64x64 tiles, us before / after: 128 x 8192 x 8192 21.5 / 17.6, 200 x 8192 x 8192 27.2 / 22.6, 512 x 4096 x 4096 18.5 / 15.3,
    // 128 x 4096 x 14336 34.6 / 27.0; 128x128 tiles 2 to 4 %.)
    v4i srd_s = {0, 0, 0, 0};
    uint32_t voff_s = 0, lds_s = 0;
    if (kScaled) {
        const int op = w & 1, srow0 = TILE == 128 ? 64 * (w >> 1) : 0;
        const int R = srow0 + lane;
        int rr = op ? b_row_to_col(R) : R;
        if (EDGE) rr = min(rr, (op ? b_rows : a_rows) - 1);
        const int pitch = op ? sc.sb_pitch : sc.sa_pitch;
        srd_s = op ? make_srd(sc.SB + (size_t)col0 * pitch, scale_rows_bytes(b_rows, pitch, sc.row_bytes))
                   : make_srd(sc.SA + (size_t)row0 * pitch, scale_rows_bytes(a_rows, pitch, sc.row_bytes));
        voff_s = (uint32_t)rr * (uint32_t)pitch;
        lds_s = to_sgpr(lds0 + kScaleBase + (uint32_t)op * (TILE * 16) + (uint32_t)srow0 * 16u);
    }
    auto issue_tile = [&](int stage, int kt_local) {
        const int kt = kt0 + kt_local;
        const uint32_t k0 = (uint32_t)kt * BK;
        const uint32_t dst = lds_wave + (uint32_t)stage * kSB;
        const uint32_t vor = kt == nk - 1 ? tail_or : 0u;
        if (kScaled && (kt & 1) == 0 && (TILE == 128 || w < 2))
            dma16(srd_s, lds_s + (uint32_t)((kt >> 1) & 3) * kScaleSlot, voff_s,
                  (uint32_t)(kt >> 1) * 16u - ((kt >> 1) == sc.tail_pair ? (uint32_t)sc.tail_shift : 0u));
#pragma unroll
        for (int i = 0; i < NDMA; ++i) dma16(srd_a, dst + i * NW * 1024, voff_a[i] | vor, k0);
#pragma unroll
        for (int i = 0; i < NDMA; ++i) dma16(srd_b, dst + kTB + i * NW * 1024, voff_b[i] | vor, k0);
    };
    // wait until at most `tiles` of the most recently issued K-steps' loads are still in flight
    auto wait_tiles = [&](int tiles) {
        switch (tiles) {
            case 0: wait_vmcnt<0>(); break;
            case 1: wait_vmcnt<LPT>(); break;
            case 2: wait_vmcnt<(STAGES > 2 ? 2 : 1) * LPT>(); break;
            case 3: wait_vmcnt<(STAGES > 3 ? 3 : 1) * LPT>(); break;
            case 4: wait_vmcnt<(STAGES > 4 ? 4 : 1) * LPT>(); break;
            case 5: wait_vmcnt<(STAGES > 5 ? 5 : 1) * LPT>(); break;
            case 6: wait_vmcnt<(STAGES > 6 ? 6 : 1) * LPT>(); break;
            default: wait_vmcnt<(STAGES > 7 ? 7 : 1) * LPT>(); break;
        }
    };

    const uint32_t r = lane & 15, g = lane >> 4;
    const uint32_t rd_lo = r * 128u + swz_chunk(r, g) * 16u;
    const uint32_t rd_hi = r * 128u + swz_chunk(r, g + 4) * 16u;
    const uint32_t a_lo0 = lds0 + wm * (TM * BK) + rd_lo, a_hi0 = lds0 + wm * (TM * BK) + rd_hi;
    const uint32_t b_lo0 = lds0 + kTB + wn * (TN * BK) + rd_lo;
    const uint32_t b_hi0 = lds0 + kTB + wn * (TN * BK) + rd_hi;

    v4f acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = v4f{0.f, 0.f, 0.f, 0.f};

    if constexpr (kScaled) {
        // K-steps kt .. kt + STAGES - 2 are in flight or in LDS while step kt is multiplied
#pragma unroll
        for (int p = 0; p < STAGES - 1; ++p)
            if (p < nkt) issue_tile(p, p);
        int st = 0;
        for (int kt = 0; kt < nkt; ++kt) {
            // this wave's part of K-step kt has landed (the loads of the steps behind it may still fly)
            wait_tiles(min(nkt - 1 - kt, STAGES - 2));
            block_barrier();  // ... everyone's; and everyone is done with the stage of K-step kt - 1
            if (kt + STAGES - 1 < nkt) issue_tile(st == 0 ? STAGES - 1 : st - 1, kt + STAGES - 1);
            const uint32_t so = (uint32_t)st * kSB;
            v8i bf[NT];
#pragma unroll
            for (int n = 0; n < NT; ++n) bf[n] = lds_frag(b_lo0 + so, b_hi0 + so, n * 16 * BK);
            {
                // the lane's scale bytes: row 16 f + r of the wave's patch, byte g of each half's dword
                const int ktg = kt0 + kt;
                const uint32_t sbase = lds0 + kScaleBase + (uint32_t)((ktg >> 1) & 3) * kScaleSlot + (uint32_t)(ktg & 1) * 8u + r * 16u +
                                       ((ktg >> 1) == sc.tail_pair ? (uint32_t)sc.tail_shift : 0u);
                const uint32_t sh = 8u * g;
                v2i bs[NT];
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    bs[n] = *(lds_v2i_t*)(uintptr_t)(sbase + TILE * 16 + (wn * TN + 16 * n) * 16);
                    bs[n].x = (int)((uint32_t)bs[n].x >> sh); bs[n].y = (int)((uint32_t)bs[n].y >> sh);
                }
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    const v8i af = lds_frag(a_lo0 + so, a_hi0 + so, m * 16 * BK);
                    v2i as = *(lds_v2i_t*)(uintptr_t)(sbase + (wm * TM + 16 * m) * 16);
                    as.x = (int)((uint32_t)as.x >> sh); as.y = (int)((uint32_t)as.y >> sh);
#pragma unroll
                    for (int n = 0; n < NT; ++n) MMA::mma(acc[m][n], bf[n], af, bs[n], as);
                }
            }
            st = st == STAGES - 1 ? 0 : st + 1;
        }
    } else {
        // The reads of the next K-step's fragments and the loads of K-step kt + STAGES are spread over the MFMAs of
        // K-step kt. One wave per SIMD runs a 128x128 tile, and LDS reads in front of the MFMAs leave the matrix cores
        // idle while the LDS delivers 64 KiB and takes in 32 KiB per K-step (768 clocks against the MFMAs' 512).
        // us, reads first / spread (and four stages instead of three with 128x128 tiles): FP8 1024^3 5.0 / 4.2, 2048^3
        // 13.2 / 10.3, 400 x 6000 x 4096 22.6 / 18.7; BF16 1024^3 7.4 / 5.6, 2048^3 22.3 / 19.0. The scaled FP4 MFMAs are
        // half as long and need two shifts per scale and fragment beside them: the same order is 5 to 12 % slower there,
        // so that form keeps its reads in front.
        // No loads go out past the last K-step: as loads of zeros that keep the waits constant they made few K-steps
        // slower than with the reads first (FP8, reads first / spread with them / spread without: 512 x 4096 x 256 3.7 / 4.2
        // / 3.5, 17 x 32512 x 1024 8.5 / 9.1 / 8.5), and many K-steps 1 to 8 % slower than without.
        struct Frags { v8i a[MT], b[NT]; };
        Frags fr[2];
        // fragment x of the K-step in stage `stage`: B's NT, then A's MT
        auto read_frag = [&](Frags& f, int stage, int x) __attribute__((always_inline)) {
            const uint32_t so = (uint32_t)stage * kSB;
            if (x < NT) f.b[x < NT ? x : 0] = lds_frag(b_lo0 + so, b_hi0 + so, x * 16 * BK);
            else f.a[x >= NT ? x - NT : 0] = lds_frag(a_lo0 + so, a_hi0 + so, (x - NT) * 16 * BK);
        };
        // load j (A's pieces, then B's) of K-step kt_local < nkt
        auto issue_load = [&](int stage, int kt_local, int j) __attribute__((always_inline)) {
            const int kt = kt0 + kt_local;
            const uint32_t k0 = (uint32_t)kt * BK, vor = kt == nk - 1 ? tail_or : 0u;
            const uint32_t dst = lds_wave + (uint32_t)stage * kSB;
            if (j < NDMA) dma16(srd_a, dst + j * NW * 1024, voff_a[j < NDMA ? j : 0] | vor, k0);
            else dma16(srd_b, dst + kTB + (j - NDMA) * NW * 1024, voff_b[j >= NDMA ? j - NDMA : 0] | vor, k0);
        };
        // all stages are filled ahead; stage kt is free for K-step kt + STAGES once everyone's fragments of K-step kt
        // are in registers
#pragma unroll
        for (int p = 0; p < STAGES; ++p)
            if (p < nkt) {
#pragma unroll
                for (int j = 0; j < LPT; ++j) issue_load(p, p, j);
            }
        wait_tiles(min(nkt, STAGES) - 1);
        block_barrier();
#pragma unroll
        for (int x = 0; x < MT + NT; ++x) read_frag(fr[0], 0, x);
        int st = 0, kt = 0;   // stage of K-step kt
        // K-step kt with its fragments in fr[P]. kMain: constant wait, the loads of K-step kt + STAGES among the MFMAs;
        // kTail: counted wait, no loads; kLast: the MFMAs alone.
        enum { kMain, kTail, kLast };
        auto step = [&]<int P, int KIND>() __attribute__((always_inline)) {
            Frags &cur = fr[P], &nxt = fr[P ^ 1];
            constexpr int kMma = MT * NT, kFirst = NT / 2;   // MFMAs in all, in front of the barrier
            constexpr int kItems = MT + NT + LPT;
            static_assert(MT + NT == LPT, "reads and loads alternate");
            const int st_next = st == STAGES - 1 ? 0 : st + 1;
#pragma unroll
            for (int q = 0; q < (KIND == kLast ? kMma : kFirst); ++q) MMA::mma(acc[q / NT][q % NT], cur.b[q % NT], cur.a[q / NT]);
            if constexpr (KIND == kLast) return;
            // this wave's part of the next K-step has landed and its fragments of this one are in registers ...
            if constexpr (KIND == kMain) wait_vmcnt<(STAGES - 2) * LPT>();
            else wait_tiles(min(nkt - kt, STAGES) - 2);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            block_barrier();   // ... and so are everyone's
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = kFirst; q < kMma; ++q) {
                MMA::mma(acc[q / NT][q % NT], cur.b[q % NT], cur.a[q / NT]);
#pragma unroll
                for (int i = (q - kFirst) * kItems / (kMma - kFirst); i < (q - kFirst + 1) * kItems / (kMma - kFirst); ++i) {
                    if ((i & 1) == 0) read_frag(nxt, st_next, i >> 1);
                    else if (KIND == kMain) issue_load(st, kt + STAGES, i >> 1);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            st = st_next;
            ++kt;
        };
        // an even count's first K-step by itself, its reads behind its MFMAs: an odd one is left, so that the last K-step's
        // fragments are in fr[0] (a last K-step in either buffer costs the 128x128 tile its registers)
        if ((nkt & 1) == 0) {
#pragma unroll
            for (int q = 0; q < MT * NT; ++q) MMA::mma(acc[q / NT][q % NT], fr[0].b[q % NT], fr[0].a[q / NT]);
            wait_tiles(min(nkt, STAGES) - 2);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            block_barrier();
            if (STAGES < nkt) {
#pragma unroll
                for (int j = 0; j < LPT; ++j) issue_load(0, STAGES, j);
            }
            st = kt = 1;
#pragma unroll
            for (int x = 0; x < MT + NT; ++x) read_frag(fr[0], 1, x);
        }
        while (kt + 1 + STAGES < nkt) {
            step.template operator()<0, kMain>();
            step.template operator()<1, kMain>();
        }
        if (kt + STAGES < nkt) {
            step.template operator()<0, kMain>();
            step.template operator()<1, kTail>();
        }
        while (kt + 1 < nkt) {
            step.template operator()<0, kTail>();
            step.template operator()<1, kTail>();
        }
        step.template operator()<0, kLast>();
    }
    if (!SPLIT) {
        store_c_tile<MT, NT, EDGE>(acc, C, M, N, row0 + wm * TM, col0 + wn * TN, alpha);
    } else {
        // fp32 partial sums: lane (r, g) holds, for row 16 m + r, columns 32 p + 8 g .. +8
        float* out = partial + (size_t)blockIdx.y * M * N;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int row = row0 + wm * TM + 16 * m + (int)r;
            if (row >= M) continue;
#pragma unroll
            for (int q = 0; q < NT / 2; ++q) {
                const int col = col0 + wn * TN + 32 * q + 8 * (int)g;
                float* dst = out + (size_t)row * N + col;
                if (col + 8 <= N && (N & 3) == 0) {
                    *(v4f*)dst = acc[m][2 * q];
                    *(v4f*)(dst + 4) = acc[m][2 * q + 1];
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (col + j < N) dst[j] = j < 4 ? acc[m][2 * q][j] : acc[m][2 * q + 1][j - 4];
                }
            }
        }
    }
}


// C = bf16(alpha * sum_s partial[s]) in split order; one thread per 4 columns.
static __global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ partial, int splits,
                                                            long long mn, float alpha,
                                                            uint16_t* __restrict__ C) {
    const long long i4 = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i4 >= mn) return;
    if (i4 + 4 <= mn && (mn & 3) == 0) {
        v4f sum = *(const v4f*)(partial + i4);
        for (int s2 = 1; s2 < splits; ++s2) sum += *(const v4f*)(partial + (size_t)s2 * mn + i4);
        sum *= alpha;
        v2i o;
        o.x = pack_bf16(sum.x, sum.y); o.y = pack_bf16(sum.z, sum.w);
        *(v2i*)(C + i4) = o;
    } else {
        for (long long i = i4; i < mn && i < i4 + 4; ++i) {
            float sum = partial[i];
            for (int s2 = 1; s2 < splits; ++s2) sum += partial[(size_t)s2 * mn + i];
            C[i] = (uint16_t)(pack_bf16(sum * alpha, 0.f) & 0xffffu);
        }
    }
}

// Which tile a GEMM gets when the caller does not pin a kernel (pick_gemm_tile): 256, 128 or 64 square, or one of the ring
// kernel's 192x256 and 256x192. A table, then a rule in two steps:
//  1. a generated table of the shapes on which a sweep found the rule's choice more than a few percent behind
//     another tile (tile_table.inc, written by `python -m hipkittens_amd.tile_sweep FORMAT --emit`; the
//     counterpart of the reference's per-shape analysis/baselines/gemm/utils/tuned.yaml). An entry is keyed by
//     the format, the numbers of 64-row / 64-column blocks of M and N and the K-step count, applies on
//     devices with the CU count the sweep ran on, and is final: it corrects the rule's estimates, so they do not judge it again;
//  2. the square tile with the smallest estimated time (pick_tile_rule). A tile kernel's workgroups run in rounds over the
//     device's CUs (one workgroup per CU for the 256- and 128-tiles, two for the 64-tile), every round costs
//     the same whether it is full or not, and a workgroup's time is a fixed part (prologue, epilogue, launch)
//     plus a part per K-step:  time = ceil(tiles / (CUs x workgroups per CU)) x (fixed + per_step x K-steps).
//     The two constants per tile and format were fitted to the sweep below on an MI355X (microseconds; they
//     enter only through their ratios, the CU count through the rounds). This captures what a threshold on the
//     tile count cannot: 72 tiles of 256 are one round where their 288 tiles of 128 are two (the large tile
//     wins by 4-12 % from a K of about 4096 elements on), 64 tiles of 256 are one round of four times the work
//     of the single round of 256 small tiles (the small tile wins by 60 %);
//  3. a shorter tile in its place where that is estimated faster (pick_shorter_tile).
// Measured against the best of the five kernels, every launch on another copy of B (a model's weights come from HBM, not from
// the memory-side cache), the rule alone is more than 5 % behind on 38 / 21 / 26 of the sweep's 414 shapes (FP8 / BF16 /
// MXFP4; without the about 40 that the skinny kernel takes), with the table on 3 / 4 / 4, by 9 % at most, and on
// 24 / 28 / 9 of 450 shapes drawn between the sweep's points (without the about 155 of the skinny kernel): the more of two sweeps.
// Table and constants were measured when a launch's last, partial span of tiles still went round robin over the XCDs (xcd_chunk_order).
// Of the 100 swept shapes that have an entry 78 are still more than 3 % ahead of the rule's choice in both sweeps, and none that a tile
// kernel takes is more than 1.1 % behind it in either; 8 / 8 / 5 shapes without one would get one in both.
struct TileRule {
    float fixed[3], per_step[3];   // 256-, 128-, 64-tile
};
enum TileFormat { kFmtFp8 = 0, kFmtBf16 = 1, kFmtMxfp4 = 2 };
struct TileTableEntry { unsigned char fmt; unsigned short m64, n64, nk; int tile; };
#include "tile_table.inc"   // kTileTableCus, kTileTable[]

int moe_num_compute_units();  // number of CUs of the current device, cached (moe_mxfp4.hip)

static inline int pick_tile_rule(int M, int N, int nk, TileRule r, int cus) {
    const int tile[3] = {BM, kSmallTile, kTinyTile};
    const int per_cu[3] = {1, 1, 2};
    int best = 0;
    double best_time = 0.0;
    for (int i = 0; i < 3; ++i) {
        const long long tiles = (((long long)M + tile[i] - 1) / tile[i]) * (((long long)N + tile[i] - 1) / tile[i]);
        const long long capacity = (long long)cus * per_cu[i];
        const double time = (double)((tiles + capacity - 1) / capacity) * ((double)r.fixed[i] + (double)r.per_step[i] * nk);
        if (i == 0 || time < best_time) { best = i; best_time = time; }   // ties go to the larger tile
    }
    return tile[best];
}
// The table's entry for a shape: 256, 128, 64 or one of the ring kernel's shorter tiles; 0: none. (The entries behind the
// first are in order; a walk over all of them, on every call, is a tenth of a microsecond.)
constexpr unsigned long long tile_key(unsigned long long fmt, unsigned long long m64, unsigned long long n64, unsigned long long nk) {
    return fmt << 48 | m64 << 32 | n64 << 16 | nk;
}
constexpr int kTileTableSize = sizeof(kTileTable) / sizeof(kTileTable[0]);
constexpr bool tile_table_in_order() {
    for (int i = 2; i < kTileTableSize; ++i) {
        const TileTableEntry &a = kTileTable[i - 1], &b = kTileTable[i];
        if (tile_key(a.fmt, a.m64, a.n64, a.nk) >= tile_key(b.fmt, b.m64, b.n64, b.nk)) return false;
    }
    return true;
}
static_assert(tile_table_in_order(), "table_tile searches it by halves");
static inline int table_tile(int fmt, int M, int N, int nk, int cus) {
    if (cus != kTileTableCus) return 0;
    const long long m64 = ((long long)M + 63) / 64, n64 = ((long long)N + 63) / 64;
    if (m64 > 0xffff || n64 > 0xffff || nk > 0xffff) return 0;
    const unsigned long long key = tile_key(fmt, m64, n64, nk);
    int lo = 1, hi = kTileTableSize;
    while (lo < hi) {
        const int mid = (lo + hi) / 2;
        const TileTableEntry& e = kTileTable[mid];
        const unsigned long long k = tile_key(e.fmt, e.m64, e.n64, e.nk);
        if (k == key) return e.tile;
        if (k < key) lo = mid + 1;
        else hi = mid;
    }
    return 0;
}
// the formats' constants (K-steps: 128 bytes of an operand row)
constexpr TileRule kTileRules[3] = {{{7.10f, 3.28f, 2.02f}, {1.060f, 0.533f, 0.385f}},      // FP8
                                    {{8.57f, 2.79f, 2.20f}, {0.983f, 0.495f, 0.336f}},      // BF16
                                    {{7.51f, 3.07f, 1.185f}, {1.316f, 0.710f, 0.587f}}};    // MXFP4

// The ring kernel's shorter tiles (gemm_ring.h): 192x256 or 256x192 in the place of the rule's square tile, where
// the same cost model, one workgroup per CU, gives them less time. The constants, and the factor on the estimate for a
// 128- or 64-tile (which is high where it is compared with these), are fitted to 91 shapes per format on an MI355X
// (M 500 ... 8192, (N, K) 4096 x 4096 ... 14336 x 4096, 2880 x 2880, 10000 x 1024, copies of B in rotation; MXFP4 again to 112
// when its small-tile kernels became faster). Over the 414 shapes of the sweep and the about 295 of 450 drawn ones that a tile kernel
// takes, a shorter tile is more than 3 % behind the square one on 3 / 2 / 3 (FP8 / BF16 / MXFP4; the more of two sweeps), and the
// geometric mean of the drawn ones falls by 2.7 / 1.9 / 2.8 %, of 3.7 / 2.9 / 3.3 that the best kernel for every shape would give. (A
// fit to all of them on the former tile order, {6.84, 0.882, 0.882}, {6.75, 0.816, 0.881}, {6.73, 1.07, 0.873}, gained 4 % where FP8 and
// BF16 choose otherwise with it, but lost up to 14 % on single shapes, 0.6 % on the average for MXFP4.) Examples, us, 256x256 /
// 256x192: BF16 4096 x 2880 x 2880 68.8 / 54.2 (192 tiles against 240); FP8 8192 x 2880 x 2880 71.8 / 59.6; MXFP4 4096 x 2880 x 2880
// 34.5 / 27.6; and not taken: BF16 4096 x 4096 x 4096 97.8 / 130.1 (256 tiles of 256x256, one round; 352 of 256x192, two). Equal
// estimates go to 256x192: with the one that pads less instead, 5 more shapes of FP8 and 16 of BF16 were behind on the former order.
constexpr int kVariant192x256 = 192256, kVariant256x192 = 256192;   // the GEMM entry points' internal numbers for them
struct ShorterTileRule { float fixed, per_step, small; };
constexpr ShorterTileRule kShorterTileRules[3] = {{5.7f, 0.87f, 0.82f}, {5.6f, 0.925f, 0.94f}, {7.37f, 1.057f, 0.974f}};
static inline int pick_shorter_tile(int M, int N, int nk, int tile, TileRule rule, ShorterTileRule shorter, long long cus) {
    auto rounds = [&](int tm, int tn, long long capacity) {
        const long long tiles = (((long long)M + tm - 1) / tm) * (((long long)N + tn - 1) / tn);
        return (double)((tiles + capacity - 1) / capacity);
    };
    const int i = tile == kTinyTile ? 2 : tile == kSmallTile ? 1 : 0;
    const double now = rounds(tile, tile, i == 2 ? 2 * cus : cus) * ((double)rule.fixed[i] + (double)rule.per_step[i] * nk) *
                       (i == 0 ? 1.0 : (double)shorter.small);
    const double one = (double)shorter.fixed + (double)shorter.per_step * nk;
    const double t0 = rounds(192, 256, cus) * one, t1 = rounds(256, 192, cus) * one;
    if ((t0 < t1 ? t0 : t1) > now) return 0;
    return t0 < t1 ? kVariant192x256 : kVariant256x192;
}
// The tile kernel of a shape: 256, 128, 64, kVariant192x256 or kVariant256x192. A measured entry of the table is final.
static inline int pick_gemm_tile(int fmt, int M, int N, int nk, bool consult_table = true) {
    const int cus = moe_num_compute_units();   // 256 when no device can be queried
    const int listed = consult_table ? table_tile(fmt, M, N, nk, cus) : 0;
    if (listed) return listed;
    const TileRule& rule = kTileRules[fmt];
    const int square = pick_tile_rule(M, N, nk, rule, cus);
    const int shorter = pick_shorter_tile(M, N, nk, square, rule, kShorterTileRules[fmt], cus);
    return shorter ? shorter : square;
}

// The GEMM entry points' variant number for a tile as hk_gemm_tile_shape names it (rows * 1000 + columns); -1: there is none.
static inline int variant_of_tile(int tile, int v256, int v128, int v64) {
    return tile == kVariant192x256 || tile == kVariant256x192 ? tile
           : tile == 256256 ? v256 : tile == 128128 ? v128 : tile == 64064 ? v64 : -1;
}

// Number of K ranges the split-K path would use: as many as fill the CUs, each at least 4
// K-steps long, at most 16; 1 = the problem has enough tiles or too short a K.
// K: the operands' row length in bytes; min_nk: the shortest K (in K-steps) that is split.
static inline int splitk_ranges(int M, int N, int K, int min_nk = 48) {
    // 64x64 tiles, two workgroups per CU
    // (64-bit: the size queries pass whatever the caller asks about)
    const long long tiles = (((long long)M + kTinyTile - 1) / kTinyTile) * (((long long)N + kTinyTile - 1) / kTinyTile);
    const long long nk = ((long long)K + BK - 1) / BK;
    const int cus = moe_num_compute_units();   // 256 when no device can be queried
    // shorter K: the 64x64-tile kernel without a second launch is as fast or faster; more than one tile for every
    // second CU: with B coming from HBM (every launch on another weight matrix) the split measured 5 to 25 % slower
    // than the plain kernel up to 128 K-steps, and within 8 % of it at 256
    if (tiles * 2 > cus || nk < min_nk) return 1;
    long long s = 2 * cus / tiles;
    if (s > nk / 4) s = nk / 4;
    if (s > 16) s = 16;
    return s < 2 ? 1 : (int)s;
}

// Launches `kern` (a small-tile kernel instantiated with SPLIT over 64x64 tiles) on `splits` K ranges
// and the reduction behind it. K in bytes.
template <typename Kern>
static inline int launch_small_tile_splitk(Kern kern, DeviceOnce& configured, const void* A, const void* B, void* C, int M,
                                           int N, int K, float alpha, int splits, float* partial,
                                           hipStream_t stream) {
    if (!set_lds_limit_once((const void*)kern, kTinyLdsBytes, configured)) return HK_ERR_LAUNCH;
    const int tiles_m = (M + kTinyTile - 1) / kTinyTile, tiles_n = (N + kTinyTile - 1) / kTinyTile;
    const int nk = (K + BK - 1) / BK;
    const int kps = (nk + splits - 1) / splits;
    const int used = (nk + kps - 1) / kps;   // ranges that hold at least one K-step
    hipLaunchKernelGGL(kern, dim3(tiles_m * tiles_n, used), dim3(256), kTinyLdsBytes, stream,
                       (const uint8_t*)A, (const uint8_t*)B, (uint16_t*)C, M, N, K, alpha, tiles_m,
                       tiles_n, kps, partial);
    const long long mn = (long long)M * N;
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)((mn / 4 + 256) / 256)), dim3(256), 0, stream,
                       (const float*)partial, used, mn, alpha, (uint16_t*)C);
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_LAUNCH;
}

}  // namespace hk
