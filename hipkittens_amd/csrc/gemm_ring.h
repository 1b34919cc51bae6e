// The 4-wave GEMM schedule with a five-slot LDS ring, written once for every operand type whose
// K-step is 128 bytes per row (FP8: 128 elements, one MFMA per fragment pair; BF16: 64 elements, two).
#pragma once
#include "gemm_tile.h"

namespace hk {

// ---------------------------------------------------------------------------------------
// 4-wave schedule with a five-slot LDS ring (all 160 KiB): two slots for A tiles, three for B
// tiles. One wave per SIMD, each owning a 128x128 patch of the 256x256 tile (8x8 MFMA tiles, 256
// accumulator registers); every LDS read, global->LDS load and MFMA has a fixed place in the
// instruction stream (one MFMA per "slot", memory operations attached to slots): A fragment m + 3 is
// read while the MFMAs of fragment m issue, the next K-step's B fragments after the single barrier per
// K-step (schedule idea after the reference's 4-wave kernel, kernels/gemm/fp8fp32/README.md:3-5,
// per-instruction helpers in FP8_4wave/utils.cpp:44-52, 131-137, 150-161). The global->LDS loads are
// spread over the whole K-step instead of being bunched behind the barrier: the address unit of a CU
// needs 16 cycles per 1 KiB load, 16 loads per wave and step, and a wave that cannot hand
// its load over also cannot issue its next MFMA. B fragments of tile kt are read one step
// early (after barrier kt-1), so with a third B slot tile kt+2 of B may be fetched during
// MFMA groups 0..PG of step kt; A tile kt+2 follows after the barrier into the A slot that
// step kt has just finished reading.
//
// MMA is the operand type's policy:
//   Frag                          a wave's registers for 16 rows x 128 bytes of an operand
//   load(lo, hi, imm) -> Frag     from the two 16-byte LDS chunks of the lane's row
//   kPasses, mma<PASS>(acc, b, a) the MFMAs of one fragment pair (PASS 1.. are issued behind the
//                                 NT PASS 0 MFMAs of the same A fragment, so that two MFMAs
//                                 into one accumulator are NT issue slots apart)
//   kScaled                       (MXFP4) every operand row has 8 e8m0 scale bytes per K-step: mma<PASS>(acc, b, a, sb, sa)
//                                 takes the lane's scale bytes in bits [7:0] of sb / sa
//   raster_group(band_n, tiles_n) tile rows per raster group
// K: operand row pitch in bytes. `smem`: the workgroup's LDS, ring_lds_bytes(). STREAM_C: the epilogue's stores carry the
// non-temporal hint (store_c_tile).
//
// TILE_M x TILE_N: 256x256, or 192 rows or columns of it (a wave then owns 96x128 or 128x96). A round of 256 CUs costs the
// same whether it is full or not, and a 256x256 tile is a coarse unit: 3001 x 4096 takes 192 of them (64 CUs idle) and
// exactly 256 of 192x256, 4096 x 2880 takes 192 with 6 % of their columns past N and 240 of 256x192. The two shorter tiles
// also leave room beside the five slots for the block scales of MXFP4, whose 256x256 kernel has two stages and no
// more (mxfp4_gemm.hip). Every element of C is summed in the same order by all three.
// Scales: the two LDS slots (pairs of K-steps) in front of the operand slots, 16 bytes per row; each pair comes in with two
// loads per wave during the even K-step before it (see mxfp4_gemm.hip for the scale rows themselves).
struct RingScales {
    const uint8_t* SA; const uint8_t* SB; int sa_pitch, sb_pitch, tail_pair, tail_shift, row_bytes;
};
constexpr int kRingScaleSlot = 2 * 256 * 16;   // A's rows, then B's (256 of each, whatever the tile)
constexpr int ring_lds_bytes(int tile_m, int tile_n, bool scaled) {
    return (2 * tile_m + 3 * tile_n) * BK + (scaled ? 2 * kRingScaleSlot : 0);
}
// Rows past M or N are not clamped: they lie outside the descriptors, fetch nothing and arrive as zeros. This depends on the
// buffers' range check counting the scalar offset, which holds the K offset and the rows of a load (i * dma_row_stride): seen with
// an offset that wrapped, whose loads returned zeros. (With a row address per load, clamped to the last row, ragged problems had
// a register and a vector instruction per load more: BF16 3001 x 4096 x 4096 on 192x256 tiles 79.0 us, now 74.9.)
// EDGE: M or N is not a multiple of the tile (only the epilogue needs to know).
template <typename MMA, bool EDGE, bool STREAM_C = false, int TILE_M = BM, int TILE_N = BN>
__device__ __forceinline__ void gemm_ring_body(uint8_t* smem, const uint8_t* __restrict__ A,
                                               const uint8_t* __restrict__ B, uint16_t* __restrict__ C,
                                               int M, int N, int K, float alpha, int tiles_m, int tiles_n,
                                               int band_n, RingScales sc = RingScales{}) {
    using Frag = typename MMA::Frag;
    constexpr bool kScaled = MMA::kScaled;
    static_assert(MMA::kPasses == 1 || MMA::kPasses == 2, "the slot plan places at most two MFMAs per fragment pair");
    constexpr int NW = 4, TM = TILE_M / 2, TN = TILE_N / 2, MT = TM / 16, NT = TN / 16;
    constexpr int kATile = TILE_M * BK, kBTile = TILE_N * BK;
    constexpr int NDMA_A = kATile / (NW * 1024), NDMA_B = kBTile / (NW * 1024);  // loads per wave and K-step
    constexpr int AD = 3, PG = MT - AD - 1;   // A fragments read ahead; the barrier stands behind group PG
    constexpr uint32_t kScaleBytes = kScaled ? 2 * kRingScaleSlot : 0;
    constexpr uint32_t kBRing = 2 * kATile;          // B slots start behind the two A slots
    static_assert((MT == 8 || MT == 6) && (NT == 8 || NT == 6), "slot plan below is written for these");
    static_assert(!kScaled || MMA::kPasses == 2, "the scaled slot plan is written for two MFMAs per fragment pair");
    static_assert(ring_lds_bytes(TILE_M, TILE_N, kScaled) <= 160 * 1024, "LDS of one CU");

    const int lane = lane_id();
    const int w = wave_id();
    const int wm = w >> 1, wn = w & 1;

    int pm, pn;
    {
        const int id = xcd_chunk_order(blockIdx.x, tiles_m * tiles_n, kCuPerXcd);
        banded_raster(id, tiles_m, tiles_n, MMA::raster_group(band_n, tiles_n), band_n, pm, pn);
    }
    const int row0 = pm * TILE_M, col0 = pn * TILE_N;

    const int a_rows = min(M - row0, TILE_M), b_rows = min(N - col0, TILE_N);
    const v4i srd_a = make_srd(A + (size_t)row0 * K, (uint32_t)a_rows * (uint32_t)K);
    const v4i srd_b = make_srd(B + (size_t)col0 * K, (uint32_t)b_rows * (uint32_t)K);

    // load i of a tile covers its rows 8 (4 i + w) .. +8 (b_row_to_col permutes within 32 rows)
    uint32_t voff_a, voff_b;
    {
        const int R = 8 * w + (lane >> 3);
        const uint32_t c = swz_chunk(R, lane & 7) * 16u;
        voff_a = (uint32_t)R * (uint32_t)K + c;
        voff_b = (uint32_t)b_row_to_col(R) * (uint32_t)K + c;
    }
    const uint32_t dma_row_stride = to_sgpr((uint32_t)(8 * NW) * (uint32_t)K);
    const uint32_t lds_scales = (uint32_t)(uintptr_t)smem;
    const uint32_t lds0 = lds_scales + kScaleBytes;
    const uint32_t lds_wave = to_sgpr(lds0 + (uint32_t)w * 1024u);

    // One global->LDS load of A (into A slot `slot`) or B (into the B slot at byte offset
    // `slot_off` of the B ring).
    // `vor` is 0, or for the last K-step of a K that is not a multiple of the K-step the lane's
    // tail_or: bit 31 moves the lanes whose 16-byte chunk lies past the end of the row out of the
    // buffer's range, and such lanes write zeros to LDS.
    auto dma_a = [&](int i, int slot, uint32_t k0, v4i srd, uint32_t vor) {
        const uint32_t dst = lds_wave + (uint32_t)slot * kATile + i * NW * 1024;
        dma16(srd, dst, voff_a | vor, k0 + i * dma_row_stride);
    };
    auto dma_b = [&](int i, uint32_t slot_off, uint32_t k0, v4i srd, uint32_t vor) {
        const uint32_t dst = lds_wave + kBRing + slot_off + i * NW * 1024;
        dma16(srd, dst, voff_b | vor, k0 + i * dma_row_stride);
    };
    // Scales: this wave loads rows 64 w .. 64 w + 63 of each operand, lane l row 64 w + l, 16 bytes = the row's scales of
    // K-steps 2 p and 2 p + 1. (Rows past a 192-row tile repeat its last one.)
    v4i srd_sa = {0, 0, 0, 0}, srd_sb = {0, 0, 0, 0};
    uint32_t voff_sa = 0, voff_sb = 0;
    const uint32_t lds_scale_wave = to_sgpr(lds_scales + (uint32_t)w * 1024u);
    if constexpr (kScaled) {
        const int R = 64 * w + lane;
        srd_sa = make_srd(sc.SA + (size_t)row0 * sc.sa_pitch, (uint32_t)(a_rows - 1) * (uint32_t)sc.sa_pitch + (uint32_t)(sc.row_bytes ? sc.row_bytes : sc.sa_pitch));
        srd_sb = make_srd(sc.SB + (size_t)col0 * sc.sb_pitch, (uint32_t)(b_rows - 1) * (uint32_t)sc.sb_pitch + (uint32_t)(sc.row_bytes ? sc.row_bytes : sc.sb_pitch));
        voff_sa = (uint32_t)min(R, TILE_M - 1) * (uint32_t)sc.sa_pitch;
        voff_sb = (uint32_t)b_row_to_col(min(R, TILE_N - 1)) * (uint32_t)sc.sb_pitch;
    }
    // this wave's scale load of operand `op` (0 = A) for the pair of K-steps `pair` (slot pair % 2)
    auto dma_scale = [&](int op, uint32_t pair, v4i srd) {
        const uint32_t dst = lds_scale_wave + (pair & 1u) * kRingScaleSlot + op * (kRingScaleSlot / 2);
        dma16(srd, dst, op ? voff_sb : voff_sa, pair * 16u - ((int)pair == sc.tail_pair ? (uint32_t)sc.tail_shift : 0u));
    };

    const uint32_t r = lane & 15, g = lane >> 4;
    const uint32_t rd_lo = r * 128u + swz_chunk(r, g) * 16u;
    const uint32_t rd_hi = r * 128u + swz_chunk(r, g + 4) * 16u;
    uint32_t a_lo[2], a_hi[2];
#pragma unroll
    for (int st = 0; st < 2; ++st) {
        a_lo[st] = lds0 + st * kATile + wm * (TM * BK) + rd_lo;
        a_hi[st] = lds0 + st * kATile + wm * (TM * BK) + rd_hi;
    }
    const uint32_t b_lo0 = lds0 + kBRing + wn * (TN * BK) + rd_lo;
    const uint32_t b_hi0 = lds0 + kBRing + wn * (TN * BK) + rd_hi;
    // scales of fragment f, K-step parity p, in the slot of the running K-step's pair: base + 256 f + 8 p
    uint32_t sa_rd = lds_scales + (wm * TM + r) * 16u;
    uint32_t sb_rd = lds_scales + kRingScaleSlot / 2 + (wn * TN + r) * 16u;
    if constexpr (kScaled) asm volatile("" : "+v"(sa_rd), "+v"(sb_rd));   // the large base in the register, offsets in immediates
    const uint32_t sh = 8u * g;   // byte g of each scale dword belongs to this lane
    auto rd_scale = [&](uint32_t base, int p, int f) -> v2i { return *(lds_v2i_t*)(uintptr_t)(base + f * 256 + p * 8); };
    auto shift_scale = [&](v2i& s) {
        s.x = (int)((uint32_t)s.x >> sh);
        s.y = (int)((uint32_t)s.y >> sh);
    };

    v4f acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = v4f{0.f, 0.f, 0.f, 0.f};
    Frag bf[2][NT];  // B fragments of the current / next K-step
    Frag af[4];      // rotating A fragments: fragment m of a K-step of parity P in af[(P MT + m) % 4]
    v2i bs[kScaled ? 2 : 1][kScaled ? NT : 1], as[kScaled ? 4 : 1];   // their scales

    const int nk = (K + BK - 1) / BK;
    // the chunk a lane fetches is the same for all of its loads: swz(row, lane % 8) with row bits
    // [1..3] = 4 w + lane / 16 (mod 8)
    const uint32_t tail_or =
        (int)(swz_chunk(8 * w + (lane >> 3), lane & 7) * 16u) >= K - (nk - 1) * BK ? 0x80000000u : 0u;

    // ---- prologue: tiles 0 and 1 in flight, first fragments in registers ------------------
    {
        const uint32_t vor = nk == 1 ? tail_or : 0u;
#pragma unroll
        for (int i = 0; i < NDMA_B; ++i) dma_b(i, 0, 0, srd_b, vor);
#pragma unroll
        for (int i = 0; i < NDMA_A; ++i) dma_a(i, 0, 0, srd_a, vor);
        if constexpr (kScaled) { dma_scale(0, 0, srd_sa); dma_scale(1, 0, srd_sb); }
    }
    wait_vmcnt<0>();
    block_barrier();
    {
        v4i sa = srd_a, sb = srd_b;
        if (nk < 2) { sa.z = 0; sb.z = 0; }
        const uint32_t vor = nk == 2 ? tail_or : 0u;
#pragma unroll
        for (int i = 0; i < NDMA_B; ++i) dma_b(i, kBTile, BK, sb, vor);
#pragma unroll
        for (int i = 0; i < NDMA_A; ++i) dma_a(i, 1, BK, sa, vor);
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        bf[0][n] = MMA::load(b_lo0, b_hi0, n * 16 * BK);
        if constexpr (kScaled) bs[0][n] = rd_scale(sb_rd, 0, n);
    }
#pragma unroll
    for (int m = 0; m < AD; ++m) {
        af[m] = MMA::load(a_lo[0], a_hi[0], m * 16 * BK);
        if constexpr (kScaled) as[m] = rd_scale(sa_rd, 0, m);
    }
    if constexpr (kScaled) {
#pragma unroll
        for (int n = 0; n < NT; ++n) shift_scale(bs[0][n]);
        shift_scale(as[0]);   // the others are shifted in the group before their first use
    }

    // B ring positions (byte offsets): tile kt+1 is read from off1, tile kt+2 is loaded to off2.
    uint32_t off1 = kBTile, off2 = 2 * kBTile;

    // One K-step with A slot / fragment parity P. Every step runs the same code: the last step's
    // prefetch reads return stale LDS contents that are never used, and refills past the end of K
    // are issued against a zero-sized buffer (out of range for every lane, no memory traffic), so
    // that no step needs a differently scheduled body.
    auto step = [&]<int P>(int kt) {
        constexpr int PA = (P * MT) & 3, PB = ((P ^ 1) * MT) & 3;   // af[] position of fragment 0 of this K-step / of the next
        const uint32_t k2 = (uint32_t)(kt + 2) * BK;
        v4i sa = srd_a, sb = srd_b, ssa = srd_sa, ssb = srd_sb;
        if (kt + 2 >= nk) { sa.z = 0; sb.z = 0; ssa.z = 0; ssb.z = 0; }
        const uint32_t vor = kt + 2 == nk - 1 ? tail_or : 0u;
        const uint32_t bl = b_lo0 + off1, bh = b_hi0 + off1;
        // scales of the next K-step: the same pair (P == 0) or the next one, in the other slot (entering the pair that was
        // fetched tail_shift bytes early)
        const uint32_t early = kScaled && P && ((kt + 1) >> 1) == sc.tail_pair ? (uint32_t)sc.tail_shift : 0u;
        const uint32_t sa_nx = P ? (sa_rd ^ (uint32_t)kRingScaleSlot) + early : sa_rd;
        const uint32_t sb_nx = P ? (sb_rd ^ (uint32_t)kRingScaleSlot) + early : sb_rd;
        // The next K-step's A fragment j: its registers are free once group PG + j is done.
        auto read_a = [&](int j) __attribute__((always_inline)) { af[(PB + j) & 3] = MMA::load(a_lo[P ^ 1], a_hi[P ^ 1], j * 16 * BK); };
        auto read_b = [&](int n) __attribute__((always_inline)) { bf[P ^ 1][n] = MMA::load(bl, bh, n * 16 * BK); };
        // Two MFMAs per fragment pair (16-cycle MFMAs, each with room for about two other instructions, where
        // the 32-cycle FP8 MFMA has room for five): the operations behind the barrier are spread over all
        // MFMAs of both passes of the last three groups instead of those of the first pass (+1.5 % for BF16 at 8192^3).
        // Slot q (0 .. 6 NT - 1) = 2 NT (m - PG - 1) + NT pass + n: LDS reads in the even slots, unit q / 2 = the B fragments,
        // A0, A1, then A2 from q = 4 NT on; the A loads at q = 1, 5, ... (Splitting a load into its M0 write and the load
        // itself, one slot apart, which also saves the wait state between them, measured the same.)
        // Scaled: a fragment's scales take a unit of their own behind it, A0 and A1 come earlier among the B fragments, and
        // the next pair's two scale loads go out at q = 3 and 7 of even K-steps. (A scaled FP4 MFMA is 16 cycles long and has
        // room for about one other instruction.)
        auto post_ops = [&](int q) __attribute__((always_inline)) {
            if ((q & 1) == 0) {
                const int u = q / 2;
                if constexpr (kScaled) {
                    // fragments in the order of their units (0..7: B, 8..10: A)
                    constexpr int kOrder8[11] = {0, 1, 2, 3, 4, 8, 5, 6, 7, 9, 10}, kOrder6[11] = {0, 1, 2, 3, 4, 8, 5, 9, 10, -1, -1};
                    const int x = u / 2 < 11 ? (NT == 8 ? kOrder8[u / 2] : kOrder6[u / 2]) : -1;
                    if (x >= 0 && x < 8) {
                        if ((u & 1) == 0) read_b(x);
                        else bs[P ^ 1][x] = rd_scale(sb_nx, P ^ 1, x);
                    } else if (x >= 8) {
                        if ((u & 1) == 0) read_a(x - 8);
                        else as[(PB + x - 8) & 3] = rd_scale(sa_nx, P ^ 1, x - 8);
                    }
                } else {
                    if (u < NT) read_b(u);
                    else if (u == NT || u == NT + 1) read_a(u - NT);
                    else if (u == 2 * NT) read_a(2);
                }
            } else if (q % 4 == 1 && q / 4 < NDMA_A) {
                dma_a(q / 4, P, k2, sa, vor);
            } else if (kScaled && P == 0 && (q == 3 || q == 7)) {
                dma_scale(q == 7, (uint32_t)(kt >> 1) + 1u, q == 7 ? ssb : ssa);
            }
        };
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            constexpr int kPre = (PG + 1) * NT;   // first-pass slots before the barrier: the B loads are spread over them
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const int ai = (PA + m) & 3;
                if constexpr (kScaled) MMA::template mma<0>(acc[m][n], bf[P][n], af[ai], bs[P][n].x, as[ai].x);
                else MMA::template mma<0>(acc[m][n], bf[P][n], af[ai]);
                if (m <= PG) {
                    const int s = m * NT + n;
                    constexpr int kEvery = kPre / NDMA_B;   // 256x256: 40 slots, B loads at 2, 7, .., 37
                    if (n == 0) af[(PA + m + AD) & 3] = MMA::load(a_lo[P], a_hi[P], (m + AD) * 16 * BK);
                    if constexpr (kScaled)
                        if (n == 1) as[(PA + m + AD) & 3] = rd_scale(sa_rd, P, m + AD);
                    if (s % kEvery == 2 && s / kEvery < NDMA_B) dma_b(s / kEvery, off2, k2, sb, vor);
                } else if (MMA::kPasses == 2) {
                    post_ops((m - PG - 1) * 2 * NT + n);
                } else {
                    const int j = (m - PG - 1) * NT + n;  // 3 NT slots after the barrier
                    if (j < NT) read_b(j);
                    else if (j == NT || j == NT + 1) read_a(j - NT);
                    else if (j == 2 * NT) read_a(2);
                    if (j < 2 * NDMA_A && (j & 1)) dma_a(j >> 1, P, k2, sa, vor);  // A loads at 1, 3, ..
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int pass = 1; pass < MMA::kPasses; ++pass)
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    const int ai = (PA + m) & 3;
                    if constexpr (kScaled) {
                        MMA::template mma<1>(acc[m][n], bf[P][n], af[ai], bs[P][n].y, as[ai].y);
                        if (m == MT - 1) shift_scale(bs[P ^ 1][n]);
                        if (n == 4) shift_scale(as[m == MT - 1 ? PB : (PA + m + 1) & 3]);   // the next group's A fragment
                    } else {
                        MMA::template mma<1>(acc[m][n], bf[P][n], af[ai]);
                    }
                    if (m > PG) post_ops((m - PG - 1) * 2 * NT + NT + n);
                    __builtin_amdgcn_sched_barrier(0);
                }
            if (m == PG) {
                // every read of A slot P by this wave has been issued; tile kt+1 (all loads
                // but the B loads of this step) must have landed for all waves
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                wait_vmcnt<NDMA_B>();
                block_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        off1 = off2;
        off2 = off2 == 2 * kBTile ? 0u : off2 + kBTile;
        if (kScaled && P) {
            sa_rd = sa_nx;
            sb_rd = sb_nx;
        }
    };

    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
        step.template operator()<0>(kt);
        step.template operator()<1>(kt + 1);
    }
    if (kt < nk) step.template operator()<0>(kt);
    wait_vmcnt<0>();  // nothing may still be writing LDS when the workgroup retires
    mfma_drain_agpr(acc);

    store_c_tile<MT, NT, EDGE, STREAM_C>(acc, C, M, N, row0 + wm * TM, col0 + wn * TN, alpha);
}

}  // namespace hk
