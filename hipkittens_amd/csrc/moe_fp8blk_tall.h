// Grouped GEMM of the FP8 block-scaled MoE on pre-shuffled weights for experts with more rows than one item of
// moe_fp8blk_stream_kernel holds (included by moe_fp8blk.hip behind that kernel, whose slot plan this one shares).
//
// What bounds the streaming kernel there is the rate at which a CU takes data in (17-21 B/clk), and it asks for every
// weight byte once per item of 144 or 160 rows. Here an item has up to 288 rows: 8 waves, two per SIMD (256 registers
// each), as two row halves x four column waves; a wave owns up to 144 rows (the row fragments 2 m + wm) x 64 weight rows =
// 36 MFMAs per K-step, 144 accumulator registers. At 256 rows per expert a CU asks for 64 KiB per K-step and 256 x 256
// patch instead of 96. Both operands go through LDS, two slots each of 36 KiB of activations and 32 KiB of weights:
//   * a wave's four weight fragments are read into registers over the last twelve MFMAs of the position before, which go
//     through the last three row fragments column by column, so that one weight fragment after the other is done with
//     (read in one go behind the last MFMA, 64 reads of the eight waves met in front of the next one: 1 % of the layer);
//     a barrier then frees the slot, and the weights of the position after the next are requested into it: they have
//     more than a K-step to arrive from HBM;
//   * the activation tile of the position after the next is requested when everyone has read this one's, ahead of the
//     position's last nine MFMAs.
// The only wait for loads is vmcnt(4) at the change of position: everything but the four weight pieces of the position
// after the next, which are the youngest loads; how many loads are older does not matter, so that waves 4..7 need not
// make up for the activation pieces they do not have (36 pieces of 8 rows over 8 waves).
// The K loop exists for items of five to nine pairs of row fragments: rows of experts that are asked for unevenly fill two
// thirds of their items (all items through the nine: 4319 us instead of 3895). The epilogue, shared, tests each fragment.
// No non-temporal hint on the weights, which an expert's second item wants from L2 (3907 / 3831 us with / without it).
// DeepSeek-V3-like layer, 8192 tokens, rows per expert 256 +- 206: 4118-4201 us with the streaming kernel, 3728-3838 with this one
// (gate+up 2595 -> 2342, down 1408 -> 1273, both traced in turn on one box); 256 +- 16: 3760 / 3269. What bounds it now is power as much as latency: the
// clock is 1.64-1.79 GHz where the streaming kernel's is 1.84-1.93, the matrix cores are busy 51-53 % of the time.
// Same MFMA, K order and scaling FMAs as the other two kernels: the same bits.
#pragma once
#include <utility>

namespace hk {

constexpr int kF8tMT = 9;                                // row fragments of a wave
constexpr int kF8tBM = 32 * kF8tMT;                      // 288 rows per item
constexpr int kF8tATile = kF8tBM * 128;
constexpr int kF8tB = 2 * kF8tATile;                     // LDS: two A slots, two B slots,
constexpr int kF8tSa = kF8tB + 2 * kF8sBTile;            // two buffers of row scales (gate+up: of four K-steps each),
constexpr int kF8tSaBuf = kF8tBM * 16;
constexpr int kF8tXch = kF8tSa + 2 * kF8tSaBuf;          // the epilogue's exchange buffer
constexpr int kF8tIds = kF8tXch + kF8tBM * 16;           // and the waves' slot ids
constexpr int kF8tLds = kF8tIds + 8 * 512;               // 153.5 KiB
typedef __attribute__((address_space(3))) const uint32_t lds_u32_t;
static_assert(kF8tLds <= 160 * 1024 && kF8tMT == 9, "LDS plan; the K loops are written out for five to nine fragments");

struct F8TallItem { int expert, row_start, rows, n_tile; };

// MODE 0: gate+up, activation rows gathered from the caller's x by token. MODE 1: down, rows of h. K >= 384.
template <int MODE>
__global__ __launch_bounds__(512) void moe_fp8blk_tall_kernel(const MoeFp8Params p) {
    constexpr bool GATHER = MODE == 0;
    constexpr int MT = kF8tMT, NT = 4, NA = 5, SR = kF8tBM / 8;
    extern __shared__ __attribute__((aligned(2048))) uint8_t smem[];
    const int lane = lane_id(), w = wave_id();
    const int wm = w >> 2, wn = w & 3;

    const int n_items = (int)to_sgpr((uint32_t)scalar_load_x1(p.num_items));
    const int xcd = blockIdx.x % kNumXcd, slot = blockIdx.x / kNumXcd;
    const int it_stride = ((int)gridDim.x - xcd + kNumXcd - 1) / kNumXcd;
    const int per_xcd = (n_items + kNumXcd - 1) / kNumXcd;
    int it = xcd * per_xcd + slot;
    int it_end_v = min(n_items, (xcd + 1) * per_xcd);
    if (it >= it_end_v) return;
    asm volatile("" : "+v"(it_end_v));   // (kept in a vector register, for want of a scalar one)
    auto it_end = [&]() __attribute__((always_inline)) { return (int)to_sgpr((uint32_t)it_end_v); };

    const int nk = p.K >> 7;
    __builtin_assume(nk >= 3);
    // Arguments that an item needs once are read again from the argument segment there: kept, they and the descriptors of
    // the K loop would be more scalar registers than there are.
    auto pointer_arg = []<int AT>() __attribute__((always_inline)) {
        uint64_t v;
        asm volatile("s_load_dwordx2 %0, %1, %2\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(__builtin_amdgcn_kernarg_segment_ptr()), "n"(AT) : "memory");
        return (uint64_t)to_sgpr((uint32_t)v) | (uint64_t)to_sgpr((uint32_t)(v >> 32)) << 32;
    };
#define HK_LATE(field) ((decltype(MoeFp8Params::field))pointer_arg.template operator()<offsetof(MoeFp8Params, field)>())
    const v4i srd_a = make_srd(p.A, GATHER ? (uint32_t)p.T * (uint32_t)p.K : (uint32_t)nk * (uint32_t)p.S * 128u);
    const v4i srd_sa = make_srd(p.SA, GATHER ? (uint32_t)p.T * (uint32_t)nk * 4u : (uint32_t)nk * (uint32_t)p.S * 4u);

    auto load_item = [&](int idx, F8TallItem& c) __attribute__((always_inline)) {
        // (past the end: the last item once more; what is fetched for it is not used)
        const v4i item = scalar_load_x4(HK_LATE(items) + min(idx, it_end() - 1));
        // (read through to_sgpr: merged over the ways through an item the results of assembly would be vector registers)
        c.expert = (int)to_sgpr((uint32_t)item.x); c.row_start = (int)to_sgpr((uint32_t)item.y);
        c.rows = (int)to_sgpr((uint32_t)item.z); c.n_tile = (int)to_sgpr((uint32_t)item.w);
    };
    // descriptor of an item's weight tile
    auto b_srd_of = [&](const F8TallItem& c) __attribute__((always_inline)) {
        return make_srd(HK_LATE(B) + (size_t)c.expert * HK_LATE(b_expert_stride) + (size_t)c.n_tile * nk * kF8sBTile, (uint32_t)nk * kF8sBTile);
    };
    // byte offset of its weight scales (gate rows / this wave's rows), K-step 0
    auto ws_of = [&](const F8TallItem& c) __attribute__((always_inline)) {
        const int block = MODE == 0 ? c.n_tile : min(2 * c.n_tile + (wn >> 1), p.N / 128 - 1);
        return to_sgpr((uint32_t)(c.expert * (int)HK_LATE(sb_expert_stride) + block * nk) * 4u);
    };

    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

    // ---- what this lane loads: rows 64 i + 8 w + lane / 8 of the activation tile (i = 4: waves 0..3), row scale SR w + lane
    // (found from the lane's number where an item needs it: kept, these would be registers too many)
    auto lane_here = []() __attribute__((always_inline)) {
        int l;
        asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
        return l;
    };
    auto piece_row = [&](int l, int i) { return 64 * i + 8 * w + (l >> 3); };
    auto scale_row_of = [&](int l) { return SR * w + min(l, SR - 1); };
    constexpr uint64_t kSaMask = (1ull << SR) - 1ull;
    // GATHER: the slot ids of the rows, a wave's 40 + SR, come through LDS as well (a conditional load into registers could be
    // merged with their old values by copies that do not wait for it)
    const uint32_t lds_ids = lds0 + kF8tIds + (uint32_t)w * 512u;
    auto issue_ids = [&](int row_start) __attribute__((always_inline)) {
        const int l = lane_here();
        const v4i srd = make_srd(HK_LATE(sorted_slots), (uint32_t)p.S * 4u);   // (ids past its end read as zero: rows that no item has)
        dma4_lanes(srd, lds_ids, (uint32_t)(row_start + 64 * (l >> 3) + 8 * w + (l & 7)) * 4u, 0u, (1ull << 40) - 1ull);
        dma4_lanes(srd, lds_ids + 256u, (uint32_t)(row_start + scale_row_of(l)) * 4u, 0u, kSaMask);
    };
    // byte offsets of the rows in x (or in an item of h) and in their scales
    uint32_t a_voff[NA], sa_voff;
    // slot / topk: with m = ceil(2^31 / topk), 2 slot m / 2^32 exceeds the quotient by slot (m topk - 2^31) / (2^31 topk),
    // less than 1 / topk while slot * topk < 2^31 (here slot < 2^24, topk <= 64)
    const uint32_t topk_m = to_sgpr((0x80000000u + (uint32_t)p.topk - 1u) / (uint32_t)p.topk);
    auto token_of = [&](uint32_t slot) { return __umulhi(2u * slot, topk_m); };
    auto make_offsets = [&](int rows) __attribute__((always_inline)) {
        asm volatile("" : "+s"(rows));
        const int l = lane_here();
        const uint32_t chunk16 = swz_chunk(8 * w + (l >> 3), l & 7) * 16u;   // the same for every piece
        if constexpr (GATHER) {
            // rows past the item's count are not fetched (bit 31: out of range, LDS gets zeros)
            uint32_t ids = lds_ids + 4u * (uint32_t)(l >> 3);
            asm volatile("" : "+v"(ids));
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                const uint32_t id = *(lds_u32_t*)(uintptr_t)(ids + 32u * i);
                a_voff[i] = piece_row(l, i) < rows ? token_of(id) * ((uint32_t)nk << 7) + chunk16 : 0x80000000u;
            }
            const uint32_t id = *(lds_u32_t*)(uintptr_t)(lds_ids + 256u + 4u * (uint32_t)min(l, SR - 1));
            sa_voff = scale_row_of(l) < rows ? token_of(id) * (uint32_t)nk * 4u : 0x80000000u;
        } else {
            a_voff[0] = (uint32_t)piece_row(l, 0) * 128u + chunk16;
            sa_voff = (uint32_t)scale_row_of(l) * 4u;
        }
    };

    const uint32_t voff_b = lane * 16;
    // GATHER: first of the four K-steps whose scales come in with K-step kt (a multiple of four): inside the row
    auto sa_first = [&](int kt) { return max(min(kt, nk - 4), 0); };
    uint32_t f_sa = 0, c_sa = 0;   // GATHER: offsets of the scale buffers that the next load fills / the next position reads

    // uniform state of the fetches of a position, made at its start
    v4i fb_srd;
    uint32_t fa_soff, fsa_soff, fb_soff, fa_dst, fb_dst;
    int fa_rows;
    bool fsa_on;
    auto set_fetch_a = [&](int row_start, int rows, int kt, uint32_t slot_a) __attribute__((always_inline)) {
        const uint32_t row_base = (uint32_t)kt * (uint32_t)p.S + (uint32_t)row_start;
        fa_soff = GATHER ? (uint32_t)kt * 128u : row_base * 128u;
        fsa_soff = GATHER ? (uint32_t)sa_first(kt) * 4u : row_base * 4u;
        fa_dst = lds0 + (uint32_t)w * 1024u + slot_a * kF8tATile;
        fa_rows = rows;
        fsa_on = !GATHER || (kt & 3) == 0;
        if (!GATHER) f_sa = slot_a * kF8tSaBuf;
    };
    auto set_fetch_b = [&](int kt, uint32_t slot_b) __attribute__((always_inline)) {
        fb_soff = (uint32_t)kt * kF8sBTile + (uint32_t)w * 4096u;
        fb_dst = lds0 + kF8tB + (uint32_t)w * 4096u + slot_b * kF8sBTile;
    };
    auto load_a = [&]<int I>() __attribute__((always_inline)) {
        if constexpr (GATHER) {
            dma16(srd_a, fa_dst + I * 8192, a_voff[I], fa_soff);
        } else {
            v4i s = srd_a;   // the piece's 8 rows lie past the item's count: nothing is fetched
            if (64 * I + 8 * w >= fa_rows) s.z = 0;
            dma16(s, fa_dst + I * 8192, a_voff[0], fa_soff + I * 8192u);
        }
    };
    auto load_sa = [&]() __attribute__((always_inline)) {
        if constexpr (GATHER) {
            if (fsa_on) {
                dma16_lanes(srd_sa, lds0 + kF8tSa + (uint32_t)w * (SR * (GATHER ? 16u : 4u)) + f_sa, sa_voff, fsa_soff, kSaMask);
                f_sa = kF8tSaBuf - f_sa;
            }
        } else {
            dma4_lanes(srd_sa, lds0 + kF8tSa + (uint32_t)w * (SR * (GATHER ? 16u : 4u)) + f_sa, sa_voff, fsa_soff, kSaMask);
        }
    };
    auto load_b = [&]<int I>() __attribute__((always_inline)) {
        dma16(fb_srd, fb_dst + I * 1024, voff_b, fb_soff + I * 1024u);
    };

    // ---- LDS -> registers ----
    const uint32_t r = lane & 15, g = lane >> 4;
    constexpr int kSaStep = 32 * (GATHER ? 16 : 4);   // bytes between the scales of a lane's consecutive fragments
    // of the compute position (chunk g + 4 of a row lies 64 bytes from chunk g, in the direction of its bit 6)
    uint32_t a_lo = lds0 + wm * 2048 + r * 128u + swz_chunk(r, g) * 16u, b_rd = lds0 + kF8tB + wn * 8192 + lane * 16u,
             a_sa = lds0 + kF8tSa + (wm * 16 + r) * (GATHER ? 16u : 4u);
    uint32_t sa_off = 0;   // GATHER: a_sa's distance from the row's first scale in the first buffer
    float acc[MT][NT][4];
    // D(16 weight rows x 16 rows) = W . A^T into fresh registers
    auto mfma = [&](v4f& d, const v8i& b, const v8i& a) __attribute__((always_inline)) {
        asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0" : "=v"(d) : "v"(b), "v"(a));
    };
    // acc += part * s; placed two MFMAs behind the one that produced `part` (the compiler does not know the MFMA's latency)
    auto fma4 = [&](float (&a)[4], const v4f& pt, float s) __attribute__((always_inline)) {
        asm volatile("v_fma_f32 %0, %4, %8, %0\n\tv_fma_f32 %1, %5, %8, %1\n\tv_fma_f32 %2, %6, %8, %2\n\tv_fma_f32 %3, %7, %8, %3"
                     : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3])
                     : "v"(pt.x), "v"(pt.y), "v"(pt.z), "v"(pt.w), "v"(s));
    };
    // weight scales of a position, requested a position earlier
    struct WScale { uint32_t gate, up; };
    auto request_ws = [&](uint32_t off, WScale& o) __attribute__((always_inline)) {
        asm volatile("s_load_dword %0, %1, %2" : "=s"(o.gate) : "s"(p.SB), "s"(off) : "memory");
        if (MODE == 0) asm volatile("s_load_dword %0, %1, %2" : "=s"(o.up) : "s"(p.SB), "s"(off + (uint32_t)(p.N / 128 * nk) * 4u) : "memory");
    };
    auto landed_ws = [&](WScale& o) __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // also: this wave's LDS reads so far have returned
        asm volatile("" : "+s"(o.gate), "+s"(o.up));
    };

    // Stores through descriptors that end at the item's last row: rows past it are dropped by the range check.
    auto epilogue = [&](const F8TallItem& a) __attribute__((always_inline)) {
        const int l = lane_here();
        const uint32_t r = l & 15, g = l >> 4;
        // fragment m has rows while 32 m < left (read back from a vector register, so that it is not tested ahead of the K loop)
        int wave = w;
        asm volatile("" : "+v"(wave));
        const uint32_t wave_col = (uint32_t)wave & 3u, row_of_lane = 16u * ((uint32_t)wave >> 2) + r;
        const int left = a.rows - (int)to_sgpr(row_of_lane - r);
        if (MODE == 1) {
            const uint32_t pitch = (uint32_t)p.N * 2u;
            const v4i srd = make_srd((uint8_t*)HK_LATE(out0) + (size_t)a.row_start * pitch, (uint32_t)a.rows * pitch);
            const int wcol0 = a.n_tile * 256 + (int)to_sgpr(wave_col) * 64;   // N % 128 == 0: a group of 32 columns is valid as a whole
            const bool ok0 = wcol0 < p.N, ok1 = wcol0 + 32 < p.N;
            uint32_t voff = row_of_lane * pitch + (uint32_t)(wcol0 + 8 * (int)g) * 2u;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (32 * m < left) {
#pragma unroll
                    for (int q = 0; q < NT / 2; ++q) {
                        const float (&x)[4] = acc[m][2 * q];
                        const float (&y)[4] = acc[m][2 * q + 1];
                        v4i o4;
                        o4.x = pack_bf16(x[0], x[1]); o4.y = pack_bf16(x[2], x[3]);
                        o4.z = pack_bf16(y[0], y[1]); o4.w = pack_bf16(y[2], y[3]);
                        if (q == 0 ? ok0 : ok1)
                            asm volatile("buffer_store_dwordx4 %0, %1, %2, 0 offen offset:%3\n\ts_nop 1"
                                         :: "v"(o4), "v"(voff), "s"(srd), "n"(q * 64) : "memory");
                    }
                    voff += 32u * pitch;
                }
            }
        } else {
            // h = silu(gate) * up for this wave's 32 of the tile's 128 h columns, which are one 1 x 128 quantization
            // block: the row maxima of the four column waves are combined through LDS
            const size_t row0 = (size_t)a.n_tile * p.S + (size_t)a.row_start;
            const v4i srd_h = make_srd((uint8_t*)HK_LATE(out0) + row0 * 128, (uint32_t)a.rows * 128u);
            const v4i srd_s = make_srd(HK_LATE(out_scales) + row0, (uint32_t)a.rows * 4u);
            uint32_t voff_h = row_of_lane * 128u + 32u * (uint32_t)wave_col + 8u * g;
            uint32_t voff_s = wave_col == 0 && g == 0 ? row_of_lane * 4u : 0x80000000u;
            const uint32_t xch = lds0 + kF8tXch + row_of_lane * 16u, xch_w = xch + 4u * (uint32_t)wave_col;
            float h[MT][8];
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (32 * m < left) {
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int j = 0; j < 4; ++j) h[m][4 * q + j] = silu_mul(acc[m][2 * q][j], acc[m][2 * q + 1][j]);
                    float amax = 0.f;
#pragma unroll
                    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(h[m][i]));
                    const uint32_t am = __float_as_uint(amax);
                    const auto s16 = __builtin_amdgcn_permlane16_swap(am, am, false, false);
                    const uint32_t m1 = __float_as_uint(fmaxf(__uint_as_float(s16[0]), __uint_as_float(s16[1])));
                    const auto s32 = __builtin_amdgcn_permlane32_swap(m1, m1, false, false);
                    amax = fmaxf(__uint_as_float(s32[0]), __uint_as_float(s32[1]));
                    if (g == 0) *(lds_f32_mut_t*)(uintptr_t)(xch_w + m * 512) = amax;
                }
            }
            __syncthreads();
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (32 * m < left) {
                    const v4f am = *(lds_v4f_t*)(uintptr_t)(xch + m * 512);
                    const float s = e4m3_block_scale(fmaxf(fmaxf(am.x, am.y), fmaxf(am.z, am.w)));
                    const v2i q8 = quant8_e4m3(h[m], s);
                    asm volatile("buffer_store_dwordx2 %0, %1, %2, 0 offen" :: "v"(q8), "v"(voff_h), "s"(srd_h) : "memory");
                    asm volatile("buffer_store_dword %0, %1, %2, 0 offen" :: "v"(s), "v"(voff_s), "s"(srd_s) : "memory");
                    voff_h += 32u * 128u;
                    voff_s += 32u * 4u;
                }
            }
            // (the next epilogue writes the buffer again: several barriers of the K loop lie between)
        }
    };

    // ---- prologue: the first two positions ----
    F8TallItem cur, nxt;
    load_item(it, cur);
    if (GATHER) {
        issue_ids(cur.row_start);
        wait_vmcnt<0>();
    }
    make_offsets(cur.rows);
    auto fetch_a = [&](int kt) __attribute__((always_inline)) {
        set_fetch_a(cur.row_start, cur.rows, kt, (uint32_t)kt);
        load_a.template operator()<0>(); load_a.template operator()<1>(); load_a.template operator()<2>(); load_a.template operator()<3>();
        if (w < 4) load_a.template operator()<4>();
        load_sa();
    };
    auto fetch_b = [&](int kt) __attribute__((always_inline)) {
        set_fetch_b(kt, (uint32_t)kt);
        load_b.template operator()<0>(); load_b.template operator()<1>(); load_b.template operator()<2>(); load_b.template operator()<3>();
    };
    fb_srd = b_srd_of(cur);
    fetch_a(0); fetch_b(0); fetch_a(1); fetch_b(1);
    load_item(it + it_stride, nxt);
    wait_vmcnt<4>();
    block_barrier();
    slot_fence();
    uint32_t st = 0;   // LDS slot of the compute position

    // The K loop of an item of up to 32 MTX rows.
    auto run_item = [&]<int MTX>() __attribute__((always_inline)) {
        WScale ws_next{};
        const uint32_t ws_row = ws_of(cur);
        request_ws(ws_row, ws_next);
        landed_ws(ws_next);
        WScale ws{to_sgpr(ws_next.gate), to_sgpr(ws_next.up)};
        v8i bf[NT];              // weight fragments of the position
        auto read_bf = [&]<int N>() __attribute__((always_inline)) { bf[N] = lds_frag(b_rd, b_rd + 1024, N * 2048); };
        v8i af[3];               // activation fragments and their rows' scales
        float xs_r[3];
        float sc[3][2] = {};     // by buffer: x_scale * w_scale of the gate (even) / up (odd) weight fragments
        v4f part[NT] = {};       // partial sums of the last four MFMAs
#pragma unroll
        for (int m = 0; m < MTX; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[m][n][e] = 0.f;
        // the first position's fragments (the last position of the item before has read them too: kept, they would be in
        // registers across the epilogue)
        af[0] = lds_frag(a_lo, a_lo ^ 64u, 0);
        xs_r[0] = *(lds_f32_t*)(uintptr_t)a_sa;
        read_bf.template operator()<0>(); read_bf.template operator()<1>(); read_bf.template operator()<2>(); read_bf.template operator()<3>();
        // A position: 4 MTX slots, one MFMA each, in an order in which a weight fragment's register is free for the next
        // position's before the end: fragment by fragment, but for the last three fragments, which go through weight
        // fragment 0 first, then 1, 2, 3. The FMAs of an MFMA follow two slots later (slots 0 and 1: of the last position).
        constexpr int TAIL = 4 * (MTX - 3);
        constexpr auto frag_of = [](int i) { return i < TAIL ? i / 4 : MTX - 3 + (i - TAIL) % 3; };
        constexpr auto col_of = [](int i) { return i < TAIL ? i % 4 : (i - TAIL) / 3; };
        // buffer of an activation fragment: the last three all in different ones, the first in that of the last but two,
        // which is the first to be free, neighbours in different ones
        constexpr auto buf_of = [](int m) {
            constexpr int x = 1 + ((MTX - 5) & 1);   // of fragment MTX - 4
            return m == 0 || m == MTX - 3 ? 0 : m < MTX - 3 ? 1 + ((m - 1) & 1) : m == MTX - 2 ? 3 - x : x;
        };
        for (int kt = 0; kt < nk; ++kt) {
            request_ws(ws_row + 4u * (uint32_t)min(kt + 1, nk - 1), ws_next);
            const bool over = kt + 2 >= nk;   // the position after the next belongs to the next item
            const int k2 = over ? kt + 2 - nk : kt + 2;
            if (kt + 2 == nk) fb_srd = b_srd_of(nxt);
            set_fetch_b(k2, st);
            set_fetch_a(over ? nxt.row_start : cur.row_start, over ? nxt.rows : cur.rows, k2, st);
            __builtin_amdgcn_sched_barrier(0);
            auto slot = [&]<int I>() __attribute__((always_inline)) {
                constexpr int M = frag_of(I), N = col_of(I), B = buf_of(M), J = I - TAIL;
                constexpr int IP = I >= 2 ? I - 2 : I + 4 * MTX - 2, MP = frag_of(IP), NP = col_of(IP), BP = buf_of(MP);
                mfma(part[I & 3], bf[N], af[B]);
                auto read_frag = [&]<int F>() __attribute__((always_inline)) {
                    af[buf_of(F)] = lds_frag(a_lo, a_lo ^ 64u, F * 4096);
                    xs_r[buf_of(F)] = *(lds_f32_t*)(uintptr_t)(a_sa + F * kSaStep);
                };
                if constexpr (J < 0 && N == 0) read_frag.template operator()<M + 1>();
                if constexpr (J == -2) read_frag.template operator()<MTX - 2>();
                if constexpr (J == 0) read_frag.template operator()<MTX - 1>();
                if constexpr (J == 2) {
                    // the change of position: its tile has landed for everyone, everyone has read this one's
                    landed_ws(ws_next);
                    wait_vmcnt<4>();
                    block_barrier();
                    slot_fence();
                    st ^= 1u;
                    a_lo += st ? kF8tATile : -kF8tATile;
                    b_rd += st ? kF8sBTile : -kF8sBTile;
                    if constexpr (GATHER) {
                        const int kn = kt + 1 < nk ? kt + 1 : 0;
                        if ((kn & 3) == 0) c_sa = kF8tSaBuf - c_sa;
                        const uint32_t off = c_sa + 4u * (uint32_t)(kn - sa_first(kn & ~3));
                        a_sa += off - sa_off;
                        sa_off = off;
                        if (kt + 2 == nk) make_offsets(nxt.rows);
                    } else {
                        a_sa += st ? kF8tSaBuf : -kF8tSaBuf;
                    }
                }
                fma4(acc[MP][NP], part[IP & 3], sc[BP][NP & 1]);
                if constexpr ((J < 0 && N == 1) || (J >= 1 && J <= 3)) {
                    constexpr int F = J < 0 ? M : MTX - 4 + J, FB = buf_of(F);
                    sc[FB][0] = xs_r[FB] * __uint_as_float(ws.gate);
                    sc[FB][1] = MODE == 0 ? xs_r[FB] * __uint_as_float(ws.up) : sc[FB][0];
                }
                if constexpr (J == 2) read_bf.template operator()<0>();
                if constexpr (J == 5) read_bf.template operator()<1>();
                if constexpr (J == 8) read_bf.template operator()<2>();
                if constexpr (J == 9) read_frag.template operator()<0>();
                if constexpr (J == 11) read_bf.template operator()<3>();
                // loads: the weights two positions on, when everyone holds its fragments of this one's; the activations two
                // positions on, when everyone has read this one's
                if constexpr (I == 5) { block_barrier(); slot_fence(); }
                constexpr int LB = MTX > 5 ? I - 7 : 2 * (I - 6);
                if constexpr (LB >= 0 && LB < 8 && (LB & 1) == 0) load_b.template operator()<LB / 2>();
                if constexpr (J == 3) load_a.template operator()<0>();
                if constexpr (J == 4) load_a.template operator()<1>();
                if constexpr (J == 6) load_a.template operator()<2>();
                if constexpr (J == 7) load_a.template operator()<3>();
                if constexpr (J == 10) { if (w < 4) load_a.template operator()<4>(); }
                if constexpr (J == 11) {
                    load_sa();
                    // (older than the next position's weights, whose wait covers them)
                    if (GATHER && kt + 3 == nk) issue_ids(nxt.row_start);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) {
                (slot.template operator()<I>(), ...);
            }(std::make_integer_sequence<int, 4 * MTX>{});
            ws = ws_next;
        }
        // the item is complete: the two FMA groups still owed
        mfma_drain();
        fma4(acc[MTX - 2][3], part[2], sc[buf_of(MTX - 2)][1]);
        fma4(acc[MTX - 1][3], part[3], sc[buf_of(MTX - 1)][1]);
        // (not used: gives the registers of the fragments that the item does not have a value on every way here)
#pragma unroll
        for (int m = MTX; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[m][n][e] = 0.f;
    };

    for (;;) {
        const int frags = (cur.rows + 31) >> 5;
        if (frags >= 9) run_item.template operator()<9>();
        else if (frags == 8) run_item.template operator()<8>();
        else if (frags == 7) run_item.template operator()<7>();
        else if (frags == 6) run_item.template operator()<6>();
        else run_item.template operator()<5>();
        epilogue(cur);
        it += it_stride;
        if (it >= it_end()) break;
        cur = nxt;
        load_item(it + it_stride, nxt);
    }
    wait_vmcnt<0>();   // nothing may still be writing LDS when the workgroup retires
}

#undef HK_LATE

}  // namespace hk
