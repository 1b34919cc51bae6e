// Grouped GEMM of the MXFP4 MoE on pre-shuffled weights for experts with more rows than one item of
// moe_mxfp4_stream4_kernel holds (included by moe_mxfp4.hip behind that kernel; MXFP4 activations in sorted order).
//
// Where several items share an expert the streaming kernel is bound by what the one wave of a SIMD issues beside its MFMAs.
// This is the structure of moe_fp8blk_tall_kernel with the scales in the MFMA: 8 waves, two per SIMD, as two row halves x four
// column waves; a wave owns up to 144 rows (the row fragments 2 m + wm) x 64 weight rows, i.e. 72 MFMAs per K-step; both operands
// and both kinds of scales go through two LDS slots each. A wave's weight fragments are read over the last 24 MFMAs of the
// position before, which go through the last three row fragments column by column; a barrier then frees the weight slot for the
// position after the next, and the activations of that position are requested at the change of position. The only wait for
// loads is vmcnt(5): everything but the weights and weight scales of the position after the next. A row's scale byte is read
// from LDS as a byte (no shift), a weight's is picked by the MFMA. The K loop exists for items of five to nine pairs of row
// fragments; the epilogue, shared, tests each fragment.
// GPT-OSS-like layer, 16384 tokens, biases and clamped SwiGLU: 1239-1274 us with the streaming kernel, 1163-1201 with this one (gate+up
// 836 -> 785, down 406 -> 394, both traced in turn on one box). What bounds it (development builds, layer, us): without epilogues 1015, on empty loads 1022, both
// 866, of which 140 are not GEMMs: MFMAs, LDS reads and two barriers a position take 1.7 times the MFMAs' own time, the epilogue of
// all eight waves at once 150, and what loads cost on top 150; matrix cores busy 41 % at 1.83 GHz.
// Same MFMA and K order as the other kernels: the same bits.
#pragma once
#include <utility>

namespace hk {

constexpr int kTlMT = 9;                                 // row fragments of a wave
constexpr int kTlBM = 32 * kTlMT;                        // 288 rows per item
constexpr int kTlATile = kTlBM * 128;
constexpr int kTlB = 2 * kTlATile;                       // LDS: two A slots, two B slots,
constexpr int kTlSa = kTlB + 2 * kMoeBTile;              // two of row scales, two of weight scales,
constexpr int kTlSaTile = kTlBM * 8;
constexpr int kTlSb = kTlSa + 2 * kTlSaTile;
constexpr int kTlBias = kTlSb + 2 * kMoeScaleB;          // each wave's 64 biases of the item
constexpr int kTlLds = kTlBias + 8 * 256;                // 146.5 KiB
static_assert(kTlLds <= 160 * 1024 && kTlMT == 9, "LDS plan; the K loops are written out for five to nine fragments");

typedef __attribute__((address_space(3))) const int lds_i32_t;
typedef __attribute__((address_space(3))) const uint8_t lds_u8_t;
typedef __attribute__((address_space(3))) const v4f lds_v4f_t;
struct MxTallItem { int expert, row_start, rows, n_tile; };

// MODE, EXT: as in moe_mxfp4_stream4_kernel. At least three K-steps.
template <int MODE, int EXT>
__global__ __launch_bounds__(512) void moe_mxfp4_tall_kernel(const MoeGemmParams p) {
    constexpr int MT = kTlMT, NT = 4, SR = kTlBM / 8;
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

    const int nk = ((p.K >> 1) + 127) >> 7;
    __builtin_assume(nk >= 3);
    // Arguments that an item needs once are read again from the argument segment there (see moe_fp8blk_tall.h).
    auto pointer_arg = []<int AT>() __attribute__((always_inline)) {
        uint64_t v;
        asm volatile("s_load_dwordx2 %0, %1, %2\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(__builtin_amdgcn_kernarg_segment_ptr()), "n"(AT) : "memory");
        return (uint64_t)to_sgpr((uint32_t)v) | (uint64_t)to_sgpr((uint32_t)(v >> 32)) << 32;
    };
#define HK_LATE(field) ((decltype(MoeGemmParams::field))pointer_arg.template operator()<offsetof(MoeGemmParams, field)>())
#define HK_LATE_INT(field) ((int)(uint32_t)pointer_arg.template operator()<offsetof(MoeGemmParams, field)>())

    auto load_item = [&](int idx, MxTallItem& c) __attribute__((always_inline)) {
        // (past the end: the last item once more; what is fetched for it is not used)
        const v4i item = scalar_load_x4(HK_LATE(items) + min(idx, it_end() - 1));
        c.expert = (int)to_sgpr((uint32_t)item.x); c.row_start = (int)to_sgpr((uint32_t)item.y);
        c.rows = (int)to_sgpr((uint32_t)item.z); c.n_tile = (int)to_sgpr((uint32_t)item.w);
    };
    // descriptors of an item's weight tile and of its scales
    v4i fb_srd, fsb_srd;
    auto set_weights = [&](const MxTallItem& c) __attribute__((always_inline)) {
        fb_srd = make_srd(HK_LATE(B) + (size_t)c.expert * HK_LATE(b_expert_stride) + (size_t)c.n_tile * nk * kMoeBTile, (uint32_t)nk * kMoeBTile);
        fsb_srd = make_srd(HK_LATE(SB) + (size_t)c.expert * HK_LATE(sb_expert_stride) + (size_t)c.n_tile * nk * kMoeScaleB, (uint32_t)nk * kMoeScaleB);
    };

    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    auto lane_here = []() __attribute__((always_inline)) {   // (once an item: kept, what follows from it would be registers too many)
        int l;
        asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
        return l;
    };
    // ---- loads of a position: this wave's rows 64 i + 8 w + lane / 8 of the activation tile (i = 4: waves 0..3), the scales of
    // rows SR w .. +SR, four 1 KiB pieces of the weight tile and its 256 bytes of weight scales ----
    const uint32_t voff_a = (uint32_t)(8 * w + (lane >> 3)) * 128u + swz_chunk(8 * w + (lane >> 3), lane & 7) * 16u;
    const uint32_t voff_b = lane * 16;
    constexpr uint64_t kSaMask = (1ull << (SR / 2)) - 1ull;
    const uint32_t tail_kill = (p.K >> 1) - (nk - 1) * 128 <= 64 ? 0x80000000u : 0u;   // a row's last K-step has no bytes in its second half
    v4i fa_srd{0, 0, 0, 0x00020000}, fsa_srd{0, 0, 0, 0x00020000};
    uint32_t fb_soff, fsa_soff, fsb_soff, fa_dst, fsa_dst, fb_dst, fsb_dst, fb_kill;
    // (what follows from the wave's number is made anew: scalar registers are short)
    auto wave_here = [&]() __attribute__((always_inline)) {
        uint32_t v = (uint32_t)w;
        asm volatile("" : "+s"(v));
        return v;
    };
    // The descriptors of the activations begin at the item's first row of the K-step and end behind its last row.
    auto set_fetch_a = [&](int row_start, int rows, int kt, uint32_t slot_a) __attribute__((always_inline)) {
        const uint32_t row_base = (uint32_t)kt * (uint32_t)p.S + (uint32_t)row_start;
        const uint64_t a0 = (uint64_t)p.A + (uint64_t)row_base * 128u, sa0 = (uint64_t)p.SA + (uint64_t)row_base * 8u;
        fa_srd.x = (int)(uint32_t)a0; fa_srd.y = (int)((uint32_t)(a0 >> 32) & 0xffffu); fa_srd.z = rows * 128;
        fsa_srd.x = (int)(uint32_t)sa0; fsa_srd.y = (int)((uint32_t)(sa0 >> 32) & 0xffffu); fsa_srd.z = rows * 8;
        const uint32_t w = wave_here();
        fa_dst = lds0 + w * 1024u + slot_a * kTlATile;
        fsa_soff = w * (SR * 8u);
        fsa_dst = lds0 + kTlSa + fsa_soff + slot_a * kTlSaTile;
    };
    auto set_fetch_b = [&](int kt, uint32_t slot_b) __attribute__((always_inline)) {
        const uint32_t w = wave_here();
        fb_soff = (uint32_t)kt * kMoeBTile + w * 4096u;
        fsb_soff = (uint32_t)kt * kMoeScaleB + w * 256u;
        fb_dst = lds0 + kTlB + w * 4096u + slot_b * kMoeBTile;
        fsb_dst = lds0 + kTlSb + w * 256u + slot_b * kMoeScaleB;
        // second half of the last K-step past the end of K: out of range (bit 31), LDS gets the zeros that the layout holds there
        fb_kill = kt == nk - 1 ? tail_kill : 0u;
    };
    auto load_a = [&]<int I>() __attribute__((always_inline)) { dma16(fa_srd, fa_dst + I * 8192, voff_a, I * 8192u); };
    auto load_sa = [&]() __attribute__((always_inline)) { dma16_lanes(fsa_srd, fsa_dst, voff_b, fsa_soff, kSaMask); };
    auto load_b = [&]<int I>() __attribute__((always_inline)) { dma16(fb_srd, fb_dst + I * 1024, voff_b, (I & 1 ? fb_soff | fb_kill : fb_soff) + I * 1024u); };
    auto load_sb = [&]() __attribute__((always_inline)) { dma4(fsb_srd, fsb_dst, voff_b >> 2, fsb_soff); };
    // EXT: the item's biases of this wave's 64 weight rows, as its epilogue wants them (MODE 0: 32 gate, 32 up). Columns past
    // N read other experts' values or, past the array, zeros; their results are dropped.
    auto load_bias = [&](const MxTallItem& c) __attribute__((always_inline)) {
        if constexpr (EXT) {
            const int l = lane_here();
            uint32_t wave = wave_here(), interleaved = (uint32_t)HK_LATE_INT(interleaved), N = (uint32_t)HK_LATE_INT(N);
            asm volatile("" : "+v"(wave), "+v"(interleaved), "+v"(N));
            const uint32_t col = wave & 3u;
            uint32_t idx;   // float index into the bias array
            if (MODE == 1) {
                idx = (uint32_t)c.expert * N + (uint32_t)c.n_tile * 256u + 64u * col + (uint32_t)l;
            } else {
                const uint32_t hcol = (uint32_t)c.n_tile * 128u + 32u * col + (uint32_t)(l & 31), up = (uint32_t)l >> 5;
                idx = (uint32_t)c.expert * 2u * N + (interleaved ? 2u * hcol + up : up * N + hcol);
            }
            const float* bias = HK_LATE(bias);
            dma4(make_srd(bias, bias ? (uint32_t)HK_LATE_INT(bias_bytes) : 0u), to_sgpr(lds0 + kTlBias + wave * 256u), idx * 4u, 0u);
        }
    };

    // ---- LDS -> registers (addresses of the compute position, advanced in place) ----
    uint32_t a_lo, b_rd = lds0 + kTlB + wn * 8192 + lane * 16u, sa_rd, sb_rd = lds0 + kTlSb + wn * 512 + lane * 4u;
    {
        const uint32_t r = lane & 15, g = lane >> 4;
        a_lo = lds0 + wm * 2048 + r * 128u + swz_chunk(r, g) * 16u;   // (chunk g + 4: bit 6 the other way round)
        sa_rd = lds0 + kTlSa + (wm * 16 + r) * 8u + g;
    }
    v4f acc[MT][NT];
    auto mfma = [&]<int BYTE>(v4f& c, const v4i& x, const v4i& y, int sx, int sy) __attribute__((always_inline)) {
        asm volatile(
            "v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel:[%5,0,0] op_sel_hi:[%6,0,0] cbsz:4 blgp:4"
            : "+v"(c)
            : "v"(x), "v"(y), "v"(sx), "v"(sy), "n"(BYTE & 1), "n"(BYTE >> 1));
    };

    // Stores through descriptors that end at the item's last row: rows past it are dropped by the range check; lanes that do not
    // store carry bit 31 in their offset.
    auto epilogue = [&](const MxTallItem& a) __attribute__((always_inline)) {
        const int l = lane_here();
        const uint32_t r = l & 15, g = l >> 4;
        int wave = w;
        asm volatile("" : "+v"(wave));
        const uint32_t wave_col = (uint32_t)wave & 3u, row_of_lane = 16u * ((uint32_t)wave >> 2) + r;
        const int left = a.rows - (int)to_sgpr(row_of_lane - r);   // fragment m has rows while 32 m < left
        // MODE 0: gate / up biases of columns 16 o + 4 g .. +4 in [2 o], [2 o + 1]; MODE 1: of columns 32 o + 8 g + 4 i .. +4 in
        // [2 o + i]. (Read for every fragment: kept, they would be registers too many.)
        v4f bias[4] = {};
        uint32_t bias_rd = lds0 + kTlBias + (uint32_t)wave * 256u + (MODE == 1 ? 32u : 16u) * g;
        auto read_bias = [&]() __attribute__((always_inline)) {
            if constexpr (EXT) {
                asm volatile("" : "+v"(bias_rd));
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    bias[q] = *(lds_v4f_t*)(uintptr_t)(bias_rd + (MODE == 1 ? 128 * (q >> 1) + 16 * (q & 1) : 128 * (q & 1) + 64 * (q >> 1)));
            }
        };
        if (MODE == 1) {
            const int N = HK_LATE_INT(N);
            const uint32_t pitch = (uint32_t)N * 2u;
            const v4i srd = make_srd((uint8_t*)HK_LATE(out0) + (size_t)a.row_start * pitch, (uint32_t)a.rows * pitch);
            const int wcol0 = a.n_tile * 256 + (int)to_sgpr(wave_col) * 64;   // N % 32 == 0: a group of 32 columns is valid as a whole
            const bool ok0 = wcol0 < N, ok1 = wcol0 + 32 < N;
            uint32_t voff = row_of_lane * pitch + (uint32_t)(wcol0 + 8 * (int)g) * 2u;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (32 * m < left) {
                    read_bias();
#pragma unroll
                    for (int o = 0; o < 2; ++o) {
                        v4f x = acc[m][2 * o], y = acc[m][2 * o + 1];
                        if (EXT)
#pragma unroll
                            for (int j = 0; j < 4; ++j) { x[j] += bias[2 * o][j]; y[j] += bias[2 * o + 1][j]; }
                        v4i o4;
                        o4.x = pack_bf16(x.x, x.y); o4.y = pack_bf16(x.z, x.w);
                        o4.z = pack_bf16(y.x, y.y); o4.w = pack_bf16(y.z, y.w);
                        if (o == 0 ? ok0 : ok1)
                            asm volatile("buffer_store_dwordx4 %0, %1, %2, 0 offen offset:%3\n\ts_nop 1"
                                         :: "v"(o4), "v"(voff), "s"(srd), "n"(o * 64) : "memory");
                    }
                    voff += 32u * pitch;
                }
            }
        } else {
            // lane (r, g) holds, for its row of fragment m, the h columns 128 n_tile + 32 wn + 16 o + 4 g .. +4 (o = 0, 1): the
            // wave's 32 columns are one MX block
            const size_t row0 = (size_t)(a.n_tile >> 1) * p.S + (size_t)a.row_start;
            const v4i srd_h = make_srd((uint8_t*)HK_LATE(out0) + row0 * 128, (uint32_t)a.rows * 128u);
            const v4i srd_s = make_srd(HK_LATE(out_scales) + row0 * 8, (uint32_t)a.rows * 8u);
            const bool ok = a.n_tile * 128 + 32 * (int)to_sgpr(wave_col) < HK_LATE_INT(N);
            uint32_t voff_h = g == 0 ? row_of_lane * 128u + (uint32_t)(a.n_tile & 1) * 64u + 16u * wave_col : 0x80000000u;
            uint32_t voff_s = g == 0 ? row_of_lane * 8u + 4u * (uint32_t)(a.n_tile & 1) + wave_col : 0x80000000u;
            static_assert(offsetof(MoeGemmParams, limit) == offsetof(MoeGemmParams, alpha) + 4, "fetched together");
            const uint64_t al = EXT == 2 ? pointer_arg.template operator()<offsetof(MoeGemmParams, alpha)>() : 0;
            const float alpha = __uint_as_float((uint32_t)al), limit = __uint_as_float((uint32_t)(al >> 32));
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (32 * m < left) {
                    read_bias();
                    float h[2][4];
#pragma unroll
                    for (int o = 0; o < 2; ++o)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const float gt = acc[m][2 * o][j], up = acc[m][2 * o + 1][j];
                            if (EXT) h[o][j] = glu_act<EXT == 2>(gt + bias[2 * o][j], up + bias[2 * o + 1][j], alpha, limit);
                            else h[o][j] = silu_mul(gt, up);
                        }
                    int e;
                    const v4i o4 = mx_block_codes<false>(h, ok, e);
                    asm volatile("buffer_store_dwordx4 %0, %1, %2, 0 offen\n\ts_nop 1" :: "v"(o4), "v"(voff_h), "s"(srd_h) : "memory");
                    asm volatile("buffer_store_byte %0, %1, %2, 0 offen" :: "v"(e + 127), "v"(voff_s), "s"(srd_s) : "memory");
                    voff_h += 32u * 128u;
                    voff_s += 32u * 8u;
                }
            }
        }
    };

    // ---- prologue: the first two positions ----
    MxTallItem cur, nxt;
    load_item(it, cur);
    auto fetch_a = [&](int kt) __attribute__((always_inline)) {
        set_fetch_a(cur.row_start, cur.rows, kt, (uint32_t)kt);
        load_a.template operator()<0>(); load_a.template operator()<1>(); load_a.template operator()<2>(); load_a.template operator()<3>();
        if (w < 4) load_a.template operator()<4>();
        load_sa();
    };
    auto fetch_b = [&](int kt) __attribute__((always_inline)) {
        set_fetch_b(kt, (uint32_t)kt);
        load_b.template operator()<0>(); load_b.template operator()<1>(); load_b.template operator()<2>(); load_b.template operator()<3>();
        load_sb();
    };
    set_weights(cur);
    fetch_a(0); fetch_b(0); fetch_a(1); fetch_b(1);
    load_item(it + it_stride, nxt);
    wait_vmcnt<5>();
    block_barrier();
    slot_fence();
    uint32_t st = 0;   // LDS slot of the compute position

    // The K loop of an item of up to 32 MTX rows.
    auto run_item = [&]<int MTX>() __attribute__((always_inline)) {
        v4i bf[NT][2];           // weight fragments of the position (K halves), the scale bytes of each pair
        int bsc[2];
        v4i af[3][2];            // activation fragments and their rows' scales
        uint32_t as[3][2];
        // buffer of an activation fragment: the last three all in different ones, the first in that of the last but two,
        // which is the first to be free, neighbours in different ones
        constexpr auto buf_of = [](int m) {
            constexpr int x = 1 + ((MTX - 5) & 1);   // of fragment MTX - 4
            return m == 0 || m == MTX - 3 ? 0 : m < MTX - 3 ? 1 + ((m - 1) & 1) : m == MTX - 2 ? 3 - x : x;
        };
        auto read_bf = [&]<int N>() __attribute__((always_inline)) {
            bf[N][0] = *(lds_v4i_t*)(uintptr_t)(b_rd + N * 2048);
            bf[N][1] = *(lds_v4i_t*)(uintptr_t)(b_rd + N * 2048 + 1024);
        };
        auto read_sb = [&]<int Q>() __attribute__((always_inline)) { bsc[Q] = *(lds_i32_t*)(uintptr_t)(sb_rd + Q * 256); };
        auto read_frag = [&]<int F>() __attribute__((always_inline)) {
            constexpr int B = buf_of(F);
            af[B][0] = *(lds_v4i_t*)(uintptr_t)(a_lo + F * 4096);
            af[B][1] = *(lds_v4i_t*)(uintptr_t)((a_lo ^ 64u) + F * 4096);
            as[B][0] = *(lds_u8_t*)(uintptr_t)(sa_rd + F * 256);
            as[B][1] = *(lds_u8_t*)(uintptr_t)(sa_rd + F * 256 + 4);
        };
#pragma unroll
        for (int m = 0; m < MTX; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[m][n] = v4f{0.f, 0.f, 0.f, 0.f};
        // the first position's fragments (the last position of the item before has read them too: kept, they would be in
        // registers across the epilogue)
        read_frag.template operator()<0>();
        read_bf.template operator()<0>(); read_bf.template operator()<1>(); read_bf.template operator()<2>(); read_bf.template operator()<3>();
        read_sb.template operator()<0>(); read_sb.template operator()<1>();
        // A position: 8 MTX MFMAs. Fragment by fragment, first K half first; the last three fragments go through weight fragment 0
        // first, then 1, 2, 3, so that a weight fragment's registers are free for the next position's one after the other.
        constexpr int TAIL = 8 * (MTX - 3);
        for (int kt = 0; kt < nk; ++kt) {
            const bool over = kt + 2 >= nk;   // the position after the next belongs to the next item
            const int k2 = over ? kt + 2 - nk : kt + 2;
            if (kt + 2 == nk) set_weights(nxt);
            set_fetch_b(k2, st);
            set_fetch_a(over ? nxt.row_start : cur.row_start, over ? nxt.rows : cur.rows, k2, st);
            __builtin_amdgcn_sched_barrier(0);
            auto slot = [&]<int I>() __attribute__((always_inline)) {
                constexpr int J = I - TAIL, J6 = J < 0 ? 0 : J % 6;
                constexpr int M = J < 0 ? I / 8 : MTX - 3 + (J6 < 4 ? (J6 & 1) : 2);
                constexpr int N = J < 0 ? I & 3 : J / 6, H = J < 0 ? (I >> 2) & 1 : (J6 < 4 ? J6 >> 1 : J6 & 1);
                constexpr int B = buf_of(M);
                mfma.template operator()<2 * H + (N & 1)>(acc[M][N], bf[N][H], af[B][H], bsc[N >> 1], (int)as[B][H]);
                if constexpr (J < 0 && I % 8 == 0) read_frag.template operator()<M + 1>();
                if constexpr (J == -4) read_frag.template operator()<MTX - 2>();
                if constexpr (J == 0) read_frag.template operator()<MTX - 1>();
                if constexpr (J == 5) {
                    // the change of position: its tile has landed for everyone, everyone has read this one's
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    wait_vmcnt<5>();
                    block_barrier();
                    slot_fence();
                    st ^= 1u;
                    a_lo += st ? kTlATile : -kTlATile;
                    b_rd += st ? kMoeBTile : -kMoeBTile;
                    sa_rd += st ? kTlSaTile : -kTlSaTile;
                    sb_rd += st ? kMoeScaleB : -kMoeScaleB;
                    read_bf.template operator()<0>();
                }
                if constexpr (J == 11) { read_bf.template operator()<1>(); read_sb.template operator()<0>(); }
                if constexpr (J == 20) read_frag.template operator()<0>();
                if constexpr (J == 17) read_bf.template operator()<2>();
                if constexpr (J == 23) { read_bf.template operator()<3>(); read_sb.template operator()<1>(); }
                // loads: the weights two positions on, when everyone holds its fragments of this one's (slot 7 is the first to
                // use, and so to wait for, the last of them: there is no other wait in front of the barrier); the activations
                // two positions on, when everyone has read this one's
                if constexpr (I == 7) { block_barrier(); slot_fence(); }
                if constexpr (I == 8) load_b.template operator()<0>();
                if constexpr (I == 10) load_b.template operator()<1>();
                if constexpr (I == 12) load_b.template operator()<2>();
                if constexpr (I == 14) load_b.template operator()<3>();
                if constexpr (I == 15) load_sb();
                if constexpr (J == 7) load_a.template operator()<0>();
                if constexpr (J == 9) load_a.template operator()<1>();
                if constexpr (J == 13) load_a.template operator()<2>();
                if constexpr (J == 15) load_a.template operator()<3>();
                if constexpr (J == 19) { if (w < 4) load_a.template operator()<4>(); }
                if constexpr (J == 18) load_sa();
                if constexpr (J == 21 && MODE == 0) { if (EXT && kt == 0) load_bias(cur); }
                __builtin_amdgcn_sched_barrier(0);
            };
            [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) {
                (slot.template operator()<I>(), ...);
            }(std::make_integer_sequence<int, 8 * MTX>{});
        }
        mfma_drain();
#pragma unroll
        for (int m = 0; m < MTX; ++m)
            asm volatile("" : "+v"(acc[m][0]), "+v"(acc[m][1]), "+v"(acc[m][2]), "+v"(acc[m][3]));
        // (not used: gives the registers of the fragments that the item does not have a value on every way here)
#pragma unroll
        for (int m = MTX; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[m][n] = v4f{0.f, 0.f, 0.f, 0.f};
    };

    for (;;) {
        if (MODE == 1) load_bias(cur);   // (older than this position's weight loads, whose wait covers it; the wave's own use of the last item's is over)
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
#undef HK_LATE_INT

}  // namespace hk
