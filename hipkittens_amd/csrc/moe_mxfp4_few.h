// Grouped GEMM of the MXFP4-weight MoE for layers whose experts get only a few rows (decode steps and small
// batches), on the pre-shuffled weights. Included by moe_mxfp4.hip.
//
// Bound: HBM (the touched experts' weights once). The persistent streaming kernel walks work items of 256 weight
// rows, one workgroup per CU: with 16 experts that is 368 items on 256 CUs, so that most CUs idle while a few
// work on their second item, and a decode step's single row fragment leaves nothing to amortize its LDS stages and
// barriers over. Here a work item's 256 weight rows are four independent waves (workgroups of one wave, 64
// weight rows each) that walk the whole K alone: no LDS, no barrier, weights and activations straight into MFMA
// operand registers through a ring of D K-steps. Two or three waves share a SIMD, so that one streams while
// another starts or finishes, and the hardware's dispatch balances them.
//   - The weight fragments of a wave and K-step are 8 KiB in one piece; two K-steps ahead and eight waves per CU
//     put 128 KiB in flight per CU (one, two or three K-steps ahead measure the same: the memory system is full).
//   - Consecutive workgroups stay on the hardware's round robin over the XCDs: a contiguous run of the list per XCD
//     streams from a part of the memory channels at a time and takes 277 instead of 216 us at 64 tokens. The
//     weights are loaded with the non-temporal hint (241 us without).
//   - The activation rows (16 MT of them at most) are fetched by every wave from L2: 2 KiB per 8 KiB of weights and row
//     fragment (MXFP8: 4 KiB).
//   - Same MFMAs in the same order per output element as the streaming kernel: identical bits.
// GPT-OSS-like layer (H = I = 2880, E = 128, top-4, biases and clamped SwiGLU; whole layer, us, streaming kernel /
// this one): 1 token 50 / 29, 4 tokens 73 / 51, 16 tokens 144 / 125, 64 tokens 232 / 216 (1.5 GB of weights at
// 7.3 TB/s), 128 tokens 279 / 262; with two row fragments (MT = 2) 128 tokens 261, 256 tokens 311 / 296 (one
// fragment 314), 400 tokens 323 / 328, 512 tokens 334 / 359. With MXFP8 activations one fragment 4 tokens 67 / 52,
// 64 tokens 239 / 225, 128 tokens 278 / 265, 256 tokens 308 / 326 (two: 317). moe_few_rows has the rule.
#pragma once

namespace hk {

__device__ __forceinline__ __amdgpu_buffer_rsrc_t few_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00020000);
}

template <int MODE, bool EXT, bool A8, int MT>
__global__ __launch_bounds__(64, 2) void moe_mxfp4_few_kernel(const MoeGemmParams p) {
    constexpr int kRow = A8 ? 256 : 128, D = MT == 1 ? 3 : 2;
    constexpr int kNt = 2;   // cache policy of the weight loads: non-temporal (they are read once)
    const int it = blockIdx.x >> 2, w = blockIdx.x & 3;
    if (it >= p.num_items[0]) return;
    const MoeItem item = p.items[it];
    const int col0 = MODE == 0 ? item.n_tile * 128 + 32 * w : item.n_tile * 256 + 64 * w;   // first output column
    if (col0 >= p.N) return;   // (the quantizer pads h's last K-step)
    const int lane = lane_id(), r = lane & 15, g = lane >> 4;
    const int Kb = p.K >> 1, nk = (Kb + 127) >> 7;

    // ---- sources ------------------------------------------------------------------------------------------
    const uint8_t* b = p.B + (size_t)item.expert * p.b_expert_stride + (size_t)item.n_tile * nk * kMoeBTile + w * 8192;
    const uint8_t* sb = p.SB + (size_t)item.expert * p.sb_expert_stride + (size_t)item.n_tile * nk * kMoeScaleB + w * 512;
    const auto rs_b = few_rsrc(b, (uint32_t)nk * kMoeBTile - (uint32_t)w * 8192u);
    const auto rs_sb = few_rsrc(sb, (uint32_t)nk * kMoeScaleB - (uint32_t)w * 512u);
    const bool gather = MODE == 0;
    const uint32_t a_rows = (uint32_t)(gather ? p.a_rows : p.S);
    const auto rs_a = few_rsrc(p.A, (uint32_t)nk * a_rows * (uint32_t)kRow);
    const auto rs_sa = few_rsrc(p.SA, gather ? (uint32_t)((nk + 15) >> 4) * a_rows * 128u : (uint32_t)nk * a_rows * 8u);
    uint32_t voff_a[MT], voff_sa[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        // rows past the item: its last row again, for fragments without any row nothing is fetched
        uint32_t row = (uint32_t)(item.row_start + min(16 * m + r, item.rows - 1));
        if (gather) {
            const uint32_t slot = (uint32_t)p.row_slots[row];
            row = p.topk_magic ? __umulhi(slot, p.topk_magic) : slot;
        }
        const uint32_t none = 16 * m >= item.rows ? 0x80000000u : 0u;
        voff_a[m] = (row * (uint32_t)kRow + 16u * g) | none;
        voff_sa[m] = (row * (gather ? 128u : 8u)) | none;
    }
    const int last_valid = Kb - (nk - 1) * 128;   // bytes of the last K-step inside K

    struct Step { v4i b[8]; int sb[2]; v4i a[MT][A8 ? 4 : 2]; v2i sa[MT]; };
    Step ring[D];
    // The loads of K-step kt; from nk on every one of them lies outside its descriptor: zeros, nothing fetched.
    auto fetch = [&](Step& q, int kt) __attribute__((always_inline)) {
#pragma unroll
        for (int f = 0; f < 8; ++f) {   // f = 4 pair + 2 fragment + K half
            const int half = f & 1;
            // lanes whose 16 bytes lie in the layout's zero padding fetch nothing
            const uint32_t kill = kt == nk - 1 && 64 * half + 16 * g >= last_valid ? 0x80000000u : 0u;
            q.b[f] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs_b, (lane * 16 + f * 1024) | kill, kt * kMoeBTile, kNt));
        }
#pragma unroll
        for (int pr = 0; pr < 2; ++pr)
            q.sb[pr] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs_sb, lane * 4 + pr * 256, kt * kMoeScaleB, kNt);
        // (a gathered row's 128 scale bytes go on past K-step nk - 1 with whatever the workspace held, a NaN scale perhaps)
        const uint32_t soff_sa = !gather ? (uint32_t)kt * a_rows * 8u
                                 : ((uint32_t)(kt >> 4) * a_rows * 128u + (uint32_t)(kt & 15) * 8u) | ((uint32_t)(nk - 1 - kt) & 0x80000000u);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
#pragma unroll
            for (int c = 0; c < (A8 ? 4 : 2); ++c)
                q.a[m][c] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs_a, voff_a[m] + 64 * c, (uint32_t)kt * a_rows * (uint32_t)kRow, 0));
            q.sa[m] = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(rs_sa, voff_sa[m], soff_sa, 0));
        }
    };
    v4f acc[MT][4];   // [row fragment][2 pair + fragment]
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m][n] = v4f{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const Step& q) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int sa = (int)((uint32_t)q.sa[m][half] >> (8 * g));
                v8i y;
                if constexpr (A8) y = __builtin_shufflevector(q.a[m][2 * half], q.a[m][2 * half + 1], 0, 1, 2, 3, 4, 5, 6, 7);
                else y = __builtin_shufflevector(q.a[m][half], q.a[m][half], 0, 1, 2, 3, 0, 1, 2, 3);
#define HK_FEW_MFMA(n)                                                                                              \
    {                                                                                                               \
        const v4i x4 = q.b[4 * ((n) >> 1) + 2 * ((n) & 1) + half];                                                  \
        const v8i x = __builtin_shufflevector(x4, x4, 0, 1, 2, 3, 0, 1, 2, 3);                                      \
        if (half == 0)                                                                                              \
            acc[m][n] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(x, y, acc[m][n], 4, A8 ? 0 : 4, (n) & 1,   \
                                                                         q.sb[(n) >> 1], 0, sa);                    \
        else                                                                                                        \
            acc[m][n] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(x, y, acc[m][n], 4, A8 ? 0 : 4,            \
                                                                         2 + ((n) & 1), q.sb[(n) >> 1], 0, sa);     \
    }
                HK_FEW_MFMA(0) HK_FEW_MFMA(1) HK_FEW_MFMA(2) HK_FEW_MFMA(3)
#undef HK_FEW_MFMA
            }
    };

#pragma unroll
    for (int d = 0; d < D - 1; ++d) {
        fetch(ring[d], d);
        __builtin_amdgcn_sched_barrier(0);   // (a K-step's loads are older than the next one's: the waits count on it)
    }
    // (bias values of the epilogue, behind the first weight loads)
    float bias_a[2][4], bias_b[2][4];   // MODE 0: [pair][j] gate / up; MODE 1: [pair][j] columns 8 g + j / 8 g + 4 + j
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
        for (int j = 0; j < 4; ++j) bias_a[o][j] = bias_b[o][j] = 0.f;
    if (EXT && p.bias) {
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (MODE == 1) {
                    const int c = min(col0 + 32 * o + 8 * g + j, p.N - 5);   // (N % 32 == 0: columns past N are not stored)
                    const float* at = p.bias + (size_t)item.expert * p.N + c;
                    bias_a[o][j] = at[0];
                    bias_b[o][j] = at[4];
                } else {
                    const int c = col0 + 16 * o + 4 * g + j;
                    const float* at = p.bias + (size_t)item.expert * 2 * p.N;
                    bias_a[o][j] = p.interleaved ? at[2 * c] : at[c];
                    bias_b[o][j] = p.interleaved ? at[2 * c + 1] : at[p.N + c];
                }
            }
    }
    for (int kt = 0; kt < nk; kt += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            fetch(ring[(d + D - 1) % D], kt + d + D - 1);
            __builtin_amdgcn_sched_barrier(0);
            compute(ring[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // ---- epilogue: as in the streaming kernel ------------------------------------------------------------
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int row = 16 * m + r;
        const bool ok = row < item.rows;
        const size_t pos = (size_t)item.row_start + row;
        if constexpr (MODE == 1) {
            if (!ok) continue;
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                if (col0 + 32 * o >= p.N) continue;
                v4f x = acc[m][2 * o], y = acc[m][2 * o + 1];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (EXT) { x[j] += bias_a[o][j]; y[j] += bias_b[o][j]; }
                *(v4i*)((uint16_t*)p.out0 + pos * p.N + col0 + 32 * o + 8 * g) =
                    v4i{(int)pack_bf16(x.x, x.y), (int)pack_bf16(x.z, x.w), (int)pack_bf16(y.x, y.y), (int)pack_bf16(y.z, y.w)};
            }
        } else {
            float h[2][4];
#pragma unroll
            for (int o = 0; o < 2; ++o)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float gt = acc[m][2 * o][j], up = acc[m][2 * o + 1][j];
                    h[o][j] = EXT ? glu_act(p.act, gt + bias_a[o][j], up + bias_b[o][j], p.alpha, p.limit) : silu_mul(gt, up);
                }
            int e;
            const v4i code = mx_block_codes<A8>(h, true, e);
            if (!ok) continue;
            const size_t out_row = (size_t)(item.n_tile >> 1) * p.S + pos;
            // MXFP4: the row's 16 bytes leave from its lane g = 0; MXFP8: its 32 bytes from lanes g = 0, 1
            if (g < (A8 ? 2 : 1))
                *(v4i*)((uint8_t*)p.out0 + out_row * kRow + (item.n_tile & 1) * (kRow / 2) + (A8 ? 32 : 16) * w + 16 * g) = code;
            if (g == 0) p.out_scales[out_row * 8 + 4 * (item.n_tile & 1) + w] = (uint8_t)(e + 127);
        }
    }
}

}  // namespace hk
