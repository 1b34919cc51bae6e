// Grouped GEMM of the FP8 block-scaled MoE for layers with few work items (decode steps, the expert that every token
// passes through), on the pre-shuffled weights. Included by moe_fp8blk.hip.
//
// Bound: HBM (the touched experts' weights once), and below that what the CUs with a work item can have in flight (a
// CU whose loads miss its L2 takes in about 60 GB/s, however many waves issue them). The persistent streaming kernel
// gives a CU an item of 256 weight rows: the shared expert of the DeepSeek-V3-like layer (4096 x 7168 and
// 7168 x 2048) is 16 and 28 such items on 256 CUs. Here the item's 256 weight rows are eight independent workgroups of
// one wave, 32 rows each (gate+up: a gate fragment and the up fragment of the same columns), that walk the whole K
// alone, weights and activations straight into MFMA operand registers through a ring of D K-steps: no LDS, no
// barrier.
//   - h's 1 x 128 quantization blocks span four columns' waves: gate+up leaves h in fp32 and a small kernel
//     quantizes it. (The eight waves as one workgroup that exchanges the blocks' maxima through LDS saves that launch
//     but keeps an item on one CU: 16 rows through the shared expert 63 us against 19.)
//   - An item's 16 activation rows are fetched by every wave from L2: 2 KiB per 4 KiB of weights. (Items of 32 or 64
//     rows were slower from 1 to 500 rows per expert.)
//   - Same MFMAs, scaling FMAs and order per output element as the streaming kernel: identical bits.
// Shared expert of that layer, its whole call, us, streaming / this kernel: 1 token 97 / 16, 16 tokens 83 / 19 (2.4
// TB/s of weights), 64 tokens 85 / 32. moe_fp8blk_few has the rule and the routed layer's figures.
#pragma once

namespace hk {

constexpr int kF8FewRows = 16;   // rows per work item

__device__ __forceinline__ __amdgpu_buffer_rsrc_t f8few_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00020000);
}

// p.items null: one expert that holds all S rows in order, item i = rows kF8FewRows (i / n_tiles).., tile i % n_tiles.
// p.sorted_slots null: row `pos` of the order is token pos.
// D: K-steps of the ring, D - 1 of them in flight.
template <int MODE, int D>
__global__ __launch_bounds__(64, 2) void moe_fp8blk_few_kernel(const MoeFp8Params p) {
    constexpr int kNt = 2;   // cache policy of the weight loads: non-temporal
    const int it = blockIdx.x >> 3, w = blockIdx.x & 7;
    MoeItem item;
    if (p.items) {
        if (it >= p.num_items[0]) return;
        item = p.items[it];
    } else {
        const int m = it / p.n_tiles_n;
        item = MoeItem{0, kF8FewRows * m, min(kF8FewRows, p.S - kF8FewRows * m), it - m * p.n_tiles_n};
    }
    const int wn = w >> 1, o = w & 1;
    const int col0 = MODE == 0 ? item.n_tile * 128 + 32 * wn : item.n_tile * 256 + 32 * w;
    if (MODE == 1 && col0 >= p.N) return;
    const int lane = lane_id(), r = lane & 15, g = lane >> 4;
    const int nk = p.K >> 7;

    const uint8_t* b = p.B + (size_t)item.expert * p.b_expert_stride + (size_t)item.n_tile * nk * kF8sBTile + w * 4096;
    const float* sb = p.SB + (size_t)item.expert * p.sb_expert_stride;
    const float* sb0 = sb + (size_t)(MODE == 0 ? item.n_tile : col0 >> 7) * nk;
    const float* sb1 = MODE == 0 ? sb + (size_t)(p.N / 128 + item.n_tile) * nk : sb0;
    // rows past the item: its last row again
    uint32_t row = (uint32_t)(item.row_start + min(r, item.rows - 1));
    if (MODE == 0 && p.sorted_slots) row = (uint32_t)p.sorted_slots[row] / (uint32_t)p.topk;
    const uint32_t voff_a = (MODE == 0 ? row * (uint32_t)p.K : row * 128u) + 16u * g;
    const uint32_t voff_sa = MODE == 0 ? row * (uint32_t)nk * 4u : row * 4u;
    const uint32_t a_bytes = (uint32_t)(MODE == 0 ? p.T : p.S) * (uint32_t)p.K;
    const uint32_t a_step = MODE == 0 ? 128u : (uint32_t)p.S * 128u, sa_step = a_step >> 5;

    struct Step { v4i b[4], a[2]; float xs, ws[2]; };
    Step ring[D];
    // The loads of K-step kt. Past the last one the descriptors are empty: zeros, nothing fetched.
    auto fetch = [&](Step& q, int kt) __attribute__((always_inline)) {
        const bool live = kt < nk;
        const uint32_t k = (uint32_t)(live ? kt : 0);
        const auto rs_b = f8few_rsrc(b, live ? (uint32_t)nk * kF8sBTile - (uint32_t)w * 4096u : 0u);
        const auto rs_a = f8few_rsrc(p.A, live ? a_bytes : 0u);
        const auto rs_sa = f8few_rsrc(p.SA, live ? a_bytes >> 5 : 0u);
#pragma unroll
        for (int f = 0; f < 4; ++f)   // f = 2 fragment + K half
            q.b[f] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs_b, lane * 16 + f * 1024, k * kF8sBTile, kNt));
#pragma unroll
        for (int c = 0; c < 2; ++c)
            q.a[c] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs_a, voff_a + 64 * c, k * a_step, 0));
        q.xs = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_sa, voff_sa, k * sa_step, 0));
        // (through the vector memory path like the rest, so that one in-order count covers a K-step)
        q.ws[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(f8few_rsrc(sb0, live ? (uint32_t)nk * 4u : 0u), 0, k * 4u, 0));
        q.ws[1] = MODE == 0 ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(f8few_rsrc(sb1, live ? (uint32_t)nk * 4u : 0u), 0, k * 4u, 0)) : 0.f;
    };
    v4f acc[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
    auto compute = [&](const Step& q) __attribute__((always_inline)) {
        const v8i af = __builtin_shufflevector(q.a[0], q.a[1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const v8i bf = __builtin_shufflevector(q.b[2 * n], q.b[2 * n + 1], 0, 1, 2, 3, 4, 5, 6, 7);
            const v4f part = mfma_fp8_16x16x128(bf, af, v4f{0.f, 0.f, 0.f, 0.f});
            const float sc = q.xs * (MODE == 0 && n ? q.ws[1] : q.ws[0]);
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[n][j] = __builtin_fmaf(part[j], sc, acc[n][j]);
        }
    };
#pragma unroll
    for (int d = 0; d < D - 1; ++d) {
        fetch(ring[d], d);
        __builtin_amdgcn_sched_barrier(0);   // (a K-step's loads are older than the next one's: the waits count on it)
    }
    int kt = 0;
    for (; kt + D < nk; kt += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            fetch(ring[(d + D - 1) % D], kt + d + D - 1);
            __builtin_amdgcn_sched_barrier(0);
            compute(ring[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // The last D K-steps at most: nothing is fetched or multiplied past nk (as loads and MFMAs of zeros, up to D - 1 of them
    // per wave, they made a narrow expert slower than the streaming kernel: H = 7168, I = 512, mean 2 rows of 256 experts,
    // streaming 440, with them 461, without 410 us; 16 experts, mean 32 rows 98 / 107 / 97).
    fetch(ring[D - 1], kt + D - 1);
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (kt + d < nk) compute(ring[d]);

    // lane (r, g) holds, for row r of the item, 8 columns of o (down) or gate and up of 4 columns of h
    if (r >= item.rows) return;
    const size_t pos = (size_t)(item.row_start + r);
    const v4f x = acc[0], y = acc[1];
    if constexpr (MODE == 1) {
        *(v4i*)((uint16_t*)p.out0 + pos * p.N + col0 + 8 * g) =
            v4i{(int)pack_bf16(x.x, x.y), (int)pack_bf16(x.z, x.w), (int)pack_bf16(y.x, y.y), (int)pack_bf16(y.z, y.w)};
    } else {
        v4f h;
#pragma unroll
        for (int j = 0; j < 4; ++j) h[j] = silu_mul(x[j], y[j]);
        *(v4f*)((float*)p.out0 + pos * p.N + col0 + 8 * g + 4 * o) = h;
    }
}

// h [S][N] fp32 -> e4m3 tiles [N / 128][S][128] and their scales [N / 128][S]: one thread per 8 elements, 16 per block.
__global__ __launch_bounds__(256) void moe_fp8blk_few_quantize_kernel(const float* __restrict__ h, int S, int N,
                                                                      uint8_t* __restrict__ q, float* __restrict__ scales) {
    const int per_row = N / 8;
    const long long gid = (long long)blockIdx.x * 256 + threadIdx.x;
    const int row = (int)(gid / per_row), c8 = (int)(gid % per_row);
    if (row >= S) return;
    const v4f lo = *(const v4f*)(h + gid * 8), hi = *(const v4f*)(h + gid * 8 + 4);
    const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    const float s = e4m3_block_scale(amax);
    const size_t tile_row = (size_t)(c8 >> 4) * S + row;
    *(v2i*)(q + tile_row * 128 + 8 * (c8 & 15)) = quant8_e4m3(v, s);
    if ((c8 & 15) == 0) scales[tile_row] = s;
}

}  // namespace hk
