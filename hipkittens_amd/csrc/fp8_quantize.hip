// Per-tensor e4m3 quantization: scale = amax / 448 (1 for an all-zero tensor or one with a NaN), codes =
// e4m3(x / scale), rounded to nearest even and saturated; NaN stays NaN. The counterpart of the host-side
// conversion in kernels/gemm/fp8fp32/profile_utils.cpp:35-45, with the amax/448 scale of the hipBLASLt
// convention that the reference benchmarks against (analysis/baselines/README.md:172-174).
//
// Bound: memory (x twice, the second time out of a cache for up to 256 MB, q once) for large tensors,
// launches and the host's wait for the scale for small ones. The maximum is taken over the bit patterns of |x| as
// unsigned integers (the order of non-negative floats, with NaN above infinity), so it does not depend on
// the order of the blocks.
//   - two launches: every block writes the maximum of its elements, then every block of the second kernel
//     reduces all of these (4 KB at most, out of L2) instead of a third launch or a pass through the host;
//   - one launch up to kOneLaunchElems elements: every block takes the maximum of the whole tensor itself.
// Block 0 stores the scale to memory of the host as soon as it knows it, before it quantizes: the caller goes on
// (to launch the GEMM that takes the scale as an argument) while the rest of the quantization runs.
#include <chrono>

#include "hk_device.h"
#include "../../include/hk355.h"

namespace hk {

constexpr int kQtThreads = 256;
constexpr int kQtChunk = 16;           // elements per thread and step: one 16-byte store of codes
constexpr int kQtMaxBlocks = 1024;     // partial maxima: 4 per thread of the second kernel
constexpr long long kOneLaunchElems = 32768;
constexpr uint32_t kScaleUnset = 0xffffffffu;   // a NaN that no amax / 448 produces

enum { kQtBf16 = 0, kQtF32 = 1, kQtF16 = 2 };

// Sixteen elements at x + 16 * chunk as floats; elements from n on read as zero (they move no maximum and are
// not stored).
template <int TYPE>
__device__ __forceinline__ void qt_load(const void* __restrict__ x, long long chunk, long long n, float (&v)[kQtChunk]) {
    const long long e0 = chunk * kQtChunk;
    if (e0 + kQtChunk <= n) {
        if constexpr (TYPE == kQtF32) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const v4f t = ((const v4f*)x)[chunk * 4 + i];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[4 * i + j] = t[j];
            }
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const v4i t = ((const v4i*)x)[chunk * 2 + i];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t u = (uint32_t)t[j];
                    if constexpr (TYPE == kQtBf16) {
                        v[8 * i + 2 * j] = __uint_as_float(u << 16);
                        v[8 * i + 2 * j + 1] = __uint_as_float(u & 0xffff0000u);
                    } else {
                        v[8 * i + 2 * j] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u & 0xffffu));
                        v[8 * i + 2 * j + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u >> 16));
                    }
                }
            }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < kQtChunk; ++i) {
        v[i] = 0.f;
        if (e0 + i < n) {
            if constexpr (TYPE == kQtF32) v[i] = ((const float*)x)[e0 + i];
            else if constexpr (TYPE == kQtBf16) v[i] = __uint_as_float((uint32_t)((const uint16_t*)x)[e0 + i] << 16);
            else v[i] = (float)((const _Float16*)x)[e0 + i];
        }
    }
}

__device__ __forceinline__ uint32_t qt_max(uint32_t m, const float (&v)[kQtChunk]) {
#pragma unroll
    for (int i = 0; i < kQtChunk; ++i) m = max(m, __float_as_uint(v[i]) & 0x7fffffffu);
    return m;
}

// Maximum over the block's threads, in every thread.
__device__ __forceinline__ uint32_t qt_block_max(uint32_t m) {
    __shared__ uint32_t part[kQtThreads / 64];
#pragma unroll
    for (int off = 32; off; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, 64));
    if (lane_id() == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kQtThreads / 64; ++i) m = max(m, part[i]);
    return m;
}

// Two quotients -> two e4m3 codes in bits [15:0].
__device__ __forceinline__ uint32_t qt_cvt2(float a, float b) {
    const float ca = __builtin_amdgcn_fmed3f(a, -448.f, 448.f), cb = __builtin_amdgcn_fmed3f(b, -448.f, 448.f);
    uint32_t c = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(ca, cb, 0, false) & 0xffffu;
    if (a != a) c = (c & 0xff00u) | 0x7fu | ((__float_as_uint(a) >> 24) & 0x80u);
    if (b != b) c = (c & 0x00ffu) | 0x7f00u | ((__float_as_uint(b) >> 16) & 0x8000u);
    return c;
}

template <int TYPE>
__global__ __launch_bounds__(kQtThreads) void fp8_tensor_amax_kernel(const void* __restrict__ x, long long n,
                                                                     uint32_t* __restrict__ partial) {
    const long long chunks = (n + kQtChunk - 1) / kQtChunk, step = (long long)gridDim.x * kQtThreads;
    uint32_t m = 0;
    for (long long c = (long long)blockIdx.x * kQtThreads + threadIdx.x; c < chunks; c += step) {
        float v[kQtChunk];
        qt_load<TYPE>(x, c, n, v);
        m = qt_max(m, v);
    }
    m = qt_block_max(m);
    if (threadIdx.x == 0) partial[blockIdx.x] = m;
}

// ONE_LAUNCH: the maximum is taken here, over the whole tensor; otherwise over `partials` of the kernel above.
template <int TYPE, bool ONE_LAUNCH>
__global__ __launch_bounds__(kQtThreads) void fp8_tensor_quantize_kernel(const void* __restrict__ x, long long n,
                                                                         const uint32_t* __restrict__ partial,
                                                                         int partials, uint8_t* __restrict__ q,
                                                                         uint32_t* __restrict__ scale_out) {
    const long long chunks = (n + kQtChunk - 1) / kQtChunk, step = (long long)gridDim.x * kQtThreads;
    uint32_t m = 0;
    if constexpr (ONE_LAUNCH) {
        for (long long c = threadIdx.x; c < chunks; c += kQtThreads) {
            float v[kQtChunk];
            qt_load<TYPE>(x, c, n, v);
            m = qt_max(m, v);
        }
    } else {
#pragma unroll
        for (int i = 0; i < kQtMaxBlocks / kQtThreads; ++i) {
            const int j = i * kQtThreads + threadIdx.x;
            if (j < partials) m = max(m, partial[j]);
        }
    }
    const float amax = __uint_as_float(qt_block_max(m));
    const float s = amax > 0.f ? __fdiv_rn(amax, 448.f) : 1.0f;
    if (blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(scale_out, __float_as_uint(s), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    for (long long c = (long long)blockIdx.x * kQtThreads + threadIdx.x; c < chunks; c += step) {
        float v[kQtChunk];
        qt_load<TYPE>(x, c, n, v);
        v4i out;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            out[i] = (int)(qt_cvt2(__fdiv_rn(v[4 * i], s), __fdiv_rn(v[4 * i + 1], s)) |
                           (qt_cvt2(__fdiv_rn(v[4 * i + 2], s), __fdiv_rn(v[4 * i + 3], s)) << 16));
        if ((c + 1) * kQtChunk <= n) {
            ((v4i*)q)[c] = out;
        } else {
            for (int i = 0; c * kQtChunk + i < n; ++i) q[c * kQtChunk + i] = (uint8_t)((uint32_t)out[i >> 2] >> (8 * (i & 3)));
        }
    }
}

template <int TYPE>
static int launch_fp8_tensor_quantize(const void* x, long long n, void* q, uint32_t* scale_out, uint32_t* partial,
                                      hipStream_t s) {
    const long long chunks = (n + kQtChunk - 1) / kQtChunk;
    const int blocks = (int)std::min<long long>((chunks + kQtThreads - 1) / kQtThreads, kQtMaxBlocks);
    if (n <= kOneLaunchElems) {
        hipLaunchKernelGGL((fp8_tensor_quantize_kernel<TYPE, true>), dim3(blocks), dim3(kQtThreads), 0, s, x, n,
                           (const uint32_t*)nullptr, 0, (uint8_t*)q, scale_out);
    } else {
        hipLaunchKernelGGL((fp8_tensor_amax_kernel<TYPE>), dim3(blocks), dim3(kQtThreads), 0, s, x, n, partial);
        hipLaunchKernelGGL((fp8_tensor_quantize_kernel<TYPE, false>), dim3(blocks), dim3(kQtThreads), 0, s, x, n,
                           (const uint32_t*)partial, blocks, (uint8_t*)q, scale_out);
    }
    return hipGetLastError() == hipSuccess ? HK_OK : HK_ERR_LAUNCH;
}

// Returns once *word differs from `unset`. The watched store is the first thing a kernel that was just launched
// does, so this polls (on an idle stream a store to host memory is seen 2-3 us earlier than the end of the kernel through
// hipStreamSynchronize) and hands over to hipStreamSynchronize when the stream has 20 ms and more to do first. The poll
// keeps its core busy, and so does the runtime's own wait: behind 10 ms of queued GEMMs this, hipStreamSynchronize and
// torch's copy of a scalar to the host each take 10.3 ms of CPU time.
static int await_host_word(const volatile uint32_t* word, uint32_t unset, hipStream_t s) {
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(20);
    for (;;) {
        for (int i = 0; i < 64; ++i) {
            if (*word != unset) return HK_OK;
            __builtin_ia32_pause();
        }
        if (std::chrono::steady_clock::now() > until) break;
    }
    if (hipStreamSynchronize(s) != hipSuccess) return HK_ERR_LAUNCH;
    return *word != unset ? HK_OK : HK_ERR_LAUNCH;
}

}  // namespace hk

extern "C" size_t hk_fp8_quantize_tensor_workspace_bytes(void) { return hk::kQtMaxBlocks * sizeof(uint32_t); }

extern "C" int hk_fp8_quantize_tensor(const void* x, int x_type, size_t n, void* q_e4m3, float* host_scale,
                                      void* workspace, size_t workspace_bytes, void* stream) {
    using namespace hk;
    if (!x || !q_e4m3 || !host_scale || !workspace) return HK_ERR_NULL_POINTER;
    if (n == 0 || n > (1ull << 40) || x_type < kQtBf16 || x_type > kQtF16) return HK_ERR_BAD_SHAPE;
    if (((uintptr_t)x | (uintptr_t)q_e4m3) & 15u) return HK_ERR_BAD_ALIGNMENT;
    if (((uintptr_t)host_scale | (uintptr_t)workspace) & 3u) return HK_ERR_BAD_ALIGNMENT;
    if (workspace_bytes < hk_fp8_quantize_tensor_workspace_bytes()) return HK_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    // a captured launch does not run: there would be no scale to wait for
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &capture) != hipSuccess) return HK_ERR_LAUNCH;
    if (capture != hipStreamCaptureStatusNone) return HK_ERR_UNSUPPORTED;
    volatile uint32_t* word = (volatile uint32_t*)host_scale;
    *word = kScaleUnset;
    const auto launch = x_type == kQtBf16 ? launch_fp8_tensor_quantize<kQtBf16>
                        : x_type == kQtF32 ? launch_fp8_tensor_quantize<kQtF32> : launch_fp8_tensor_quantize<kQtF16>;
    const int st = launch(x, (long long)n, q_e4m3, (uint32_t*)host_scale, (uint32_t*)workspace, s);
    return st != HK_OK ? st : await_host_word(word, kScaleUnset, s);
}
