// The row-wise and element-wise parts of a decoder layer over many tokens: RMS norm and silu(gate) * up,
// each one launch that reads its inputs and writes its output once, with the roundings of the torch ops
// they replace (four launches for the norm, through fp32 copies of x, and two for the product).
// Bound by memory. fp16, us (GB/s): norm of 2048 x 4096 41 -> 8.6 (3900), silu(gate) * up of 2048 x 11008
// 42.7 -> 25.4 (5300, what a large copy reaches on the part).
#include "nq_common.h"

namespace nq {
namespace {

constexpr int kThreads = 256;

__device__ inline u32x4 load16(const uint16_t* p) { return *reinterpret_cast<const u32x4*>(p); }

// Both 16-bit halves of a dword through f, which takes and returns floats already rounded to T by the caller.
template <typename T, typename F>
__device__ inline uint32_t halves(uint32_t a, uint32_t b, F f) {
    const uint16_t lo = f(T::to_float(static_cast<uint16_t>(a)), T::to_float(static_cast<uint16_t>(b)));
    const uint16_t hi = f(T::to_float(static_cast<uint16_t>(a >> 16)), T::to_float(static_cast<uint16_t>(b >> 16)));
    return static_cast<uint32_t>(lo) | (static_cast<uint32_t>(hi) << 16);
}

// One block per row of n = 8 c columns, CH 16-byte chunks a thread held in registers between the sum and the
// scaling: y = T(g * T(x * rsqrt(mean(x^2) + eps))), mean and first product in fp32. y may be x.
template <typename T, int CH>
__global__ __launch_bounds__(kThreads) void rms_norm_kernel(const uint16_t* x, const uint16_t* __restrict__ g, uint16_t* y,
                                                            int n, float eps) {
    __shared__ float part[kThreads / 64];
    const int t = threadIdx.x;
    const size_t row = static_cast<size_t>(blockIdx.x) * static_cast<size_t>(n);
    const int chunks = n / 8;
    u32x4 v[CH], gv[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = t + i * kThreads;
        v[i] = c < chunks ? load16(x + row + 8 * c) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = t + i * kThreads;
        gv[i] = c < chunks ? load16(g + 8 * c) : u32x4{0u, 0u, 0u, 0u};
    }
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float lo = T::to_float(static_cast<uint16_t>(v[i][q]));
            const float hi = T::to_float(static_cast<uint16_t>(v[i][q] >> 16));
            ss += lo * lo;
            ss += hi * hi;
        }
    ss = wave_sum(ss);
    if ((t & 63) == 0) part[t >> 6] = ss;
    __syncthreads();
    const float r = rsqrtf((part[0] + part[1] + part[2] + part[3]) / static_cast<float>(n) + eps);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = t + i * kThreads;
        if (c >= chunks) continue;
        u32x4 o;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            o[q] = halves<T>(v[i][q], gv[i][q],
                             [&](float xe, float ge) { return T::from_float(ge * T::to_float(T::from_float(xe * r))); });
        *reinterpret_cast<u32x4*>(y + row + 8 * c) = o;
    }
}

// y = T(T(silu(gate)) * up), silu in fp32; eight elements a thread. y may be gate or up.
template <typename T>
__global__ __launch_bounds__(kThreads) void silu_mul_kernel(const uint16_t* gate, const uint16_t* up, uint16_t* y,
                                                            int64_t chunks) {
    const int64_t c = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (c >= chunks) return;
    const u32x4 a = load16(gate + 8 * c), b = load16(up + 8 * c);
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        o[q] = halves<T>(a[q], b[q], [](float g, float u) {
            return T::from_float(T::to_float(T::from_float(g / (1.0f + expf(-g)))) * u);
        });
    *reinterpret_cast<u32x4*>(y + 8 * c) = o;
}

template <typename T>
void launch_norm(const uint16_t* x, const uint16_t* g, uint16_t* y, int64_t rows, int n, float eps, hipStream_t st) {
    const dim3 grid(static_cast<unsigned>(rows));
    const int chunks = n / 8;
    if (chunks <= kThreads) rms_norm_kernel<T, 1><<<grid, kThreads, 0, st>>>(x, g, y, n, eps);
    else if (chunks <= 2 * kThreads) rms_norm_kernel<T, 2><<<grid, kThreads, 0, st>>>(x, g, y, n, eps);
    else if (chunks <= 4 * kThreads) rms_norm_kernel<T, 4><<<grid, kThreads, 0, st>>>(x, g, y, n, eps);
    else rms_norm_kernel<T, 8><<<grid, kThreads, 0, st>>>(x, g, y, n, eps);
}

constexpr int64_t kMaxNormColumns = 8 * 8 * kThreads;

}  // namespace
}  // namespace nq

using namespace nq;

extern "C" {

int nq_rms_norm(int dtype, const void* x, const void* weight, void* y, int64_t rows, int64_t n, float eps,
                nq_stream_t stream) {
    const char* name = "nq_rms_norm";
    if (dtype != NQ_F16 && dtype != NQ_BF16) return fail(NQ_ERR_DTYPE, "%s: unsupported dtype %d", name, dtype);
    if (rows < 0 || n <= 0) return fail(NQ_ERR_INVALID_ARGUMENT, "%s: bad sizes", name);
    if (n % 8) return fail(NQ_ERR_SHAPE, "%s: n must be a multiple of 8, got %lld", name, (long long)n);
    if (n > kMaxNormColumns || rows > INT32_MAX)
        return fail(NQ_ERR_UNSUPPORTED, "%s: sizes too large (n at most %lld)", name, (long long)kMaxNormColumns);
    if (rows == 0) return NQ_OK;
    if (!x || !weight || !y) return fail(NQ_ERR_INVALID_ARGUMENT, "%s: null pointer", name);
    if (!aligned(x, 16) || !aligned(weight, 16) || !aligned(y, 16))
        return fail(NQ_ERR_ALIGNMENT, "%s: x, weight and y must be 16-byte aligned", name);
    const auto* xp = static_cast<const uint16_t*>(x);
    const auto* gp = static_cast<const uint16_t*>(weight);
    auto* yp = static_cast<uint16_t*>(y);
    if (dtype == NQ_F16) launch_norm<F16>(xp, gp, yp, rows, static_cast<int>(n), eps, as_stream(stream));
    else launch_norm<BF16>(xp, gp, yp, rows, static_cast<int>(n), eps, as_stream(stream));
    return check_launch(name);
}

int nq_silu_mul(int dtype, const void* gate, const void* up, void* y, int64_t count, nq_stream_t stream) {
    const char* name = "nq_silu_mul";
    if (dtype != NQ_F16 && dtype != NQ_BF16) return fail(NQ_ERR_DTYPE, "%s: unsupported dtype %d", name, dtype);
    if (count < 0) return fail(NQ_ERR_INVALID_ARGUMENT, "%s: negative size", name);
    if (count % 8) return fail(NQ_ERR_SHAPE, "%s: count must be a multiple of 8, got %lld", name, (long long)count);
    const int64_t chunks = count / 8;
    if (ceil_div(chunks, kThreads) > INT32_MAX) return fail(NQ_ERR_UNSUPPORTED, "%s: sizes too large", name);
    if (count == 0) return NQ_OK;
    if (!gate || !up || !y) return fail(NQ_ERR_INVALID_ARGUMENT, "%s: null pointer", name);
    if (!aligned(gate, 16) || !aligned(up, 16) || !aligned(y, 16))
        return fail(NQ_ERR_ALIGNMENT, "%s: gate, up and y must be 16-byte aligned", name);
    const auto* gp = static_cast<const uint16_t*>(gate);
    const auto* up_ = static_cast<const uint16_t*>(up);
    auto* yp = static_cast<uint16_t*>(y);
    const dim3 grid(static_cast<unsigned>(ceil_div(chunks, kThreads)));
    if (dtype == NQ_F16) silu_mul_kernel<F16><<<grid, kThreads, 0, as_stream(stream)>>>(gp, up_, yp, chunks);
    else silu_mul_kernel<BF16><<<grid, kThreads, 0, as_stream(stream)>>>(gp, up_, yp, chunks);
    return check_launch(name);
}

}  // extern "C"
