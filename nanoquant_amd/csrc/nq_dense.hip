// Dense GEMV of several batch rows (a decode step's lm_head for a batch of sequences):
// y[b][j] = T(sum_k W[j][k] xn[b][k]), xn = x or its RMS norm rounded as the decoder's torch path does,
// T(g[k] * T(x[k] * rsqrt(mean(x^2) + eps))).
//
// W is read once from HBM whatever the batch, so the launch is bound by streaming it, provided that the
// arithmetic stays out of the way: v_mfma_f32_16x16x32 with A = 16 rows of W x 32 k and B = 16 batch rows of
// x. The eight waves of a block split k, and each keeps its slice of x in registers (NF fragments per 16 batch
// rows) while the block walks over 16-row tiles of W (a grid of one block per CU, every grid-th tile): x is
// read and normalised once per block. Each wave streams its columns of W by DMA through a ring of its own in
// LDS, stages of four fragments, three of four stages in flight across tile ends (96 KB a CU; no wave waits
// for another). The waves' partial tiles meet in LDS (two buffers, one barrier per tile).
//
// Measured (MI355X, cold weights, 32000 rows, norm prologue, float32 out; us at 3 / 16 / 32 rows), against
// loads into registers eight fragments ahead (64 bytes of a row an instruction instead of 256, 64 KB in flight):
//   n = 2048 32 / 35 / 44 -> 27 / 30 / 35, n = 4096 54 / 58 / 67 -> 44 / 50 / 61,
//   n = 6144 85 / 91 / 183 -> 66 / 74 / 145, n = 8192 101 / 110 / 220 -> 90 / 98 / 191 (524 MB: 5.3 TB/s).
// The VALU kernel, which takes up to four batch rows a pass over W: n = 4096 86 / 239 / 470, n = 8192 164 / 608.
// The non-temporal hint is worth 7% at n = 8192.
#include <algorithm>

#include "nq_dense.h"

namespace nq {
namespace {

constexpr int kWaves = 8;
// The barrier between the waves' LDS writes and their reads: waits for this wave's LDS accesses only (W's
// loads stay in flight).
__device__ inline void lds_barrier() { barrier_keep_dma(); }

template <typename T, int NF, int CT, bool kNorm>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(2))) void dense_mfma_kernel(
    const DenseArgs a) {
    static_assert(NF % 4 == 0, "whole stages of four fragments");
    constexpr int NS = NF / 4;                  // stages of a tile
    constexpr int kStages = CT == 1 ? 4 : 3;    // of a wave's ring, as the LDS holds beside the partial tiles
    __shared__ f32x4 part[2][kWaves][CT][64];
    __shared__ float ssum[kWaves][16 * CT];
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int c = lane & 15;
    const int g = lane >> 4;
    const int nf = a.n / (32 * kWaves);  // fragments of this wave's k slice, <= NF
    const int k0 = wave * nf * 32;
    const int b0 = static_cast<int>(blockIdx.y) * 16 * CT;
    const int tiles = (a.m + 15) / 16;

    // a stage is four fragments of a tile, 16 rows x 256 bytes, each DMA taking four rows; LDS chunk p of row r
    // holds the row's 16-byte chunk p ^ r, so that a fragment's reads (one chunk of 16 rows) have no bank conflicts.
    // Rows past m fetch row m - 1 (their sums are not stored), columns past the row its end (not multiplied).
    __shared__ __attribute__((aligned(16))) uint16_t ring[kWaves][kStages][16 * 128];
    const uint32_t lring =
        __builtin_amdgcn_readfirstlane(lds_addr(&ring[0][0][0]) + static_cast<uint32_t>(wave) * sizeof(ring[0]));
    auto issue_stage = [&](int tile, int grp, int slot) {
        const int row0 = min(tile, tiles - 1) * 16;
        const uint16_t* base = a.w + static_cast<size_t>(row0) * static_cast<size_t>(a.n);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = 4 * j + (lane >> 4);
            const int col = min(k0 + 128 * grp + 8 * ((lane & 15) ^ r), a.n - 8);
            dma16_lds_stream(base, 2u * (static_cast<uint32_t>(min(r, a.m - 1 - row0)) * static_cast<uint32_t>(a.n) +
                                         static_cast<uint32_t>(col)),
                             lring + static_cast<uint32_t>(slot) * (16u * 256u) + static_cast<uint32_t>(j) * 1024u);
        }
    };
    int tile = static_cast<int>(blockIdx.x);
    const int stride = static_cast<int>(gridDim.x);
#pragma unroll
    for (int st = 0; st < kStages; ++st) issue_stage(tile + st / NS * stride, st % NS, st);

    // the mean square of each batch row: every wave sums its slice, the slices meet in LDS
    auto load_x = [&](int b, int i) {
        const uint16_t* xr = a.x + static_cast<size_t>(min(b, a.batch - 1)) * static_cast<size_t>(a.n) + k0 + 8 * g;
        return *reinterpret_cast<const u32x4*>(xr + 32 * i);
    };
    float rs[CT];
    if (kNorm) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            float ss = 0.0f;
#pragma unroll 4
            for (int i = 0; i < nf; ++i) {
                const u32x4 v = load_x(b0 + 16 * ct + c, i);
                const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float lo = T::to_float(static_cast<uint16_t>(d[q] & 0xFFFFu));
                    const float hi = T::to_float(static_cast<uint16_t>(d[q] >> 16));
                    ss += lo * lo;
                    ss += hi * hi;
                }
            }
            ss += __shfl_xor(ss, 16, 64);
            ss += __shfl_xor(ss, 32, 64);
            if (g == 0) ssum[wave][16 * ct + c] = ss;
        }
        lds_barrier();
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            float tot = 0.0f;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) tot += ssum[w][16 * ct + c];
            rs[ct] = rsqrtf(tot / static_cast<float>(a.n) + a.eps);
        }
    }
    // this wave's slice of x (or xn): lane (c, g) holds row b0 + 16 ct + c, columns k0 + 32 i + 8 g .. +7; rows
    // past the batch are zero
    u32x4 xf[CT][NF];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int b = b0 + 16 * ct + c;
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            // a few fragments' loads at a time: all at once they would take the registers of the slice again
            if (kNorm && i % 2 == 0) __builtin_amdgcn_sched_barrier(0);
            u32x4 v = u32x4{0u, 0u, 0u, 0u};
            if (i < nf) {
                v = load_x(b, i);
                if (kNorm) {
                    const u32x4 gv = *reinterpret_cast<const u32x4*>(a.norm_w + k0 + 32 * i + 8 * g);
                    uint32_t d[4] = {v.x, v.y, v.z, v.w};
                    const uint32_t gd[4] = {gv.x, gv.y, gv.z, gv.w};
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        uint16_t h[2];
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            const float xe = T::to_float(static_cast<uint16_t>(d[q] >> (16 * e)));
                            const float ge = T::to_float(static_cast<uint16_t>(gd[q] >> (16 * e)));
                            h[e] = T::from_float(ge * T::to_float(T::from_float(xe * rs[ct])));
                        }
                        d[q] = static_cast<uint32_t>(h[0]) | (static_cast<uint32_t>(h[1]) << 16);
                    }
                    v = u32x4{d[0], d[1], d[2], d[3]};
                }
                if (b >= a.batch) v = u32x4{0u, 0u, 0u, 0u};
            }
            xf[ct][i] = v;
        }
    }

    int slot = 0;
    for (int it = 0; tile < tiles; ++it) {
        f32x4 acc[CT][2];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[ct][0] = acc[ct][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < NS; ++st) {
            wait_vmcnt<4 * (kStages - 1)>();  // the oldest stage's four DMAs (a store in flight only waits longer)
            asm volatile("" ::: "memory");    // (the compiler does not know that the reads depend on it)
            const uint16_t* src = &ring[wave][slot][128 * c];
            u32x4 f[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) f[i] = *reinterpret_cast<const u32x4*>(src + 8 * ((4 * i + g) ^ c));
            __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));  // lgkmcnt(0): read before the slot is filled again
            asm volatile("" ::: "memory");
            issue_stage(tile + (st + kStages) / NS * stride, (st + kStages) % NS, slot);
            slot = slot + 1 == kStages ? 0 : slot + 1;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (4 * st + i < nf)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct)
                        acc[ct][i & 1] = mfma16x16x32<T>(f[i], xf[ct][4 * st + i], acc[ct][i & 1]);
        }
        // C: lane (c, g) holds rows 4 g + i of the tile for batch row c
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
            part[it & 1][wave][ct][lane] = f32x4{acc[ct][0].x + acc[ct][1].x, acc[ct][0].y + acc[ct][1].y,
                                                 acc[ct][0].z + acc[ct][1].z, acc[ct][0].w + acc[ct][1].w};
        lds_barrier();
        if (t < 256 * CT) {
            const float* p = reinterpret_cast<const float*>(&part[it & 1][0][0][0]) + t;
            float s = 0.0f;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) s += p[w * 256 * CT];
            const int l = (t & 255) >> 2;
            const int b = b0 + 16 * (t >> 8) + (l & 15);
            const int row = tile * 16 + 4 * (l >> 4) + (t & 3);
            if (b < a.batch && row < a.m) {
                const uint16_t v = T::from_float(s);
                const size_t at = static_cast<size_t>(b) * static_cast<size_t>(a.ldy) + static_cast<size_t>(row);
                if (a.y_f32) static_cast<float*>(a.y)[at] = T::to_float(v);
                else static_cast<uint16_t*>(a.y)[at] = v;
            }
        }
        tile += stride;
    }
    wait_vmcnt<0>();  // the re-fetches past the last tile land before the block's LDS is released
}

template <typename T, int NF, int CT>
void launch_nf(const DenseArgs& a, hipStream_t st) {
    const unsigned tiles = static_cast<unsigned>(ceil_div(a.m, 16));
    const dim3 grid(std::min(tiles, 256u), static_cast<unsigned>(ceil_div(a.batch, 16 * CT)));
    if (a.norm_w) dense_mfma_kernel<T, NF, CT, true><<<grid, kWaves * 64, 0, st>>>(a);
    else dense_mfma_kernel<T, NF, CT, false><<<grid, kWaves * 64, 0, st>>>(a);
}

// Sixteen batch rows a pass over W; 32 where two slices of x fit the registers beside the loads in flight
// (n up to 4096: 32 rows 61 us in one pass, n = 8192 191 in two).
template <typename T>
void launch_dense(const DenseArgs& a, hipStream_t st) {
    const int nf = a.n / (32 * kWaves);
    if (a.batch > 16 && nf <= 16) {
        if (nf <= 8) launch_nf<T, 8, 2>(a, st);
        else launch_nf<T, 16, 2>(a, st);
        return;
    }
    if (nf <= 8) launch_nf<T, 8, 1>(a, st);
    else if (nf <= 16) launch_nf<T, 16, 1>(a, st);
    else if (nf <= 24) launch_nf<T, 24, 1>(a, st);
    else launch_nf<T, 32, 1>(a, st);
}

}  // namespace

// From three batch rows: at one or two the VALU kernel streams W faster (n = 4096 41.5, n = 8192 82 us, against
// 44 and 90 here). Whole fragments per wave, as many as its registers hold; any other n keeps the VALU kernel.
bool dense_mfma_applies(int64_t batch, int64_t n) { return batch >= 3 && n % (32 * kWaves) == 0 && n <= 32 * 32 * kWaves; }

void launch_dense_mfma(int dtype, const DenseArgs& a, hipStream_t st) {
    if (dtype == NQ_F16) launch_dense<F16>(a, st);
    else launch_dense<BF16>(a, st);
}

}  // namespace nq
