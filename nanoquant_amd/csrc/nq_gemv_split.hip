// Stage 2 of the decode GEMV for a few batch rows, the rank split over a block's waves:
//
//   y[b][i] = sat(s_out[i] * sum_j sign(U[i,j]) (z_hi[b][j] + z_lo[b][j]))
//
// as v_mfma_f32_16x16x32_bf16 tiles: A = 16 rows of U x 32 j, the word shifted left by 4g + d carrying pair 4g + d's
// signs for the +-1 pair; B = 32 j x 16 columns, eight batch rows of which column 2b holds z_hi and 2b + 1 z_lo.
//
// What bounds this stage at these sizes is a chain of latencies, not bytes (m = 8192, r = 3520 reads 3.6 MB of U): a
// kernel that streams the intermediate through LDS for the whole block meets a barrier every two to four words of the
// rank, 0.17-0.2 us each, and one that holds the intermediate in LDS passes over U again for every two to eight batch
// rows. Here no wave waits for another until the end. The block's rows of U come into LDS by DMA in one go; then wave w
// runs all of the block's row tiles over its own run of words, the intermediate coming by DMA in chunks of two words
// (whole 128-byte lines) through a ring of the wave's own, the next chunk's operands in registers before the current
// one's MFMAs; the waves' sums meet in LDS once, added in wave order (deterministic). (Fragments loaded from L2
// straight into registers touch 16 lines a load and took 9.3 us where this takes 6.05; a ring of four or three chunks
// took 0-15% more than one of two, whose blocks are smaller and start sooner.)
//
// Measured, bf16, rotating copies of U, us, the kernels it replaced against this one: m = 8192, r = 3520 at 8 / 16 / 32
// rows 7.0 / 5.15, 12.4 / 6.05, 11.6 / 8.7; r = 2240 at 8 / 16 / 32 5.35 / 4.45, 7.55 / 5.1, 8.2 / 6.9; r = 4224 at 4 / 16
// 9.1 / 5.7, 26.9 / 6.7; m = 28672, r = 3520 at 4 / 8 rows 12.6 / 10.45, 12.5 / 10.6; m = 11008, r = 1632 at 16 6.6 /
// 5.65; gated pairs: 28672 x 3520 at 4 / 16 27.2 / 19.4, 29.7 / 26.9, 11008 x 1632 at 4 / 16 9.8 / 8.0, 13.7 / 9.6,
// 8192 x 2240 at 4 / 16 11.6 / 7.45, 16.9 / 8.5, 4096 x 1632 at 8 / 16 7.25 / 5.4, 11.9 / 6.4.
#include <algorithm>

#include "nq_gemv_split.h"

namespace nq {
namespace {

constexpr int kSplitLds = 160 * 1024;
constexpr int kSplitRing = 2;  // chunks of the intermediate in flight per wave

// LDS dwords of one item's tile of U: whole 16-byte DMAs of a wave.
__host__ __device__ inline int split_tile_words(int row_tiles, int wr) { return (row_tiles * wr * 16 + 1 + 255) / 256 * 256; }

__device__ inline float silu_of(float g) { return g / (1.0f + expf(-g)); }

template <typename T, int RT, int CT, int NW, int EPI>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2, 4))) void s2k_kernel(const SplitTable tab,
                                                                                              int batch) {
    constexpr int P = EPI == kSplitGated ? 2 : 1;  // items of a block (over the same rows)
    constexpr int kDma = 2 * CT;                   // DMAs of a wave per chunk: 8 CT rows x (hi, lo) x 128 bytes
    constexpr uint32_t kChunk = kDma * 1024u;
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    SplitItem it[P];
    it[0] = tab.item[P == 2 ? 0 : blockIdx.z];
    if (P == 2) it[P - 1] = tab.item[1];
    if (static_cast<int>(blockIdx.x) >= it[0].blocks) return;
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int c = lane & 15;
    const int g = lane >> 4;
    const int m = it[0].m, wr = it[0].wr;
    const int i0 = static_cast<int>(blockIdx.x) * 16 * RT;
    const int bb = static_cast<int>(blockIdx.y) * 8 * CT;
    const int tile = split_tile_words(RT, wr);
    uint32_t* zb = lds + P * tile + wave * (kSplitRing * kDma * 256);
    const uint32_t lz = __builtin_amdgcn_readfirstlane(lds_addr(zb));

    // 1. the block's rows of U, row-major as in memory (the last block's rows past m repeat U's last word)
    const uint32_t total = static_cast<uint32_t>(m) * static_cast<uint32_t>(wr);
    const uint32_t base = static_cast<uint32_t>(i0) * static_cast<uint32_t>(wr);
    const int words = 16 * RT * wr;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const uint32_t lu = __builtin_amdgcn_readfirstlane(lds_addr(lds + p * tile));
        if (base + static_cast<uint32_t>(words) <= total) {
            for (int l0 = wave * 64; l0 < words / 4; l0 += NW * 64)
                dma16_lds(it[p].u_bits + base, 16u * static_cast<uint32_t>(min(l0 + lane, words / 4 - 1)), lu + 16u * l0);
        } else {
            for (int l0 = wave * 64; l0 < words; l0 += NW * 64)
                dma4_lds(it[p].u_bits, 4u * min(base + static_cast<uint32_t>(l0 + lane), total - 1u), lu + 4u * l0);
        }
    }

    // 2. this wave's run of chunks (two words, 64 j) and the DMAs of its first ones. Row R = 2 b + (0 hi, 1 lo) of a
    //    chunk has eight pieces of 16 bytes, piece p at p ^ (R % 8).
    const int chunks = (wr + 1) / 2;
    const int lo = chunks * wave / NW, len = chunks * (wave + 1) / NW - lo;
    uint32_t zoff[kDma];  // byte offset of the lane's piece from the item's z_hi
#pragma unroll
    for (int d = 0; d < kDma; ++d) {
        const int l = d * 64 + lane, R = l >> 3;
        const uint32_t b = static_cast<uint32_t>(min(bb + (R >> 1), batch - 1));
        zoff[d] = 2u * (b * static_cast<uint32_t>(it[0].zpitch) + 8u * static_cast<uint32_t>((l & 7) ^ (R & 7)));
    }
    const bool odd = (lane >> 3) & 1;  // R & 1 of every piece of the lane
    uint32_t lo_off[P];
#pragma unroll
    for (int p = 0; p < P; ++p) lo_off[p] = odd ? static_cast<uint32_t>((it[p].z_lo - it[p].z_hi) * 2) : 0u;
    auto issue = [&](int f) {  // chunk f of the run(s) into the ring (past the end: the last one again)
        const int p = P == 2 && f >= len ? 1 : 0;
        const int ch = max(min(lo + f - p * len, lo + len - 1), 0);
        const uint16_t* src = (P == 2 && p ? it[P - 1].z_hi : it[0].z_hi) + 64 * ch;
        const uint32_t add = P == 2 && p ? lo_off[P - 1] : lo_off[0];
        const uint32_t dst = lz + static_cast<uint32_t>(f % kSplitRing) * kChunk;
#pragma unroll
        for (int d = 0; d < kDma; ++d) dma16_lds(src, zoff[d] + add, dst + 1024u * d);
    };
#pragma unroll
    for (int f = 0; f < kSplitRing; ++f) issue(f);
    wait_vmcnt<(kSplitRing - 1) * kDma>();  // U's words and the first chunk
    barrier_keep_dma();

    // 3. the run(s), the next chunk's operands read before the current one's MFMAs
    const uint32_t mask = 0x80008000u;
    // (no inline assembly on values that an MFMA reads or has read: the compiler keeps the wait states between the two
    // only for instructions that it knows)
    uint32_t one = BF16::ONE_PAIR;
    asm volatile("" : "+v"(one));
    const int sh = 4 * g;
    f32x4 acc[P][RT][CT];
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int j = 0; j < RT; ++j)
#pragma unroll
            for (int q = 0; q < CT; ++q) acc[p][j][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    struct Ops {
        u32x4 z[2][CT];
        uint32_t w[2][RT];
    };
    auto read = [&](Ops& o, int f) {
        const int p = P == 2 && f >= len ? 1 : 0;
        const int ch = max(min(lo + f - p * len, lo + len - 1), 0);
        const uint32_t* zr = zb + (f % kSplitRing) * (kDma * 256) + c * 32;
        const uint32_t* ur = lds + p * tile + c * wr + 2 * ch;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int q = 0; q < CT; ++q)
                o.z[s][q] = *reinterpret_cast<const u32x4*>(zr + 512 * q + 4 * ((4 * s + g) ^ (c & 7)));
#pragma unroll
            for (int j = 0; j < RT; ++j) o.w[s][j] = ur[16 * j * wr + s];
        }
    };
    Ops cur, nxt;
    read(cur, 0);
#pragma unroll
    for (int p = 0; p < P; ++p) {
#pragma unroll 2
        for (int i = 0; i < len; ++i) {
            const int f = p * len + i;
            __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4));  // lgkmcnt(0): the chunk is in registers
            issue(f + kSplitRing);
            wait_vmcnt<(kSplitRing - 1) * kDma>();
            asm volatile("" ::: "memory");  // the reads depend on it, which the compiler does not know
            read(nxt, f + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int j = 0; j < RT; ++j) {
                    const uint32_t v = cur.w[s][j] << sh;
                    const u32x4 a = u32x4{one ^ (v & mask), one ^ (v << 1 & mask), one ^ (v << 2 & mask), one ^ (v << 3 & mask)};
#pragma unroll
                    for (int q = 0; q < CT; ++q) acc[p][j][q] = mfma16x16x32<BF16>(a, cur.z[s][q], acc[p][j][q]);
                }
            __builtin_amdgcn_sched_barrier(0);
            cur = nxt;
        }
    }
    wait_vmcnt<0>();  // the re-fetches land before the sums take the ring's place
    __syncthreads();

    // 4. the waves' sums through LDS, then lane (c, g) of a tile holds rows 4g .. 4g+3 of column c
    f32x4* red = reinterpret_cast<f32x4*>(lds);
    constexpr int NT = P * RT * CT;
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int j = 0; j < RT; ++j)
#pragma unroll
            for (int q = 0; q < CT; ++q) red[(wave * NT + (p * RT + j) * CT + q) * 64 + lane] = acc[p][j][q];
    __syncthreads();
#pragma unroll
    for (int k0 = 0; k0 < RT * CT; k0 += NW) {
        const int k = k0 + wave;
        if (k >= RT * CT) break;
        const int j = k / CT, q = k % CT;
        const int row = i0 + 16 * j + 4 * g;
        const int b = bb + 8 * q + (c >> 1);
        float out[P][4];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            f32x4 s = red[((p * RT + j) * CT + q) * 64 + lane];
#pragma unroll
            for (int wv = 1; wv < NW; ++wv) s += red[(wv * NT + (p * RT + j) * CT + q) * 64 + lane];
            const float v[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {  // the odd lane's lo to the even lane's hi
                const float l = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v[e]), 0xB1, 0xF, 0xF, false));
                out[p][e] = v[e] + l;
            }
        }
        if ((c & 1) || b >= batch) continue;
        const size_t at = static_cast<size_t>(b) * it[0].ystride + row;
        uint16_t y[4], res[4] = {0, 0, 0, 0};
        const bool vec = it[0].vec4 && row + 3 < m;
        if (EPI == kSplitResidual) {
            if (vec) {
                const uint2 r = *reinterpret_cast<const uint2*>(it[0].resid + at);
                res[0] = static_cast<uint16_t>(r.x);
                res[1] = static_cast<uint16_t>(r.x >> 16);
                res[2] = static_cast<uint16_t>(r.y);
                res[3] = static_cast<uint16_t>(r.y >> 16);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (row + e < m) res[e] = it[0].resid[at + e];
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int r = min(row + e, m - 1);
            y[e] = saturate_to<T>(out[0][e] * T::to_float(it[0].s_out[r]), T::SAT);
            if (EPI == kSplitResidual) y[e] = T::from_float(T::to_float(res[e]) + T::to_float(y[e]));
            if (EPI == kSplitGated) {
                const float up = T::to_float(saturate_to<T>(out[P - 1][e] * T::to_float(it[P - 1].s_out[r]), T::SAT));
                y[e] = T::from_float(T::to_float(T::from_float(silu_of(T::to_float(y[e])))) * up);
            }
        }
        uint16_t* dst = it[0].y + at;
        if (vec) {
            *reinterpret_cast<uint2*>(dst) = uint2{y[0] | (uint32_t(y[1]) << 16), y[2] | (uint32_t(y[3]) << 16)};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (row + e < m) dst[e] = y[e];
        }
    }
}

inline size_t split_lds_bytes(const SplitPlan& p, int items, int wr) {
    const size_t stage = static_cast<size_t>(items) * split_tile_words(p.row_tiles, wr) * 4 +
                         static_cast<size_t>(p.waves) * kSplitRing * p.col_tiles * 2048;
    return std::max<size_t>(stage, static_cast<size_t>(p.waves) * items * p.row_tiles * p.col_tiles * 1024);
}

template <typename T, int RT, int CT, int NW, int EPI>
int launch_one(const SplitTable& tab, int batch, const SplitPlan& p, hipStream_t st) {
    constexpr int P = EPI == kSplitGated ? 2 : 1;
    int blocks = 0, wr = 0;
    for (int k = 0; k < tab.count; ++k) {
        blocks = std::max(blocks, tab.item[k].blocks);
        wr = std::max(wr, tab.item[k].wr);
    }
    const size_t bytes = split_lds_bytes(p, P, wr);
    if (wr > kSplitMaxWords || bytes > static_cast<size_t>(kSplitLds)) return fail(NQ_ERR_UNSUPPORTED, "stage 2: shape does not fit");
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&s2k_kernel<T, RT, CT, NW, EPI>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, kSplitLds);
    if (attr != hipSuccess) return fail(NQ_ERR_HIP, "stage 2: LDS limit: %s", hipGetErrorString(attr));
    const dim3 grid(static_cast<unsigned>(blocks), static_cast<unsigned>(ceil_div(batch, 8 * CT)),
                    static_cast<unsigned>(P == 2 ? 1 : tab.count));
    s2k_kernel<T, RT, CT, NW, EPI><<<grid, NW * 64, bytes, st>>>(tab, batch);
    return check_launch("stage 2");
}

template <typename T, int RT, int CT, int NW>
int launch_epi(const SplitTable& tab, int batch, SplitEpilogue epi, const SplitPlan& p, hipStream_t st) {
    switch (epi) {
        case kSplitStore: return launch_one<T, RT, CT, NW, kSplitStore>(tab, batch, p, st);
        case kSplitResidual: return launch_one<T, RT, CT, NW, kSplitResidual>(tab, batch, p, st);
        case kSplitGated: return launch_one<T, RT, CT, NW, kSplitGated>(tab, batch, p, st);
    }
    return fail(NQ_ERR_INVALID_ARGUMENT, "stage 2: unknown epilogue");
}

template <typename T, int RT, int CT>
int launch_waves(const SplitTable& tab, int batch, SplitEpilogue epi, const SplitPlan& p, hipStream_t st) {
    // the shapes of split_plan: four waves on four column tiles, eight on four row tiles by two column tiles
    if constexpr (CT == 4) return launch_epi<T, RT, CT, 4>(tab, batch, epi, p, st);
    else if constexpr (RT == 4 && CT == 2) return launch_epi<T, RT, CT, 8>(tab, batch, epi, p, st);
    else if (p.waves == 4) return launch_epi<T, RT, CT, 4>(tab, batch, epi, p, st);
    else return launch_epi<T, RT, CT, 8>(tab, batch, epi, p, st);
}

template <typename T, int RT>
int launch_cols(const SplitTable& tab, int batch, SplitEpilogue epi, const SplitPlan& p, hipStream_t st) {
    if (p.col_tiles == 1) return launch_waves<T, RT, 1>(tab, batch, epi, p, st);
    if (p.col_tiles == 2) return launch_waves<T, RT, 2>(tab, batch, epi, p, st);
    return launch_waves<T, RT, 4>(tab, batch, epi, p, st);
}

template <typename T>
int launch_rows(const SplitTable& tab, int batch, SplitEpilogue epi, const SplitPlan& p, hipStream_t st) {
    if (p.row_tiles == 1) return launch_cols<T, 1>(tab, batch, epi, p, st);
    if (p.row_tiles == 2) return launch_cols<T, 2>(tab, batch, epi, p, st);
    return launch_cols<T, 4>(tab, batch, epi, p, st);
}

}  // namespace

// Row tiles: four from 640 tiles on ranks of 64 words (m = 11008, r = 2976 at 16 rows 7.1 us, two 7.5; below, r = 1632,
// 5.9 and 5.65), else two, and one up to 256 tiles (m = 4096, r = 2976 at 16 rows 5.4, two 5.5; r = 1632 at 32 rows 5.1,
// 5.7). Eight waves share a rank of 64 words or more while their rings are small (m = 8192, r = 3520 at 16 rows 6.05 us,
// four waves 6.5; r = 1120 4.7 and 4.27; at 32 rows 8.86 and 8.72), but for grids of several rounds, where four leave
// room for more blocks (the pair of m = 28672, r = 3520 at 8 rows 21.5 and 19.5; at 16, one block a CU either way, 26.9
// and 31.2).
SplitPlan split_plan(int batch, int m, int wr) {
    SplitPlan p;
    const int64_t tiles = ceil_div(m, 16);
    p.col_tiles = batch <= 8 ? 1 : (batch <= 16 ? 2 : 4);
    p.row_tiles = tiles >= 640 && wr >= 64 ? 4 : (tiles > 256 ? 2 : 1);
    p.waves = wr >= 64 && p.col_tiles < 4 && (p.col_tiles == 2 || tiles < 1600) ? 8 : 4;
    return p;
}

int launch_split(int dtype, SplitTable& tab, int batch, SplitEpilogue epi, const SplitPlan& p, hipStream_t st) {
    for (int k = 0; k < tab.count; ++k) {
        SplitItem& it = tab.item[k];
        it.blocks = static_cast<int>(ceil_div(it.m, 16 * p.row_tiles));
        it.vec4 = it.ystride % 4 == 0 && aligned(it.y, 8) && (epi != kSplitResidual || aligned(it.resid, 8));
    }
    return dtype == NQ_F16 ? launch_rows<F16>(tab, batch, epi, p, st) : launch_rows<BF16>(tab, batch, epi, p, st);
}

}  // namespace nq
